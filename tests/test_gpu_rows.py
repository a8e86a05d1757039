"""Row movers (K4 / K6 / index_add) through pcl_xpu_customops against the C restatement of the
SYCL kernels.  Bar: bit-exact, except routing_weights_grad (a dot product whose summation order
differs: wavefront tree vs serial) which is held to 2e-3 relative."""
import numpy as np
import pytest
import torch

from util import bits, from_bits, routed_experts

pytestmark = pytest.mark.gpu


def _setup(T, N, K, E, start, end, dtype, oracle_lib, seed=0):
    se = routed_experts(T, N, K, seed=seed + 1)
    idx = oracle_lib.index_construction(se.numpy(), end - start, start, end)
    g = torch.Generator().manual_seed(seed)
    TR = idx["num_routed_tokens"]
    x = torch.randn(T, E, generator=g).to(dtype)
    y = torch.randn(TR, E, generator=g).to(dtype)
    w = torch.rand(T, K, generator=g)
    return se, idx, x, y, w


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T,N,K,E,start,end", [(64, 8, 2, 256, 0, 8), (512, 64, 8, 2048, 0, 64),
                                              (256, 32, 4, 136, 8, 24), (128, 8, 2, 100, 0, 8)])
def test_gather_reduce_combine(cuda, oracle_lib, dtype, T, N, K, E, start, end):
    import pcl_xpu_customops as ops
    se, idx, x, y, w = _setup(T, N, K, E, start, end, dtype, oracle_lib)
    TR = idx["num_routed_tokens"]
    d = lambda a: torch.from_numpy(a).to(cuda)
    ii, oi, si, ce = d(idx["input_indices"]), d(idx["output_indices"]), d(idx["selected_experts_indices"]), d(idx["cum_expert_counts_ep"])
    # K4 forward
    out = torch.empty(TR, E, dtype=dtype, device=cuda)
    assert ops.index_gather(x.to(cuda), ii, out) is out
    assert np.array_equal(bits(out), oracle_lib.index_gather(bits(x), idx["input_indices"]))
    # K4 backward
    hg = torch.empty(T, E, dtype=dtype, device=cuda)
    ops.shuffle_sub_matrix_reduce(y.to(cuda), ce, oi, hg)
    assert np.array_equal(bits(hg), oracle_lib.shuffle_sub_matrix_reduce(bits(y), idx["cum_expert_counts_ep"], idx["output_indices"], T))
    # K6 forward: weights in the activation dtype, and fp32 weights with bf16 activations
    for wdt in ([dtype] if dtype == torch.float32 else [torch.bfloat16, torch.float32]):
        ww = w.to(wdt)
        fin = torch.empty(T, E, dtype=dtype, device=cuda)
        ops.reduce_ggemm_output(y.to(cuda), ww.to(cuda), ce, si, oi, fin, False)
        ref = oracle_lib.reduce_ggemm_output(bits(y), bits(ww), idx["cum_expert_counts_ep"], idx["selected_experts_indices"], idx["output_indices"])
        assert np.array_equal(bits(fin), ref)
        # K6 backward
        dout = torch.randn(T, E, generator=torch.Generator().manual_seed(3)).to(dtype)
        dy = torch.empty(TR, E, dtype=dtype, device=cuda)
        dw = torch.zeros(T, K, dtype=wdt, device=cuda)
        ops.reduce_ggemm_output_backward(dout.to(cuda), y.to(cuda), ww.to(cuda), ce, si, ii, oi, dy, dw)
        rdy, rdw = oracle_lib.reduce_ggemm_output_backward(bits(dout), bits(y), bits(ww), idx["selected_experts_indices"], idx["input_indices"], idx["output_indices"])
        assert np.array_equal(bits(dy), rdy)
        a, b = dw.float().cpu(), from_bits(rdw, wdt).float()
        tol = 2e-2 if wdt == torch.bfloat16 else 2e-3
        assert float((a - b).abs().max()) <= tol * float(b.abs().max())
        # not-local entries stay zero
        local = ((se >= start) & (se < end))
        assert float(a[~local].abs().max() if (~local).any() else 0.0) == 0.0
    # skip_weights_scaling
    fin = torch.empty(T, E, dtype=dtype, device=cuda)
    ops.reduce_ggemm_output(y.to(cuda), w.to(dtype).to(cuda), ce, si, oi, fin, True)
    assert np.array_equal(bits(fin), oracle_lib.shuffle_sub_matrix_reduce(bits(y), idx["cum_expert_counts_ep"], idx["output_indices"], T))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_index_add_and_autograd_function(cuda, oracle_lib, dtype):
    from optimus.custom_ops import IndexAddOpFunction
    g = torch.Generator().manual_seed(0)
    C, E, S = 96, 72, 40
    inp = torch.randn(C, E, generator=g).to(dtype)
    base = torch.randn(S, E, generator=g).to(dtype)
    idx = torch.randperm(S, generator=g)[:C % S].tolist() + list(range(S)) + torch.randperm(S, generator=g)[: C - S - C % S].tolist()
    idx = torch.tensor(idx[:C], dtype=torch.int32)
    uniq = torch.randperm(S, generator=g)[:32].to(torch.int32)   # distinct: bit-exact case
    out = base.clone().to(cuda)
    import pcl_xpu_customops as ops
    ops.index_add_op(inp[:32].contiguous().to(cuda), out, uniq.to(cuda))
    ref = bits(base).copy()
    oracle_lib.index_add(bits(inp[:32].contiguous()), ref, uniq.numpy())
    assert np.array_equal(bits(out), ref)
    # duplicates: sums are order-dependent in the last bit; compare in fp32 with tolerance
    out = base.clone().to(cuda)
    ops.index_add_op(inp.to(cuda), out, idx.to(cuda))
    want = base.float().index_add(0, idx.long(), inp.float())
    tol = 1e-5 if dtype == torch.float32 else 6e-2
    assert float((out.float().cpu() - want).abs().max()) <= tol
    # autograd wrapper: gradient wrt expert_output is a gather of grad_output
    eo = inp[:32].contiguous().to(cuda).requires_grad_(True)
    fo = base.clone().to(cuda)
    res = IndexAddOpFunction.apply(eo, fo, uniq.to(cuda))
    gout = torch.randn(S, E, generator=g).to(dtype).to(cuda)
    res.backward(gout)
    assert torch.equal(eo.grad, gout[uniq.long().to(cuda)])


@pytest.mark.parametrize("dtype,wdtype", [(torch.bfloat16, torch.bfloat16), (torch.bfloat16, torch.float32),
                                          (torch.float32, torch.float32)])
@pytest.mark.parametrize("T,N,K,E,start,end", [(64, 8, 2, 256, 0, 8), (512, 64, 8, 2048, 0, 64),
                                              (256, 32, 4, 136, 8, 24), (128, 8, 2, 100, 0, 8)])
def test_combine_with_residual_equals_two_steps(cuda, oracle_lib, dtype, wdtype, T, N, K, E, start, end):
    """reduce_ggemm_output_residual = reduce_ggemm_output (already bit-exact against the restatement
    of the SYCL kernel) followed by the tensor addition the callers perform: the same bits, for an
    expert window (tokens without a local expert get residual + 0) and row lengths that are not a
    multiple of the vector width."""
    import pcl_xpu_customops as ops
    se, idx, x, y, w = _setup(T, N, K, E, start, end, dtype, oracle_lib, seed=5)
    d = lambda a: torch.from_numpy(a).to(cuda)
    oi, si, ce = d(idx["output_indices"]), d(idx["selected_experts_indices"]), d(idx["cum_expert_counts_ep"])
    yd, wd, res = y.to(cuda), w.to(wdtype).to(cuda), x.to(cuda)
    two = torch.empty(T, E, dtype=dtype, device=cuda)
    ops.reduce_ggemm_output(yd, wd, ce, si, oi, two, False)
    two = res + two
    one = torch.empty(T, E, dtype=dtype, device=cuda)
    ops.reduce_ggemm_output_residual(yd, wd, ce, si, oi, res, one)
    assert np.array_equal(bits(one), bits(two))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T,N,K,E", [(8, 16, 9, 8), (16, 16, 9, 520), (512, 24, 17, 264), (520, 8, 3, 4104), (3000, 8, 3, 264),
                                     (1600, 8, 3, 1416)])
def test_token_sums_on_both_sides_of_the_few_tokens_line(cuda, oracle_lib, dtype, T, N, K, E):
    """Few tokens run a wavefront per 64-vector chunk with eight rows in flight: more rows per token than that
    and a remainder, one vector more than a chunk, an expert window that leaves tokens without rows, and
    sizes on either side of the line.  Same order of the sums: bit-exact."""
    import pcl_xpu_customops as ops
    start, end = N // 4, N // 2
    for lo, hi in ((0, N), (start, end)):
        se, idx, x, y, w = _setup(T, N, K, E, lo, hi, dtype, oracle_lib)
        ce, oi = torch.from_numpy(idx["cum_expert_counts_ep"]).to(cuda), torch.from_numpy(idx["output_indices"]).to(cuda)
        if idx["num_routed_tokens"] == 0:
            continue
        hg = torch.empty(T, E, dtype=dtype, device=cuda)
        ops.shuffle_sub_matrix_reduce(y.to(cuda), ce, oi, hg)
        assert np.array_equal(bits(hg), oracle_lib.shuffle_sub_matrix_reduce(bits(y), idx["cum_expert_counts_ep"], idx["output_indices"], T))


@pytest.mark.parametrize("T,N,K,E,I,start,end,dtype,wdt", [
    (8, 4, 2, 8, 8, 0, 4, torch.bfloat16, torch.bfloat16), (80, 8, 3, 264, 200, 0, 8, torch.bfloat16, torch.bfloat16),
    (704, 16, 8, 1000, 1048, 4, 6, torch.bfloat16, torch.float32), (600, 130, 70, 2048, 64, 0, 130, torch.bfloat16, torch.float32),
    (40, 12, 3, 12, 520, 6, 12, torch.float32, torch.float32), (24, 8, 2, 64, 72, 0, 1, torch.bfloat16, torch.bfloat16)])
def test_row_sum_with_the_routing_weights_gradient(cuda, oracle_lib, T, N, K, E, I, start, end, dtype, wdt):
    """One launch against om_sum_ggemm_output and the column ranges added in order; `rows` is a bound under a window."""
    from optimus import _native as n
    se, idx, _, y, _ = _setup(T, N, K, E, start, end, dtype, oracle_lib, seed=T)
    TR = idx["num_routed_tokens"]
    rows = T * K if end - start < N else TR
    parts = n.lib().om_merged_mlp_row_dot_parts(I)
    dot = torch.randn(parts, rows, generator=torch.Generator().manual_seed(4))
    d = lambda a: torch.from_numpy(a).to(cuda)
    oi, si, ce = d(idx["output_indices"]), d(idx["selected_experts_indices"]), d(idx["cum_expert_counts_ep"])
    yg, dotg, residual = y.to(cuda), dot.to(cuda), torch.randn(T, E, generator=torch.Generator().manual_seed(5)).to(dtype).to(cuda)
    for res in (None, residual):
        want, got = torch.empty(T, E, dtype=dtype, device=cuda), torch.empty(T, E, dtype=dtype, device=cuda)
        dw = torch.full((T, K), 7.0, dtype=wdt, device=cuda)
        n.check(n.lib().om_sum_ggemm_output(n.ptr(yg), n.ptr(ce), n.ptr(oi), n.ptr(res), n.ptr(want), T, E, n.dtype_code(yg), n.stream()), "sum")
        n.check(n.lib().om_sum_ggemm_output_row_weights_grad(n.ptr(yg), n.ptr(ce), n.ptr(oi), n.ptr(res), n.ptr(got), T, E,
                                                             n.dtype_code(yg), n.ptr(dotg), parts, rows, n.ptr(si), n.ptr(dw), K,
                                                             n.dtype_code(dw), n.stream()), "sum and gradient")
        assert torch.equal(got.view(torch.uint8), want.view(torch.uint8))
        sums = torch.zeros(rows)
        for part in dot:
            sums += part
        token = np.repeat(np.arange(T), np.diff(idx["cum_expert_counts_ep"]))
        ref = torch.zeros(T, K)
        ref[torch.from_numpy(token), torch.from_numpy(idx["selected_experts_indices"]).long()] = sums[torch.from_numpy(idx["output_indices"]).long()]
        assert torch.equal(dw.cpu(), ref.to(wdt))


@pytest.mark.parametrize("T,N,K,I,start,end,wdt", [(8, 4, 2, 8, 0, 4, torch.bfloat16), (80, 8, 3, 200, 0, 8, torch.float32), (704, 16, 8, 1048, 4, 6, torch.float32),
                                                   (600, 130, 70, 64, 0, 130, torch.bfloat16)])
def test_routing_weights_gradient_alone(cuda, oracle_lib, T, N, K, I, start, end, wdt):
    """om_moe_row_weights_grad: the column ranges added in order; entries of pairs outside the window keep what they held."""
    from optimus import _native as n
    _, idx, _, _, _ = _setup(T, N, K, 8, start, end, torch.bfloat16, oracle_lib, seed=T)
    TR, parts = idx["num_routed_tokens"], n.lib().om_merged_mlp_row_dot_parts(I)
    dot = torch.randn(parts, TR, generator=torch.Generator().manual_seed(4))
    ii, oi, si = (torch.from_numpy(idx[k]).to(cuda) for k in ("input_indices", "output_indices", "selected_experts_indices"))
    dotg, dw = dot.to(cuda), torch.full((T, K), 7.0, dtype=wdt, device=cuda)
    n.check(n.lib().om_moe_row_weights_grad(n.ptr(dotg), parts, n.ptr(si), n.ptr(ii), n.ptr(oi), n.ptr(dw), TR, K, n.dtype_code(dw), n.stream()), "gradient")
    sums = torch.zeros(TR)
    for part in dot:
        sums += part
    pos = torch.from_numpy(idx["output_indices"]).long()
    ref = torch.full((T, K), 7.0)
    ref[torch.from_numpy(idx["input_indices"]).long()[pos], torch.from_numpy(idx["selected_experts_indices"]).long()] = sums[pos]
    assert torch.equal(dw.cpu(), ref.to(wdt))
