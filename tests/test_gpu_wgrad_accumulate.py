"""Weight gradients accumulated into a live gradient buffer inside the GEMM epilogue.

In the reference every p.grad is a view of the optimizer's flat gradient buffer
(optimus/optimizers.py:105-111) that is zeroed in place (:117-118) and accumulated into over the
micro-batches of a step (dist_train.py:154), so autograd ends each weight-gradient GEMM with an
in-place `p.grad += dW`.  The *_accumulate entry points do that sum in the epilogue.  The bar is
bit equality with the two-step form: the same GEMM writing a fresh dW, then torch's in-place add.
"""
import pytest
import torch

from util import bits
from test_gpu_ggemm import _counts

pytestmark = pytest.mark.gpu


def _call(name, *args):
    from optimus import _native as n
    n.check(getattr(n.lib(), name)(*args, n.stream()), name)


# (kind, G, rows, N, K): both tile shapes (256x256 needs N, K multiples of 256 and enough tiles),
# odd row counts (single trailing contraction step), experts without rows
ABI_CASES = [("ragged", 64, 4096, 256, 512), ("empties", 16, 777, 128, 256), ("uniform", 8, 1000, 512, 256),
             ("onehot", 9, 3000, 512, 256), ("ragged", 3, 5, 128, 128), ("ragged", 150, 6000, 128, 128),
             ("ragged", 8, 1000, 192, 320)]   # partial last tiles along both extents of dW


@pytest.mark.parametrize("kind,G,rows,N,K", ABI_CASES)
@pytest.mark.parametrize("form", ["plain", "gathered", "gathered_out"])
def test_accumulate_entry_points_equal_gemm_then_add(cuda, form, kind, G, rows, N, K):
    from optimus import _native as n
    g = torch.Generator().manual_seed(rows + N)
    T = max(rows // 2, 8)
    idx = torch.randint(0, T, (rows,), generator=g, dtype=torch.int32).to(cuda)
    dout_rows = T if form == "gathered_out" else rows
    in_rows = T if form == "gathered" else rows
    dout = torch.randn(dout_rows, N, generator=g).to(torch.bfloat16).to(cuda)
    x = torch.randn(in_rows, K, generator=g).to(torch.bfloat16).to(cuda)
    cum = _counts(kind, G, rows).to(cuda)
    pitch = N * K + 64                       # per-expert matrices at a constant pitch inside one buffer
    old = torch.randn(G * pitch, generator=g).to(torch.bfloat16).to(cuda)
    P = n.ptr

    def run(suffix, out):
        if form == "plain":
            _call("om_grouped_gemm_wgrad" + suffix, P(dout), P(x), P(out), P(cum), rows, G, N, K, pitch)
        elif form == "gathered":
            _call("om_grouped_gemm_wgrad_gathered" + suffix, P(dout), P(x), P(idx), T, P(out), P(cum), rows, G,
                  N, K, pitch)
        else:
            _call("om_grouped_gemm_wgrad_gathered_out" + suffix, P(dout), P(idx), T, P(x), P(out), P(cum), rows,
                  G, N, K, pitch)

    fresh = torch.zeros_like(old)
    run("", fresh)
    acc = old.clone()
    run("_accumulate", acc)
    view = lambda t: torch.as_strided(t, (G, N, K), (pitch, K, 1))
    expect = old.clone()
    view(expect).add_(view(fresh))           # torch's in-place bf16 add: fp32 sum, one rounding
    torch.cuda.synchronize()
    assert (bits(acc) == bits(expect)).all()
    # the padding between the experts' matrices is not touched
    gap = torch.as_strided(acc, (G, 64), (pitch, 1), N * K)
    assert (bits(gap) == bits(torch.as_strided(old, (G, 64), (pitch, 1), N * K))).all()
    # a second accumulation on top of the first
    run("_accumulate", acc)
    view(expect).add_(view(fresh))
    torch.cuda.synchronize()
    assert (bits(acc) == bits(expect)).all()


# both tile shapes, one launch and three, extents that no tile divides, experts without rows, one with more rows than the
# block keeps indices of in LDS
@pytest.mark.parametrize("kind,G,rows,I,H", [("ragged", 8, 4096, 512, 256), ("ragged", 12, 9003, 712, 1000), ("empties", 16, 777, 128, 256),
                                             ("ragged", 64, 4096, 1024, 2048), ("uniform", 22, 11000, 512, 1024), ("onehot", 5, 5000, 256, 512),
                                             ("uniform", 1, 300, 264, 136), ("ragged", 3, 5, 8, 72), ("uniform", 4, 0, 128, 128),
                                             # (more than 16 rounds of tiles: three launches that write, one that adds)
                                             ("ragged", 700, 2000, 136, 136)])
@pytest.mark.parametrize("indexed", [False, True])
def test_three_weight_gradients_of_a_merged_mlp(cuda, indexed, kind, G, rows, I, H):
    """One bf16 rounding of a float32 sum over an expert's rows (2^-8 of the value, and the order of the sum); the
    accumulating form equals torch's in-place add of what the writing form gives, bit for bit."""
    from optimus import _native as n
    g = torch.Generator().manual_seed(rows + I)
    T = max(rows // 2, 8)
    rnd = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16).to(cuda)
    dout, x, h, dg, du = rnd(T if indexed else max(rows, 1), H), rnd(T if indexed else max(rows, 1), H), rnd(max(rows, 1), I), rnd(max(rows, 1), I), rnd(max(rows, 1), I)
    idx = torch.randint(0, T, (max(rows, 1),), generator=g, dtype=torch.int32).to(cuda)
    cum = _counts(kind, G, rows) if rows else torch.zeros(G + 1, dtype=torch.int32)
    d, P, ix = cum.to(cuda), n.ptr, idx if indexed else None
    pitch = I * H + 64
    old = [rnd(G * pitch) for _ in range(3)]
    fresh, acc = [torch.full_like(o, 7.0) for o in old], [o.clone() for o in old]
    p = lambda t: None if t is None else P(t)
    for suffix, out in (("", fresh), ("_accumulate", acc)):
        _call("om_grouped_gemm_wgrad_merged" + suffix, P(dout), p(ix), P(h), P(dg), P(du), P(x), p(ix), T, *(P(o) for o in out),
              P(d), rows, G, I, H, pitch, pitch, pitch)
    torch.cuda.synchronize()
    dr, xr = (t[idx.long()] if indexed else t for t in (dout, x))
    for i, (a, b, m, k) in enumerate(((dr, h, H, I), (dg, xr, I, H), (du, xr, I, H))):
        view = lambda t: torch.as_strided(t, (G, m, k), (pitch, k, 1))
        for e in range(G):
            s = slice(int(cum[e]), int(cum[e + 1]))
            want = a[s].float().t() @ b[s].float()
            err = (view(fresh[i])[e].float() - want).abs()
            assert (err <= want.abs() * 2 ** -8 + 2e-5 * max(s.stop - s.start, 1) ** 0.5).all(), (i, e)
        expect = old[i].clone()
        view(expect).add_(view(fresh[i]))
        assert (bits(acc[i]) == bits(expect)).all(), i
        assert (torch.as_strided(fresh[i], (G, 64), (pitch, 1), I * H) == 7.0).all()


# matrices of 96 and more 256x256 tiles, a multiple of eight of them: the XCDs share every expert's tiles, the experts come
# by rows.  Equal rows, one expert (with fewer than 128 tiles: the 128x128 kernel), more experts than a round has blocks, all
# rows on one, wide and tall matrices.
@pytest.mark.parametrize("kind,G,rows,N,K", [("uniform", 1, 100, 2048, 3072), ("uniform", 1, 100, 4096, 2048), ("ragged", 33, 1500, 2048, 3072), ("empties", 6, 900, 3072, 2048),
                                             ("onehot", 5, 700, 4096, 2048), ("uniform", 4, 512, 3072, 2048), ("uniform", 3, 0, 2048, 3072),
                                             # (the line below which only the accumulating form is shared)
                                             ("ragged", 33, 527, 2048, 3072), ("ragged", 33, 528, 2048, 3072)])
@pytest.mark.parametrize("gathered", [False, True])
def test_weight_gradients_spread_over_the_xcds(cuda, gathered, kind, G, rows, N, K):
    """The same bound as above: one bf16 rounding of a float32 sum over the expert's rows; accumulated bit for bit as
    torch's in-place add of it."""
    from optimus import _native as n
    g = torch.Generator().manual_seed(rows + G)
    T = max(rows // 2, 8)
    rnd = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16).to(cuda)
    dout, x = rnd(max(rows, 1), N), rnd(T if gathered else max(rows, 1), K)
    idx = torch.randint(0, T, (max(rows, 1),), generator=g, dtype=torch.int32).to(cuda)
    cum = _counts(kind, G, rows) if rows else torch.zeros(G + 1, dtype=torch.int32)
    d, P = cum.to(cuda), n.ptr
    old = torch.randn(G, N, K, device=cuda).to(torch.bfloat16)
    fresh, acc = torch.full_like(old, 7.0), old.clone()
    for suffix, out in (("", fresh), ("_accumulate", acc)):
        if gathered:
            _call("om_grouped_gemm_wgrad_gathered" + suffix, P(dout), P(x), P(idx), T, P(out), P(d), rows, G, N, K, 0)
        else:
            _call("om_grouped_gemm_wgrad" + suffix, P(dout), P(x), P(out), P(d), rows, G, N, K, 0)
    xr = x[idx.long()] if gathered else x
    for e in range(G):
        s = slice(int(cum[e]), int(cum[e + 1]))
        want = dout[s].float().t() @ xr[s].float()
        err = (fresh[e].float() - want).abs()
        assert (err <= want.abs() * 2 ** -8 + 2e-5 * max(s.stop - s.start, 1) ** 0.5).all(), e
    assert (bits(acc) == bits(old.add_(fresh))).all()


def _launches(fn):
    """Kernels that fn launches."""
    import ctypes
    from optimus import _native as n
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph):
        fn()
    nodes = ctypes.c_size_t()
    count = ctypes.CDLL(n.LIB_PATH).hipGraphGetNodes       # (the runtime that the library is linked with)
    assert count(ctypes.c_void_p(graph.raw_cuda_graph()), None, ctypes.byref(nodes)) == 0
    return nodes.value


# 16 experts of 32 tiles a product: as many rounds in one launch as in three, so that only few rows take one launch
@pytest.mark.parametrize("suffix", ["", "_accumulate"])
@pytest.mark.parametrize("expected,launches", [(0, 1), (520, 1), (4096, 1), (4097, 3), (4160, 3)])
def test_launches_go_by_the_rows_to_expect(cuda, suffix, expected, launches):
    """Where `rows` is a bound, three times and more what there is, the choice is the one that the plain form makes for
    the rows to expect, and the results are its results."""
    from optimus import _native as n
    G, bound, I, H = 16, 4160, 1024, 2048
    cum = _counts("ragged", G, 520)
    torch.manual_seed(2)
    rnd = lambda *s: torch.randn(*s, device=cuda).to(torch.bfloat16)
    dout, x, h, dg, du, d, P = rnd(bound, H), rnd(bound, H), rnd(bound, I), rnd(bound, I), rnd(bound, I), cum.to(cuda), n.ptr
    old = [rnd(G, I * H) for _ in range(3)]
    got, want = [o.clone() for o in old], [o.clone() for o in old]
    args = lambda out, *rows: (P(dout), None, P(h), P(dg), P(du), P(x), None, 0, *(P(o) for o in out), P(d), *rows, G, I, H, 0, 0, 0)
    _call("om_grouped_gemm_wgrad_merged" + suffix, *args(want, 520))
    name = "om_grouped_gemm_wgrad_merged" + suffix + "_bound"
    _call(name, *args(got, bound, expected))
    torch.cuda.synchronize()
    for a, b in zip(got, want):
        assert (bits(a) == bits(b)).all()
    assert _launches(lambda: _call(name, *args(got, bound, expected))) == launches


# 33 rounds of 256x256 tiles: from 128 rows an expert on the writing form makes three launches
@pytest.mark.parametrize("rows,suffix,launches", [(3711, "", 1), (3712, "", 3), (3712, "_accumulate", 1)])
def test_launches_of_large_experts(cuda, rows, suffix, launches):
    from optimus import _native as n
    G, I, H = 29, 2048, 3072
    torch.manual_seed(4)
    rnd = lambda *s: torch.randn(*s, device=cuda).to(torch.bfloat16)
    dout, x, h, dg, du, d, P = rnd(rows, H), rnd(rows, H), rnd(rows, I), rnd(rows, I), rnd(rows, I), _counts("ragged", G, rows).to(cuda), n.ptr
    got = [rnd(G, I * H) for _ in range(3)]
    want = [o.clone() for o in got]
    run = lambda: _call("om_grouped_gemm_wgrad_merged" + suffix, P(dout), None, P(h), P(dg), P(du), P(x), None, 0, *(P(o) for o in got),
                        P(d), rows, G, I, H, 0, 0, 0)
    run()
    for o, a, b, m, k in zip(want, (dout, dg, du), (h, x, x), (H, I, I), (I, H, H)):
        _call("om_grouped_gemm_wgrad" + suffix, P(a), P(b), P(o), P(d), rows, G, m, k, 0)
    torch.cuda.synchronize()
    for a, b in zip(got, want):
        assert torch.equal(a, b)
    assert _launches(run) == launches


@pytest.mark.parametrize("offset", [0, 8, 32])
def test_large_gradients_off_a_line(cuda, offset):
    """Gradients that the caches cannot hold, on a 128-byte line (stored past the caches) and off it: the same bits."""
    from optimus import _native as n
    G, rows, I, H = 45, 500, 1024, 1024
    torch.manual_seed(1)
    rnd = lambda *s: torch.randn(*s, device=cuda).to(torch.bfloat16)
    dout, x, h, dg, du, d, P = rnd(rows, H), rnd(rows, H), rnd(rows, I), rnd(rows, I), rnd(rows, I), _counts("ragged", G, rows).to(cuda), n.ptr
    out = [torch.full((G * I * H + 64,), 7.0, dtype=torch.bfloat16, device=cuda) for _ in range(3)]
    _call("om_grouped_gemm_wgrad_merged", P(dout), None, P(h), P(dg), P(du), P(x), None, 0, *(P(o[offset:]) for o in out), P(d), rows, G, I, H, 0, 0, 0)
    for o, a, b in zip(out, (dout, dg, du), (h, x, x)):
        one = torch.empty(G, I, H, dtype=torch.bfloat16, device=cuda)
        _call("om_grouped_gemm_wgrad", P(a), P(b), P(one), P(d), rows, G, H, I, 0)
        assert torch.equal(o[offset:offset + one.numel()].view_as(one), one)
        assert (o[:offset] == 7.0).all() and (o[offset + one.numel():] == 7.0).all()


def test_accumulate_f32(cuda):
    from optimus import _native as n
    g = torch.Generator().manual_seed(5)
    G, rows, N, K = 6, 700, 128, 64
    dout = torch.randn(rows, N, generator=g).to(cuda)
    x = torch.randn(rows, K, generator=g).to(cuda)
    cum = _counts("empties", G, rows).to(cuda)
    old = torch.randn(G, N, K, generator=g).to(cuda)
    fresh = torch.empty_like(old)
    P = n.ptr
    _call("om_grouped_gemm_wgrad_f32", P(dout), P(x), P(fresh), P(cum), rows, G, N, K, 0)
    acc = old.clone()
    _call("om_grouped_gemm_wgrad_f32_accumulate", P(dout), P(x), P(acc), P(cum), rows, G, N, K, 0)
    torch.cuda.synchronize()
    assert torch.equal(acc, old + fresh)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("tied", [(0, 0, 1), (0, 1, 0), (0, 1, 1), (0, 0, 0)])     # gate, up, down: which parameter
@pytest.mark.parametrize("G,rows,I", [(8, 700, 256), (3, 3000, 512), (1, 129, 200)])
def test_weights_that_are_one_parameter(cuda, G, rows, I, tied, dtype):
    """Projections that share a parameter add into one live gradient: the sum of the gradients that separate parameters get,
    in the order down, gate, up; bit for bit."""
    from optimus.models.common.moe import MergedMLPFunction
    g = torch.Generator().manual_seed(rows + sum(tied))
    H = I if tied[2] in tied[:2] else I + 56
    rnd = lambda *s, f=1.0: (torch.randn(*s, generator=g) * f).to(dtype).to(cuda)
    x, dy, cum = rnd(rows, H), rnd(rows, H), _counts("ragged", G, rows).to(cuda)
    shapes = [(G, I, H), (G, I, H), (G, H, I)]
    values = {t: rnd(*shapes[tied.index(t)], f=0.05) for t in sorted(set(tied))}
    old = {t: rnd(*values[t].shape) for t in values}

    def run(weights):
        xd = x.clone().requires_grad_(True)
        MergedMLPFunction.apply(xd, *weights, cum).backward(dy)
        torch.cuda.synchronize()
        return xd.grad

    def live(value, grad):                   # a parameter whose gradient lies in a larger buffer
        p = torch.nn.Parameter(value.clone())
        flat = torch.full((grad.numel() + 64,), 7.0, dtype=dtype, device=cuda)
        p.grad = flat[:grad.numel()].view_as(grad)
        p.grad.copy_(grad)
        return p

    separate = [torch.nn.Parameter(values[t].clone()) for t in tied]
    dx = run(separate)
    for _ in range(3):
        one = {t: live(values[t], old[t]) for t in values}
        buffers = {t: one[t].grad.data_ptr() for t in one}
        assert torch.equal(run([one[t] for t in tied]), dx)
        for t in values:
            want = old[t].clone()
            for i in (2, 0, 1):
                if tied[i] == t:
                    want += separate[i].grad
            assert one[t].grad.data_ptr() == buffers[t] and (bits(one[t].grad) == bits(want)).all(), t


# gate, up and down gradients of each expert between one another in one buffer, and the same with gate and up in one place
@pytest.mark.parametrize("pitches,offsets", [((3, 3, 3), (0, 1, 2)), ((3, 3, 3), (0, 0, 2)), ((2, 2, 1), (0, 1, 12)), ((2, 4, 1), (0, 0, 24))])
def test_interleaved_gradients(cuda, pitches, offsets):
    """bf16 and float32 entry points on gradients at multiples of I * H in one buffer, against one product at a time."""
    from optimus import _native as n
    G, rows, I, H = 6, 500, 128, 192
    for dtype in (torch.bfloat16, torch.float32):
        g = torch.Generator().manual_seed(sum(pitches))
        rnd = lambda *s: torch.randn(*s, generator=g).to(dtype).to(cuda)
        dout, x, h, dg, du, wg, wu = rnd(rows, H), rnd(rows, H), rnd(rows, I), rnd(rows, I), rnd(rows, I), rnd(G, I, H), rnd(G, I, H)
        cum, P, M, dx, f = _counts("ragged", G, rows).to(cuda), n.ptr, I * H, torch.empty_like(x), "_f32" if dtype == torch.float32 else ""
        got = rnd(32 * M)
        want = got.clone()
        at = lambda t: [P(t[o * M:]) for o in offsets]
        if f:
            _call("om_grouped_gemm_wgrad_merged_dgrad_f32_accumulate", P(dout), P(h), P(dg), P(du), P(x), None, 0, P(wg), P(wu), P(dx),
                  at(got)[2], at(got)[0], at(got)[1], P(cum), rows, G, I, H, 0, 0, pitches[2] * M, pitches[0] * M, pitches[1] * M)
        else:
            _call("om_grouped_gemm_wgrad_merged_accumulate", P(dout), None, P(h), P(dg), P(du), P(x), None, 0, at(got)[2], at(got)[0],
                  at(got)[1], P(cum), rows, G, I, H, pitches[2] * M, pitches[0] * M, pitches[1] * M)
        for i, a, b, N, K in ((2, dout, h, H, I), (0, dg, x, I, H), (1, du, x, I, H)):
            _call(f"om_grouped_gemm_wgrad{f}_accumulate", P(a), P(b), at(want)[i], P(cum), rows, G, N, K, pitches[i] * M)
        torch.cuda.synchronize()
        assert (bits(got) == bits(want)).all()
        if f:
            two = want.clone()
            got = want.clone()
            _call("om_merged_mlp_gate_up_wgrad_f32", P(dg), P(du), P(x), None, 0, at(got)[0], at(got)[1], P(cum), rows, G, I, H,
                  pitches[0] * M, pitches[1] * M, 3)
            for i, a in ((0, dg), (1, du)):
                _call("om_grouped_gemm_wgrad_f32_accumulate", P(a), P(x), at(two)[i], P(cum), rows, G, I, H, pitches[i] * M)
            torch.cuda.synchronize()
            assert (bits(got) == bits(two)).all()


def _olmoe_block(cuda, merged, fast=True, dtype=torch.bfloat16, seed=3):
    from optimus.mapper import ParallelDpPpEpTpMapper
    from optimus.models.common.moe import FastOlmoeParallelSparseMoeBlock
    from optimus.models.olmoe.configuration_olmoe import OlmoeParallelConfig
    from optimus.models.olmoe.modeling_olmoe import OlmoeParallelSparseMoeBlock
    cfg = OlmoeParallelConfig(hidden_size=256, intermediate_size=256, num_experts=8, num_experts_per_tok=2,
                              norm_topk_prob=True, use_fast_moe=True, use_merged_mlp_in_fast_moe=merged)
    cfg.router_logits_fp32 = True
    torch.manual_seed(seed)
    cls = FastOlmoeParallelSparseMoeBlock if fast else OlmoeParallelSparseMoeBlock
    blk = cls(cfg, ParallelDpPpEpTpMapper())
    for p in blk.parameters():
        torch.nn.init.normal_(p, std=0.05)
    return blk.to(cuda).to(dtype)


def _dsv3_block(cuda, seed=4):
    from optimus.mapper import ParallelDpPpEpTpMapper
    from optimus.models.deepseek_v3.configuration_deepseek_v3 import DeepseekV3ParallelConfig
    from optimus.models.deepseek_v3.modeling_deepseek_v3 import DeepseekV3ParallelMoE
    cfg = DeepseekV3ParallelConfig(hidden_size=256, moe_intermediate_size=128, n_routed_experts=16,
                                   num_experts_per_tok=4, n_group=4, topk_group=2, expert_parallelism=2)
    torch.manual_seed(seed)
    blk = DeepseekV3ParallelMoE(cfg, ParallelDpPpEpTpMapper(expert_parallelism=2, rank=1))
    for p in blk.parameters():
        torch.nn.init.normal_(p, std=0.05)
    return blk.to(cuda).to(torch.bfloat16)


def _two_backwards(blk, cuda, dtype, in_place):
    """flat_grad after two backward passes without zero_grad under MixedPrecisionAdamW, and the
    names of the C-ABI entry points the second pass launched."""
    from optimus import _native
    from optimus.models.common import moe
    from optimus.optimizers import MixedPrecisionAdamW
    opt = MixedPrecisionAdamW(blk.parameters(), blk, lr=1e-3, dtype=dtype, device=cuda)
    g = torch.Generator().manual_seed(11)
    xs = [torch.randn(2, 192, 256, generator=g).to(dtype).to(cuda) for _ in range(2)]
    ds = [torch.randn(2, 192, 256, generator=g).to(dtype).to(cuda) for _ in range(2)]
    moe.accumulate_weight_grads_in_place = in_place
    try:
        opt.zero_grad()
        names = []
        for i, (x, d) in enumerate(zip(xs, ds)):
            if i == 1:
                _native.launch_log = []
            out = blk(x)
            out = out[0] if isinstance(out, tuple) else out
            out.backward(d)
        torch.cuda.synchronize()
        names = [nm for nm, _, _ in _native.launch_log]
    finally:
        _native.launch_log = None
        moe.accumulate_weight_grads_in_place = True
    for p in blk.parameters():          # every gradient still is its view of the flat buffer
        assert p.grad.untyped_storage().data_ptr() == opt.flat_grad.untyped_storage().data_ptr()
    return opt.flat_grad.clone(), names


BLOCKS = {
    "fast_merged": lambda cuda: (_olmoe_block(cuda, True), torch.bfloat16),
    "fast_per_expert": lambda cuda: (_olmoe_block(cuda, False), torch.bfloat16),
    "slow_per_expert": lambda cuda: (_olmoe_block(cuda, False, fast=False), torch.bfloat16),
    "fast_merged_f32": lambda cuda: (_olmoe_block(cuda, True, dtype=torch.float32), torch.float32),
    "dsv3_window_and_shared": lambda cuda: (_dsv3_block(cuda), torch.bfloat16),
}


@pytest.mark.parametrize("which", sorted(BLOCKS))
def test_block_under_flat_buffer_optimizer_accumulates_in_the_epilogue(cuda, which):
    """Two backward passes without zero_grad: the flat gradient buffer is bit-identical whether the
    weight-gradient GEMMs add into it themselves or autograd adds their fresh results, and in the
    first form no plain weight-gradient launch (hence no separate accumulation pass) is left."""
    blk_a, dtype = BLOCKS[which](cuda)
    blk_b, _ = BLOCKS[which](cuda)
    fused, names_fused = _two_backwards(blk_a, cuda, dtype, True)
    plain, names_plain = _two_backwards(blk_b, cuda, dtype, False)
    assert (bits(fused) == bits(plain)).all()
    assert float(fused.float().abs().max()) > 0
    wgrads = [nm for nm in names_fused if nm.startswith("om_grouped_gemm_wgrad")]
    assert wgrads and all(nm.endswith("_accumulate") for nm in wgrads), wgrads
    assert not any(nm.endswith("_accumulate") for nm in names_plain)


def test_fresh_gradients_without_a_live_buffer(cuda):
    """Without an optimizer that owns the gradients (p.grad is None, or a tensor of its own) the
    functions return fresh gradients and autograd accumulates as usual."""
    from optimus import _native
    blk = _olmoe_block(cuda, True)
    x = torch.randn(1, 128, 256).to(torch.bfloat16).to(cuda)
    _native.launch_log = []
    try:
        for _ in range(2):
            blk(x)[0].backward(torch.ones_like(x))
        torch.cuda.synchronize()
        names = [nm for nm, _, _ in _native.launch_log]
    finally:
        _native.launch_log = None
    assert not any(nm.endswith("_accumulate") for nm in names)
    assert all(p.grad is not None for p in blk.parameters())


def test_accumulation_under_activation_checkpointing(cuda):
    """With the block's expert computation under torch's activation checkpoint (the reference's
    use_activation_checkpointing bit 0, moe.py:430-432, :612-616) the recomputed forward's backward
    still adds into the live gradient buffer, with the same bits as without checkpointing."""
    from optimus.optimizers import MixedPrecisionAdamW
    res = []
    for ckpt in (False, True):
        blk = _olmoe_block(cuda, True)
        blk.use_activation_checkpointing_for_moe = ckpt
        opt = MixedPrecisionAdamW(blk.parameters(), blk, lr=1e-3, dtype=torch.bfloat16, device=cuda)
        g = torch.Generator().manual_seed(21)
        opt.zero_grad()
        for _ in range(2):
            x = torch.randn(2, 128, 256, generator=g).to(torch.bfloat16).to(cuda).requires_grad_(True)
            blk(x)[0].backward(torch.randn(2, 128, 256, generator=g).to(torch.bfloat16).to(cuda))
        torch.cuda.synchronize()
        res.append(opt.flat_grad.clone())
    assert (bits(res[0]) == bits(res[1])).all() and float(res[0].float().abs().max()) > 0
