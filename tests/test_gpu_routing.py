"""Router parity through the module-level autograd Functions (-> C-ABI om_route_*).

Bar: expert indices bit-exact on fixtures whose top-(K+1) scores are separated by more than 4 fp32
ulp (so a last-ulp difference between two exp() implementations cannot reorder a row); weights
within 1 bf16 ulp / 1e-6 relative in fp32; gradients against autograd of the torch restatement."""
import numpy as np
import pytest
import torch

from oracle import routing as R

pytestmark = pytest.mark.gpu


def _valid_logits(T, N, K, seed, scale=1.0, bias=None):
    while True:
        g = torch.Generator().manual_seed(seed)
        logits = torch.randn(T, N, generator=g) * scale
        if bias is not None:
            logits = logits + bias
        if R.min_topk_gap_ulps(torch.softmax(logits, 1), K) > 4.0:
            return logits
        seed += 1000


@pytest.mark.parametrize("T,N,K,renorm,ldt,wdt", [
    (2048, 8, 2, True, torch.float32, torch.float32),      # C1
    (16384, 64, 8, False, torch.float32, torch.bfloat16),  # C3: fp32 logits
    (512, 64, 8, False, torch.float32, torch.bfloat16),    # C4 shape
    (300, 100, 5, True, torch.float32, torch.float32),     # N not a multiple of 64
    (257, 256, 8, True, torch.float32, torch.float32),
    (64, 384, 6, False, torch.float32, torch.float32),
])
def test_softmax_topk_forward(cuda, T, N, K, renorm, ldt, wdt):
    from optimus.models.common.moe import SoftmaxTopkRouterFunction as F
    logits = _valid_logits(T, N, K, seed=T + N)
    w_ref, e_ref, _ = R.olmoe_router(logits, K, renorm, wdt)
    w, e = F.apply(logits.to(ldt).to(cuda), K, renorm, wdt)
    assert e.dtype == torch.int64 and torch.equal(e.cpu(), e_ref)
    if wdt == torch.bfloat16:
        # at most one bf16 ulp apart
        a = w.cpu().view(torch.int16).int(); b = w_ref.view(torch.int16).int()
        assert int((a - b).abs().max()) <= 1
    else:
        assert float(((w.cpu() - w_ref).abs() / w_ref).max()) <= 2e-6


@pytest.mark.parametrize("seed", list(range(16)))
def test_softmax_topk_random_shapes(cuda, seed):
    """Seeded sweep over expert counts (one to eight experts per lane), top-k up to 64, odd token
    counts, logit scales (sharp and flat distributions), both weight dtypes."""
    from optimus.models.common.moe import SoftmaxTopkRouterFunction as F
    rng = np.random.RandomState(31 + seed)
    N = int(rng.choice([2, 3, 8, 60, 64, 65, 128, 200, 256, 512]))
    K = int(rng.choice([1, 2, min(8, N), min(64, N)]))
    T = int(rng.choice([1, 7, 100, 1023, 5000]))
    renorm = bool(seed % 2)
    wdt = [torch.float32, torch.bfloat16][(seed // 2) % 2]
    g = torch.Generator().manual_seed(seed)
    logits = torch.randn(T, N, generator=g) * float(rng.choice([0.3, 1.0, 4.0]))
    # rows whose top-(K+1) probabilities are more than 4 ulp apart: there a last-ulp difference in
    # exp() cannot change the choice, and the result must be the restatement's
    probs = torch.softmax(logits, 1)
    top = torch.sort(probs, dim=1, descending=True).values[:, :min(K + 1, N)]
    ok = ((top[:, :-1] - top[:, 1:]) > 4 * top[:, :-1] * 2.0 ** -23).all(dim=1) if N > 1 else torch.ones(T, dtype=torch.bool)
    w_ref, e_ref, _ = R.olmoe_router(logits, K, renorm, wdt)
    w, e = F.apply(logits.to(cuda), K, renorm, wdt)
    tag = (T, N, K, renorm, wdt)
    assert int(ok.sum()) >= T // 2, tag
    assert torch.equal(e.cpu()[ok], e_ref[ok]), tag
    if wdt == torch.bfloat16:
        a = w.cpu()[ok].view(torch.int16).int(); b = w_ref[ok].view(torch.int16).int()
        assert int((a - b).abs().max()) <= 1, tag
    else:
        assert float(((w.cpu()[ok] - w_ref[ok]).abs() / w_ref[ok].clamp_min(1e-30)).max()) <= 4e-6, tag
    # every row, tie or not: K distinct experts, none of them worse than an unselected one
    sel = probs.gather(1, e.cpu())
    rest = probs.scatter(1, e.cpu(), -1.0)
    assert bool((sel.min(1).values >= rest.max(1).values * (1 - 1e-6)).all()), tag
    srt = torch.sort(e.cpu(), 1).values
    assert bool((srt[:, 1:] != srt[:, :-1]).all()), tag


def test_softmax_topk_bf16_logits_and_ties(cuda):
    """bf16 logits tie often; the rule is (probability desc, expert index asc) = stable sort."""
    from optimus.models.common.moe import SoftmaxTopkRouterFunction as F
    g = torch.Generator().manual_seed(0)
    logits = torch.randn(4096, 64, generator=g).to(torch.bfloat16)
    logits[:64] = 0.0            # all equal: experts 0..K-1 in order
    logits[64:128] = logits[64:128].clamp(max=2.0)
    logits[64:128, 10:20] = 3.0  # ten-way tie above the rest: 10..17
    w, e = F.apply(logits.to(cuda), 8, False, torch.float32)
    e = e.cpu()
    assert torch.equal(e[:64], torch.arange(8).expand(64, 8))
    assert torch.equal(e[64:128], torch.arange(10, 18).expand(64, 8))
    # rows whose fp32 probabilities have no near-ties must match the oracle exactly
    probs = torch.softmax(logits.float(), 1)
    top = torch.sort(probs, dim=1, descending=True).values[:, :9]
    ok = ((top[:, :-1] - top[:, 1:]) > 4 * top[:, :-1] * 2.0 ** -23).all(dim=1)
    _, e_ref, _ = R.olmoe_router(logits, 8, False, torch.float32)
    assert int(ok.sum()) > 1000 and torch.equal(e[ok], e_ref[ok])
    # every row: a valid top-K set (K-th selected prob >= best unselected prob, up to 4 ulp)
    sel = probs.gather(1, e)
    rest = probs.scatter(1, e, -1.0)
    assert bool((sel.min(1).values >= rest.max(1).values * (1 - 1e-6)).all())
    assert bool((torch.sort(e, 1).values[:, 1:] != torch.sort(e, 1).values[:, :-1]).all())


@pytest.mark.parametrize("N,K,renorm,ldt", [(8, 2, True, torch.float32), (64, 8, False, torch.float32),
                                           (64, 8, True, torch.bfloat16), (256, 8, True, torch.float32)])
def test_softmax_topk_backward(cuda, N, K, renorm, ldt):
    from optimus.models.common.moe import SoftmaxTopkRouterFunction as F
    T = 512
    logits = _valid_logits(T, N, K, seed=N).to(ldt)
    g = torch.Generator().manual_seed(1)
    dw = torch.randn(T, K, generator=g)
    x = logits.to(cuda).requires_grad_(True)
    w, e = F.apply(x, K, renorm, torch.float32)
    w.backward(dw.to(cuda))
    xr = logits.float().requires_grad_(True)
    wr, er, _ = R.olmoe_router(xr, K, renorm, torch.float32)
    wr.backward(dw)
    tol = 1e-5 if ldt == torch.float32 else 1e-2
    err = (x.grad.float().cpu() - xr.grad).abs().max() / xr.grad.abs().max()
    assert float(err) <= tol, float(err)


def _dsv3_case(T, N, n_group, seed):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(T, N, generator=g) * 0.5, torch.randn(N, generator=g) * 0.1


@pytest.mark.parametrize("T,N,n_group,topk_group,K,renorm", [
    (8192, 256, 8, 4, 8, True),      # C5
    (512, 16, 4, 2, 2, True),        # tiny brute-force shape
    (512, 64, 8, 3, 6, False),
    (100, 256, 1, 1, 8, True),       # one group = plain top-K
])
def test_sigmoid_group_topk(cuda, T, N, n_group, topk_group, K, renorm):
    from optimus.models.deepseek_v3.modeling_deepseek_v3 import SigmoidGroupTopkRouterFunction as F
    logits, bias = _dsv3_case(T, N, n_group, seed=N + K)
    scores = logits.sigmoid()
    e_ref, choice = R.dsv3_topk_indices(scores, bias, n_group, topk_group, K)
    w_ref = scores.gather(1, e_ref)
    if renorm:
        w_ref = w_ref / (w_ref.sum(-1, keepdim=True) + 1e-20)
    w_ref = w_ref * 2.5
    x = logits.to(cuda).requires_grad_(True)
    e, w = F.apply(x, bias.to(cuda), n_group, topk_group, K, renorm, 2.5)
    # rows where group scores and choice scores are well separated must match exactly
    gs = R._topk_stable((scores + bias).view(T, n_group, -1), 2)[0].sum(-1)
    gtop = torch.sort(gs, dim=1, descending=True).values
    gap_g = (gtop[:, topk_group - 1] - gtop[:, topk_group]) if topk_group < n_group else torch.ones(T)
    ctop = torch.sort(choice, dim=1, descending=True).values[:, :K + 1]
    gap_c = (ctop[:, :-1] - ctop[:, 1:]).min(1).values
    ok = (gap_g > 1e-5) & (gap_c > 1e-5)
    assert int(ok.sum()) > 0.9 * T
    assert torch.equal(e.cpu()[ok], e_ref[ok])          # same order: choice desc
    assert float((w.detach().cpu()[ok] - w_ref[ok]).abs().max()) <= 1e-5
    if renorm:
        assert float((w.detach().sum(1).cpu() - 2.5).abs().max()) <= 1e-5
    # gradient through gather -> renorm -> scale -> sigmoid
    dw = torch.randn(T, K, generator=torch.Generator().manual_seed(2))
    w.backward(dw.to(cuda))
    lr = logits.clone().requires_grad_(True)
    sr = lr.sigmoid()
    wr = sr.gather(1, e.cpu())
    if renorm:
        wr = wr / (wr.sum(-1, keepdim=True) + 1e-20)
    (wr * 2.5).backward(dw)
    assert float((x.grad.cpu() - lr.grad).abs().max()) <= 1e-5 * max(1.0, float(lr.grad.abs().max()))


# ---- gate projection fused with the routing (om_router_gate_logits / om_router_gate_softmax_topk) --
def _gate_inputs(T, H, N, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(T, H, generator=g).to(torch.bfloat16)
    w = (torch.randn(N, H, generator=g) * 0.02).to(torch.bfloat16)
    return x, w


@pytest.mark.parametrize("T,H,N", [(1000, 2048, 64), (64, 512, 8), (33, 1024, 128), (300, 7168, 256),
                                   (4096, 2048, 60), (200, 2304, 8), (77, 192, 60),   # hidden sizes the one-pass kernel does not take
                                   # more than 64 experts: the kernel that shares the weight tile
                                   # through LDS and splits H (odd step counts, padded expert rows,
                                   # a partial last 128-token block, one and several slices)
                                   (8192, 7168, 256), (1000, 1024, 130), (129, 320, 96), (5, 64, 200),
                                   # hidden sizes that are multiples of 8 only: a last step with fewer than 64 columns
                                   (300, 72, 8), (129, 328, 96), (1000, 1000, 130), (5, 8, 200), (2048, 200, 64)])
def test_gate_logits_match_fp32_matmul(cuda, T, H, N):
    """fp32 logits from bf16 operands: the products are exact, only the order of the fp32 sum differs
    from the CPU matmul of the up-cast operands."""
    from optimus.models.common.moe import fp32_logits
    x, w = _gate_inputs(T, H, N, seed=T + N)
    got = fp32_logits(x.to(cuda), w.to(cuda)).cpu()
    ref = x.float() @ w.float().t()
    exact = (x.double() @ w.double().t())
    assert got.dtype == torch.float32 and got.shape == (T, N)
    # both are fp32 sums of the same exact products: compare their distance to the fp64 value
    err_got = float((got.double() - exact).abs().max()); err_ref = float((ref.double() - exact).abs().max())
    assert err_got <= max(4 * err_ref, 2e-6), (err_got, err_ref)


@pytest.mark.parametrize("T,H,N,K,renorm,wdt", [
    (16384, 2048, 64, 8, False, torch.bfloat16),    # C3
    (1000, 2048, 64, 8, True, torch.float32),       # ragged token count
    (512, 1024, 128, 6, True, torch.float32),
    (96, 512, 8, 2, True, torch.bfloat16),
])
def test_gate_softmax_topk_equals_two_step_on_its_own_logits(cuda, T, H, N, K, renorm, wdt):
    """The routing half of the fused kernel is the same code as om_route_softmax_topk: on the logits
    the kernel itself returns, experts and weights must be identical bit for bit, and the experts
    equal the CPU oracle's on rows without near-ties."""
    from optimus.models.common.moe import GateSoftmaxTopkFunction, SoftmaxTopkRouterFunction
    x, w = _gate_inputs(T, H, N, seed=7 * T + N)
    wts, exp, logits, x_out = GateSoftmaxTopkFunction.apply(x.to(cuda), w.to(cuda), K, renorm, wdt)
    assert x_out.data_ptr() != 0 and torch.equal(x_out.cpu(), x)      # the pass-through of the hidden states
    w2, e2 = SoftmaxTopkRouterFunction.apply(logits.contiguous(), K, renorm, wdt)
    assert torch.equal(exp, e2) and torch.equal(wts.view(torch.int16 if wdt == torch.bfloat16 else torch.int32),
                                                w2.view(torch.int16 if wdt == torch.bfloat16 else torch.int32))
    lg = logits.cpu()
    w_ref, e_ref, _ = R.olmoe_router(lg, K, renorm, wdt)
    probs = torch.softmax(lg, 1)
    top = torch.sort(probs, dim=1, descending=True).values[:, :K + 1]
    ok = ((top[:, :-1] - top[:, 1:]) > 4 * top[:, :-1] * 2.0 ** -23).all(dim=1)
    assert int(ok.sum()) >= 0.99 * T and torch.equal(exp.cpu()[ok], e_ref[ok])


def test_gate_softmax_topk_backward(cuda):
    """dx and dW of the fused router against autograd of the fp32 restatement (the gradient of the
    logits is rounded to bf16 before the two GEMMs, as a bf16 router's backward does)."""
    from optimus.models.common.moe import GateSoftmaxTopkFunction
    T, H, N, K = 2048, 1024, 64, 8
    x, w = _gate_inputs(T, H, N, seed=5)
    g = torch.Generator().manual_seed(6)
    dw_out = torch.randn(T, K, generator=g)
    dlogit_out = torch.randn(T, N, generator=g) * 0.1
    xg = x.to(cuda).requires_grad_(True); wg = w.to(cuda).requires_grad_(True)
    dx_other = torch.randn(T, H, generator=g).to(torch.bfloat16)     # a gradient arriving through the pass-through
    wts, exp, logits, x_out = GateSoftmaxTopkFunction.apply(xg, wg, K, True, torch.float32)
    (wts * dw_out.to(cuda)).sum().backward(retain_graph=True)
    gx1, gw1 = xg.grad.clone(), wg.grad.clone()
    xg.grad = None; wg.grad = None
    ((wts * dw_out.to(cuda)).sum() + (logits * dlogit_out.to(cuda)).sum()).backward(retain_graph=True)
    # reference in fp32 on the CPU with the kernel's own expert choice
    xr = x.float().requires_grad_(True); wr = w.float().requires_grad_(True)
    lr = xr @ wr.t()
    pr = torch.softmax(lr, 1).gather(1, exp.cpu())
    pr = pr / pr.sum(1, keepdim=True)
    ((pr * dw_out).sum() + (lr * dlogit_out).sum()).backward()
    rel = lambda a, b: float((a.float().cpu() - b).abs().mean() / b.abs().mean())
    assert rel(xg.grad, xr.grad) < 1e-2 and rel(wg.grad, wr.grad) < 1e-2
    assert not torch.equal(gx1, xg.grad)     # the logits' own gradient takes part
    # a gradient through the pass-through output is added inside the kernel with autograd's two
    # roundings: bf16(float(other) + float(gate dx)) bit for bit
    gate_dx = xg.grad.clone()
    xg.grad = None; wg.grad = None
    ((wts * dw_out.to(cuda)).sum() + (logits * dlogit_out.to(cuda)).sum()
     + (x_out.float() * dx_other.to(cuda).float()).sum()).backward()
    want = (dx_other.to(cuda).float() + gate_dx.float()).to(torch.bfloat16)
    assert torch.equal(xg.grad, want)


@pytest.mark.parametrize("T,H,N,wdt", [(16384, 2048, 64, torch.bfloat16), (1, 128, 32, torch.float32),
                                       (100, 256, 64, torch.float32), (5000, 1024, 128, torch.bfloat16),
                                       (777, 7168, 256, torch.float32), (64, 2048, 64, torch.float32),
                                       # expert counts that are no multiple of 32 or of 4
                                       (300, 256, 8, torch.bfloat16), (1000, 384, 60, torch.float32),
                                       (500, 128, 130, torch.float32), (257, 512, 7, torch.float32),
                                       # hidden sizes that end in a partial 128-column slice
                                       (700, 192, 8, torch.bfloat16), (2048, 320, 64, torch.float32),
                                       (333, 72, 5, torch.float32)])
def test_gate_weight_grad_matches_fp32_matmul(cuda, T, H, N, wdt):
    """om_router_gate_wgrad against the product it replaces: dlogits rounded to bf16, multiplied in
    fp32.  The bf16 x bf16 products are exact in fp32, so only the order of the fp32 sum differs
    (float64 reference; bound = a few fp32 roundings of the absolute sum), plus one final rounding
    for a bf16 weight.  Token counts that are not multiples of the 64-token stage or of the split."""
    from optimus.models.common.moe import _gate_weight_grad
    g = torch.Generator().manual_seed(T + N)
    x = torch.randn(T, H, generator=g).to(torch.bfloat16)
    dl = torch.randn(T, N, generator=g) * 0.3
    w = torch.empty(N, H, dtype=wdt)
    out = _gate_weight_grad(x.to(cuda), w.to(cuda), dl.to(cuda))
    assert out.dtype == wdt and out.shape == (N, H)
    d16 = dl.to(torch.bfloat16).double()
    ref = d16.t() @ x.double()
    bound = 1e-6 * (d16.abs().t() @ x.double().abs()) + 1e-30
    err = (out.double().cpu() - ref).abs()
    if wdt == torch.bfloat16:
        bound = bound + ref.abs() * 2.0 ** -8      # one bf16 rounding
    assert bool((err <= bound).all()), float((err / bound).max())
    # deterministic: same bits on a second run
    out2 = _gate_weight_grad(x.to(cuda), w.to(cuda), dl.to(cuda))
    assert torch.equal(out, out2)


# ---- auxiliary load-balancing loss (om_router_balance_stats / _bwd) ---------------------------------
@pytest.mark.parametrize("L,T,N,K", [(3, 4096, 64, 8), (2, 1000, 100, 5), (1, 77, 256, 8), (4, 512, 8, 2)])
def test_balance_losses_match_the_reference_expressions(cuda, L, T, N, K):
    from optimus.models.common.ral_functions import (layer_level_load_balancing_loss_func,
                                                     load_balancing_loss_func,
                                                     single_input_load_balancing_loss_func)
    layers = tuple(_valid_logits(T, N, K, seed=31 * l + T) for l in range(L))
    dev = tuple(l.to(cuda) for l in layers)
    got = float(load_balancing_loss_func(dev, N, K)); want = float(R.load_balancing_loss(layers, N, K))
    assert abs(got - want) <= 2e-5 * want
    got = float(layer_level_load_balancing_loss_func(dev, N, K))
    want = float(R.layer_level_load_balancing_loss(layers, N, K))
    assert abs(got - want) <= 2e-5 * want
    got = float(single_input_load_balancing_loss_func(dev[0], N, K))
    want = float(R.load_balancing_loss(layers[:1], N, K))
    assert abs(got - want) <= 2e-5 * want
    assert load_balancing_loss_func(None, N, K) == 0 and load_balancing_loss_func(dev[0], N, K) == 0


def test_balance_loss_gradient_and_bf16_logits(cuda):
    from optimus.models.common.ral_functions import load_balancing_loss_func
    L, T, N, K = 2, 2048, 64, 8
    layers = [_valid_logits(T, N, K, seed=77 + l) for l in range(L)]
    ref = [l.clone().requires_grad_(True) for l in layers]
    R.load_balancing_loss(tuple(ref), N, K).backward()
    dev = [l.to(cuda).requires_grad_(True) for l in layers]
    load_balancing_loss_func(tuple(dev), N, K).backward()
    for a, b in zip(dev, ref):
        assert float((a.grad.cpu() - b.grad).abs().max()) <= 1e-5 * float(b.grad.abs().max())
    # bf16 logits: probabilities are kept in fp32 here, rounded to bf16 in the reference
    b16 = tuple(l.to(torch.bfloat16) for l in layers)
    got = float(load_balancing_loss_func(tuple(l.to(cuda) for l in b16), N, K))
    want = float(R.load_balancing_loss(tuple(l.float() for l in b16), N, K))
    assert abs(got - want) <= 1e-3 * want


@pytest.mark.parametrize("T,H,N,with_other", [(16384, 2048, 64, True), (1, 128, 32, False), (100, 264, 60, True),
                                              (5000, 1024, 128, False), (777, 7168, 256, True), (130, 2304, 7, True),
                                              (64, 8, 5, False)])
def test_gate_input_grad_matches_fp32_matmul(cuda, T, H, N, with_other):
    """om_router_gate_dgrad against the product it replaces, mm(bf16(dlogits), W): exact products,
    fp32 sums in another order, one bf16 rounding; with `other` the second rounding of the
    accumulation.  Partial token blocks, partial column blocks, expert counts that need padding."""
    from optimus.models.common.moe import _gate_input_grad
    g = torch.Generator().manual_seed(3 * T + N)
    w = (torch.randn(N, H, generator=g) * 0.05).to(torch.bfloat16)
    dl = torch.randn(T, N, generator=g) * 0.3
    other = torch.randn(T, H, generator=g).to(torch.bfloat16) if with_other else None
    got = _gate_input_grad(w.to(cuda), dl.to(cuda), None if other is None else other.to(cuda))
    assert got.dtype == torch.bfloat16 and got.shape == (T, H)
    d16 = dl.to(torch.bfloat16).double()
    exact = d16 @ w.double()
    bound = 1e-6 * (d16.abs() @ w.double().abs()) + exact.abs() * 2.0 ** -8 + 1e-30     # order of the sum + one rounding
    if other is None:
        err = (got.double().cpu() - exact).abs()
        assert bool((err <= bound).all()), float((err / bound).max())
    else:
        total = other.double() + exact
        err = (got.double().cpu() - total).abs()
        bound = bound + total.abs() * 2.0 ** -8
        assert bool((err <= bound).all()), float((err / bound).max())
        # exactly the two roundings: round the kernel's own product, add, round
        alone = _gate_input_grad(w.to(cuda), dl.to(cuda))
        assert torch.equal(got, (other.to(cuda).float() + alone.float()).to(torch.bfloat16))
    assert torch.equal(got, _gate_input_grad(w.to(cuda), dl.to(cuda), None if other is None else other.to(cuda)))


def test_gate_shapes_without_a_kernel_raise(cuda):
    """No library fallback behind the gate: a bf16 gate whose shape the kernels do not take raises."""
    from optimus._native import NativeLibraryError
    from optimus.models.common.moe import _gate_backward, fp32_logits
    x = torch.zeros(16, 100, dtype=torch.bfloat16, device=cuda)
    with pytest.raises(NativeLibraryError):
        fp32_logits(x, torch.zeros(8, 100, dtype=torch.bfloat16, device=cuda))            # H % 64
    x = torch.zeros(16, 128, dtype=torch.bfloat16, device=cuda)
    with pytest.raises(NativeLibraryError):
        fp32_logits(x, torch.zeros(300, 128, dtype=torch.bfloat16, device=cuda))          # more than 256 experts
    x = torch.zeros(16, 196, dtype=torch.bfloat16, device=cuda)
    with pytest.raises(NativeLibraryError):
        _gate_backward(x, torch.zeros(8, 196, dtype=torch.bfloat16, device=cuda),
                       torch.zeros(16, 8, device=cuda), (False, True))                      # weight gradient: H % 8
    x = torch.zeros(16, 192, dtype=torch.bfloat16, device=cuda)
    with pytest.raises(TypeError):
        fp32_logits(x, torch.zeros(8, 192, dtype=torch.float32, device=cuda))              # mixed dtypes


@pytest.mark.parametrize("L,B,S,N,K,dtype", [(3, 4, 1024, 64, 8, torch.float32), (2, 5, 200, 100, 5, torch.float32),
                                             (1, 1, 77, 256, 8, torch.float32), (2, 2, 48, 16, 2, torch.bfloat16),
                                             (4, 2, 256, 8, 2, torch.float32)])
def test_masked_balance_loss_matches_the_reference_expression(cuda, L, B, S, N, K, dtype):
    """load_balancing_loss_func with an attention mask (modeling_olmoe.py:58-83): value against the
    oracle's restatement of the masked branch, gradient against autograd through it; masked tokens get
    exactly zero gradient; an all-ones mask gives the unmasked loss."""
    from optimus.models.common.ral_functions import load_balancing_loss_func
    T = B * S
    def layer_logits(seed):
        if dtype == torch.float32:
            return _valid_logits(T, N, K, seed=seed)
        while True:    # the ROUNDED logits must order every token's top-(K+1) without ties
            lg = (torch.randn(T, N, generator=torch.Generator().manual_seed(seed)) * 4.0).to(dtype).float()
            if R.min_topk_gap_ulps(torch.softmax(lg, 1), K) > 4.0:
                return lg
            seed += 1000
    layers = tuple(layer_logits(17 * l + T + N) for l in range(L))
    g = torch.Generator().manual_seed(L + N)
    mask = (torch.rand(B, S, generator=g) > 0.3).long()
    mask[0, 0] = 1
    dev = tuple(l.to(dtype).to(cuda).requires_grad_(True) for l in layers)
    got = load_balancing_loss_func(dev, N, K, attention_mask=mask.to(cuda))
    got.backward()
    ref_in = tuple(l.to(dtype).float().requires_grad_(True) for l in layers)
    want = R.load_balancing_loss(ref_in, N, K, attention_mask=mask.float())
    want.backward()
    tol = 2e-5 if dtype == torch.float32 else 2e-3
    assert abs(float(got.detach()) - float(want.detach())) <= tol * float(want.detach())
    keep = mask.reshape(-1).bool()
    for a, b in zip(dev, ref_in):
        ga = a.grad.float().cpu()
        assert float(ga[~keep].abs().max()) == 0.0 if bool((~keep).any()) else True
        err = float((ga - b.grad).abs().max())
        assert err <= (1e-3 if dtype == torch.float32 else 2e-2) * float(b.grad.abs().max()) + 1e-12, err
    ones = load_balancing_loss_func(tuple(d.detach() for d in dev), N, K, attention_mask=torch.ones(B, S, device=cuda))
    plain = load_balancing_loss_func(tuple(d.detach() for d in dev), N, K)
    assert abs(float(ones) - float(plain)) <= 1e-6 * float(plain)


@pytest.mark.parametrize("T,H,N", [(2048, 256, 8), (1, 7, 3), (777, 100, 130), (5000, 2048, 64)])
def test_float32_gate_kernels_match_float64_products(cuda, T, H, N):
    """The float32 module's gate (om_router_gate_logits_f32 and its two backward products) against
    float64 products of the same float32 values: only the order of the float32 sums differs, so the
    bound is a few float32 roundings of the absolute sum (the weight gradient, summed in double,
    one rounding of the result)."""
    from optimus.models.common.moe import GateLogitsF32Function
    g = torch.Generator().manual_seed(T + H + N)
    x = torch.randn(T, H, generator=g)
    w = torch.randn(N, H, generator=g) * 0.1
    dl = torch.randn(T, N, generator=g)
    xd, wd = x.to(cuda).requires_grad_(True), w.to(cuda).requires_grad_(True)
    logits = GateLogitsF32Function.apply(xd, wd)
    logits.backward(dl.to(cuda))
    eps = 2.0 ** -23
    cases = (("logits", logits, x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t(), 8.0),
             ("dx", xd.grad, dl.double() @ w.double(), dl.double().abs() @ w.double().abs(), 8.0),
             ("dw", wd.grad, dl.double().t() @ x.double(), dl.double().abs().t() @ x.double().abs(), 1.0))
    for name, got, ref, absum, k in cases:
        err = (got.detach().double().cpu() - ref).abs()
        bound = k * eps * absum + 1e-30
        assert bool((err <= bound).all()), (name, float((err / bound).max()))


@pytest.mark.parametrize("T,H,N,K", [(1, 2048, 64, 8), (129, 512, 32, 4), (33, 1000, 12, 3), (5, 8, 3, 3), (300, 7168, 256, 8),
                                     (64, 64, 100, 1)])
@pytest.mark.parametrize("bf16_logits", [False, True])
def test_split_gate_router_equals_its_steps(cuda, T, H, N, K, bf16_logits):
    """om_router_gate_split_softmax_topk against the projection (to the fp32 order of the sum) and, bit for
    bit, against the router on its own logits; the logits are rounded to bf16 where asked for."""
    from optimus import _native as n
    from optimus.models.common.moe import SoftmaxTopkRouterFunction, fp32_logits
    x, w = _gate_inputs(T, H, N, seed=T + H)
    x, w = x.to(cuda), w.to(cuda)
    we, e, logits, x_out = n.host().route_softmax(x, w, K, True, torch.bfloat16, False, bf16_logits)
    assert logits.dtype == (torch.bfloat16 if bf16_logits else torch.float32) and x_out.data_ptr() == x.data_ptr()
    w2, e2 = SoftmaxTopkRouterFunction.apply(logits, K, True, torch.bfloat16)
    assert torch.equal(e, e2) and torch.equal(we.view(torch.int16), w2.view(torch.int16))
    ref = x.double() @ w.double().t()
    # fp32 sum of H exact products in another order, then (bf16) one rounding of 2^-9
    bound = 8 * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t()) + (2.0 ** -8 * ref.abs() if bf16_logits else 0)
    assert bool(((logits.double() - ref).abs() <= bound + 1e-30).all())
    if not bf16_logits and N <= 64 and H % 512 == 0:
        assert torch.equal(logits, fp32_logits(x, w))       # eight slices in order: the one-pass kernel's bits


@pytest.mark.parametrize("T,H,N,K", [(1, 512, 64, 8), (31, 1024, 33, 16), (33, 512, 17, 1), (65, 1536, 64, 17), (64, 2048, 32, 32),
                                     (95, 512, 5, 4), (513, 4608, 50, 6), (512, 4608, 50, 6),
                                     (8200, 512, 64, 8)])
@pytest.mark.parametrize("renorm", [False, True])
@pytest.mark.parametrize("one_pass,bf16_logits", [(True, False), (False, False), (False, True)])
def test_one_launch_gate_router(cuda, T, H, N, K, renorm, one_pass, bf16_logits):
    """The one-launch router of up to 64 experts: edges of its 32 tokens, experts that do not fill their
    block of 32, the selections on rows of 16 lanes and (more than 16) on whole wavefronts, equal
    logits (two experts with the same weights) and a token without a number.  The logits against
    float64 products, the routing bit for bit against the router on the same logits."""
    from optimus import _native as n
    from optimus.models.common.moe import SoftmaxTopkRouterFunction
    x, w = _gate_inputs(T, H, N, seed=T + H + N)
    w[N // 2] = w[0]
    if T > 2:
        x[T // 2, 3] = float("nan")
    x, w = x.to(cuda), w.to(cuda)
    we, e, logits, _ = n.host().route_softmax(x, w, K, renorm, torch.float32, one_pass, bf16_logits)
    w2, e2 = SoftmaxTopkRouterFunction.apply(logits, K, renorm, torch.float32)
    assert torch.equal(e, e2) and torch.equal(we.view(torch.int32), w2.view(torch.int32))
    ok = torch.ones(T, dtype=torch.bool, device=cuda)
    if T > 2:
        ok[T // 2] = False
        assert bool(logits[T // 2].isnan().all())
    assert torch.equal(logits[ok, N // 2], logits[ok, 0])
    ref = x[ok].double() @ w.double().t()
    # an fp32 sum of H exact products in any order, then (bf16) one rounding of 2^-9
    bound = 8 * 2.0 ** -24 * (x[ok].double().abs() @ w.double().abs().t()) + (2.0 ** -8 * ref.abs() if bf16_logits else 0)
    assert bool(((logits[ok].double() - ref).abs() <= bound + 1e-30).all())


@pytest.mark.parametrize("T,H,N,K,one", [(513, 1024, 64, 16, True), (513, 1024, 64, 17, False), (16, 512, 40, 20, True), (17, 512, 40, 20, False),
                                         (6144, 512, 33, 33, False), (6145, 512, 33, 33, True), (8192, 1024, 64, 17, True),
                                         (8193, 512, 64, 40, False), (8192, 512, 32, 17, False)])
def test_router_of_many_selections(cuda, T, H, N, K, one):
    """Where more than 16 experts are selected the two launches stay where they are the faster ones (seen by the workspace, which
    one launch leaves alone); the same bits either way."""
    from optimus import _native as n
    x, w = (t.to(cuda) for t in _gate_inputs(T, H, N, seed=T + K))
    size = n.lib().om_router_gate_route_workspace_bytes(T, H, N)
    ws = torch.full((size,), 77, dtype=torch.uint8, device=cuda)
    new = lambda *s, dt=torch.float32: torch.empty(*s, dtype=dt, device=cuda)
    a, b = ((new(T, N), new(T, K), new(T, K, dt=torch.int64)) for _ in range(2))
    P = n.ptr
    n.check(n.lib().om_router_gate_split_softmax_topk(P(x), P(w), T, H, N, K, 1, P(a[0]), n.OM_F32, P(a[1]), n.OM_F32, P(a[2]), P(ws), size,
                                                      n.stream()), "split")
    n.check(n.lib().om_router_gate_softmax_topk(P(x), P(w), T, H, N, K, 1, P(b[0]), P(b[1]), n.OM_F32, P(b[2]), n.stream()), "one pass")
    for u, v in zip(a, b):
        assert torch.equal(u, v)
    assert bool((ws == 77).all()) == one


@pytest.mark.parametrize("T,H,N,slices", [(4096, 1000, 12, 8), (4097, 1000, 12, 6), (6677, 4928, 40, 8), (8193, 1000, 12, 6), (11000, 4104, 8, 5), (18000, 4104, 8, 3), (18000, 336, 61, 1),
                                          (16513, 2920, 61, 3), (33000, 72, 64, 1)])
def test_gate_of_many_tokens(cuda, T, H, N, slices):
    """Up to 64 experts: as many slices of the hidden size as the busiest CU is done with soonest; the logits against float64."""
    from optimus import _native as n
    L, P = n.lib(), n.ptr
    x, w = (t.to(cuda) for t in _gate_inputs(T, H, N, seed=T + N))
    size = L.om_router_gate_logits_split_workspace_bytes(T, H, N)
    assert size == slices * T * N * 4
    ws, logits = torch.empty(size, dtype=torch.uint8, device=cuda), torch.full((T + 1, N), 7.0, device=cuda)
    n.check(L.om_router_gate_logits_split(P(x), P(w), T, H, N, P(logits), P(ws), size, n.stream()), "logits")
    bound = (H / 16 + 33) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t()) + 1e-30   # as in test_gate_of_many_experts
    assert bool(((logits[:T].double() - x.double() @ w.double().t()).abs() <= bound).all()) and bool((logits[T] == 7.0).all())


@pytest.mark.parametrize("T,H,N", [(1, 8, 65), (127, 72, 100), (129, 64, 128), (257, 128, 129), (256, 1624, 256), (640, 200, 160), (300, 7168, 80),
                                   (33000, 136, 256), (700, 264, 132), (1000, 520, 250), (700, 192, 96)])
@pytest.mark.parametrize("base", [False, True])
def test_gate_of_many_experts(cuda, T, H, N, base):
    """Projection and both gradients of more than 64 experts: edges of the blocks of 128 and 256 tokens, one to three steps
    of 64 columns and a partial last one, slices of unequal length, experts that do not fill their tiles; with `base` the
    sum has a second rounding."""
    from optimus import _native as n
    L, P = n.lib(), n.ptr
    x, w = _gate_inputs(T, H, N, seed=T + H + N)
    g = torch.Generator().manual_seed(N)
    dl = torch.randn(T, N, generator=g)
    x, w, dl = x.to(cuda), w.to(cuda), dl.to(cuda)
    logits, dx = torch.full((T, N), 7.0, device=cuda), torch.full((T + 1, H), 7.0, dtype=torch.bfloat16, device=cuda)
    size = L.om_router_gate_logits_split_workspace_bytes(T, H, N)
    ws = torch.empty(size, dtype=torch.uint8, device=cuda)
    n.check(L.om_router_gate_logits_split(P(x), P(w), T, H, N, P(logits), P(ws), size, n.stream()), "logits")
    n.check(L.om_router_gate_dgrad(P(dl), P(w), P(x) if base else None, P(dx), T, H, N, n.stream()), "dgrad")
    # a rounding of 2^-24 of the sum so far for every 16 columns and every slice
    bound = (H / 16 + 33) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t()) + 1e-30
    assert bool(((logits.double() - x.double() @ w.double().t()).abs() <= bound).all())
    d16 = dl.to(torch.bfloat16).double()
    exact = d16 @ w.double()
    total = exact + x.double() if base else exact
    bound = 2e-6 * (d16.abs() @ w.double().abs()) + exact.abs() * 2.0 ** -8 + (total.abs() * 2.0 ** -8 if base else 0) + 1e-30
    assert bool(((dx[:T].double() - total).abs() <= bound).all())
    assert bool((dx[T] == 7.0).all())
    if base:
        return
    dw = torch.full((N + 1, H), 7.0, device=cuda)
    size = L.om_router_gate_wgrad_workspace_bytes(T, H, N)
    ws = torch.empty(size, dtype=torch.uint8, device=cuda)
    n.check(L.om_router_gate_wgrad(P(x), P(dl), T, H, N, P(dw), 0, P(ws), size, n.stream()), "wgrad")
    bound = (T / 16 + 300) * 2.0 ** -24 * (d16.abs().t() @ x.double().abs()) + 1e-30
    assert bool(((dw[:N].double() - d16.t() @ x.double()).abs() <= bound).all())
    assert bool((dw[N] == 7.0).all())


@pytest.mark.parametrize("T,H,N,K,renorm,ldt,wdt", [
    (1, 8, 1, 1, False, torch.float32, torch.bfloat16), (127, 136, 8, 2, True, torch.float32, torch.bfloat16),
    (2048, 256, 8, 2, True, torch.float32, torch.bfloat16), (512, 2048, 64, 8, False, torch.float32, torch.bfloat16),
    (129, 264, 12, 12, True, torch.float32, torch.float32), (65, 1000, 33, 9, False, torch.float32, torch.bfloat16),
    (300, 512, 64, 20, True, torch.bfloat16, torch.bfloat16), (9000, 2048, 64, 8, False, torch.float32, torch.bfloat16), (3001, 1000, 13, 3, False, torch.bfloat16, torch.float32)])
@pytest.mark.parametrize("extra", [False, True])
def test_softmax_router_backward_in_one_call(cuda, T, H, N, K, renorm, ldt, wdt, extra):
    """The bits of the separate calls, whether the token ranges are added in the launch or behind it; a workspace of any content."""
    from optimus import _native as n
    lib = n.lib()
    g = torch.Generator().manual_seed(T + H + N)
    x, w = _gate_inputs(T, H, N, seed=T)
    logits = (x.float() @ w.float().t()).to(ldt)
    experts = torch.topk(torch.softmax(logits.float(), 1), K, dim=1).indices
    d = lambda t: None if t is None else t.to(cuda).contiguous()
    xg, wg, lg, eg, dg = map(d, (x, w, logits, experts, torch.randn(T, K, generator=g).to(wdt)))
    more = d((torch.randn(T, N, generator=g) * 0.1).to(ldt)) if extra else None
    base = d(torch.randn(T, H, generator=g).to(torch.bfloat16)) if extra else None
    st = n.stream()
    dl = torch.empty_like(lg)
    n.check(lib.om_route_softmax_topk_bwd(n.ptr(lg), n.dtype_code(lg), n.ptr(eg), n.ptr(dg), n.dtype_code(dg), T, N, K, int(renorm), n.ptr(dl), st), "softmax")
    dl = (dl if more is None else dl + more).float()
    for dw_dtype in (torch.bfloat16, torch.float32):
        want_dx, want_dw, dx, dw = torch.empty_like(xg), torch.empty_like(wg, dtype=dw_dtype), torch.empty_like(xg), torch.empty_like(wg, dtype=dw_dtype)
        ws = torch.empty(max(lib.om_router_gate_wgrad_workspace_bytes(T, H, N), 16), dtype=torch.uint8, device=cuda)
        n.check(lib.om_router_gate_dgrad(n.ptr(dl), n.ptr(wg), n.ptr(base), n.ptr(want_dx), T, H, N, st), "dgrad")
        n.check(lib.om_router_gate_wgrad(n.ptr(xg), n.ptr(dl), T, H, N, n.ptr(want_dw), n.dtype_code(want_dw), n.ptr(ws), ws.numel(), st), "wgrad")
        ws = torch.full((lib.om_router_softmax_bwd_workspace_bytes(T, H, N),), 255, dtype=torch.uint8, device=cuda)
        for _ in range(2):
            n.check(lib.om_router_softmax_bwd(n.ptr(xg), n.ptr(wg), n.ptr(lg), n.dtype_code(lg), n.ptr(eg), n.ptr(dg), n.dtype_code(dg), n.ptr(more),
                                              n.ptr(base), n.ptr(dx), n.ptr(dw), n.dtype_code(dw), T, H, N, K, int(renorm), n.ptr(ws), ws.numel(), st),
                    "om_router_softmax_bwd")
        assert torch.equal(dx, want_dx) and torch.equal(dw, want_dw)


def test_softmax_router_backward_keeps_what_is_not_finite(cuda):
    """A token whose logits hold NaN or +inf has NaN gradients, as in the separate kernels, and the others are untouched."""
    from optimus.models.common.moe import GateSoftmaxTopkFunction
    T, H, N, K = 130, 512, 64, 4
    x, w = _gate_inputs(T, H, N, seed=8)
    x[3, 5] = float("nan")
    x[77, 1] = float("inf")
    xg, wg = x.to(cuda).requires_grad_(True), w.to(cuda).requires_grad_(True)
    weights, _, _, _ = GateSoftmaxTopkFunction.apply(xg, wg, K, False, torch.float32)
    weights.sum().backward()
    bad = torch.isnan(xg.grad).all(1).cpu()
    assert bad[3] and bad[77] and int(torch.isnan(xg.grad).any(1).sum()) == 2 and torch.isnan(wg.grad).any()


@pytest.mark.parametrize("T,H,N,K", [(1, 8, 1, 1), (15, 64, 64, 16), (17, 72, 33, 8), (16, 256, 32, 16), (2049, 256, 8, 2), (4113, 256, 64, 8),
                                     (33, 264, 31, 5), (300, 1000, 12, 3), (4097, 1000, 61, 16), (2000, 1096, 59, 4), (64, 2040, 32, 8), (5000, 5000, 13, 6)])
@pytest.mark.parametrize("bf16_logits", [False, True])
def test_small_gate_router_in_one_launch(cuda, T, H, N, K, bf16_logits):
    """Bit for bit the split projection and the routing of its logits: partial groups of tokens and experts, slices and pieces that end early."""
    from optimus import _native as n
    lib, st = n.lib(), n.stream()
    x, w = (t.to(cuda) for t in _gate_inputs(T, H, N, seed=T + H))
    ldt = torch.bfloat16 if bf16_logits else torch.float32
    ref = torch.empty(T, N, device=cuda)
    ws = torch.empty(max(lib.om_router_gate_logits_split_workspace_bytes(T, H, N), 16), dtype=torch.uint8, device=cuda)
    n.check(lib.om_router_gate_logits_split(n.ptr(x), n.ptr(w), T, H, N, n.ptr(ref), n.ptr(ws), ws.numel(), st), "logits")
    ref = ref.to(ldt)
    for renorm in (0, 1):
        want_w, want_e = torch.empty(T, K, dtype=torch.bfloat16, device=cuda), torch.empty(T, K, dtype=torch.int64, device=cuda)
        n.check(lib.om_route_softmax_topk(n.ptr(ref), n.dtype_code(ref), T, N, K, renorm, n.ptr(want_w), n.dtype_code(want_w), n.ptr(want_e), st), "route")
        logits, got_w, got_e = torch.empty_like(ref), torch.empty_like(want_w), torch.empty_like(want_e)
        ws = torch.empty(max(lib.om_router_gate_route_workspace_bytes(T, H, N), 16), dtype=torch.uint8, device=cuda)
        n.check(lib.om_router_gate_split_softmax_topk(n.ptr(x), n.ptr(w), T, H, N, K, renorm, n.ptr(logits), n.dtype_code(logits), n.ptr(got_w),
                                                      n.dtype_code(got_w), n.ptr(got_e), n.ptr(ws), ws.numel(), st), "one launch")
        assert torch.equal(logits, ref) and torch.equal(got_e, want_e) and torch.equal(got_w, want_w)


@pytest.mark.parametrize("T,H,N,n_group,topk_group,K", [(1, 7168, 256, 8, 4, 8), (64, 7168, 256, 8, 4, 8), (1025, 512, 256, 1, 1, 12), (300, 264, 16, 4, 2, 2),
                                                        (77, 512, 64, 8, 3, 6), (500, 72, 24, 3, 1, 8), (40, 512, 96, 8, 3, 5), (2000, 1000, 128, 32, 9, 16)])
@pytest.mark.parametrize("bias_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("ties", [False, True])
def test_group_router_behind_the_split_projection(cuda, T, H, N, n_group, topk_group, K, bias_dtype, ties):
    """Bit for bit the router on the logits that it writes, also where experts and groups tie."""
    from optimus import _native as n
    lib, st = n.lib(), n.stream()
    x, w = _gate_inputs(T, H, N, seed=T + N)
    bias = torch.randn(N, generator=torch.Generator().manual_seed(2)).mul(0.1).to(bias_dtype)
    if ties:
        w, bias = w[: max(N // n_group // 2, 1)].repeat(2 * n_group, 1)[:N], torch.zeros(N, dtype=bias_dtype)
    xg, wg, bg = x.to(cuda), w.to(cuda).contiguous(), bias.to(cuda)
    logits = torch.empty(T, N, device=cuda)
    got_e, got_w = torch.empty(T, K, dtype=torch.int64, device=cuda), torch.empty(T, K, device=cuda)
    ws = torch.empty(max(lib.om_router_gate_route_workspace_bytes(T, H, N), 16), dtype=torch.uint8, device=cuda)
    for renorm in (0, 1):
        n.check(lib.om_router_gate_split_sigmoid_group_topk_bias(n.ptr(xg), n.ptr(wg), n.ptr(bg), n.dtype_code(bg), T, H, N, n_group, topk_group, K,
                                                                 renorm, 2.5, n.ptr(logits), n.ptr(got_e), n.ptr(got_w), n.ptr(ws), ws.numel(), st), "fused")
        bf, want_e, want_w = bg.float(), torch.empty_like(got_e), torch.empty_like(got_w)
        n.check(lib.om_route_sigmoid_group_topk(n.ptr(logits), n.ptr(bf), T, N, n_group, topk_group, K, renorm, 2.5, n.ptr(want_e), n.ptr(want_w), st), "router")
        assert torch.equal(got_e, want_e) and torch.equal(got_w, want_w)
    ref = x.double() @ w.double().t()
    assert bool(((logits.cpu().double() - ref).abs() <= 8 * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t()) + 1e-30).all())


@pytest.mark.parametrize("T,H,N,K", [(1, 7, 1, 1), (5, 64, 8, 2), (2048, 256, 8, 2), (777, 100, 13, 13), (513, 520, 64, 9), (3, 1000, 33, 4)])
def test_float32_router_launches_equal_their_steps(cuda, T, H, N, K):
    """Projection with routing, and both gradients of the gate, in one launch: the bits of the separate calls."""
    from optimus import _native as n
    lib, st = n.lib(), n.stream()
    g = torch.Generator().manual_seed(T + H + N)
    x, w, dl, base = (torch.randn(*s, generator=g).to(cuda) for s in ((T, H), (N, H), (T, N), (T, H)))
    new = lambda *s: torch.empty(*s, device=cuda)
    logits, got_logits = new(T, N), new(T, N)
    n.check(lib.om_router_gate_logits_f32(n.ptr(x), n.ptr(w), T, H, N, n.ptr(logits), st), "logits")
    for wdt in (torch.float32, torch.bfloat16):
        want_w, got_w = new(T, K).to(wdt), new(T, K).to(wdt)
        want_e, got_e = (torch.empty(T, K, dtype=torch.int64, device=cuda) for _ in range(2))
        for renorm in (0, 1):
            n.check(lib.om_route_softmax_topk(n.ptr(logits), n.OM_F32, T, N, K, renorm, n.ptr(want_w), n.dtype_code(want_w), n.ptr(want_e), st), "route")
            n.check(lib.om_router_gate_softmax_topk_f32(n.ptr(x), n.ptr(w), T, H, N, K, renorm, n.ptr(got_logits), n.ptr(got_w),
                                                        n.dtype_code(got_w), n.ptr(got_e), st), "one launch")
            assert torch.equal(got_logits, logits) and torch.equal(got_e, want_e) and torch.equal(got_w, want_w)
    for b in (None, base):
        want_dx, want_dw, dx, dw = new(T, H), new(N, H), new(T, H), new(N, H)
        n.check(lib.om_router_gate_dgrad_f32_add(n.ptr(dl), n.ptr(w), n.ptr(b), T, H, N, n.ptr(want_dx), st), "dx")
        n.check(lib.om_router_gate_wgrad_f32(n.ptr(x), n.ptr(dl), T, H, N, n.ptr(want_dw), st), "dw")
        n.check(lib.om_router_gate_bwd_f32(n.ptr(x), n.ptr(dl), n.ptr(w), n.ptr(b), T, H, N, n.ptr(dx), n.ptr(dw), st), "both")
        assert torch.equal(dx, want_dx) and torch.equal(dw, want_dw)


@pytest.mark.parametrize("T,H,N,K,start,end", [(1, 2048, 64, 8, 0, 64), (3, 1024, 33, 16, 0, 33), (4, 4096, 17, 1, 5, 9), (5, 7168, 8, 8, 0, 1), (37, 2048, 64, 8, 0, 64),
                                               (64, 1536, 32, 16, 8, 24), (63, 3000, 64, 3, 60, 64)])
@pytest.mark.parametrize("bf16_logits", [False, True])
def test_router_that_sorts_its_selections(cuda, T, H, N, K, start, end, bf16_logits):
    """Bit for bit the router and the sort of what it selects."""
    from optimus import _native as n
    lib, st = n.lib(), n.stream()
    assert lib.om_router_gate_softmax_topk_sort_fits(T, H, N, K) == 1
    x, w = (t.to(cuda) for t in _gate_inputs(T, H, N, seed=T + H))
    ldt = torch.bfloat16 if bf16_logits else torch.float32
    ws = torch.empty(max(lib.om_router_gate_route_workspace_bytes(T, H, N), 16), dtype=torch.uint8, device=cuda)
    i32 = lambda k: torch.full((k,), -7, dtype=torch.int32, device=cuda)
    NR = end - start
    for renorm, wdt in ((0, torch.bfloat16), (1, torch.float32)):
        def buffers():
            return ([torch.empty(T, N, dtype=ldt, device=cuda), torch.empty(T, K, dtype=wdt, device=cuda), torch.empty(T, K, dtype=torch.int64, device=cuda)],
                    [i32(NR + 1), i32(T + 1), i32(T * K), i32(T * K), i32(T * K), torch.full((T * K,), -7.0, device=cuda)])
        (logits, weights, experts), index = buffers()
        n.check(lib.om_router_gate_split_softmax_topk(n.ptr(x), n.ptr(w), T, H, N, K, renorm, n.ptr(logits), n.dtype_code(logits), n.ptr(weights),
                                                      n.dtype_code(weights), n.ptr(experts), n.ptr(ws), ws.numel(), st), "router")
        sort_ws = i32(max(lib.om_moe_sort_workspace_bytes(T, K, NR) // 4, 1))
        n.check(lib.om_moe_sort_weighted(n.ptr(experts), n.OM_I64, T, K, start, end, *(n.ptr(t) for t in index[:5]), n.ptr(weights), n.dtype_code(weights),
                                         n.ptr(index[5]), n.ptr(sort_ws), sort_ws.numel() * 4, st), "sort")
        (g_logits, g_weights, g_experts), g_index = buffers()
        n.check(lib.om_router_gate_softmax_topk_sort(n.ptr(x), n.ptr(w), T, H, N, K, renorm, n.ptr(g_logits), n.dtype_code(g_logits), n.ptr(g_weights),
                                                     n.dtype_code(g_weights), n.ptr(g_experts), start, end, *(n.ptr(t) for t in g_index), n.ptr(ws),
                                                     ws.numel(), st), "router and sort")
        for got, want in zip([g_logits, g_weights, g_experts] + g_index, [logits, weights, experts] + index):
            assert torch.equal(got, want)


@pytest.mark.parametrize("H,N", [(1024, 64), (2048, 61), (4608, 50), (7168, 17), (1536, 1)])
def test_few_tokens_have_the_logits_of_many(cuda, H, N):
    """Up to 512 tokens a wavefront takes 16 tokens and experts of a slice, above them a block goes through it: the same eight sums in order."""
    from optimus import _native as n
    x, w = (t.to(cuda) for t in _gate_inputs(513, H, N, seed=H + N))
    _, _, many, _ = n.host().route_softmax(x, w, 1, False, torch.bfloat16, False, False)
    for T in (1, 16, 17, 512):
        _, _, few, _ = n.host().route_softmax(x[:T], w, 1, False, torch.bfloat16, False, False)
        assert torch.equal(few, many[:T])


# one token, a partial block of 64, more partial rows than a round of loads a wavefront, several groups of 64 experts
@pytest.mark.parametrize("T,N,K", [(1, 8, 2), (63, 64, 8), (1025, 100, 5), (4097, 512, 8), (16384 + 64 * 17, 64, 8), (300, 2, 1)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_balance_loss_in_one_function_is_the_composed_one(cuda, T, N, K, dtype):
    """single_input_load_balancing_loss_func against the same expression of RouterBalanceStatsFunction's sums, loss and gradient."""
    from optimus.models.common.ral_functions import RouterBalanceStatsFunction, single_input_load_balancing_loss_func
    base = _valid_logits(T, N, K, seed=T + N).to(dtype).to(cuda)
    a, b = base.clone().requires_grad_(True), base.clone().requires_grad_(True)
    loss = single_input_load_balancing_loss_func(a, N, K)
    prob_sum, count = RouterBalanceStatsFunction.apply(b, K, None)
    want = torch.sum((count / T) * (prob_sum / T)) * N
    # N products' sum in another order, and one rounding of each of them
    assert loss.shape == () and loss.dtype == torch.float32
    assert abs(float(loss.detach().double() - want.detach().double())) <= (N + 4) * 2.0 ** -24 * float(want.detach())
    (want * 0.01).backward()
    loss *= 0.01                                   # in place, as a caller may
    loss.backward()
    # dlogits = p (g - sum p g), where g = 0.01 N (count / T) / T: the tensor expression multiplies by 1 / T, so each of g and the sum is
    # off by at most 2 + 2 roundings of g's size, which the difference may cancel down to; in bf16 one rounding of the result
    p = torch.softmax(base.float(), 1).max()
    g = 0.01 * N * float(count.max()) / T / T
    bound = float(p) * g * 2 * 4 * 2.0 ** -24 + (2.0 ** -8 * float(b.grad.abs().max()) if dtype == torch.bfloat16 else 0.0)
    assert float((a.grad.float() - b.grad.float()).abs().max()) <= bound


@pytest.mark.parametrize("H,N", [(7168, 256), (2048, 256), (1624, 160), (1000, 65), (264, 200), (8, 100)])
def test_few_tokens_of_many_experts_have_the_logits_of_many(cuda, H, N):
    """Up to 64 tokens of more than 64 experts, around the tiles of 16, slices of one to several chunks: the bits that the same tokens
    have among 128 (as many slices)."""
    from optimus import _native as n
    L = n.lib()
    x = torch.randn(128, H, device=cuda).bfloat16()
    w = (torch.randn(N, H, device=cuda) * 0.1).bfloat16()

    def logits(T):
        out = torch.full((T, N), 7.0, device=cuda)
        ws = torch.empty(L.om_router_gate_logits_split_workspace_bytes(T, H, N), dtype=torch.uint8, device=cuda)
        n.check(L.om_router_gate_logits_split(n.ptr(x), n.ptr(w), T, H, N, n.ptr(out), n.ptr(ws), ws.numel(), n.stream()), "logits")
        return out

    many = logits(128)
    exact = x.double() @ w.double().T
    # float32 sums of H exact products: at most H roundings of the largest partial sum
    assert bool(((many.double() - exact).abs() <= H * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)).all())
    for T in (1, 15, 16, 17, 63, 64, 65):
        assert torch.equal(logits(T), many[:T]), T


@pytest.mark.parametrize("renorm", [0, 1])
def test_sigmoid_router_backward_of_numbers_that_are_no_experts(cuda, renorm):
    """A selection outside the experts has no weight and no gradient: the others' gradients are those of the token without it."""
    from optimus import _native as n
    lib, st, T, N, K = n.lib(), n.stream(), 5, 72, 3
    g = torch.Generator().manual_seed(3)
    logits, dw = torch.randn(T, N, generator=g), torch.randn(T, K, generator=g)
    experts = torch.tensor([[1, 70, 9], [0x7fffffff, 71, 0], [5, -1, N], [0x7fffffff] * 3, [2 ** 32 + 1, 2, 71]])
    lg, eg, dg = logits.to(cuda), experts.to(cuda), dw.to(cuda)
    got = torch.full((T, N), 7.0, device=cuda)
    n.check(lib.om_route_sigmoid_topk_bwd(n.ptr(lg), n.ptr(eg), n.ptr(dg), T, N, K, renorm, 2.5, n.ptr(got), st), "backward")
    x = logits.double().requires_grad_(True)
    loss = 0.0
    for t in range(T):
        kept = [k for k in range(K) if 0 <= experts[t, k] < N]
        s = torch.sigmoid(x[t, experts[t, kept]])
        loss = loss + (dw[t, kept].double() * 2.5 * (s / (s.sum() + 1e-20) if renorm else s)).sum()
    loss.backward()
    # a dozen float32 operations of terms no larger than 2.5 |dw| each
    assert float((got.cpu().double() - x.grad).abs().max()) <= 16 * 2.0 ** -24 * 2.5 * float(dw.abs().max()) * K


# (groups of one lane, of several, all kept, a single group, more selections than the groups that are left have experts)
@pytest.mark.parametrize("T,H,N,n_group,topk_group,K", [(9, 512, 256, 8, 4, 8), (1030, 264, 64, 8, 3, 6), (40, 512, 96, 3, 3, 5), (33, 72, 24, 1, 1, 8),
                                                        (12, 512, 16, 4, 2, 16), (10, 512, 12, 4, 2, 5)])
@pytest.mark.parametrize("bad", ["token", "expert", "group", "expert bias", "-inf biases", "-inf bias of all", "+inf alone"])
def test_group_router_of_what_is_not_finite(cuda, T, H, N, n_group, topk_group, K, bad):
    """Scores that do not compare: K different experts of the model for every token, those that om_route_sigmoid_group_topk selects; tokens
    with finite scores as without the others; and NaN gradients where the weights are NaN."""
    from optimus import _native as n
    lib, st, gs, nan = n.lib(), n.stream(), N // n_group, float("nan")
    x, w = _gate_inputs(T, H, N, seed=T + N)
    bias = torch.randn(N, generator=torch.Generator().manual_seed(2)).mul(0.1)

    def route(x, w, bias):
        xg, wg, bg = x.to(cuda), w.to(cuda).contiguous(), bias.to(cuda)
        logits, e, wt = torch.empty(T, N, device=cuda), torch.empty(T, K, dtype=torch.int64, device=cuda), torch.empty(T, K, device=cuda)
        ws = torch.empty(max(lib.om_router_gate_route_workspace_bytes(T, H, N), 16), dtype=torch.uint8, device=cuda)
        n.check(lib.om_router_gate_split_sigmoid_group_topk(n.ptr(xg), n.ptr(wg), n.ptr(bg), T, H, N, n_group, topk_group, K, 1, 2.5, n.ptr(logits),
                                                            n.ptr(e), n.ptr(wt), n.ptr(ws), ws.numel(), st), "fused")
        want_e, want_w = torch.empty_like(e), torch.empty_like(wt)
        n.check(lib.om_route_sigmoid_group_topk(n.ptr(logits), n.ptr(bg), T, N, n_group, topk_group, K, 1, 2.5, n.ptr(want_e), n.ptr(want_w), st), "router")
        assert torch.equal(e, want_e) and torch.equal(torch.isnan(wt), torch.isnan(want_w)) and torch.equal(wt.nan_to_num(7.0), want_w.nan_to_num(7.0))
        assert bool(((e >= 0) & (e < N)).all()) and bool((e.sort(1).values.diff(dim=1) > 0).all())
        return logits, e, wt
    good_logits, good_e, good_w = route(x, w, bias)
    if bad == "token":
        x[T // 2, 3] = nan
    elif bad == "expert":
        w[N // 2] = nan
    elif bad == "group":
        w[N - gs:] = nan
    elif bad == "expert bias":
        bias[1] = nan
    elif bad == "-inf biases":
        bias[torch.randperm(N, generator=torch.Generator().manual_seed(4))[:N - 3]] = float("-inf")
    elif bad == "-inf bias of all":
        bias[:] = float("-inf")
    else:
        bias[:gs] = float("-inf")
        bias[0] = float("inf")
    logits, e, wt = route(x, w, bias)
    if bad != "token":
        return
    # the NaN token: no group compares, so the first is kept, and the zeros of the others come first
    order = list(range(gs, N)) + list(range(gs))
    if n_group == 1:
        order = list(range(N))
    assert e[T // 2].tolist() == order[:K] and bool(torch.isnan(wt[T // 2]).all())
    others = torch.arange(T, device=cuda) != T // 2
    assert torch.equal(logits[others], good_logits[others]) and torch.equal(e[others], good_e[others]) and torch.equal(wt[others], good_w[others])
    dw, dl = torch.ones(T, K, device=cuda), torch.full((T, N), 7.0, device=cuda)
    n.check(lib.om_route_sigmoid_topk_bwd(n.ptr(logits), n.ptr(e), n.ptr(dw), T, N, K, 1, 2.5, n.ptr(dl), st), "backward")
    assert bool(torch.isnan(dl[T // 2][e[T // 2]]).all()) and bool(torch.isfinite(dl[others]).all())


def test_float32_gate_gradients_of_more_tokens_than_one_grid_holds(cuda):
    """A launch holds less than 2^32 threads: from there on the two gradients are launches of their own, with the same results."""
    from optimus import _native as n
    lib, st, T, H, N = n.lib(), n.stream(), (1 << 24) + 3, 8, 2
    g = torch.Generator(device=cuda).manual_seed(1)
    x, dl = (torch.randn(T, k, generator=g, device=cuda) for k in (H, N))
    w = torch.randn(N, H, generator=g, device=cuda)
    dx, dw = torch.full((T, H), 7.0, device=cuda), torch.full((N, H), 7.0, device=cuda)
    n.check(lib.om_router_gate_bwd_f32(n.ptr(x), n.ptr(dl), n.ptr(w), None, T, H, N, n.ptr(dx), n.ptr(dw), st), "both")
    want_dx, want_dw = torch.empty_like(dx), torch.empty_like(dw)
    n.check(lib.om_router_gate_dgrad_f32(n.ptr(dl), n.ptr(w), T, H, N, n.ptr(want_dx), st), "dx")
    n.check(lib.om_router_gate_wgrad_f32(n.ptr(x), n.ptr(dl), T, H, N, n.ptr(want_dw), st), "dw")
    assert torch.equal(dx, want_dx) and torch.equal(dw, want_dw)
    # two products and their sum, a rounding each
    ref = dl[-5:].double() @ w.double()
    assert bool(((dx[-5:].double() - ref).abs() <= 3 * 2.0 ** -24 * (dl[-5:].double().abs() @ w.double().abs())).all())


# slices of 64, 128, 192 and 256 columns, whole ones and shorter last ones, taken in pieces of 64, 128 and 256 columns; both kinds of kernel
@pytest.mark.parametrize("T,H,N,K", [(1, 1536, 64, 8), (37, 1536, 17, 3), (64, 2880, 128, 4), (5, 1088, 96, 2), (3, 2048, 64, 8), (33, 1096, 65, 2),
                                     (40, 776, 40, 8), (300, 1000, 12, 3), (2049, 1088, 20, 4), (50, 256, 8, 2)])
def test_infinite_gate_weights_meet_their_own_tokens_only(cuda, T, H, N, K):
    """An expert whose weights are all infinite, behind positive tokens: its logits are infinite (not NaN, as by a column past a slice's end, whose
    token counts as zero), the others' are those of any weight there."""
    from optimus import _native as n
    lib, st = n.lib(), n.stream()
    x, w = (t.to(cuda) for t in _gate_inputs(T, H, N, seed=T + H))
    x = x.abs() + 0.125
    bad = w.clone()
    bad[N // 2] = float("inf")
    others = [i for i in range(N) if i != N // 2]
    got = []
    for weight in (w, bad):
        logits, ws = torch.empty(T, N, device=cuda), torch.empty(lib.om_router_gate_logits_split_workspace_bytes(T, H, N), dtype=torch.uint8, device=cuda)
        if N > 64 or T <= 512:
            n.check(lib.om_router_gate_logits_split(n.ptr(x), n.ptr(weight), T, H, N, n.ptr(logits), n.ptr(ws), ws.numel(), st), "logits")
            got.append(logits)
        if N <= 64:
            logits, experts = torch.empty(T, N, device=cuda), torch.empty(T, K, dtype=torch.int64, device=cuda)
            weights = torch.empty(T, K, device=cuda)
            ws = torch.empty(max(lib.om_router_gate_route_workspace_bytes(T, H, N), 16), dtype=torch.uint8, device=cuda)
            n.check(lib.om_router_gate_split_softmax_topk(n.ptr(x), n.ptr(weight), T, H, N, K, 0, n.ptr(logits), n.OM_F32, n.ptr(weights), n.OM_F32,
                                                          n.ptr(experts), n.ptr(ws), ws.numel(), st), "router")
            got.append(logits)
    half = len(got) // 2
    for fine, infinite in zip(got[:half], got[half:]):
        assert bool(torch.isposinf(infinite[:, N // 2]).all()) and torch.equal(infinite[:, others], fine[:, others])
