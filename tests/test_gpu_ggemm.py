"""Grouped expert GEMMs through optimus.models.common.moe (-> C-ABI om_grouped_gemm_*,
om_merged_mlp_*) against per-expert torch.matmul in fp32 on the same bf16 inputs — the special
case the reference itself uses as its check (optimus/kernels/grouped_linear_forward.py:104-112,
moe.py:174-178).  Bar: a product's output is ONE bf16 rounding of an fp32-accumulated sum, so its
distance from the fp32 reference must be that of the ideally rounded reference (mean_rel 1.41e-3
for Gaussian results) plus fp32 summation-order noise: util.assert_bf16_parity with an excess
factor just above 1 (ONE_ROUNDING), and max-abs <= 2e-2 of the largest magnitude.  The merged MLP
rounds g, u, h (and y) on the way like the reference, hence the wider MLP_BARS."""
import numpy as np
import pytest
import torch

from util import assert_bf16_parity, max_abs, mean_rel

# (excess over the bf16 floor, absolute cap on mean_rel); measured: single products 1.00 x the floor,
# the merged MLP 1.6 x (y) and 1.5-2.5 x (gradients)
ONE_ROUNDING = (1.03, 1.8e-3)
MLP_BARS = {"out": (1.9, 2.7e-3), "grad": (2.9, 4.1e-3)}

pytestmark = pytest.mark.gpu


def _counts(kind, G, rows, seed=0):
    g = torch.Generator().manual_seed(seed)
    if kind == "uniform":
        c = torch.full((G,), rows // G)
        c[: rows - int(c.sum())] += 1
    elif kind == "ragged":
        p = torch.rand(G, generator=g) ** 3
        c = torch.floor(p / p.sum() * rows).long()
        c[0] += rows - int(c.sum())
    elif kind == "empties":
        c = torch.zeros(G, dtype=torch.long)
        hot = torch.randperm(G, generator=g)[: max(1, G // 4)]
        c[hot] = rows // len(hot)
        c[hot[0]] += rows - int(c.sum())
    elif kind == "onehot":   # every row belongs to one expert in the middle
        c = torch.zeros(G, dtype=torch.long)
        c[G // 2] = rows
    cum = torch.zeros(G + 1, dtype=torch.int32)
    cum[1:] = torch.cumsum(c, 0)
    return cum


def _ref_fwd(x, w, cum):
    out = torch.zeros(x.shape[0], w.shape[1])
    for g in range(w.shape[0]):
        s, e = int(cum[g]), int(cum[g + 1])
        out[s:e] = x[s:e].float() @ w[g].float().t()
    return out


CASES = [# few rows per expert with extents that are multiples of 256 (skewed small batches): most tiles hold
         # a handful of valid rows; one expert with many row tiles among empty ones
         ("ragged", 64, 4096, 1024, 2048), ("empties", 64, 3000, 256, 512), ("onehot", 16, 1000, 256, 256),
         ("uniform", 20, 640, 512, 256), ("ragged", 300, 9000, 256, 256), ("ragged", 512, 4097, 256, 512),
         ("uniform", 4, 512, 256, 128), ("ragged", 8, 1000, 256, 512), ("empties", 16, 777, 128, 256),
         ("ragged", 64, 4096, 1024, 2048), ("uniform", 1, 300, 256, 256), ("ragged", 3, 5, 128, 128),
         # several tiles per persistent block, on both tile shapes, with empty experts in between
         ("ragged", 8, 20000, 512, 768), ("ragged", 8, 20000, 384, 640), ("empties", 32, 9000, 512, 1024),
         # more experts than lanes in a wavefront: the per-block tile table is built in several
         # rounds with a carry, the last one partial
         ("ragged", 150, 6000, 128, 128), ("empties", 200, 70000, 256, 256),
         # all the work in one expert: the weight gradient's work-balanced split of the tiles over the
         # XCDs then cuts that expert's tiles eight ways and the zero tiles of the others ride along
         ("onehot", 70, 5000, 256, 512), ("onehot", 9, 3000, 512, 256), ("onehot", 2, 130, 128, 128),
         # extents that are multiples of 64 but not of 128: partial last tiles along the output columns
         # (and, for the weight gradient, along both extents of dW), odd numbers of contraction steps
         ("ragged", 8, 1000, 320, 192), ("uniform", 4, 512, 64, 64), ("empties", 16, 777, 192, 448),
         ("ragged", 64, 20000, 320, 2048), ("onehot", 5, 700, 2048, 320),
         # extents that are multiples of 8 only: partial 16-byte-chunk column masks in the last tile, a
         # last contraction step with fewer than 64 indices (zero-filled in LDS), tiny extents
         ("ragged", 8, 1000, 200, 136), ("uniform", 4, 512, 72, 40), ("empties", 16, 777, 8, 8),
         ("ragged", 6, 900, 328, 1000), ("onehot", 5, 700, 1000, 328), ("ragged", 3, 50, 24, 264)]


@pytest.mark.parametrize("kind,G,rows,N,K", CASES)
def test_grouped_gemm_fwd_dgrad_wgrad(cuda, kind, G, rows, N, K):
    from optimus.models.common.moe import GroupedGemmFunction
    g = torch.Generator().manual_seed(rows)
    x = torch.randn(rows, K, generator=g).to(torch.bfloat16)
    w = (torch.randn(G, N, K, generator=g) * 0.05).to(torch.bfloat16)
    dout = torch.randn(rows, N, generator=g).to(torch.bfloat16)
    cum = _counts(kind, G, rows)
    xd = x.to(cuda).requires_grad_(True)
    wd = w.to(cuda).requires_grad_(True)
    # the reference passes a CPU int32 tensor of offsets and max_tokens_per_expert (moe.py:397-398)
    out = GroupedGemmFunction.apply(xd, wd, cum, int((cum[1:] - cum[:-1]).max()), False)
    out.backward(dout.to(cuda))
    ref = _ref_fwd(x, w, cum)
    assert max_abs(out.float().cpu(), ref) <= 2e-2 * max(1.0, float(ref.abs().max()))
    tag = f"ggemm[{kind},{G},{rows},{N},{K}]"
    assert_bf16_parity(out, ref, *ONE_ROUNDING, tag=tag + " fwd")
    dx_ref = torch.zeros(rows, K); dw_ref = torch.zeros(G, N, K)
    for e in range(G):
        s, t = int(cum[e]), int(cum[e + 1])
        dx_ref[s:t] = dout[s:t].float() @ w[e].float()
        dw_ref[e] = dout[s:t].float().t() @ x[s:t].float()
    assert_bf16_parity(xd.grad, dx_ref, *ONE_ROUNDING, tag=tag + " dgrad")
    assert_bf16_parity(wd.grad, dw_ref, *ONE_ROUNDING, tag=tag + " wgrad")
    assert max_abs(wd.grad.float().cpu(), dw_ref) <= 1e-2 * max(1.0, float(dw_ref.abs().max()))
    # experts without rows get exactly zero weight gradient
    empty = (cum[1:] == cum[:-1])
    if empty.any():
        assert float(wd.grad[empty.to(cuda)].abs().max()) == 0.0


@pytest.mark.parametrize("kind,G,rows,I,H", [("uniform", 4, 512, 128, 256), ("ragged", 8, 1500, 512, 256),
                                            # skewed small batches: a few rows per expert
                                            ("ragged", 64, 4096, 1024, 2048), ("empties", 32, 700, 256, 512),
                                            ("onehot", 8, 500, 128, 256), ("ragged", 40, 1000, 384, 256),
                                            ("empties", 64, 4096, 1024, 2048), ("ragged", 2, 7, 128, 128),
                                            # hidden / ffn sizes that are multiples of 64 only
                                            ("ragged", 8, 1500, 192, 320), ("uniform", 4, 300, 64, 64),
                                            ("empties", 16, 9000, 320, 1088),
                                            # ... and of 8 only
                                            ("ragged", 8, 1500, 200, 328), ("uniform", 4, 300, 8, 8),
                                            ("empties", 16, 2000, 72, 1000), ("ragged", 5, 600, 1000, 72)])
def test_merged_mlp_fused(cuda, kind, G, rows, I, H):
    """MergedMLP (fused gate+up+SwiGLU, fused down-dgrad+SwiGLU-backward, dual dgrad) against the
    fp32 composition silu(x Wg^T) * (x Wu^T) Wd^T under autograd."""
    from optimus.models.common.moe import MergedMLPFunction
    g = torch.Generator().manual_seed(rows + 1)
    x = torch.randn(rows, H, generator=g).to(torch.bfloat16)
    wg = (torch.randn(G, I, H, generator=g) * 0.05).to(torch.bfloat16)
    wu = (torch.randn(G, I, H, generator=g) * 0.05).to(torch.bfloat16)
    wd = (torch.randn(G, H, I, generator=g) * 0.05).to(torch.bfloat16)
    dy = torch.randn(rows, H, generator=g).to(torch.bfloat16)
    cum = _counts(kind, G, rows)
    dev = [t.to(cuda).requires_grad_(True) for t in (x, wg, wu, wd)]
    y = MergedMLPFunction.apply(*dev, cum.to(cuda))
    y.backward(dy.to(cuda))
    ref = [t.float().requires_grad_(True) for t in (x, wg, wu, wd)]
    outs = []
    for e in range(G):
        s, t = int(cum[e]), int(cum[e + 1])
        xe = ref[0][s:t]
        outs.append((torch.nn.functional.silu(xe @ ref[1][e].t()) * (xe @ ref[2][e].t())) @ ref[3][e].t())
    yr = torch.cat(outs)
    yr.backward(dy.float())
    tag = f"merged_mlp[{kind},{G},{rows},{I},{H}]"
    assert_bf16_parity(y, yr, *MLP_BARS["out"], tag=tag + " y")
    assert max_abs(y.float().cpu(), yr.detach()) <= 2e-2 * max(1.0, float(yr.detach().abs().max()))
    for name, a, b in zip(("dx", "dwg", "dwu", "dwd"), dev, ref):
        assert_bf16_parity(a.grad, b.grad, *MLP_BARS["grad"], tag=f"{tag} {name}")


@pytest.mark.parametrize("T,K,N,start,end,I,H,skew", [
    (4096, 8, 64, 0, 64, 512, 512, 0.0),      # 256x256 tiles, forward and weight gradient
    (512, 2, 8, 0, 8, 128, 384, 0.0),         # 128x128 tiles
    (3000, 4, 16, 4, 12, 256, 256, 1.5),      # expert window: only part of the pairs is routed; skew
    (70, 8, 64, 0, 64, 128, 128, 3.0),        # most experts empty, a few rows each
    (16384, 8, 64, 0, 64, 1024, 2048, 0.0),   # C3
])
def test_gathered_merged_mlp_is_bit_identical(cuda, T, K, N, start, end, I, H, skew):
    """The token gather folded into the GEMM loads (om_merged_mlp_gate_up_fwd_gathered,
    om_grouped_gemm_wgrad_gathered) against gather-then-GEMM (om_index_gather + the plain entry
    points): the same products are summed in the same order, so outputs and every gradient must be
    equal bit for bit."""
    from optimus.models.common.moe import (GatheredMergedMLPFunction, MergedMLPFunction,
                                           PrepareInputForGroupGemmFunction, build_token_permutation)
    from util import routed_experts
    G = end - start
    g = torch.Generator().manual_seed(T + I)
    se = routed_experts(T, N, K, seed=T + K, skew=skew).to(cuda)
    cum, cum_ep, ii, oi, _ = build_token_permutation(se, start, end)
    rows = int(cum[-1].item())
    ii, oi = ii[:rows], oi[:rows]
    x = torch.randn(T, H, generator=g).to(torch.bfloat16)
    ws = [(torch.randn(G, I, H, generator=g) * 0.05).to(torch.bfloat16),
          (torch.randn(G, I, H, generator=g) * 0.05).to(torch.bfloat16),
          (torch.randn(G, H, I, generator=g) * 0.05).to(torch.bfloat16)]
    dy = torch.randn(rows, H, generator=g).to(torch.bfloat16).to(cuda)
    results = []
    for gathered in (False, True):
        xd = x.to(cuda).requires_grad_(True)
        wd = [w.to(cuda).requires_grad_(True) for w in ws]
        if gathered:
            y = GatheredMergedMLPFunction.apply(xd, ii, cum_ep, oi, *wd, cum)
        else:
            y = MergedMLPFunction.apply(PrepareInputForGroupGemmFunction.apply(xd, ii, cum_ep, oi), *wd, cum)
        y.backward(dy)
        results.append([y.detach(), xd.grad] + [w.grad for w in wd])
    for name, a, b in zip(("y", "dx", "dw_gate", "dw_up", "dw_down"), *results):
        assert torch.equal(a, b), name
    assert results[0][0].shape == (rows, H) and bool(torch.isfinite(results[1][0].float()).all())


def test_gathered_merged_mlp_with_no_routed_rows(cuda):
    """An expert window that receives no token: empty output, zero weight gradients, zero input
    gradient, no launch on empty index arrays."""
    from optimus.models.common.moe import GatheredMergedMLPFunction, build_token_permutation
    T, K, H, I, G = 64, 2, 128, 128, 2
    se = torch.zeros(T, K, dtype=torch.int64, device=cuda)
    se[:, 1] = 1                                     # every token picks experts 0 and 1
    cum, cum_ep, ii, oi, _ = build_token_permutation(se, 4, 6)   # window [4, 6): nothing routed
    assert int(cum[-1].item()) == 0
    x = torch.randn(T, H, device=cuda).to(torch.bfloat16).requires_grad_(True)
    ws = [torch.randn(G, I, H, device=cuda).to(torch.bfloat16).requires_grad_(True),
          torch.randn(G, I, H, device=cuda).to(torch.bfloat16).requires_grad_(True),
          torch.randn(G, H, I, device=cuda).to(torch.bfloat16).requires_grad_(True)]
    y = GatheredMergedMLPFunction.apply(x, ii[:0], cum_ep, oi[:0], *ws, cum)
    assert y.shape == (0, H)
    y.sum().backward()
    assert float(x.grad.abs().max()) == 0.0
    for w in ws:
        assert float(w.grad.abs().max()) == 0.0


@pytest.mark.parametrize("kind,G,rows,N,K", [("uniform", 4, 512, 256, 128), ("ragged", 8, 1000, 192, 320),
                                            ("empties", 16, 777, 64, 64), ("ragged", 3, 5, 128, 64),
                                            ("uniform", 8, 4096, 512, 256),
                                            # extents that are multiples of 8 only
                                            ("ragged", 8, 1000, 200, 136), ("uniform", 4, 300, 8, 8),
                                            ("empties", 6, 500, 72, 328)])
def test_grouped_gemm_float32(cuda, kind, G, rows, N, K):
    """float32 modules (the reference's GroupedGemmFunction runs in the module's dtype): the fp32
    kernels against per-expert matmul in float64.  fp32 products and sums, so only the order of
    summation differs from torch's fp32 matmul: errors of a few fp32 roundings of the absolute sum."""
    from optimus.models.common.moe import GroupedGemmFunction
    g = torch.Generator().manual_seed(rows + 7)
    x = torch.randn(rows, K, generator=g)
    w = torch.randn(G, N, K, generator=g) * 0.05
    dout = torch.randn(rows, N, generator=g)
    cum = _counts(kind, G, rows)
    xd = x.to(cuda).requires_grad_(True)
    wd = w.to(cuda).requires_grad_(True)
    out = GroupedGemmFunction.apply(xd, wd, cum, int((cum[1:] - cum[:-1]).max()), False)
    assert out.dtype == torch.float32
    out.backward(dout.to(cuda))
    X, W, D = x.double(), w.double(), dout.double()
    ref = torch.zeros(rows, N, dtype=torch.float64)
    dx_ref = torch.zeros(rows, K, dtype=torch.float64)
    dw_ref = torch.zeros(G, N, K, dtype=torch.float64)
    ref_abs, dx_abs, dw_abs = torch.zeros_like(ref), torch.zeros_like(dx_ref), torch.zeros_like(dw_ref)
    for e in range(G):
        s, t = int(cum[e]), int(cum[e + 1])
        ref[s:t] = X[s:t] @ W[e].t(); ref_abs[s:t] = X[s:t].abs() @ W[e].abs().t()
        dx_ref[s:t] = D[s:t] @ W[e]; dx_abs[s:t] = D[s:t].abs() @ W[e].abs()
        dw_ref[e] = D[s:t].t() @ X[s:t]; dw_abs[e] = D[s:t].abs().t() @ X[s:t].abs()
    for name, got, want, scale in (("out", out, ref, ref_abs), ("dx", xd.grad, dx_ref, dx_abs),
                                   ("dw", wd.grad, dw_ref, dw_abs)):
        err = (got.detach().double().cpu() - want).abs()
        assert bool((err <= 2e-6 * scale + 1e-30).all()), (name, float((err / (scale + 1e-30)).max()))
    empty = (cum[1:] == cum[:-1])
    if empty.any():
        assert float(wd.grad[empty.to(cuda)].abs().max()) == 0.0


def test_float32_backward_of_many_experts(cuda):
    """30000 experts, a few of them with rows: bounded by the launch's blocks alone."""
    from optimus import _native as n
    G, rows, I, H = 30000, 64, 8, 16
    g = torch.Generator().manual_seed(1)
    owner = torch.sort(torch.randint(0, G, (rows,), generator=g)).values
    cum = torch.cat([torch.zeros(1, dtype=torch.long), torch.bincount(owner, minlength=G).cumsum(0)]).to(torch.int32).to(cuda)
    x, dy, wg, wu, wd = (torch.randn(*s, generator=g).to(cuda) for s in ((rows, H), (rows, H), (G, I, H), (G, I, H), (G, H, I)))
    ws = [torch.nn.Parameter(w) for w in (wg, wu, wd)]
    from optimus.models.common.moe import MergedMLPFunction
    xd = x.clone().requires_grad_(True)
    MergedMLPFunction.apply(xd, *ws, cum).backward(dy)
    D, ref = (lambda t: t.detach().double()), [torch.zeros_like(w, dtype=torch.float64) for w in ws]
    for r in range(rows):
        e = int(owner[r])
        a, b = D(wg[e]) @ D(x[r]), D(wu[e]) @ D(x[r])
        s = torch.sigmoid(a)
        dh = D(wd[e]).t() @ D(dy[r])
        da, db = dh * b * s * (1 + a * (1 - s)), dh * a * s
        ref[0][e] += torch.outer(da, D(x[r]))
        ref[1][e] += torch.outer(db, D(x[r]))
        ref[2][e] += torch.outer(D(dy[r]), a * s * b)
        want = D(wg[e]).t() @ da + D(wu[e]).t() @ db
        # float32 sums of 8 to 16 products behind three of their own: 2e-6 of the largest, as elsewhere, times their number
        assert (D(xd.grad[r]) - want).abs().max() <= 1e-5 * (1 + want.abs().max())
    for w, want in zip(ws, ref):
        assert (D(w.grad) - want).abs().max() <= 1e-5 * (1 + want.abs().max())


# contractions of which the last step (32) is partial, of both operands; one and two row-tile heights
@pytest.mark.parametrize("counts,I,H", [([40, 7, 0, 33], 72, 40), ([700, 129], 264, 328), ([1, 2, 3, 95], 8, 104)])
def test_float32_infinities_stay_infinities(cuda, counts, I, H):
    """An infinity in the last contraction index of either operand gives what float64 products give: it meets no zero that
    stands for an index past the end."""
    from optimus import _native as n
    g = torch.Generator().manual_seed(I)
    G, rows = len(counts), sum(counts)
    cum = torch.zeros(G + 1, dtype=torch.int32)
    cum[1:] = torch.cumsum(torch.tensor(counts), 0)
    inf, P, L, d, st = float("inf"), n.ptr, n.lib(), cum.to(cuda), n.stream()
    last = (cum[1:] - 1)[torch.tensor(counts) > 0].long()     # each expert's last row
    mats = lambda r, c: torch.rand(r, c, generator=g) + 0.5   # (no zero beside an infinity)
    x, dy, h, dg, du = mats(rows, H), mats(rows, H), mats(rows, I), mats(rows, I), mats(rows, I)
    wg, wu, wd = (torch.rand(G, *s, generator=g) + 0.5 for s in ((I, H), (I, H), (H, I)))
    wg[:, I // 2, H - 1], wu[:, I - 1, H - 1], wd[:, H - 1, 0] = inf, -inf, inf
    same = lambda got, want, name: (torch.testing.assert_close(got.double().cpu(), want, rtol=1e-5, atol=0.0, equal_nan=True, msg=name))

    def run(name, *a):
        n.check(getattr(L, name)(*a, st), name)
        torch.cuda.synchronize()
    dev = lambda *ts: [t.to(cuda) for t in ts]
    new = lambda *s: torch.full(s, 7.0, device=cuda)
    X, DY, HH, DG, DU, WG, WU, WD = dev(x, dy, h, dg, du, wg, wu, wd)
    per_expert = lambda f: torch.cat([f(slice(int(cum[e]), int(cum[e + 1])), e) for e in range(G)])
    up = lambda t: t.double()
    # the weights' infinities: forward, input gradient of one matrix, gate and up, both of them in one accumulation
    y = new(rows, I)
    run("om_grouped_gemm_fwd_f32", P(X), P(WG), P(y), P(d), rows, G, I, H, 0)
    same(y, per_expert(lambda s, e: up(x[s]) @ up(wg[e]).t()), "fwd")
    dx = new(rows, I)
    run("om_grouped_gemm_dgrad_f32", P(DY), P(WD), P(dx), P(d), rows, G, H, I, 0)
    same(dx, per_expert(lambda s, e: up(dy[s]) @ up(wd[e])), "dgrad")
    gq, uq, hq = new(rows, I), new(rows, I), new(rows, I)
    run("om_merged_mlp_gate_up_fwd_f32", P(X), None, 0, P(WG), P(WU), P(gq), P(uq), P(hq), P(d), rows, G, I, H, 0, 0)
    same(gq, per_expert(lambda s, e: up(x[s]) @ up(wg[e]).t()), "gate")
    same(uq, per_expert(lambda s, e: up(x[s]) @ up(wu[e]).t()), "up")
    dx = new(rows, H)
    run("om_merged_mlp_gate_up_dgrad_f32", P(DG), P(DU), P(WG), P(WU), P(dx), P(d), rows, G, I, H, 0, 0)
    same(dx, per_expert(lambda s, e: up(dg[s]) @ up(wg[e]) + up(du[s]) @ up(wu[e])), "dx")
    # the activations' infinities: weight gradients, alone and in the backward's one launch
    x[last, 3], h[last, I - 1], dg[last, 1] = inf, -inf, -inf
    X, HH, DG = dev(x, h, dg)
    dw = lambda a, b: torch.stack([up(a[s]).t() @ up(b[s]) for s in (slice(int(cum[e]), int(cum[e + 1])) for e in range(G))])
    out = new(G, H, I)
    run("om_grouped_gemm_wgrad_f32", P(DY), P(HH), P(out), P(d), rows, G, H, I, 0)
    same(out, dw(dy, h), "wgrad")
    index = torch.arange(rows, dtype=torch.int32, device=cuda)
    for ix in (None, P(index)):
        down, gate, upw = new(G, H, I), new(G, I, H), new(G, I, H)
        run("om_grouped_gemm_wgrad_merged_dgrad_f32", P(DY), P(HH), P(DG), P(DU), P(X), ix, rows, P(WG), P(WU), P(dx), P(down), P(gate),
            P(upw), P(d), rows, G, I, H, 0, 0, 0, 0, 0)
        for name, got, want in (("down", down, dw(dy, h)), ("gate", gate, dw(dg, x)), ("up", upw, dw(du, x))):
            same(got, want, name)


# row tiles of 32 and of 64, contractions of 1 to 5 steps of 32 and partial ones, more rows in an expert than the kernel keeps
# indices of in LDS, no rows at all
@pytest.mark.parametrize("counts,I,H", [([31, 32, 33, 0, 1, 63, 64, 65], 40, 72), ([96, 97, 128, 160, 159, 5], 160, 96), ([1100, 7, 300], 64, 32),
                                        ([512, 530, 490, 515, 700, 300, 512, 537], 512, 256), ([2000, 2048], 136, 520), ([0, 0, 0], 64, 64)])
@pytest.mark.parametrize("indexed", [False, True])
def test_float32_input_and_weight_gradients_in_one_launch(cuda, indexed, counts, I, H):
    """dx and the three weight gradients (written, and added to old values) against float64, and forward and SwiGLU backward of
    the same sizes: a few float32 roundings of the absolute sum."""
    from optimus import _native as n
    g = torch.Generator().manual_seed(sum(counts) + I)
    G, rows = len(counts), sum(counts)
    R, T = max(rows, 1), max(rows // 2, 4)
    cum = torch.zeros(G + 1, dtype=torch.int32)
    cum[1:] = torch.cumsum(torch.tensor(counts), 0)
    rnd = lambda *s: torch.randn(*s, generator=g).to(cuda)
    x, idx = rnd(T if indexed else R, H), torch.randint(0, T, (R,), generator=g, dtype=torch.int32).to(cuda)
    dy, h, dg, du, wg, wu, wd = rnd(R, H), rnd(R, I), rnd(R, I), rnd(R, I), rnd(G, I, H) * 0.05, rnd(G, I, H) * 0.05, rnd(G, H, I) * 0.05
    gq, uq, hq, dgq, duq, dx = rnd(R, I), rnd(R, I), rnd(R, I), rnd(R, I), rnd(R, I), rnd(R, H)
    shapes = ((G, H, I), (G, I, H), (G, I, H))
    fresh, old = [torch.full(s, 7.0, device=cuda) for s in shapes], [rnd(*s) for s in shapes]
    acc, d, P, L = [o.clone() for o in old], cum.to(cuda), n.ptr, n.lib()
    ix = P(idx) if indexed else None
    for suffix, out in (("", fresh), ("_accumulate", acc)):
        n.check(getattr(L, "om_grouped_gemm_wgrad_merged_dgrad_f32" + suffix)(
            P(dy), P(h), P(dg), P(du), P(x), ix, T, P(wg), P(wu), P(dx), *(P(o) for o in out), P(d), rows, G, I, H, 0, 0, 0, 0, 0, n.stream()), "bwd")
    n.check(L.om_merged_mlp_gate_up_fwd_f32(P(x), ix, T, P(wg), P(wu), P(gq), P(uq), P(hq), P(d), rows, G, I, H, 0, 0, n.stream()), "fwd")
    n.check(L.om_merged_mlp_down_dgrad_f32(P(dy), P(wd), P(gq), P(uq), P(dgq), P(duq), P(d), rows, G, I, H, 0, n.stream()), "dgrad")
    torch.cuda.synchronize()
    D = lambda t: t.double()

    def close(name, got, want, scale, roundings=2e-6):
        assert ((D(got) - want).abs() <= roundings * scale + 1e-30).all(), name
    xr = x[idx.long()] if indexed else x
    for e in range(G):
        s = slice(int(cum[e]), int(cum[e + 1]))
        for i, (a, b) in enumerate(((dy, h), (dg, xr), (du, xr))):
            want, scale = D(a[s]).t() @ D(b[s]), D(a[s]).abs().t() @ D(b[s]).abs()
            close(("dw", i, e), fresh[i][e], want, scale)
            assert torch.equal(acc[i][e], old[i][e] + fresh[i][e])
        close(("dx", e), dx[s], D(dg[s]) @ D(wg[e]) + D(du[s]) @ D(wu[e]), D(dg[s]).abs() @ D(wg[e]).abs() + D(du[s]).abs() @ D(wu[e]).abs())
        for name, got, w in (("g", gq, wg), ("u", uq, wu)):
            close((name, e), got[s], D(xr[s]) @ D(w[e]).t(), D(xr[s]).abs() @ D(w[e]).abs().t())
        dh, G64, U64 = D(dy[s]) @ D(wd[e]), D(gq[s]), D(uq[s])
        sg, size = torch.sigmoid(G64), D(dy[s]).abs() @ D(wd[e]).abs()
        # (the factors beside dh: a few roundings of their own)
        close(("du", e), duq[s], dh * G64 * sg, size * (G64 * sg).abs(), 4e-6)
        close(("dg", e), dgq[s], dh * U64 * sg * (1 + G64 * (1 - sg)), size * U64.abs() * sg * (1 + G64.abs()), 4e-6)
        close(("h", e), hq[s], G64 * sg * U64, (G64 * U64).abs() * sg, 4e-6)


# sizes of the seeded sweeps: multiples of 128, and multiples of 8 only (partial last tiles along every
# extent, a last contraction step with 8 to 56 indices)
SWEEP_SIZES = {"multiples_of_128": ([128, 256, 384, 512, 1024], [128, 256, 384, 640, 1024]),
               "multiples_of_8": ([8, 24, 72, 136, 200, 264, 328, 520, 1000], [8, 40, 72, 136, 200, 264, 328, 584, 1000])}


@pytest.mark.parametrize("sizes", sorted(SWEEP_SIZES))
@pytest.mark.parametrize("seed", list(range(24)))
def test_grouped_gemm_random_shapes(cuda, seed, sizes):
    """Seeded sweep over expert counts, row counts and sizes: exercises the persistent-block
    partition (fewer tiles than blocks, remainders over the 8 XCDs, experts without rows, one or many
    tiles per expert) on both tile shapes, against per-expert fp32 matmul."""
    from optimus.models.common.moe import GroupedGemmFunction
    rng = np.random.RandomState(1234 + seed)
    G = int(rng.choice([1, 2, 3, 7, 16, 33, 64, 70]))
    rows = int(rng.choice([1, 17, 255, 256, 257, 1000, 3333, 6000, 20000]))
    N = int(rng.choice(SWEEP_SIZES[sizes][0]))
    K = int(rng.choice(SWEEP_SIZES[sizes][1]))
    kind = ["uniform", "ragged", "empties"][seed % 3]
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(rows, K, generator=g).to(torch.bfloat16)
    w = (torch.randn(G, N, K, generator=g) * 0.05).to(torch.bfloat16)
    dout = torch.randn(rows, N, generator=g).to(torch.bfloat16)
    cum = _counts(kind, G, rows, seed=seed)
    assert int(cum[-1]) == rows
    xd = x.to(cuda).requires_grad_(True)
    wd = w.to(cuda).requires_grad_(True)
    out = GroupedGemmFunction.apply(xd, wd, cum, int((cum[1:] - cum[:-1]).max()), False)
    out.backward(dout.to(cuda))
    ref = _ref_fwd(x, w, cum)
    dx_ref = torch.zeros(rows, K); dw_ref = torch.zeros(G, N, K)
    for e in range(G):
        s, t = int(cum[e]), int(cum[e + 1])
        dx_ref[s:t] = dout[s:t].float() @ w[e].float()
        dw_ref[e] = dout[s:t].float().t() @ x[s:t].float()
    tag = (G, rows, N, K, kind)
    assert max_abs(out.float().cpu(), ref) <= 2e-2 * max(1.0, float(ref.abs().max())), tag
    assert_bf16_parity(out, ref, *ONE_ROUNDING, tag=f"ggemm_random{tag} fwd")
    assert_bf16_parity(xd.grad, dx_ref, *ONE_ROUNDING, tag=f"ggemm_random{tag} dgrad")
    assert max_abs(wd.grad.float().cpu(), dw_ref) <= 1e-2 * max(1.0, float(dw_ref.abs().max())), tag
    if float(dw_ref.abs().mean()) > 0:
        assert_bf16_parity(wd.grad, dw_ref, *ONE_ROUNDING, tag=f"ggemm_random{tag} wgrad")


@pytest.mark.parametrize("sizes", sorted(SWEEP_SIZES))
@pytest.mark.parametrize("seed", list(range(12)))
def test_gathered_merged_mlp_random_shapes(cuda, seed, sizes):
    """Seeded sweep of the bit-identity between the GEMMs that read tokens through input_indices and
    gather-then-GEMM, over token counts, top-k, expert windows and sizes."""
    from optimus.models.common.moe import (GatheredMergedMLPFunction, MergedMLPFunction,
                                           PrepareInputForGroupGemmFunction, build_token_permutation)
    from util import routed_experts
    rng = np.random.RandomState(99 + seed)
    N = int(rng.choice([4, 8, 16, 64]))
    K = int(rng.choice([1, 2, min(4, N)]))
    T = int(rng.choice([5, 64, 300, 1024, 5000]))
    H = int(rng.choice([128, 256, 384, 512] if sizes == "multiples_of_128" else [8, 72, 200, 328, 520]))
    I = int(rng.choice([128, 256, 384] if sizes == "multiples_of_128" else [8, 40, 136, 264]))
    start = int(rng.choice([0, N // 4]))
    end = int(rng.choice([N, max(start + 1, N - N // 4)]))
    G = end - start
    g = torch.Generator().manual_seed(seed)
    se = routed_experts(T, N, K, seed=seed, skew=float(rng.choice([0.0, 1.0]))).to(cuda)
    cum, cum_ep, ii, oi, _ = build_token_permutation(se, start, end)
    rows = int(cum[-1].item())
    ii, oi = ii[:rows], oi[:rows]
    x = torch.randn(T, H, generator=g).to(torch.bfloat16)
    ws = [(torch.randn(G, I, H, generator=g) * 0.05).to(torch.bfloat16),
          (torch.randn(G, I, H, generator=g) * 0.05).to(torch.bfloat16),
          (torch.randn(G, H, I, generator=g) * 0.05).to(torch.bfloat16)]
    dy = torch.randn(rows, H, generator=g).to(torch.bfloat16).to(cuda)
    results = []
    for gathered in (False, True):
        xd = x.to(cuda).requires_grad_(True)
        wd = [w.to(cuda).requires_grad_(True) for w in ws]
        if gathered:
            y = GatheredMergedMLPFunction.apply(xd, ii, cum_ep, oi, *wd, cum)
        else:
            y = MergedMLPFunction.apply(PrepareInputForGroupGemmFunction.apply(xd, ii, cum_ep, oi), *wd, cum)
        y.backward(dy)
        results.append([y.detach(), xd.grad] + [w.grad for w in wd])
    for name, a, b in zip(("y", "dx", "dw_gate", "dw_up", "dw_down"), *results):
        assert torch.equal(a, b), (name, T, K, N, start, end, I, H)


@pytest.mark.parametrize("G,rows,N,K", [(4096, 9000, 128, 256), (4097, 9000, 256, 128), (5000, 6000, 128, 128)])
def test_wgrad_with_thousands_of_experts(cuda, G, rows, N, K):
    """The weight gradient has no limit on the number of experts (the forward/dgrad tile table has).
    Up to 4096 experts its tiles are split over the XCDs by estimated work, above that by count:
    both sides of that threshold, most experts with 0-3 rows, against per-expert fp32 matmul."""
    from optimus import _native as n
    g = torch.Generator().manual_seed(G)
    c = torch.bincount(torch.randint(0, G, (rows,), generator=g), minlength=G)
    cum = torch.zeros(G + 1, dtype=torch.int32)
    cum[1:] = torch.cumsum(c, 0)
    dy = torch.randn(rows, N, generator=g).to(torch.bfloat16)
    x = torch.randn(rows, K, generator=g).to(torch.bfloat16)
    dyd, xd, cumd = dy.to(cuda), x.to(cuda), cum.to(cuda)
    dw = torch.full((G, N, K), float("nan"), dtype=torch.bfloat16, device=cuda)
    n.check(n.lib().om_grouped_gemm_wgrad(n.ptr(dyd), n.ptr(xd), n.ptr(dw), n.ptr(cumd), rows, G, N, K, 0,
                                          n.stream()), "om_grouped_gemm_wgrad")
    got = dw.float().cpu()
    assert bool(torch.isfinite(got).all())      # every tile of every expert was written
    ref = torch.zeros(G, N, K)
    for e in torch.nonzero(c).flatten().tolist():
        s, t = int(cum[e]), int(cum[e + 1])
        ref[e] = dy[s:t].float().t() @ x[s:t].float()
    assert max_abs(got, ref) <= 1e-2 * max(1.0, float(ref.abs().max()))
    assert float(got[c == 0].abs().max()) == 0.0


def test_operands_beyond_2_31_elements(cuda):
    """Activations of 1.1M rows x 2048 (2.25e9 elements, 4.5 GB): every product of the merged MLP,
    forward and backward, reads or writes a tensor past the 2^31-element mark.  Rows at the start,
    around the mark and at the end are checked against fp32 per-expert products, and so are the
    weight gradients of the expert whose rows straddle the mark and of the last one."""
    from optimus.models.common.moe import MergedMLPFunction
    rows, H, I, G = 1_100_000, 2048, 128, 4
    assert rows * H > (1 << 31)
    cum = torch.tensor([0, 500_000, 1_000_000, 1_099_000, rows], dtype=torch.int32)
    gen = torch.Generator(device=cuda).manual_seed(77)
    x = torch.randn(rows, H, device=cuda, dtype=torch.bfloat16, generator=gen).requires_grad_(True)
    dy = torch.randn(rows, H, device=cuda, dtype=torch.bfloat16, generator=gen)
    ws = [(torch.randn(shape, device=cuda, dtype=torch.float32, generator=gen) * 0.03).to(torch.bfloat16).requires_grad_(True)
          for shape in ((G, I, H), (G, I, H), (G, H, I))]
    y = MergedMLPFunction.apply(x, *ws, cum.to(cuda))
    y.backward(dy)
    torch.cuda.synchronize()
    mark = (1 << 31) // H
    picks = torch.cat([torch.arange(0, 48), torch.arange(mark - 40, mark + 40), torch.arange(999_980, 1_000_020),
                       torch.arange(rows - 48, rows)])
    expert_of = torch.bucketize(picks, cum[1:].long(), right=True)
    wf = [w.detach().float().cpu() for w in ws]
    for e in range(G):
        sel = picks[expert_of == e]
        if sel.numel() == 0:
            continue
        xr = x.detach()[sel.to(cuda)].float().cpu().requires_grad_(True)
        yr = (torch.nn.functional.silu(xr @ wf[0][e].t()) * (xr @ wf[1][e].t())) @ wf[2][e].t()
        yr.backward(dy[sel.to(cuda)].float().cpu())
        assert_bf16_parity(y.detach()[sel.to(cuda)], yr, *MLP_BARS["out"], tag=f"beyond2^31 expert {e} y")
        assert_bf16_parity(x.grad[sel.to(cuda)], xr.grad, *MLP_BARS["grad"], tag=f"beyond2^31 expert {e} dx")
    for e in (2, 3):       # rows 1,000,000..1,099,000 straddle the mark; 1,099,000.. lie beyond it
        s0, s1 = int(cum[e]), int(cum[e + 1])
        xr = x.detach()[s0:s1].float().cpu()
        p = [w[e].clone().requires_grad_(True) for w in wf]
        yr = (torch.nn.functional.silu(xr @ p[0].t()) * (xr @ p[1].t())) @ p[2].t()
        yr.backward(dy[s0:s1].float().cpu())
        for name, w, r in zip(("dwg", "dwu", "dwd"), ws, p):
            assert_bf16_parity(w.grad[e], r.grad, *MLP_BARS["grad"], tag=f"beyond2^31 expert {e} {name}")


@pytest.mark.parametrize("N,K", [(320, 192), (192, 2048), (1000, 328)])
def test_few_rows_kernels_give_the_bits_of_the_direct_load_kernels(cuda, N, K):
    """Experts with few rows run kernels that stage their operands through registers (the weights two
    contraction steps ahead); they are meant to change when data arrives in LDS, not what is summed.
    The same light experts are computed twice through the C ABI: alone (fewer than 256 rows per expert
    on average: the register-staged kernels), and followed by one heavy expert that lifts the average
    above 256 rows (the direct-load kernels; sizes that keep both launches on the 128x128 tile).  The
    light experts' rows must agree bit for bit, forward and input gradient."""
    from optimus import _native as n
    from util import bits
    g = torch.Generator().manual_seed(N + K)
    G = 12
    light = torch.randint(0, 90, (G,), generator=g)
    light[3] = 0
    rows_light = int(light.sum())
    heavy = (G + 1) * 256 + 64 - rows_light          # lifts the mean above 256 rows per expert
    cum_a = torch.zeros(G + 1, dtype=torch.int32); cum_a[1:] = torch.cumsum(light, 0)
    cum_b = torch.cat([cum_a, torch.tensor([rows_light + heavy], dtype=torch.int32)])
    rows_b = rows_light + heavy
    x = torch.randn(rows_b, K, generator=g).to(torch.bfloat16).to(cuda)
    dout = torch.randn(rows_b, N, generator=g).to(torch.bfloat16).to(cuda)
    w = (torch.randn(G + 1, N, K, generator=g) * 0.05).to(torch.bfloat16).to(cuda)
    P = n.ptr
    res = []
    for cum, rows, experts in ((cum_a, rows_light, G), (cum_b, rows_b, G + 1)):
        cum = cum.to(cuda)
        out = torch.zeros(rows_b, N, dtype=torch.bfloat16, device=cuda)
        dx = torch.zeros(rows_b, K, dtype=torch.bfloat16, device=cuda)
        n.check(n.lib().om_grouped_gemm_fwd(P(x), P(w), P(out), P(cum), rows, experts, N, K, 0, n.stream()), "fwd")
        n.check(n.lib().om_grouped_gemm_dgrad(P(dout), P(w), P(dx), P(cum), rows, experts, N, K, 0, n.stream()), "dgrad")
        torch.cuda.synchronize()
        res.append((out[:rows_light], dx[:rows_light]))
    assert rows_light < G * 256 and rows_b >= (G + 1) * 256
    assert float(res[0][0].float().abs().max()) > 0
    assert (bits(res[0][0]) == bits(res[1][0])).all()
    assert (bits(res[0][1]) == bits(res[1][1])).all()


@pytest.mark.parametrize("T,K,N,start,end,I,H", [
    (1, 1, 1, 0, 1, 8, 8),              # one row, one 8-wide step
    (65, 2, 4, 0, 4, 72, 40),           # one row past a 64-row tile; extents between 32 and 64 and above
    (300, 3, 12, 2, 9, 264, 136),       # an expert window; remainders along every extent
    (40, 4, 80, 0, 80, 32, 64),         # more experts than a wavefront has lanes, some empty
])
@pytest.mark.parametrize("live", [False, True])
def test_merged_mlp_float32_gathered(cuda, T, K, N, start, end, I, H, live):
    """The float32 merged MLP through the token gather (om_merged_mlp_*_f32), forward and backward, against
    float64.  Bound: a float32 dot product of n terms is off by about sqrt(n) 2^-24 of its norm (n <= 300:
    1e-6), three products and the sigmoid in a chain: 1e-5 of the 2-norm.  `live`: the gate weight's
    gradient is a view of a larger buffer and gets added into it, the others are fresh."""
    from optimus.models.common.moe import GatheredMergedMLPFunction, build_token_permutation
    g = torch.Generator().manual_seed(T + I)
    G = end - start
    se = torch.stack([torch.randperm(N, generator=g)[:K] for _ in range(T)])
    cum, cum_ep, ii, oi, _ = build_token_permutation(se.to(cuda), start, end)
    rows = int(cum[-1].item())
    x = torch.randn(T, H, generator=g)
    ws = [torch.randn(s, generator=g) * 0.2 for s in ((G, I, H), (G, I, H), (G, H, I))]
    xd = x.to(cuda).requires_grad_(True)
    wd = [w.to(cuda).requires_grad_(True) for w in ws]
    before = torch.randn(G, I, H, generator=g)
    if live:
        wd[0].grad = torch.cat([before.flatten(), torch.zeros(8)]).to(cuda)[:-8].view(G, I, H)
    y = GatheredMergedMLPFunction.apply(xd, ii[:rows], cum_ep, oi[:rows], *wd, cum)
    dy = torch.randn(rows, H, generator=g)
    y.backward(dy.to(cuda))
    x64 = x.double().requires_grad_(True)
    w64 = [w.double().requires_grad_(True) for w in ws]
    c, idx = cum.cpu().tolist(), ii[:rows].cpu().long()
    parts = []
    for e in range(G):
        xe = x64[idx[c[e]:c[e + 1]]]
        parts.append((torch.nn.functional.silu(xe @ w64[0][e].t()) * (xe @ w64[1][e].t())) @ w64[2][e].t())
    ref = torch.cat(parts)
    ref.backward(dy.double())
    want_gate = w64[0].grad + (before.double() if live else 0)
    for got, want in ((y, ref), (xd.grad, x64.grad), (wd[0].grad, want_gate), (wd[1].grad, w64[1].grad),
                      (wd[2].grad, w64[2].grad)):
        err = (got.detach().double().cpu() - want.detach()).norm()
        assert float(err) <= 1e-5 * float(want.detach().norm()) + 1e-12


STREAM_COUNTS = [[1], [16], [64], [0, 1, 0, 15, 16, 17, 0, 3], [0] * 170 + [32, 33, 1] + [0] * 30 + [64, 65, 130], [0, 0, 72]]


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("N,K", [(8, 8), (40, 72), (200, 512), (328, 1000), (256, 1088)])
@pytest.mark.parametrize("counts", STREAM_COUNTS, ids=lambda c: f"{len(c)}x{max(c)}")
def test_few_row_products_stream_the_weights(cuda, counts, N, K, weighted):
    """The kernels for a handful of rows per expert (at most 64 + 16 per expert in all): row tiles of 64 in
    fragments of 16, a contraction shared by eight wavefronts in pieces of 64, column tiles of 16 + 16.
    Counts on both sides of each edge, experts beyond one scan of 64, a pitch between the experts'
    weights, rows through an index, extents that no tile divides.  Each product is one rounding of a
    float32 sum; h adds the rounding-free weight."""
    from optimus import _native as n
    G, rows = len(counts), sum(counts)
    # (the rule: otherwise the tiled kernels run)
    assert rows <= 64 + 16 * G and (rows < 2 * G or (min(rows, G) + rows // 128) * ((2 * N + 127) // 128) <= 256)
    g = torch.Generator().manual_seed(rows + N + K)
    cum = torch.zeros(G + 1, dtype=torch.int32)
    cum[1:] = torch.cumsum(torch.tensor(counts), 0)
    T, pitch = 37, N * K + 64
    x = torch.randn(T, K, generator=g).to(torch.bfloat16)
    index = torch.randint(0, T, (rows,), generator=g).int()
    scale = torch.rand(rows, generator=g)
    store = [(torch.randn(G * pitch, generator=g) * 0.05).to(torch.bfloat16) for _ in range(2)]
    w = [s.view(G, pitch)[:, :N * K].view(G, N, K).float() for s in store]
    d = dict(x=x, index=index, scale=scale, cum=cum, wg=store[0], wu=store[1])
    d = {k: v.to(cuda) for k, v in d.items()}
    P = n.ptr
    guard = 3
    out = [torch.full((rows + guard, N), 7.0, dtype=torch.bfloat16, device=cuda) for _ in range(4)]
    xr = x[index.long()]
    d["xr"] = xr.to(cuda)
    if weighted:
        n.check(n.lib().om_merged_mlp_gate_up_fwd_weighted(P(d["x"]), P(d["index"]), T, P(d["wg"]), P(d["wu"]), P(d["scale"]),
                                                          P(out[0]), P(out[1]), P(out[2]), P(d["cum"]), rows, G, N, K, pitch,
                                                          n.stream()), "gate_up")
    else:
        n.check(n.lib().om_merged_mlp_gate_up_fwd(P(d["xr"]), P(d["wg"]), P(d["wu"]), P(out[0]), P(out[1]), P(out[2]),
                                                 P(d["cum"]), rows, G, N, K, pitch, n.stream()), "gate_up")
    n.check(n.lib().om_grouped_gemm_fwd(P(d["xr"]), P(d["wg"]), P(out[3]), P(d["cum"]), rows, G, N, K, pitch, n.stream()), "fwd")
    torch.cuda.synchronize()
    ref = [_ref_fwd(xr, m, cum) for m in w]
    h = torch.nn.functional.silu(ref[0]) * ref[1] * (scale[:, None] if weighted else 1.0)
    for name, got, want in zip(("g", "u", "h", "y"), out, (ref[0], ref[1], h, ref[0])):
        assert (got[rows:] == 7.0).all(), name
        # one bf16 rounding (2^-9 of the value), and sums of K products in another order; h from unrounded g, u
        err = (got[:rows].float().cpu() - want).abs()
        assert (err <= want.abs() * 2 ** -8 + 1e-6 * K ** 0.5).all(), (name, float(err.max()))


@pytest.mark.parametrize("counts", [[128, 129, 256, 384, 385, 1, 0, 639], [255, 257, 0, 512, 127, 130, 300, 300]], ids=str)
def test_half_row_tiles_of_the_256_kernels(cuda, counts):
    """The 256x256 kernels give a row tile with at most 128 rows to half of a block's wavefronts: remainders
    on both sides of 0, 128 and 256, experts with such a tile only, without one, and without rows; more tiles than blocks.  One bf16 rounding of
    a float32 sum of at most 1024 products (2^-8 of the value, and the order of the sum)."""
    from optimus import _native as n
    counts = counts * 6
    G, N, K, rows = len(counts), 1024, 512, sum(counts)
    assert rows >= 192 * G and (rows // 256) * (min(N, K) // 256) * 2 >= 256 // 2
    g = torch.Generator().manual_seed(rows)
    cum = torch.zeros(G + 1, dtype=torch.int32)
    cum[1:] = torch.cumsum(torch.tensor(counts), 0)
    x = torch.randn(rows, K, generator=g).to(torch.bfloat16).to(cuda)
    dy = torch.randn(rows, N, generator=g).to(torch.bfloat16).to(cuda)
    w = (torch.randn(G, N, K, generator=g) * 0.05).to(torch.bfloat16).to(cuda)
    y, dx = torch.full((rows, N), 7.0, dtype=torch.bfloat16, device=cuda), torch.full((rows, K), 7.0, dtype=torch.bfloat16, device=cuda)
    d, P = cum.to(cuda), n.ptr
    n.check(n.lib().om_grouped_gemm_fwd(P(x), P(w), P(y), P(d), rows, G, N, K, 0, n.stream()), "fwd")
    n.check(n.lib().om_grouped_gemm_dgrad(P(dy), P(w), P(dx), P(d), rows, G, N, K, 0, n.stream()), "dgrad")
    torch.cuda.synchronize()
    for e in range(G):
        s = slice(int(cum[e]), int(cum[e + 1]))
        for name, got, want, k in (("fwd", y[s], x[s].float() @ w[e].float().t(), K), ("dgrad", dx[s], dy[s].float() @ w[e].float(), N)):
            assert ((got.float() - want).abs() <= want.abs() * 2 ** -8 + 1e-6 * k ** 0.5).all(), (name, e)


@pytest.mark.parametrize("K", [64, 128, 192, 256, 320])
def test_row_units_and_step_counts_of_the_256_kernels(cuda, K):
    """1 to 5 contraction steps (the loads run two steps ahead, so the first and last two of a tile are special), rows on
    both sides of every multiple of 64 (the units in which a tile's rows are worked), and in the weight gradient
    contractions of 0 to 513 rows.  One bf16 rounding of a float32 sum (2^-8 of the value, and the order of the sum)."""
    from optimus import _native as n
    counts = [64, 65, 127, 129, 191, 192, 193, 255, 256, 257, 320, 0, 1, 448, 513, 300] * 3
    G, N, rows = len(counts), 1024, sum(counts)
    assert rows >= 192 * G and (rows // 256) * (N // 256) * 2 >= 256
    g = torch.Generator().manual_seed(K)
    cum = torch.zeros(G + 1, dtype=torch.int32)
    cum[1:] = torch.cumsum(torch.tensor(counts), 0)
    x = torch.randn(rows, K, generator=g).to(torch.bfloat16).to(cuda)
    z = torch.randn(rows, N, generator=g).to(torch.bfloat16).to(cuda)
    w = (torch.randn(G, N, K, generator=g) * 0.05).to(torch.bfloat16).to(cuda)
    wt = (torch.randn(G, K, N, generator=g) * 0.05).to(torch.bfloat16).to(cuda)
    y, dx = (torch.full((rows, N), 7.0, dtype=torch.bfloat16, device=cuda) for _ in range(2))
    dw = torch.full((G, N, 512), 7.0, dtype=torch.bfloat16, device=cuda)
    d, P = cum.to(cuda), n.ptr
    n.check(n.lib().om_grouped_gemm_fwd(P(x), P(w), P(y), P(d), rows, G, N, K, 0, n.stream()), "fwd")
    n.check(n.lib().om_grouped_gemm_dgrad(P(x), P(wt), P(dx), P(d), rows, G, K, N, 0, n.stream()), "dgrad")
    v = z[:, :512].contiguous()
    n.check(n.lib().om_grouped_gemm_wgrad(P(z), P(v), P(dw), P(d), rows, G, N, 512, 0, n.stream()), "wgrad")
    torch.cuda.synchronize()
    for e in range(G):
        s = slice(int(cum[e]), int(cum[e + 1]))
        for name, got, want, k in (("fwd", y[s], x[s].float() @ w[e].float().t(), K), ("dgrad", dx[s], x[s].float() @ wt[e].float(), K),
                                   ("wgrad", dw[e], z[s].float().t() @ v[s].float(), counts[e])):
            assert ((got.float() - want).abs() <= want.abs() * 2 ** -8 + 2e-5 * max(k, 1) ** 0.5).all(), (name, e)


# weights of 8 M elements and more: several XCDs share an expert, four with 16 experts or more, all eight with fewer.  Both
# tile sizes, columns of tiles that neither divides, more experts than a wavefront has lanes, experts without rows, one with all.
@pytest.mark.parametrize("kind,G,rows,N,K", [("uniform", 16, 4000, 4096, 2048), ("ragged", 33, 6500, 4096, 2048), ("ragged", 17, 700, 4104, 2056),
                                             ("empties", 20, 5000, 2048, 4096), ("onehot", 3, 900, 4352, 2048), ("ragged", 5, 1700, 2056, 4104),
                                             ("ragged", 70, 9000, 2048, 4096), ("uniform", 2, 64, 4096, 2048),
                                             # (not shared, but too much for the caches: experts with one row tile, with several)
                                             ("ragged", 64, 3000, 1024, 2048), ("onehot", 40, 129, 2056, 1640), ("ragged", 40, 129, 2056, 1664),
                                             ("ragged", 64, 33, 1024, 2048), ("uniform", 64, 31, 1024, 2048)])
def test_row_products_of_shared_experts(cuda, kind, G, rows, N, K):
    """Every tile once: forward, input gradient and the gate/up product against float32 products of each expert's
    rows; one bf16 rounding of a float32 sum (2^-8 of the value, and the order of the sum)."""
    from optimus import _native as n
    cum = _counts(kind, G, rows)
    bf = lambda *s, f=1.0: (torch.randn(*s, device=cuda) * f).to(torch.bfloat16)
    torch.manual_seed(G)
    x, dy, w, w2 = bf(rows, K), bf(rows, N), bf(G, N, K, f=0.02), bf(G, N, K, f=0.02)
    y, g, u, h = (torch.full((rows, N), 7.0, dtype=torch.bfloat16, device=cuda) for _ in range(4))
    dx, d, P = torch.full((rows, K), 7.0, dtype=torch.bfloat16, device=cuda), cum.to(cuda), n.ptr
    n.check(n.lib().om_grouped_gemm_fwd(P(x), P(w), P(y), P(d), rows, G, N, K, 0, n.stream()), "fwd")
    n.check(n.lib().om_grouped_gemm_dgrad(P(dy), P(w), P(dx), P(d), rows, G, N, K, 0, n.stream()), "dgrad")
    n.check(n.lib().om_merged_mlp_gate_up_fwd(P(x), P(w), P(w2), P(g), P(u), P(h), P(d), rows, G, N, K, 0, n.stream()), "gate/up")
    for e in range(G):
        s = slice(int(cum[e]), int(cum[e + 1]))
        first = x[s].float() @ w[e].float().t()
        for name, got, want, k in (("fwd", y[s], first, K), ("dgrad", dx[s], dy[s].float() @ w[e].float(), N), ("gate", g[s], first, K),
                                   ("up", u[s], x[s].float() @ w2[e].float().t(), K)):
            assert ((got.float() - want).abs() <= want.abs() * 2 ** -8 + 1e-6 * k ** 0.5).all(), (name, e)
    silu = torch.nn.functional.silu(g.float()) * u.float()    # h is formed before g and u are rounded: three roundings
    assert ((h.float() - silu).abs() <= silu.abs() * 2 ** -6 + (g.float().abs() + 1) * (u.float().abs() + 1) * 2 ** -7).all()


# four XCDs (16 experts and more) and all eight to an expert, 256x256 and 128x128 tiles, extents that neither divides
@pytest.mark.parametrize("kind,G,rows,I,H", [("ragged", 16, 6000, 2048, 4096), ("ragged", 5, 3300, 4096, 2048), ("ragged", 16, 1500, 2056, 4104),
                                             ("empties", 6, 600, 2048, 4096), ("onehot", 3, 900, 2056, 4104)])
def test_backward_products_of_shared_experts(cuda, kind, G, rows, I, H):
    """SwiGLU backward (rows through an index, weighted, with the partial sums of the weights' gradient) and the two-phase
    input gradient over a bound of the rows: bounds as in test_products_over_a_bound_of_the_rows, nothing past the last row."""
    from optimus import _native as n
    torch.manual_seed(rows)
    bf = lambda *s, f=1.0: (torch.randn(*s, device=cuda) * f).to(torch.bfloat16)
    bound, cum = rows + 45, _counts(kind, G, rows)
    dy, wg, wu, wd, g, u = bf(rows // 2, H), bf(G, I, H, f=0.02), bf(G, I, H, f=0.02), bf(G, H, I, f=0.02), bf(bound, I), bf(bound, I)
    index = torch.randint(0, rows // 2, (bound,), device=cuda, dtype=torch.int32)
    scale, new = torch.rand(bound, device=cuda), lambda c: torch.full((bound, c), 7.0, dtype=torch.bfloat16, device=cuda)
    dg, du, dx, d, P, L = new(I), new(I), new(H), cum.to(cuda), n.ptr, n.lib()
    dot = torch.full((L.om_merged_mlp_row_dot_parts(I), bound), 7.0, device=cuda)
    n.check(L.om_merged_mlp_down_dgrad_weighted_bound(P(dy), P(index), rows // 2, P(wd), P(g), P(u), P(scale), P(dg), P(du), P(dot), P(d), bound,
                                                      rows, G, I, H, 0, n.stream()), "down dgrad")
    n.check(L.om_merged_mlp_gate_up_dgrad_bound(P(dg), P(du), P(wg), P(wu), P(dx), P(d), bound, rows, G, I, H, 0, n.stream()), "dx")
    torch.cuda.synchronize()
    assert all((t[rows:] == 7.0).all() for t in (dg, du, dx)) and (dot[:, rows:] == 7.0).all()
    for e in range(G):
        s = slice(int(cum[e]), int(cum[e + 1]))
        gb, ub, dh = g[s].float(), u[s].float(), dy[index[s].long()].float() @ wd[e].float()
        sig, pre = torch.sigmoid(gb), scale[s, None] * dh
        factor = 1 + gb.abs() + ub.abs() * (1 + gb.abs())
        for name, got, want, rel, room in (("du", du[s], pre * gb * sig, 2 ** -7 + 2 ** -12, H ** 0.5 * factor),
                                           ("dg", dg[s], pre * ub * sig * (1 + gb * (1 - sig)), 2 ** -7 + 2 ** -12, H ** 0.5 * factor),
                                           ("dx", dx[s], dg[s].float() @ wg[e].float() + du[s].float() @ wu[e].float(), 2 ** -8, (2 * I) ** 0.5)):
            assert ((got.float() - want).abs() <= want.abs() * rel + 1e-6 * room).all(), (name, e)
        terms = dh * gb * sig * ub
        assert ((dot[:, s].sum(0) - terms.sum(1)).abs() <= (2 ** -8 + 1e-5) * terms.abs().sum(1) + 1e-6).all(), e


# (rows per expert: enough to share, on 128x128 tiles; extents that tiles and steps divide and do not)
@pytest.mark.parametrize("kind,G,rows,I,H", [("ragged", 16, 1500, 2048, 4096), ("empties", 5, 500, 2056, 4104), ("ragged", 33, 1100, 2056, 4104)])
def test_sharing_experts_leaves_the_bits(cuda, kind, G, rows, I, H):
    """Experts divided among XCDs or not (fewer rows expected): the products of the merged MLP add in the same order."""
    from optimus import _native as n
    torch.manual_seed(G)
    bf = lambda *s, f=1.0: (torch.randn(*s, device=cuda) * f).to(torch.bfloat16)
    x, dy, wg, wu, wd = bf(rows, H), bf(rows, H), bf(G, I, H, f=0.02), bf(G, I, H, f=0.02), bf(G, H, I, f=0.02)
    d, index, scale = _counts(kind, G, rows).to(cuda), torch.randperm(rows, device=cuda, dtype=torch.int32), torch.rand(rows, device=cuda)
    P, L, parts, out = n.ptr, n.lib(), n.lib().om_merged_mlp_row_dot_parts(I), []
    for expected in (32 * G - 1, rows):
        g, u, h, dg, du = (torch.empty(rows, I, dtype=torch.bfloat16, device=cuda) for _ in range(5))
        y, dx, dot = torch.empty_like(x), torch.empty_like(x), torch.empty(parts, rows, device=cuda)
        n.check(L.om_merged_mlp_gate_up_fwd_weighted_bound(P(x), P(index), rows, P(wg), P(wu), P(scale), P(g), P(u), P(h), P(d), rows,
                                                           expected, G, I, H, 0, n.stream()), "gate/up")
        n.check(L.om_grouped_gemm_fwd_bound(P(h), P(wd), P(y), P(d), rows, expected, G, H, I, 0, n.stream()), "down")
        n.check(L.om_merged_mlp_down_dgrad_weighted_bound(P(dy), P(index), rows, P(wd), P(g), P(u), P(scale), P(dg), P(du), P(dot), P(d),
                                                          rows, expected, G, I, H, 0, n.stream()), "down dgrad")
        n.check(L.om_merged_mlp_gate_up_dgrad_bound(P(dg), P(du), P(wg), P(wu), P(dx), P(d), rows, expected, G, I, H, 0, n.stream()), "dx")
        out.append((g, u, h, y, dg, du, dot, dx))
    torch.cuda.synchronize()
    for i, (a, b) in enumerate(zip(*out)):
        assert torch.equal(a, b), i


def test_sharing_experts_leaves_the_bits_of_large_tiles(cuda):
    """The same on 256x256 tiles: an expert's rows as the last row tiles of a launch of one expert, which is not shared;
    as many tiles before them, modulo the period of the steps that sums begin at (8)."""
    from optimus import _native as n
    G, rows, N, K = 9, 4500, 2048, 4096
    torch.manual_seed(3)
    x, w = torch.randn(rows, K, device=cuda).to(torch.bfloat16), (torch.randn(G, N, K, device=cuda) * 0.02).to(torch.bfloat16)
    cum, y, P, before = _counts("ragged", G, rows), torch.empty(rows, N, dtype=torch.bfloat16, device=cuda), n.ptr, 0
    n.check(n.lib().om_grouped_gemm_fwd(P(x), P(w), P(y), P(cum.to(cuda)), rows, G, N, K, 0, n.stream()), "fwd")
    for e in range(G):
        s = slice(int(cum[e]), int(cum[e + 1]))
        xe = torch.cat([torch.zeros((before % 8 + 16) * 256, K, dtype=torch.bfloat16, device=cuda), x[s]])
        ye, ce = torch.empty(len(xe), N, dtype=torch.bfloat16, device=cuda), torch.tensor([0, len(xe)], dtype=torch.int32, device=cuda)
        n.check(n.lib().om_grouped_gemm_fwd(P(xe), P(w[e]), P(ye), P(ce), len(xe), 1, N, K, 0, n.stream()), "one expert")
        assert torch.equal(ye[len(xe) - (s.stop - s.start):], y[s]), e
        before += (s.stop - s.start + 255) // 256


@pytest.mark.parametrize("expected", [0, 9, 100, 1087, 3000, 9000])
@pytest.mark.parametrize("N,K", [(1024, 512), (200, 328)])
def test_products_over_a_bound_of_the_rows(cuda, expected, N, K):
    """Outputs sized by a bound of the rows, the kernel chosen by the rows to expect (streamed weights, both loads
    of the 128x128 tile, 256x256): right for any expectation, nothing written past the rows there are.  A row far
    from the expected ones included; bounds as in test_few_row_products_stream_the_weights."""
    from optimus import _native as n
    counts, bound = [0, 1, 300, 0, 17, 64, 700, 5], 9000
    G, rows, T = len(counts), sum(counts), 211
    g = torch.Generator().manual_seed(expected + N)
    cum = torch.zeros(G + 1, dtype=torch.int32)
    cum[1:] = torch.cumsum(torch.tensor(counts), 0)
    bf = lambda *s, f=1.0: (torch.randn(*s, generator=g) * f).to(torch.bfloat16).to(cuda)
    x, dy = bf(T, K), bf(T, K)
    index = torch.zeros(bound, dtype=torch.int32)
    index[:rows] = torch.randint(0, T, (rows,), generator=g).int()
    scale = torch.rand(bound, generator=g).to(cuda)
    wg, wu, wd = bf(G, N, K, f=0.05), bf(G, N, K, f=0.05), bf(G, K, N, f=0.05)
    new = lambda c: torch.full((bound, c), 7.0, dtype=torch.bfloat16, device=cuda)
    G_, U, Hh, dG, dU, Y, dX = new(N), new(N), new(N), new(N), new(N), new(K), new(K)
    parts = n.lib().om_merged_mlp_row_dot_parts(N)
    dot = torch.full((parts, bound), 7.0, device=cuda)
    d, ix, P, st = cum.to(cuda), index.to(cuda), n.ptr, n.stream()
    L = n.lib()
    n.check(L.om_merged_mlp_gate_up_fwd_weighted_bound(P(x), P(ix), T, P(wg), P(wu), P(scale), P(G_), P(U), P(Hh), P(d), bound,
                                                       expected, G, N, K, 0, st), "gate_up")
    n.check(L.om_grouped_gemm_fwd_bound(P(Hh), P(wd), P(Y), P(d), bound, expected, G, K, N, 0, st), "down")
    n.check(L.om_merged_mlp_down_dgrad_weighted_bound(P(dy), P(ix), T, P(wd), P(G_), P(U), P(scale), P(dG), P(dU), P(dot), P(d),
                                                      bound, expected, G, N, K, 0, st), "down_dgrad")
    n.check(L.om_merged_mlp_gate_up_dgrad_bound(P(dG), P(dU), P(wg), P(wu), P(dX), P(d), bound, expected, G, N, K, 0, st), "dx")
    torch.cuda.synchronize()
    for t in (G_, U, Hh, dG, dU, Y, dX):
        assert (t[rows:] == 7.0).all()
    assert (dot[:, rows:] == 7.0).all()
    xr, dyr, sc = x[ix[:rows].long()].float(), dy[ix[:rows].long()].float(), scale[:rows, None]
    for e in range(G):
        s = slice(int(cum[e]), int(cum[e + 1]))
        g_, u_ = xr[s] @ wg[e].float().t(), xr[s] @ wu[e].float().t()
        gb, ub = G_[s].float(), U[s].float()
        sig = torch.sigmoid(gb)
        dh = dyr[s] @ wd[e].float()
        pre = sc[s] * dh
        want = {"g": (G_[s], g_, K), "u": (U[s], u_, K), "h": (Hh[s], sc[s] * torch.nn.functional.silu(g_) * u_, K),
                "y": (Y[s], Hh[s].float() @ wd[e].float().t(), N), "du": (dU[s], pre * gb * sig, K),
                "dg": (dG[s], pre * ub * sig * (1 + gb * (1 - sig)), K),
                "dx": (dX[s], dG[s].float() @ wg[e].float() + dU[s].float() @ wu[e].float(), 2 * N)}
        for name, (got, ref, k) in want.items():
            rel = 2 ** -7 + 2 ** -12 if name in ("du", "dg") else 2 ** -8
            # (the order of the sum enters du and dg through a factor of at most |g|, |u| (1 + |g|))
            factor = 1 + (gb.abs() + ub.abs() * (1 + gb.abs()) if name in ("du", "dg") else 0)
            assert ((got.float() - ref).abs() <= ref.abs() * rel + 1e-6 * k ** 0.5 * factor).all(), (name, e)
        terms = dh * gb * sig * ub
        assert ((dot[:, s].sum(0) - terms.sum(1)).abs() <= (2 ** -8 + 1e-5) * terms.abs().sum(1) + 1e-6).all(), e


# rows an expert: streamed, 128x128 tiles with remainders and extents that no tile divides, 256x256 tiles with partial ones
@pytest.mark.parametrize("rows_e,I,H", [((1, 0, 3), 64, 128), ((1, 0, 3), 72, 200), ((140, 0, 129, 64), 712, 200),
                                        ((300, 97, 256, 0, 513, 400, 330, 290), 2048, 512)])
@pytest.mark.parametrize("form", ["plain", "gathered", "weighted"])
def test_hidden_alone_is_the_h_of_the_full_product(cuda, rows_e, I, H, form):
    """om_merged_mlp_hidden_fwd: the bits of h, for each kernel that can take the product, and no g and u."""
    from optimus import _native as n
    L, P, G, rows, T = n.lib(), n.ptr, len(rows_e), sum(rows_e), 77
    gen = torch.Generator().manual_seed(rows)
    bf = lambda *s: torch.randn(*s, generator=gen).mul(0.2).bfloat16().to(cuda)
    x = bf(rows if form == "plain" else T, H)
    wg, wu = bf(G, I, H), bf(G, I, H)
    cum = torch.tensor([0] + list(torch.tensor(rows_e).cumsum(0)), dtype=torch.int32, device=cuda)
    index = torch.randint(0, T, (rows,), generator=gen, dtype=torch.int32).to(cuda)
    scale = torch.rand(rows, generator=gen).to(cuda)
    out = [torch.full((rows, I), 7.0, dtype=torch.bfloat16, device=cuda) for _ in range(4)]
    g, u, h, alone = out
    args = (rows, G, I, H, 0, n.stream())
    if form == "plain":
        n.check(L.om_merged_mlp_gate_up_fwd(P(x), P(wg), P(wu), P(g), P(u), P(h), P(cum), *args), "full")
    elif form == "gathered":
        n.check(L.om_merged_mlp_gate_up_fwd_gathered(P(x), P(index), T, P(wg), P(wu), P(g), P(u), P(h), P(cum), *args), "full")
    else:
        n.check(L.om_merged_mlp_gate_up_fwd_weighted(P(x), P(index), T, P(wg), P(wu), P(scale), P(g), P(u), P(h), P(cum), *args), "full")
    n.check(L.om_merged_mlp_hidden_fwd(P(x), None if form == "plain" else P(index), T, P(wg), P(wu), P(scale) if form == "weighted" else None,
                                       P(alone), P(cum), rows, rows, G, I, H, 0, None, n.stream()), "alone")
    torch.cuda.synchronize()
    assert torch.equal(alone, h) and not torch.equal(g, h)
    assert L.om_merged_mlp_hidden_fwd(P(x), None, T, P(wg), P(wu), P(scale), P(alone), P(cum), rows, rows, G, I, H, 0, None,
                                      n.stream()) == L.om_merged_mlp_gate_up_fwd(P(x), P(wg), P(wu), None, P(u), P(h), P(cum), *args) != 0


@pytest.mark.parametrize("tokens", [1, 37, 200, 4000])
@pytest.mark.parametrize("parallel", [1, 4])
def test_layer_without_gradients_gives_the_same_bits(cuda, tokens, parallel):
    """A layer with a shared expert, alone or in the routed experts' launch, and a window of the experts: with and without autograd."""
    from optimus.models.deepseek_v3.modeling_deepseek_v3 import DeepseekV3ParallelMoE
    from optimus.models.deepseek_v3.configuration_deepseek_v3 import DeepseekV3ParallelConfig
    from optimus.mapper import ParallelDpPpEpTpMapper
    cfg = DeepseekV3ParallelConfig(hidden_size=256, moe_intermediate_size=264, n_routed_experts=16, n_group=4, topk_group=2,
                                   num_experts_per_tok=4, expert_parallelism=parallel)
    torch.manual_seed(tokens)
    block = DeepseekV3ParallelMoE(cfg, ParallelDpPpEpTpMapper(expert_parallelism=parallel, rank=0)).to(torch.bfloat16).to(cuda)
    x = torch.randn(tokens, 1, 256, device=cuda, dtype=torch.bfloat16)
    with torch.no_grad():
        alone = block(x)
    assert torch.equal(alone, block(x).detach())


# experts without rows, partial tiles of both extents, one tile in all, more row tiles than blocks, sizes that do not join
@pytest.mark.parametrize("rows_e,I,H", [((0, 3, 0), 8, 16), ((130, 0, 1, 257), 200, 136), ((64,) * 8, 512, 256), ((700, 0, 129, 500, 3000), 712, 1000),
                                        ((20000, 5000), 264, 520), ((300, 500), 1024, 2048)])
@pytest.mark.parametrize("accumulate", [0, 1])
@pytest.mark.parametrize("shared_memory", [False, True])
def test_input_and_weight_gradients_in_one_call_are_those_of_two(cuda, rows_e, I, H, accumulate, shared_memory):
    """om_grouped_gemm_wgrad_merged_dgrad: the bits of the two entry points, in one launch or in several (the gradients of gate and up
    one buffer), and what those refuse is refused."""
    from optimus import _native as n
    L, P, G, rows, T = n.lib(), n.ptr, len(rows_e), sum(rows_e), 501
    gen = torch.Generator(device=cuda).manual_seed(rows + I)
    bf = lambda *s: (torch.randn(*s, generator=gen, device=cuda) * 0.1).bfloat16()
    x, dy, h, dg, du = bf(T, H), bf(T, H), bf(rows, I), bf(rows, I), bf(rows, I)
    wg, wu = bf(G, I, H), bf(G, I, H)
    cum = torch.tensor([0] + list(torch.tensor(rows_e).cumsum(0)), dtype=torch.int32, device=cuda)
    index = torch.randint(0, T, (rows,), generator=gen, device=cuda, dtype=torch.int32)
    start = [bf(G, H, I), bf(G, I, H), bf(G, I, H)]
    got, want = [t.clone() for t in start], [t.clone() for t in start]
    if shared_memory:
        got[2], want[2] = got[1], want[1]
    dx, dx_want = torch.full((2, rows, H), 7.0, dtype=torch.bfloat16, device=cuda)
    wgrad = L.om_grouped_gemm_wgrad_merged_accumulate_bound if accumulate else L.om_grouped_gemm_wgrad_merged_bound
    n.check(wgrad(P(dy), P(index), P(h), P(dg), P(du), P(x), P(index), T, *(P(t) for t in want), P(cum), rows, rows, G, I, H, 0, 0, 0,
                  n.stream()), "weights")
    n.check(L.om_merged_mlp_gate_up_dgrad_bound(P(dg), P(du), P(wg), P(wu), P(dx_want), P(cum), rows, rows, G, I, H, 0, n.stream()), "input")
    both = L.om_grouped_gemm_wgrad_merged_dgrad_accumulate if accumulate else L.om_grouped_gemm_wgrad_merged_dgrad
    call = lambda r, i: both(P(dy), P(index), P(h), P(dg), P(du), P(x), P(index), T, P(wg), P(wu), P(dx), *(P(t) for t in got),
                             P(cum), r, min(r, rows), G, i, H, 0, 0, 0, 0, n.stream())
    n.check(call(rows, I), "both")
    torch.cuda.synchronize()
    assert torch.equal(dx, dx_want) and all(torch.equal(a, b) for a, b in zip(got, want))
    assert call(0, I) == call(rows, I + 4) == L.om_merged_mlp_gate_up_dgrad(P(dg), P(du), P(wg), P(wu), P(dx), P(cum), rows, G, I + 4, H, 0,
                                                                          n.stream())
    assert L.om_merged_mlp_backward_joins(rows, G, I, H) == (0 if (I, H) == (1024, 2048) else 1)


@pytest.mark.parametrize("rows_e,I,H", [((0, 3, 0), 8, 16), ((130, 0, 1, 257), 200, 136), ((700, 0, 129, 500, 1000), 712, 1000), ((300, 500), 1024, 2048)])
@pytest.mark.parametrize("accumulate", [0, 1])
def test_input_and_weight_gradients_in_one_call_over_a_bound_of_the_rows(cuda, rows_e, I, H, accumulate):
    """As under an expert window: the buffers and `rows` are those of all pairs, `expected` lies between, below or above what the device counts.
    The bits of the two entry points over the same bound, rows past the routed ones neither read (they hold NaN) nor written."""
    from optimus import _native as n
    L, P, G, routed, T = n.lib(), n.ptr, len(rows_e), sum(rows_e), 501
    rows = 4 * routed + 61
    gen = torch.Generator(device=cuda).manual_seed(routed + I)
    bf = lambda *s: (torch.randn(*s, generator=gen, device=cuda) * 0.1).bfloat16()
    x, dy, h, dg, du = bf(T, H), bf(T, H), bf(rows, I), bf(rows, I), bf(rows, I)
    for t in (h, dg, du):
        t[routed:] = float("nan")
    wg, wu = bf(G, I, H), bf(G, I, H)
    cum = torch.tensor([0] + list(torch.tensor(rows_e).cumsum(0)), dtype=torch.int32, device=cuda)
    index = torch.randint(0, T, (rows,), generator=gen, device=cuda, dtype=torch.int32)
    index[routed:] = 0
    start = [bf(G, H, I), bf(G, I, H), bf(G, I, H)]
    wgrad = L.om_grouped_gemm_wgrad_merged_accumulate_bound if accumulate else L.om_grouped_gemm_wgrad_merged_bound
    both = L.om_grouped_gemm_wgrad_merged_dgrad_accumulate if accumulate else L.om_grouped_gemm_wgrad_merged_dgrad
    for expected in (routed // 2, (routed + rows) // 2, rows):
        got, want = [t.clone() for t in start], [t.clone() for t in start]
        dx, dx_want = torch.full((2, rows, H), 7.0, dtype=torch.bfloat16, device=cuda)
        n.check(wgrad(P(dy), P(index), P(h), P(dg), P(du), P(x), P(index), T, *(P(t) for t in want), P(cum), rows, expected, G, I, H, 0, 0, 0,
                      n.stream()), "weights")
        n.check(L.om_merged_mlp_gate_up_dgrad_bound(P(dg), P(du), P(wg), P(wu), P(dx_want), P(cum), rows, expected, G, I, H, 0, n.stream()), "input")
        n.check(both(P(dy), P(index), P(h), P(dg), P(du), P(x), P(index), T, P(wg), P(wu), P(dx), *(P(t) for t in got), P(cum), rows, expected,
                     G, I, H, 0, 0, 0, 0, n.stream()), "both")
        assert torch.equal(dx, dx_want) and all(torch.equal(a, b) for a, b in zip(got, want)), expected
        assert bool((dx[routed:] == 7.0).all()) and bool(torch.isfinite(dx).all()) and all(bool(torch.isfinite(t).all()) for t in got)
