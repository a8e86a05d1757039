"""The shared expert in the routed experts' launches (om_*_dense): the routed outputs are the bits of the calls without it,
and the shared expert's those of a call of its own, wherever that runs on the same tiles."""
import ctypes

import pytest
import torch

from util import assert_bf16_parity

pytestmark = pytest.mark.gpu


class Dense(ctypes.Structure):
    _fields_ = [("a", ctypes.c_void_p * 2), ("w", ctypes.c_void_p * 2), ("c", ctypes.c_void_p * 3), ("g", ctypes.c_void_p),
                ("u", ctypes.c_void_p), ("cum", ctypes.c_void_p), ("rows", ctypes.c_int64)]


def _ptrs(n, *ts):
    return (ctypes.c_void_p * n)(*([t.data_ptr() for t in ts] + [None] * (n - len(ts))))


# tokens at the edges of 64-row units and 128-row tiles; extents that no tile divides; one expert; experts without rows; a
# bound of the rows above those routed; 2200 tokens, whose shared expert takes 256x256 tiles of its own; 128 M weights a matrix,
# from which on they are loaded past the caches where one row tile reads them: one, and three, of the shared expert
@pytest.mark.parametrize("T,G,I,H,rows,bound", [(17, 8, 72, 40, 9, 34), (64, 32, 256, 1024, 64, 512), (128, 1, 136, 328, 5, 5),
                                                (129, 12, 200, 264, 387, 387), (300, 5, 512, 256, 0, 600), (2200, 3, 1024, 2048, 40, 40),
                                                (64, 16, 2048, 4096, 200, 200), (300, 16, 2048, 4096, 200, 250)])
def test_dense_expert_beside_the_routed_ones(cuda, T, G, I, H, rows, bound):
    from optimus import _native
    lib, st = _native.lib(), torch.cuda.current_stream().cuda_stream
    gen = torch.Generator().manual_seed(T + G)

    large = G * I * H >= 128 << 20
    on_device = torch.Generator(device=cuda).manual_seed(T + G)

    def rnd(*s, scale=1.0):
        if large:
            return torch.empty(*s, dtype=torch.bfloat16, device=cuda).normal_(0.0, scale, generator=on_device)
        return (torch.randn(*s, generator=gen) * scale).to(torch.bfloat16).to(cuda)

    def new(*s):
        return torch.full(s, float("nan"), dtype=torch.bfloat16, device=cuda)

    cuts = torch.sort(torch.randint(0, rows + 1, (G - 1,), generator=gen)).values
    cum = torch.cat([torch.zeros(1), cuts, torch.full((1,), rows)]).to(torch.int32).to(cuda)
    idx = torch.randint(0, T, (bound,), generator=gen).to(torch.int32).to(cuda)
    w = torch.rand(bound, generator=gen).to(cuda)
    one = torch.tensor([0, T], dtype=torch.int32, device=cuda)
    x, dy = rnd(T, H), rnd(T, H)
    wg, wu, wd = rnd(G, I, H, scale=0.1), rnd(G, I, H, scale=0.1), rnd(G, H, I, scale=0.1)
    sg, su, sd = rnd(I, H, scale=0.1), rnd(I, H, scale=0.1), rnd(H, I, scale=0.1)
    P = lambda t: t.data_ptr()
    parts = lib.om_merged_mlp_row_dot_parts(I)
    expected = max(rows, 1) if bound > rows else bound
    if large:
        assert lib.om_merged_mlp_dense_products(expected, G, I, H, T) == 15     # all four products

    def run(dense):
        r = {k: new(bound, I) for k in ("g", "u", "h", "dg", "du")} | {k: new(bound, H) for k in ("y", "dx")}
        s = {k: new(T, I) for k in ("g", "u", "h", "dg", "du")} | {k: new(T, H) for k in ("y", "dx")}
        r["dot"] = torch.zeros(parts, bound, device=cuda)
        tail = (P(cum), bound, expected, G)

        def call(name, args, dims, a, ws, cs, alone):
            if dense:
                d = Dense(_ptrs(2, *a), _ptrs(2, *ws), _ptrs(3, *cs), P(s["g"]), P(s["u"]), P(one), T)
                assert getattr(lib, name + "_dense")(*args, *tail, *dims, 0, ctypes.addressof(d), st) == 0
            else:
                assert getattr(lib, name + "_bound")(*args, *tail, *dims, 0, st) == 0
                assert alone() == 0

        call("om_merged_mlp_gate_up_fwd_weighted", (P(x), P(idx), T, P(wg), P(wu), P(w), P(r["g"]), P(r["u"]), P(r["h"])), (I, H),
             (x,), (sg, su), (s["g"], s["u"], s["h"]),
             lambda: lib.om_merged_mlp_gate_up_fwd(P(x), P(sg), P(su), P(s["g"]), P(s["u"]), P(s["h"]), P(one), T, 1, I, H, 0, st))
        call("om_grouped_gemm_fwd", (P(r["h"]), P(wd), P(r["y"])), (H, I), (s["h"],), (sd,), (s["y"],),
             lambda: lib.om_grouped_gemm_fwd(P(s["h"]), P(sd), P(s["y"]), P(one), T, 1, H, I, 0, st))
        call("om_merged_mlp_down_dgrad_weighted",
             (P(dy), P(idx), T, P(wd), P(r["g"]), P(r["u"]), P(w), P(r["dg"]), P(r["du"]), P(r["dot"])), (I, H),
             (dy,), (sd,), (s["dg"], s["du"]),
             lambda: lib.om_merged_mlp_down_dgrad(P(dy), P(sd), P(s["g"]), P(s["u"]), P(s["dg"]), P(s["du"]), P(one), T, 1, I, H, 0, st))
        call("om_merged_mlp_gate_up_dgrad", (P(r["dg"]), P(r["du"]), P(wg), P(wu), P(r["dx"])), (I, H), (s["dg"], s["du"]),
             (sg, su), (s["dx"],),
             lambda: lib.om_merged_mlp_gate_up_dgrad(P(s["dg"]), P(s["du"]), P(sg), P(su), P(s["dx"]), P(one), T, 1, I, H, 0, st))
        torch.cuda.synchronize()
        return r, s

    (r, s), (r0, s0) = run(True), run(False)
    for k in r:
        got, want = (r[k][:, :rows], r0[k][:, :rows]) if k == "dot" else (r[k][:rows], r0[k][:rows])
        assert torch.equal(got, want), k
        if k != "dot":
            assert r[k][rows:].isnan().all(), k          # nothing past the routed rows
    f = lambda *ts: [t.float().cpu() for t in ts]
    xf, gf, uf, hf, dgf, duf = f(x, s["g"], s["u"], s["h"], s["dg"], s["du"])
    sgf, suf, sdf = f(sg, su, sd)
    # each product against float32 on the operands that it had (the bar of a single rounding, as for the other entry points)
    assert_bf16_parity(s["g"], xf @ sgf.t(), 1.03, 1.8e-3, "dense g")
    assert_bf16_parity(s["u"], xf @ suf.t(), 1.03, 1.8e-3, "dense u")
    assert_bf16_parity(s["y"], hf @ sdf.t(), 1.03, 1.8e-3, "dense y")
    assert_bf16_parity(s["dx"], dgf @ sgf + duf @ suf, 1.03, 1.8e-3, "dense dx")
    # h from the sums themselves, one rounding; dg and du from the gradient of h rounded, two: independent, sqrt(2) of one at most
    silu = lambda t: t * torch.sigmoid(t)
    assert_bf16_parity(s["h"], silu(xf @ sgf.t()) * (xf @ suf.t()), 1.03, 1.8e-3, "dense h")
    dh, sig = dy.float().cpu() @ sdf, torch.sigmoid(gf)
    assert_bf16_parity(s["dg"], dh * uf * sig * (1 + gf * (1 - sig)), 1.46, 2.6e-3, "dense dg")
    assert_bf16_parity(s["du"], dh * silu(gf), 1.46, 2.6e-3, "dense du")
    if T > 80:   # (a launch of its own with fewer rows adds a forward product up in another order)
        for k in s:
            assert torch.equal(s[k], s0[k]), k


@pytest.mark.parametrize("T,products", [(8192, 0), (600, 15)])
def test_shared_expert_goes_first_where_nothing_of_it_rides(cuda, T, products):
    """All of its forward, and all of its backward, stand ahead of the routed experts' then."""
    from optimus import _native
    G, K, H, I = 8, 1, 1024, 1024
    assert _native.lib().om_merged_mlp_dense_products(T * K, G, I, H, T) == products
    gen = torch.Generator().manual_seed(T)

    def leaf(*s, scale=0.05):
        return (torch.randn(*s, generator=gen) * scale).to(torch.bfloat16).to(cuda).requires_grad_(True)

    x, rw = leaf(T, H, scale=1.0), torch.rand(T, K, generator=gen).to(cuda).requires_grad_(True)
    experts = torch.randint(0, G, (T, K), generator=gen).to(cuda)
    leaves = [leaf(G, I, H), leaf(G, I, H), leaf(G, H, I), leaf(I, H), leaf(I, H), leaf(H, I)]
    one = torch.tensor([0, T], dtype=torch.int32, device=cuda)
    _native.launch_log = []
    try:
        out = _native.host().moe_experts(x, rw, experts, 0, G, G, False, None, True, leaves, True, one)
        out.backward(torch.ones_like(out))
        torch.cuda.synchronize()
    finally:
        names, _native.launch_log = [e[0] for e in _native.launch_log], None
    assert any(n.endswith("_dense") for n in names) == (products != 0)
    if not products:
        for last_shared, first_routed in (("om_grouped_gemm_fwd", "om_merged_mlp_gate_up_fwd_weighted"),
                                          ("om_merged_mlp_gate_up_dgrad", "om_merged_mlp_down_dgrad_weighted")):
            assert names.index(last_shared) < names.index(first_routed), names
