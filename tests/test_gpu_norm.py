"""RMSNorm kernels (om_rmsnorm_fwd / om_rmsnorm_bwd) through the reference-shaped modules.

Bars: fp32 within 2e-6 relative of the CPU restatement; bf16 identical except where the last ulp of
rsqrt / of the fp32 sum of squares moves the first of the two bf16 roundings (the product with a
weight above 1 can then land two bf16 steps away; under 1 % of the elements differ at all); the residual sum h bit-exact; gradients against autograd of the
restatement run in fp32."""
import pytest
import torch

from oracle.moe_layer import rmsnorm

pytestmark = pytest.mark.gpu


def _inputs(rows, E, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    x = (torch.randn(rows, E, generator=g) * 2).to(dtype)
    res = torch.randn(rows, E, generator=g).to(dtype)
    w = (1 + 0.1 * torch.randn(E, generator=g)).to(dtype)
    return x, res, w


def _close_bf16(a, b, frac=0.01):
    ai = a.view(torch.int16).int(); bi = b.view(torch.int16).int()
    d = (ai - bi).abs()
    assert int(d.max()) <= 2 and float((d > 0).float().mean()) <= frac, (int(d.max()), float((d > 0).float().mean()))


@pytest.mark.parametrize("rows,E", [(1000, 2048), (64, 7168), (5, 256), (300, 4104)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("fused", [False, True])
def test_forward(cuda, rows, E, dtype, fused):
    from optimus.models.olmoe.modeling_olmoe import OlmoeParallelRMSNorm
    x, res, w = _inputs(rows, E, dtype, seed=rows + E)
    m = OlmoeParallelRMSNorm(E, eps=1e-5).to(dtype).to(cuda)
    with torch.no_grad():
        m.weight.copy_(w)
    if fused:
        y, h = m.forward_with_residual(x.to(cuda), res.to(cuda))
        y_ref, h_ref = rmsnorm(x, w, 1e-5, residual=res)
        assert torch.equal(h.cpu(), h_ref)
    else:
        y = m(x.to(cuda))
        y_ref, _ = rmsnorm(x, w, 1e-5)
    if dtype == torch.float32:
        torch.testing.assert_close(y.cpu(), y_ref, rtol=2e-6, atol=1e-7)
    else:
        _close_bf16(y.cpu(), y_ref)


@pytest.mark.parametrize("rows,E,dtype", [(777, 2048, torch.bfloat16), (130, 7168, torch.bfloat16),
                                          (257, 512, torch.float32)])
def test_backward(cuda, rows, E, dtype):
    from optimus.models.deepseek_v3.modeling_deepseek_v3 import DeepseekV3ParallelRMSNorm
    x, res, w = _inputs(rows, E, dtype, seed=3 * rows + E)
    g = torch.Generator().manual_seed(9)
    gy = torch.randn(rows, E, generator=g).to(dtype); gh = torch.randn(rows, E, generator=g).to(dtype)
    m = DeepseekV3ParallelRMSNorm(E, eps=1e-6).to(dtype).to(cuda)
    with torch.no_grad():
        m.weight.copy_(w)
    xg = x.to(cuda).requires_grad_(True); rg = res.to(cuda).requires_grad_(True)
    y, h = m.forward_with_residual(xg, rg)
    (y.float() * gy.to(cuda).float()).sum().add((h.float() * gh.to(cuda).float()).sum()).backward()
    xr = x.float().requires_grad_(True); rr = res.float().requires_grad_(True); wr = w.float().requires_grad_(True)
    yr, hr = rmsnorm(xr, wr, 1e-6, residual=rr)
    ((yr * gy.float()).sum() + (hr * gh.float()).sum()).backward()
    rel = lambda a, b: float((a.float().cpu() - b).abs().mean() / b.abs().mean())
    tol = 2e-6 if dtype == torch.float32 else 6e-3
    assert rel(xg.grad, xr.grad) <= tol and rel(rg.grad, rr.grad) <= tol
    assert rel(m.weight.grad, wr.grad) <= (1e-5 if dtype == torch.float32 else 6e-3)
    assert torch.equal(xg.grad, rg.grad)


# one to four vectors a lane, one lane short and over, the first row length that a wavefront does not hold; less than a wavefront's
# rows, a partial chunk (four rows up to 2048, then eight), both ways of loading (more than 8 M elements)
@pytest.mark.parametrize("rows,vecs", [(1, 1), (3, 64), (5, 65), (2047, 129), (2049, 192), (2051, 193), (4100, 256), (70, 257), (4099, 250),
                                       (16387, 64)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_rows_that_a_wavefront_holds(cuda, rows, vecs, dtype):
    from optimus.models.olmoe.modeling_olmoe import OlmoeParallelRMSNorm
    E = vecs * (8 if dtype == torch.bfloat16 else 4)
    x, res, w = _inputs(rows, E, dtype, seed=rows + vecs)
    dy = torch.randn(rows, E, generator=torch.Generator().manual_seed(4)).to(dtype)
    m = OlmoeParallelRMSNorm(E, eps=1e-5).to(dtype).to(cuda)
    with torch.no_grad():
        m.weight.copy_(w)
    xg = x.to(cuda).requires_grad_(True)
    y, h = m.forward_with_residual(xg, res.to(cuda))
    gh = torch.randn(rows, E, generator=torch.Generator().manual_seed(5)).to(dtype)
    dx_alone, dw_alone = torch.autograd.grad(y, (xg, m.weight), dy.to(cuda), retain_graph=True)
    torch.autograd.backward([y, h], [dy.to(cuda), gh.to(cuda)])
    assert torch.equal(xg.grad, dx_alone + gh.to(cuda)) and torch.equal(m.weight.grad, dw_alone)
    y_ref, h_ref = rmsnorm(x, w, 1e-5, residual=res)
    assert torch.equal(h.detach().cpu(), h_ref)
    if dtype == torch.float32:
        torch.testing.assert_close(y.detach().cpu(), y_ref, rtol=2e-6, atol=1e-7)
    else:
        _close_bf16(y.detach().cpu(), y_ref)
    # the gradients in float64, from the sum as the dtype holds it and (the weight's) the normalised value as it rounds it
    hd, gd, wd = h_ref.double(), dy.double(), w.double()
    r = (hd.pow(2).mean(1, keepdim=True) + 1e-5).rsqrt()
    xn, dxn = hd * r, gd * wd
    dx = r * (dxn - xn * (dxn * xn).mean(1, keepdim=True))
    # one rounding of the result (2^-9 / 2^-24 of it) and the float32 sums before it: at most E + rows terms' relative 2^-24 each
    eps = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -21
    assert float((dx_alone.cpu().double() - dx).norm() / dx.norm()) <= eps
    terms = gd * xn.to(dtype).double()
    bound = eps * terms.sum(0).abs() + terms.abs().sum(0) * (2.0 ** -24 * (rows / 4 + 8) + (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -22))
    assert bool(((m.weight.grad.cpu().double() - terms.sum(0)).abs() <= bound).all())


@pytest.mark.parametrize("E", [256, 2056])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_residual_gradients_that_the_kernel_does_not_read(cuda, E, dtype):
    """A gradient of h between 16-byte boundaries (a part of a larger tensor's) and a batch of them: dx + gh, as with one that it reads."""
    from optimus.models.olmoe.modeling_olmoe import OlmoeParallelRMSNorm
    rows = 7
    x, res, w = (t.to(cuda) for t in _inputs(rows, E, dtype, seed=E))
    m = OlmoeParallelRMSNorm(E, eps=1e-5).to(dtype).to(cuda)
    with torch.no_grad():
        m.weight.copy_(w)
    x.requires_grad_(True)
    y, h = m.forward_with_residual(x, res)
    gen = torch.Generator(device=cuda).manual_seed(1)
    gy, gh = (torch.randn(rows, E, generator=gen, device=cuda).to(dtype) for _ in range(2))
    want = torch.autograd.grad([y, h], [x, m.weight], [gy, gh], retain_graph=True)
    shifted = torch.empty(rows * E + 1, dtype=dtype, device=cuda)[1:].view(rows, E).copy_(gh)
    assert shifted.data_ptr() % 16 and shifted.is_contiguous()
    got = torch.autograd.grad([y, h], [x, m.weight], [gy, shifted], retain_graph=True)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    joined = torch.cat([torch.ones(1, device=cuda, dtype=dtype), h.flatten()])    # its gradient's part is such a tensor
    got = torch.autograd.grad([y, joined], [x], [gy, torch.cat([gh[0, :1], gh.flatten()])], retain_graph=True)
    assert torch.equal(got[0], want[0])
    batch = torch.stack([gh, 2 * gh, gh - 1])
    got, = torch.autograd.grad(h, x, batch, is_grads_batched=True)
    assert torch.equal(got, batch)                                                # (nothing comes through y)


@pytest.mark.parametrize("rows,vecs", [(1, 1), (131, 64), (700, 250), (2100, 256), (300, 257), (17 * 128, 3)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("add", [False, True])
def test_backward_with_the_least_workspace(cuda, rows, vecs, dtype, add):
    """om_rmsnorm_bwd_workspace_bytes, where the other size spreads the rows over more chunks: the same bits of dx, the weight gradient's
    sums in another order."""
    from optimus import _native as n
    L, st, E = n.lib(), n.stream(), vecs * (8 if dtype == torch.bfloat16 else 4)
    gen = torch.Generator(device=cuda).manual_seed(rows + vecs)
    dy, h, gh = (torch.randn(rows, E, generator=gen, device=cuda).to(dtype) for _ in range(3))
    w, rstd = torch.randn(E, generator=gen, device=cuda).to(dtype), torch.rand(rows, generator=gen, device=cuda) + 0.5
    got = []
    for size in (L.om_rmsnorm_bwd_workspace_bytes(rows, E), L.om_rmsnorm_bwd_workspace_spread_bytes(rows, E)):
        dx, dw = torch.full_like(h, 7.0), torch.full_like(w, 7.0)
        ws = torch.empty(size, dtype=torch.uint8, device=cuda)
        n.check(L.om_rmsnorm_bwd_residual(n.ptr(dy), n.ptr(h), n.ptr(w), n.ptr(rstd), n.ptr(gh) if add else None, n.ptr(dx), n.ptr(dw), n.ptr(ws),
                                          size, rows, E, n.dtype_code(h), st), "backward")
        got.append((dx, dw))
    assert torch.equal(got[0][0], got[1][0])
    # either is within one rounding of the result and a float32 rounding a term of the sum of dy * cast(h * rstd)
    terms = dy.double() * (h.float() * rstd[:, None]).to(dtype).double()
    eps = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -23
    for _, dw in got:
        assert bool(((dw.double() - terms.sum(0)).abs() <= eps * terms.sum(0).abs() + rows * 2.0 ** -24 * terms.abs().sum(0)).all())
    with_ws = lambda size: L.om_rmsnorm_bwd(n.ptr(dy), n.ptr(h), n.ptr(w), n.ptr(rstd), n.ptr(got[0][0]), n.ptr(got[0][1]), n.ptr(ws), size, rows, E,
                                            n.dtype_code(h), st)
    assert with_ws(L.om_rmsnorm_bwd_workspace_bytes(rows, E) - 1) != 0


@pytest.mark.parametrize("rows,vecs", [(130, 65), (515, 128), (1000, 129), (257, 192), (900, 193)])
def test_backward_with_the_least_workspace_for_every_length_that_fits(cuda, rows, vecs):
    """Two, three and four vectors a lane, whole and partial."""
    for dtype in (torch.bfloat16, torch.float32):
        for add in (False, True):
            test_backward_with_the_least_workspace(cuda, rows, vecs, dtype, add)
