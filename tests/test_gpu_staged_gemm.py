"""GPU: the register-staged grouped GEMM (fp32 of any shape; bf16 / fp16 whose
rows are not whole aligned 16-byte chunks) against float64.

Bound, per element: a reduction of length R over products rounded to fp32
errs by at most (R + 8) 2^-24 sum |a||b| (any summation order; the 8 covers
fp32's split operands, whose dropped terms are below 2^-24 of a product), and
the result is rounded once more to its own type of p significant bits, by at
most 2^-p of its value (p = 8 bf16, 11 fp16, 24 fp32), or 2^-25 at fp16's
subnormals."""

import pytest
import torch

pytestmark = pytest.mark.gpu

HALF_ULP = {torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11, torch.float32: 2.0**-24}
COUNTS = [130, 0, 1, 257, 63]


def _bound(ref, mag, R, dtype):
    return (R + 8) * 2.0**-24 * mag + HALF_ULP[dtype] * (ref.abs() + (R + 8) * 2.0**-24 * mag) + 2.0**-25


def _check(out, ref, mag, R, dtype, what):
    err = (out.cpu().double() - ref).abs()
    assert bool((err <= _bound(ref, mag, R, dtype)).all()), (
        what, float((err / _bound(ref, mag, R, dtype)).max()))


def _misaligned(shape, dtype, g, shift):
    """Contiguous tensor whose storage starts `shift` elements off a 256-byte boundary."""
    n = 1
    for s in shape:
        n *= s
    t = torch.randn(n, generator=g).to(dtype)
    buf = torch.empty(n + shift, dtype=dtype, device="cuda")
    buf[shift:] = t.cuda()
    return t.view(shape), buf[shift:].view(shape)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("K,N,shift", [(1, 9, 0), (9, 1, 1), (7, 129, 0), (66, 127, 1),
                                       (129, 65, 0), (128, 64, 1), (200, 683, 0)])
def test_staged_gemms_match_float64(ext, dtype, K, N, shift):
    g = torch.Generator().manual_seed(100 * K + N)
    E, A = len(COUNTS), sum(COUNTS)
    offs = [0]
    for c in COUNTS:
        offs.append(offs[-1] + c)
    offsets = torch.tensor(offs, dtype=torch.int32, device="cuda")
    X, Xg = _misaligned((A, K), dtype, g, shift)
    W, Wg = _misaligned((E, K, N), dtype, g, shift)
    W2, W2g = _misaligned((E, K, N), dtype, g, shift)
    D, Dg = _misaligned((A, N), dtype, g, shift)
    D2, D2g = _misaligned((A, N), dtype, g, shift)
    seg = [(e, slice(offs[e], offs[e + 1])) for e in range(E)]
    Xd, Wd, W2d, Dd, D2d = (t.double() for t in (X, W, W2, D, D2))

    def rows(f):
        return torch.cat([f(e, s) for e, s in seg])

    fwd = ext.grouped_gemm_kernel(Xg, offsets, Wg)
    _check(fwd, rows(lambda e, s: Xd[s] @ Wd[e]), rows(lambda e, s: Xd[s].abs() @ Wd[e].abs()),
           K, dtype, "fwd")
    dX = ext.bwd_grouped_gemm_dX_kernel(Wg, offsets, Dg)
    _check(dX, rows(lambda e, s: Dd[s] @ Wd[e].t()),
           rows(lambda e, s: Dd[s].abs() @ Wd[e].abs().t()), N, dtype, "dX")
    dX2 = ext.bwd_grouped_gemm_dX2(Wg, W2g, offsets, Dg, D2g)
    _check(dX2, rows(lambda e, s: Dd[s] @ Wd[e].t() + D2d[s] @ W2d[e].t()),
           rows(lambda e, s: Dd[s].abs() @ Wd[e].abs().t() + D2d[s].abs() @ W2d[e].abs().t()),
           2 * N, dtype, "dX2")
    dW = ext.bwd_grouped_gemm_dW_kernel(Xg, offsets, Dg)
    _check(dW, torch.stack([Xd[s].t() @ Dd[s] for e, s in seg]),
           torch.stack([Xd[s].abs().t() @ Dd[s].abs() for e, s in seg]), max(COUNTS), dtype, "dW")

    # fused epilogues: the same products, then the activation on rounded values
    act, dact = ext.grouped_gemm_gelu(Xg, offsets, Wg)
    h = fwd.cpu().double().requires_grad_()
    gelu = torch.nn.functional.gelu(h)
    (dg,) = torch.autograd.grad(gelu.sum(), h)
    tol = dict(rtol=4 * HALF_ULP[dtype], atol=2e-6 * float(h.detach().abs().max()))
    torch.testing.assert_close(act.cpu().double(), gelu.detach(), **tol)
    torch.testing.assert_close(dact.cpu().double(), dg, **tol)
    dH = ext.bwd_grouped_gemm_dX_gelu(Wg, offsets, Dg, Xg)
    assert torch.equal(dH, (dX.float() * Xg.float()).to(dtype))
    hid, gate, val = ext.grouped_gemm_swiglu(Xg, offsets, Wg, W2g)
    assert torch.equal(gate, fwd)
    assert torch.equal(val, ext.grouped_gemm_kernel(Xg, offsets, W2g))
    silu = torch.nn.functional.silu(gate.float()).to(dtype).float()
    torch.testing.assert_close(hid.float(), (silu * val.float()).to(dtype).float(),
                               rtol=8 * HALF_ULP[dtype], atol=1e-6)


@pytest.mark.parametrize("mode", ["fwd", "dX", "dW"])
def test_staged_f32_non_finite(ext, mode):
    """Infinities, NaN and values past bf16's largest propagate as fp32 products do."""
    g = torch.Generator().manual_seed(5)
    A, K, N = 200, 132, 140
    offsets = torch.tensor([0, A], dtype=torch.int32, device="cuda")
    X = torch.randn(A, K, generator=g)
    W = torch.randn(1, K, N, generator=g)
    D = torch.randn(A, N, generator=g)
    for t in (X, D):
        t[3, 5] = float("inf")
        t[131, 7] = float("nan")
        t[150, 131] = 3.4e38  # finite in fp32, rounds to infinity in bf16
        t[151, 130] = -3.4e38
    W.clamp_(-0.9, 0.9)
    if mode == "fwd":
        out = ext.grouped_gemm_kernel(X.cuda(), offsets, W.cuda()).cpu()
        ref = X.double() @ W[0].double()
    elif mode == "dX":
        out = ext.bwd_grouped_gemm_dX_kernel(W.cuda(), offsets, D.cuda()).cpu()
        ref = D.double() @ W[0].double().t()
    else:
        X.clamp_(-0.9, 0.9)
        out = ext.bwd_grouped_gemm_dW_kernel(X.cuda(), offsets, D.cuda()).cpu()[0]
        ref = X.double().t() @ D.double()
    ref = ref.float()
    assert torch.equal(torch.isnan(out), torch.isnan(ref))
    assert torch.equal(torch.isinf(out), torch.isinf(ref))
    ok = torch.isfinite(ref)
    assert torch.equal(out[torch.isinf(ref)], ref[torch.isinf(ref)])
    torch.testing.assert_close(out[ok], ref[ok], rtol=1e-4, atol=1e-3)


@pytest.mark.parametrize("mode", ["fwd", "dX", "dW"])
@pytest.mark.parametrize("R", [1, 132])
@pytest.mark.parametrize("ex,ew,rows", [
    (-110, 0, None), (-111, 0, None), (-114, 0, None), (-126, 0, None), (0, -114, None),
    (0, -126, None), (-126, 60, None), (-60, -60, None), (-118, 0, 3)])
def test_staged_f32_small_operands(ext, mode, R, ex, ew, rows):
    """Operands whose last bits no third bf16 term holds (below 2^-110) keep
    24 bits: the same relative bound at every magnitude, without an absolute
    term (products of values in [2^e, 2^(e+1)) stay normal here). rows: only
    that row of the left operand is small, between ordinary ones. A sum of one
    product (R = 1) shows a loss from 2^-114 on, long sums from 2^-126."""
    g = torch.Generator().manual_seed(6)
    A, K, N = 200, 132, 140
    A, K, N = {"fwd": (A, R, N), "dX": (A, K, R), "dW": (R, K, N)}[mode]
    offsets = torch.tensor([0, A], dtype=torch.int32, device="cuda")

    def values(*shape):
        return torch.randn(shape, generator=g).sign() * (1 + torch.rand(shape, generator=g))

    a, b = {"fwd": ((A, K), (K, N)), "dX": ((A, N), (K, N)), "dW": ((A, K), (A, N))}[mode]
    a, b = values(*a), values(*b)
    b = torch.ldexp(b, torch.tensor(ew))
    if rows is None:
        a = torch.ldexp(a, torch.tensor(ex))
    elif mode == "dW":
        a[:, rows] = torch.ldexp(a[:, rows], torch.tensor(ex))
    else:
        a[rows] = torch.ldexp(a[rows], torch.tensor(ex))
    ad, bd = a.double(), b.double()
    if mode == "fwd":
        out = ext.grouped_gemm_kernel(a.cuda(), offsets, b.cuda()[None])
        ref, mag = ad @ bd, ad.abs() @ bd.abs()
    elif mode == "dX":
        out = ext.bwd_grouped_gemm_dX_kernel(b.cuda()[None], offsets, a.cuda())
        ref, mag = ad @ bd.t(), ad.abs() @ bd.abs().t()
    else:
        out = ext.bwd_grouped_gemm_dW_kernel(a.cuda(), offsets, b.cuda())[0]
        ref, mag = ad.t() @ bd, ad.abs().t() @ bd.abs()
    err = (out.cpu().double() - ref).abs()
    assert bool((err <= (R + 8) * 2.0**-24 * mag).all()), float((err / mag).max())
