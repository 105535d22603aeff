"""GPU: the register-staged grouped GEMM (fp32 of any shape; bf16 / fp16 whose
rows are not whole aligned 16-byte chunks) against float64.

Bound, per element: a reduction of length R over products rounded to fp32
errs by at most (R + 8) 2^-24 sum |a||b| (any summation order; the 8 covers
fp32's split operands, whose dropped terms are below 2^-25 of a product), and
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
