"""GPU: grouped GEMMs of few rows per expert (64-row tiles) at the tile edges,
against float64. Bound as for any 16-bit GEMM here: (R + 8) 2^-24 sum |a||b| of
fp32 accumulation, then one rounding to p significant bits (2^-p of the value;
2^-25 at fp16's subnormals)."""

import pytest
import torch

pytestmark = pytest.mark.gpu

HALF_ULP = {torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11}
COUNTS = [0, 1, 63, 64, 65, 0, 7, 16, 17, 3, 130, 2]  # mean 30.7


def _check(out, ref, mag, R, dtype):
    acc = (R + 8) * 2.0**-24 * mag
    bound = acc + HALF_ULP[dtype] * (ref.abs() + acc) + 2.0**-25
    assert bool(((out.cpu().double() - ref).abs() <= bound).all())


MID = [0, 127, 128, 129, 64, 200, 1, 100]  # mean 93.6


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("counts,K,N", [
    (COUNTS, 64, 128), (COUNTS, 8, 136), (COUNTS, 200, 264), (COUNTS, 72, 8456),
    # 128-row SwiGLU tiles; with weights past 256 MB the plain ones too
    (MID, 136, 264), (MID, 200, 88000)])
def test_few_rows_per_expert(ext, dtype, counts, K, N):
    g = torch.Generator().manual_seed(K + N)
    E, A = len(counts), sum(counts)
    # the 64-row rule (N = 8456 takes its 256-column form), the 128-row rule
    assert A <= 32 * E if counts is COUNTS else 48 * E < A <= 112 * E
    if N == 88000:  # few columns are compared: the rest is the same tile again
        return _wide(ext, dtype, counts, K, N, g)
    offs = torch.tensor([0, *torch.tensor(counts).cumsum(0).tolist()], dtype=torch.int32)
    X = torch.randn(A, K, generator=g).to(dtype)
    W = torch.randn(E, K, N, generator=g).to(dtype)
    V = torch.randn(E, K, N, generator=g).to(dtype)
    D = torch.randn(A, N, generator=g).to(dtype)
    Xg, Wg, Vg, Dg, og = (t.cuda() for t in (X, W, V, D, offs))
    seg = [(e, slice(int(offs[e]), int(offs[e + 1]))) for e in range(E)]

    def rows(a, b):
        return torch.cat([a[s].double() @ b[e].double() for e, s in seg])

    fwd = ext.grouped_gemm_kernel(Xg, og, Wg)
    _check(fwd, rows(X, W), rows(X.abs(), W.abs()), K, dtype)
    Wt = W.transpose(1, 2)
    dX = ext.bwd_grouped_gemm_dX_kernel(Wg, og, Dg)
    _check(dX, rows(D, Wt), rows(D.abs(), Wt.abs()), N, dtype)
    act, dact = ext.grouped_gemm_gelu(Xg, og, Wg)
    h = fwd.cpu().double().requires_grad_()
    (dg,) = torch.autograd.grad(torch.nn.functional.gelu(h).sum(), h)
    tol = dict(rtol=2 * HALF_ULP[dtype], atol=1e-6)
    torch.testing.assert_close(act.cpu().double(), torch.nn.functional.gelu(h).detach(), **tol)
    torch.testing.assert_close(dact.cpu().double(), dg, **tol)
    hid, gate, val = ext.grouped_gemm_swiglu(Xg, og, Wg, Vg)
    assert torch.equal(gate, fwd) and torch.equal(val, ext.grouped_gemm_kernel(Xg, og, Vg))
    silu = torch.nn.functional.silu(gate.float()).to(dtype).float()
    torch.testing.assert_close(hid.float(), silu * val.float(), rtol=6 * HALF_ULP[dtype], atol=1e-6)


def _wide(ext, dtype, counts, K, N, g):
    E, A = len(counts), sum(counts)
    offs = torch.tensor([0, *torch.tensor(counts).cumsum(0).tolist()], dtype=torch.int32)
    X = torch.randn(A, K, generator=g).to(dtype)
    W = torch.empty(E, K, N, dtype=dtype, device="cuda").normal_()
    D = torch.empty(A, N, dtype=dtype, device="cuda").normal_()
    cols = torch.tensor([0, 1, 255, 256, 511, 40000, N - 257, N - 256, N - 2, N - 1])
    Wc = W[:, :, cols.cuda()].cpu()
    seg = [(e, slice(int(offs[e]), int(offs[e + 1]))) for e in range(E)]

    def rows(a, b):
        return torch.cat([a[s].double() @ b[e].double() for e, s in seg])

    fwd = ext.grouped_gemm_kernel(X.cuda(), offs.cuda(), W)
    _check(fwd[:, cols.cuda()], rows(X, Wc), rows(X.abs(), Wc.abs()), K, dtype)
    act, _ = ext.grouped_gemm_gelu(X.cuda(), offs.cuda(), W)
    h = fwd[:, cols.cuda()].cpu().double()
    torch.testing.assert_close(act[:, cols.cuda()].cpu().double(), torch.nn.functional.gelu(h),
                               rtol=2 * HALF_ULP[dtype], atol=1e-6)
    dX = ext.bwd_grouped_gemm_dX_kernel(W, offs.cuda(), D)
    Wd, Dd = W.double(), D.double()
    ref = torch.cat([Dd[s] @ Wd[e].t().contiguous() for e, s in seg]).cpu()
    mag = torch.cat([Dd[s].abs() @ Wd[e].abs().t().contiguous() for e, s in seg]).cpu()
    _check(dX, ref, mag, N, dtype)
