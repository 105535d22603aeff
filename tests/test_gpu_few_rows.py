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


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("K,N", [(64, 128), (8, 136), (200, 264), (72, 8456)])
def test_few_rows_per_expert(ext, dtype, K, N):
    g = torch.Generator().manual_seed(K + N)
    E, A = len(COUNTS), sum(COUNTS)
    assert A <= 32 * E  # the 64-row rule; N = 8456 takes its 256-column form
    offs = torch.tensor([0, *torch.tensor(COUNTS).cumsum(0).tolist()], dtype=torch.int32)
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
