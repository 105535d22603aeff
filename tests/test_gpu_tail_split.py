"""GPU: forward / dX GEMMs whose last round of tiles is cut along the reduction
(one piece per idle workgroup, partials summed in piece order): against
float64, run to run, against a call without a workspace, and under graph
replay with eager calls in between.

Bound as for the uncut GEMM, the order of a sum does not enter it:
(R + 8) 2^-24 sum |a||b|, then one rounding to p significant bits (2^-p of the
value; 2^-25 at fp16's subnormals)."""

import pytest
import torch

from nanotitan_amd import capi

pytestmark = pytest.mark.gpu

HALF_ULP = {torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11, torch.float32: 2.0**-24}
COUNTS = [200, 0, 129, 128, 300, 1, 0, 255, 77, 256, 90, 131, 140, 127, 2, 260, 130]  # mean 131


def _check(out, ref, mag, R, dtype):
    acc = (R + 8) * 2.0**-24 * mag
    bound = acc + HALF_ULP[dtype] * (ref.abs() + acc) + 2.0**-25
    assert bool(((out.cpu().double() - ref).abs() <= bound).all())


def _case(dtype, K, N, counts=COUNTS, seed=0):
    g = torch.Generator().manual_seed(seed + K + N)
    offs = torch.tensor([0, *torch.tensor(counts).cumsum(0).tolist()], dtype=torch.int32)
    A, E = sum(counts), len(counts)
    X = torch.randn(A, K, generator=g).to(dtype)
    W = torch.randn(E, K, N, generator=g).to(dtype)
    return offs, X, W, [(e, slice(int(offs[e]), int(offs[e + 1]))) for e in range(E)]


@pytest.mark.parametrize("dtype,K,N", [
    (torch.bfloat16, 4096, 64), (torch.float16, 4104, 264), (torch.bfloat16, 2056, 136),
    (torch.float32, 512, 130), (torch.float32, 1001, 64), (torch.bfloat16, 1365, 300)])
def test_tail_pieces(ext, dtype, K, N):
    offs, X, W, seg = _case(dtype, K, N)
    A, E = X.shape[0], W.shape[0]
    code = capi.dtype_code(dtype)
    assert capi.load().nt_grouped_gemm_tail_workspace_bytes(code, 0, E, A, K, N) > 0
    assert capi.load().nt_grouped_gemm_tail_workspace_bytes(code, 1, E, A, N, K) > 0
    og, Xg, Wg = offs.cuda(), X.cuda(), W.cuda()

    def rows(a, b):
        return torch.cat([a[s].double() @ b[e].double() for e, s in seg])

    ref, mag = rows(X, W), rows(X.abs(), W.abs())
    out = ext.grouped_gemm_kernel(Xg, og, Wg)
    _check(out, ref, mag, K, dtype)
    assert torch.equal(out, ext.grouped_gemm_kernel(Xg, og, Wg))
    # without a workspace: whole tiles
    whole = torch.empty_like(out)
    capi.call("nt_grouped_gemm", code, capi.ptr(Xg), capi.ptr(og), capi.ptr(Wg), E, A, K, N,
              capi.ptr(whole), None, 0, capi.current_stream())
    _check(whole, ref, mag, K, dtype)
    # dX of an up projection N -> K, one and two parts, alone and beside its dW
    Wt = W.transpose(1, 2).contiguous().cuda()  # [E, N, K]: dX = X @ Wt^T, N columns
    dX = ext.bwd_grouped_gemm_dX_kernel(Wt, og, Xg)
    _check(dX, ref, mag, K, dtype)
    H = torch.randn(A, N, generator=torch.Generator().manual_seed(1)).to(dtype).cuda()
    assert torch.equal(ext.bwd_grouped_gemm_dW_dX(H, Wt, og, Xg)[1], dX)
    G, V = (torch.randn(A, N, generator=torch.Generator().manual_seed(s)).to(dtype).cuda()
            for s in (2, 3))
    dH = ext.bwd_grouped_gemm_dX_gelu(Wt, og, Xg, H)
    assert torch.equal(dH, (dX.float() * H.float()).to(dtype))
    assert torch.equal(ext.bwd_grouped_gemm_dW_dX_gelu(H, Wt, og, Xg, H)[1], dH)
    dS = ext.bwd_grouped_gemm_dX_swiglu(Wt, og, Xg, G, V)
    for a, b in zip(ext.bwd_grouped_gemm_dW_dX_swiglu(H, Wt, og, Xg, G, V)[1:], dS):
        assert torch.equal(a, b)
    dX2 = ext.bwd_grouped_gemm_dX2(Wt, Wt, og, Xg, Xg)
    _check(dX2, 2 * ref, 2 * mag, 2 * K, dtype)
    assert torch.equal(ext.bwd_grouped_gemm_dW_dX2(H, Wt, Wt, og, Xg, Xg)[1], dX2)


@pytest.mark.parametrize("dtype,K,N", [(torch.bfloat16, 4096, 128), (torch.float32, 777, 130)])
def test_tail_pieces_under_graph_replay(ext, dtype, K, N):
    offs, X, W, _ = _case(dtype, K, N)
    og, Xg, Wg = offs.cuda(), X.cuda(), W.cuda()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        ext.grouped_gemm_kernel(Xg, og, Wg)
    torch.cuda.current_stream().wait_stream(s)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = ext.grouped_gemm_kernel(Xg, og, Wg)
    for seed in range(4):
        Xg.copy_(_case(dtype, K, N, seed=10 * seed)[1])
        graph.replay()
        eager = ext.grouped_gemm_kernel(Xg, og, Wg)
        torch.cuda.synchronize()
        assert torch.equal(out, eager), seed


@pytest.mark.parametrize("K,N", [(512, 130), (1001, 64)])
def test_tail_pieces_f32_special_values(ext, K, N):
    """The fp32 repair (non-finite results, operands below 2^-110) runs per piece:
    values of one k index each, so that other pieces of their tile are ordinary."""
    offs, X, W, seg = _case(torch.float32, K, N, seed=3)
    E, A = W.shape[0], X.shape[0]
    assert capi.load().nt_grouped_gemm_tail_workspace_bytes(capi.dtype_code(X.dtype), 0, E, A, K,
                                                            N) > 0
    W.clamp_(-0.9, 0.9)
    X[3, 5] = float("inf")
    X[131, K - 1] = float("nan")
    X[250, 7] = 3.4e38  # finite in fp32, rounds to infinity in bf16
    X[400] = torch.ldexp(X[400], torch.tensor(-120))
    out = ext.grouped_gemm_kernel(X.cuda(), offs.cuda(), W.cuda())
    out = out.cpu()
    ref = torch.cat([X[s].double() @ W[e].double() for e, s in seg])
    mag = torch.cat([X[s].double().abs() @ W[e].double().abs() for e, s in seg])
    assert torch.equal(torch.isnan(out), torch.isnan(ref))
    inf = torch.isinf(ref)
    assert torch.equal(torch.isinf(out), inf) and torch.equal(out[inf], ref[inf].float())
    ok = torch.isfinite(ref)
    err = (out.double() - ref).abs()
    assert bool((err[ok] <= (K + 8) * 2.0**-24 * mag[ok] + 2.0**-24 * ref[ok].abs()).all())


# (E, rows per expert, K = dX columns, N = reduction): the plain dX runs on
# 64-row tiles, on 128x256 ones (weights past 256 MiB), on 256x256 ones
WHOLE = [(32, 16, 768, 4096), (32, 64, 512, 8960), (17, 2892, 512, 2112)]


@pytest.mark.parametrize("E,rows,K,N", WHOLE)
def test_fused_dx_equals_dx_where_dx_is_not_cut(ext, E, rows, K, N):
    """The fused dX runs on other tiles there: it is not cut either."""
    g = torch.Generator(device="cuda").manual_seed(E + K)
    A = E * rows

    def randn(*shape):
        return torch.randn(shape, generator=g, device="cuda").to(torch.bfloat16)

    offs = torch.arange(0, A + 1, rows, dtype=torch.int32, device="cuda")
    W, D, H, V = randn(E, K, N), randn(A, N), randn(A, K), randn(A, K)
    G = torch.full_like(H, 64)  # silu(64) is 64: dvalue is 64 dX
    assert capi.load().nt_grouped_gemm_tail_workspace_bytes(capi.dtype_code(W.dtype), 1, E, A, K,
                                                            N) == 0
    dX = ext.bwd_grouped_gemm_dX_kernel(W, offs, D)
    dH = ext.bwd_grouped_gemm_dX_gelu(W, offs, D, H)
    assert torch.equal(dH, (dX.float() * H.float()).to(W.dtype))
    assert torch.equal(ext.bwd_grouped_gemm_dX_swiglu(W, offs, D, G, V)[1], 64 * dX)
    assert torch.equal(ext.bwd_grouped_gemm_dW_dX_gelu(H, W, offs, D, H)[1], dH)


@pytest.mark.parametrize("dtype,K,N", [(torch.bfloat16, 512, 4096), (torch.float32, 300, 1001)])
def test_dw_dx_follows_the_workspace_it_is_given(ext, dtype, K, N):
    """The C ABI's dW + dX call equals a dX without a workspace when it has the
    dW's alone (however large that is), and a dX with its own when it has both."""
    code, lib, s = capi.dtype_code(dtype), capi.load(), capi.current_stream()
    counts = [3900] + [350 + 11 * e for e in range(31)]  # more than 16: not paired
    E, A = len(counts), sum(counts)
    g = torch.Generator(device="cuda").manual_seed(K)
    offs = torch.tensor([0, *torch.tensor(counts).cumsum(0).tolist()], dtype=torch.int32,
                        device="cuda")

    def randn(*shape):
        return torch.randn(shape, generator=g, device="cuda").to(dtype)

    X, W, D = randn(A, K), randn(E, K, N), randn(A, N)
    dw = lib.nt_grouped_gemm_workspace_bytes(code, E, A, K, N)
    tail = lib.nt_grouped_gemm_tail_workspace_bytes(code, 1, E, A, K, N)
    assert tail > 0 and (dw > tail or dtype == torch.float32)
    ws = torch.empty(dw + 255 + tail, dtype=torch.uint8, device="cuda")

    def dx(size):
        out = torch.full_like(X, 7)
        capi.call("nt_grouped_gemm_dx", code, capi.ptr(W), capi.ptr(offs), capi.ptr(D), E, A, K,
                  N, capi.ptr(out), capi.ptr(ws) if size else None, size, s)
        return out

    def dw_dx(size):
        out, dW = torch.full_like(X, 7), torch.empty_like(W)
        capi.call("nt_grouped_gemm_dw_dx", code, capi.ptr(X), capi.ptr(W), capi.ptr(offs),
                  capi.ptr(D), E, A, K, N, capi.ptr(dW), capi.ptr(out), capi.ptr(ws), size, s)
        return out

    whole, cut = dx(0), dx(tail)
    assert not torch.equal(whole, cut)  # the sizes are cut
    assert torch.equal(dw_dx(dw), whole)
    assert torch.equal(dw_dx((dw + 255) // 256 * 256 + tail), cut)
    assert torch.equal(ext.bwd_grouped_gemm_dX_kernel(W, offs, D), cut)
    assert torch.equal(ext.bwd_grouped_gemm_dW_dX(X, W, offs, D)[1], cut)


UNEVEN = [1371, 0, 1203, 1280, 1, 2049, 1999, 1408, 900, 1155, 1666, 1537, 1024, 1290, 1811, 1300]


@pytest.mark.parametrize("dtype,op,K,N,scale", [
    (torch.bfloat16, "fwd", 4096, 512, 1), (torch.float16, "dx2", 512, 2048, 1.6),
    (torch.bfloat16, "dx2", 512, 2112, 1)])
def test_whole_tiles_then_pieces(ext, dtype, op, K, N, scale):
    """More tiles than workgroups: a workgroup multiplies whole tiles first and
    loads its piece of the last round behind their stores. The same bounds; the
    uncut tiles' bits; run to run; and under graph replay."""
    counts = [int(c * scale) for c in UNEVEN]
    E, A = len(counts), sum(counts)
    assert sum(-(-c // 128) for c in counts) * 4 > 512  # 512 columns; two workgroups per CU
    g = torch.Generator(device="cuda").manual_seed(N)
    offs = torch.tensor([0, *torch.tensor(counts).cumsum(0).tolist()], dtype=torch.int32,
                        device="cuda")
    seg = [(e, slice(int(offs[e]), int(offs[e + 1]))) for e in range(E)]
    R = K if op == "fwd" else N  # reduction of one part

    def randn(*shape):
        return torch.randn(shape, generator=g, device="cuda").to(dtype)

    a = [randn(A, R) for _ in range(1 if op == "fwd" else 2)]
    W = [randn(E, K, N) for _ in a]

    def call():
        if op == "fwd":
            return ext.grouped_gemm_kernel(a[0], offs, W[0])
        return ext.bwd_grouped_gemm_dX2(*W, offs, *a)

    whole = call()
    args = [capi.dtype_code(dtype)]
    if op == "fwd":
        args += [capi.ptr(a[0]), capi.ptr(offs), capi.ptr(W[0])]
    else:
        args += [capi.ptr(W[0]), capi.ptr(W[1]), capi.ptr(offs), capi.ptr(a[0]), capi.ptr(a[1])]
    capi.call("nt_grouped_gemm" if op == "fwd" else "nt_grouped_gemm_dx2", *args, E, A, K, N,
              capi.ptr(whole), None, 0, capi.current_stream())

    out = call()
    assert not torch.equal(out, whole)  # some tiles are cut
    assert float((out == whole).float().mean()) > 0.9  # single roundings differ

    def rows(f):
        return torch.cat([sum(f(x[s].double()) @ f(w[e].double() if op == "fwd" else
                                                  w[e].double().t().contiguous())
                              for x, w in zip(a, W)) for e, s in seg]).cpu()

    ref, mag = rows(lambda t: t), rows(torch.abs)
    _check(out, ref, mag, R * len(a), dtype)
    _check(whole, ref, mag, R * len(a), dtype)
    assert torch.equal(call(), out)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        again = call()
    for _ in range(3):
        a[0].copy_(randn(A, R))
        graph.replay()
        eager = call()
        torch.cuda.synchronize()
        assert torch.equal(again, eager)


@pytest.mark.parametrize("dtype,K,N", [(torch.bfloat16, 4096, 136), (torch.float32, 512, 130),
                                       (torch.bfloat16, 1365, 300)])
def test_fused_forward_holds_the_bits_of_whole_tiles(ext, dtype, K, N):
    """An up projection narrower than its input: the plain forward is cut with a
    workspace, the fused ones never are."""
    offs, X, W, _ = _case(dtype, K, N)
    A, E = X.shape[0], W.shape[0]
    og, Xg, Wg = offs.cuda(), X.cuda(), W.cuda()
    Vg = Wg.flip(2).contiguous()

    def whole(w):
        out = torch.empty(A, N, dtype=dtype, device="cuda")
        capi.call("nt_grouped_gemm", capi.dtype_code(dtype), capi.ptr(Xg), capi.ptr(og),
                  capi.ptr(w), E, A, K, N, capi.ptr(out), None, 0, capi.current_stream())
        return out

    assert not torch.equal(ext.grouped_gemm_kernel(Xg, og, Wg), whole(Wg))  # cut
    _, gate, value = ext.grouped_gemm_swiglu(Xg, og, Wg, Vg)
    assert torch.equal(gate, whole(Wg)) and torch.equal(value, whole(Vg))
