"""GPU: token segments of the token-id surface (combine, pack backward) at the
edges of their row batches: fan-ins of 0, one batch (2 or 8 rows) and one more,
the LDS-sorted limit (256) and past it, and token ids out of range."""

import numpy as np
import pytest
import torch

from oracle import moe_oracle as O
from tests.test_gpu_dispatch import bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("pad", [0, 2000])  # empty tokens: mean fan-in above / below 2
@pytest.mark.parametrize("d", [24, 600])
def test_token_segments(ext, dtype, pad, d):
    g = torch.Generator().manual_seed(d + pad)
    fan = [0, 1, 2, 3, 0, 7, 8, 9, 64, 65, 255, 256, 257, 700] + [0] * pad
    T = len(fan)
    tid = torch.cat([torch.full((n,), t, dtype=torch.int32) for t, n in enumerate(fan)])
    tid = torch.cat([tid, torch.tensor([-1, T, T + 5], dtype=torch.int32)])
    A = tid.numel()
    tid = tid[torch.randperm(A, generator=g)].contiguous()
    y = torch.randn(A, d, generator=g).to(dtype)
    w = torch.randn(A, generator=g)
    out = ext.combine_tokens_kernel(y.cuda(), tid.cuda(), w.cuda(), T, d)
    assert torch.equal(bits(out), bits(torch.from_numpy(O.combine_tokens(y, tid, w, T))))

    # pack backward: every row's gradient, ascending packed order; gate
    # gradients to the first slot of the row's expert
    topk = torch.stack([torch.randperm(6, generator=g)[:3] for _ in range(T)]).to(torch.int32)
    expert = torch.randint(0, 6, (A,), generator=g, dtype=torch.int32)
    dX, dw = ext.pack_kernel_backward(y.cuda(), w.cuda(), tid.cuda(), expert.cuda(), topk.cuda())
    ref = torch.zeros(T, d, dtype=torch.float32)
    dwr = torch.zeros(T, 3, dtype=torch.float32)
    for p in range(A):
        t = int(tid[p])
        if 0 <= t < T:
            ref[t] += y[p].float()
            for j in range(3):
                if topk[t, j] == expert[p]:
                    dwr[t, j] += w[p]
                    break
    assert torch.equal(dX.cpu(), ref.to(dtype))
    assert torch.equal(dw.cpu(), dwr)


# more than 256 rows a token (sorted by a wave): two passes of the sort up to
# 65,536 rows in all, four above; lengths at the edges of its rounds of 256
@pytest.mark.parametrize("fan", [
    [257, 511, 512, 513, 0, 1, 1000], [65536 - 300, 300], [65536 - 300, 301],
    [300] * 90 + [5000, 257], [70000, 3, 40000]])
def test_long_token_segments(ext, fan):
    g = torch.Generator().manual_seed(len(fan))
    T, d = len(fan), 8
    tid = torch.repeat_interleave(torch.arange(T, dtype=torch.int32), torch.tensor(fan))
    A = tid.numel()
    tid = tid[torch.randperm(A, generator=g)].contiguous()
    y = torch.randn(A, d, generator=g)
    w = torch.randn(A, generator=g)
    out = ext.combine_tokens_kernel(y.cuda(), tid.cuda(), w.cuda(), T, d).cpu()
    expert = torch.zeros(A, dtype=torch.int32)
    dX, dw = ext.pack_kernel_backward(y.cuda(), w.cuda(), tid.cuda(), expert.cuda(),
                                      torch.zeros(T, 1, dtype=torch.int32, device="cuda"))
    dX, dw = dX.cpu(), dw.cpu()
    for t in range(T):  # sequential fp32 sums in ascending packed order
        rows = (tid == t).nonzero().flatten()
        assert len(rows) == fan[t]
        if fan[t] == 0:
            assert not out[t].any() and not dX[t].any() and not dw[t].any()
            continue
        yr, wr = y[rows].numpy(), w[rows].numpy()
        assert np.array_equal(out[t].numpy(), np.cumsum(wr[:, None] * yr, axis=0)[-1])
        assert np.array_equal(dX[t].numpy(), np.cumsum(yr, axis=0)[-1])
        assert np.array_equal(dw[t].numpy(), np.cumsum(wr)[-1:])
