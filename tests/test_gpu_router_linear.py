"""GPU: the router's statistics and linear backward against float64, and the
layer's single router pass against the two-pass dataflow it replaces.

Bounds: a sum of n fp32 products in any order errs by at most
(n + 8) 2^-24 sum |a||b|; dx is then rounded to p significant bits (2^-p of its
value, 2^-25 at fp16's subnormals). Probabilities come from one fp32 softmax
(a few 2^-24 each), means and sums over T of them."""

from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu

HALF_ULP = {torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11, torch.float32: 2.0**-24}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("T,E,d", [(1, 1, 1), (5, 3, 7), (64, 8, 64), (65, 16, 130),
                                   (257, 17, 1031), (1000, 32, 300), (40000, 9, 36)])
def test_router_linear_backward(ext, dtype, T, E, d):
    g = torch.Generator().manual_seed(T + E + d)
    x = torch.randn(T, d, generator=g).to(dtype)
    W, dl, da = (torch.randn(*s, generator=g) for s in ((E, d), (T, E), (T, E)))
    xg, Wg, dlg, dag = (t.cuda() for t in (x, W, dl, da))
    xd, Wd = x.double(), W.double()
    for a, b in ((dlg, dag), (dlg, None), (None, dag)):
        dx, dW = ext.router_linear_backward(xg, Wg, a, b, a is not None, True)
        gw = sum(t.cpu().double() for t in (a, b) if t is not None)
        mag = gw.abs().t() @ xd.abs()
        assert bool(((dW.cpu().double() - gw.t() @ xd).abs() <= (T + 8) * 2.0**-24 * mag).all())
        if a is None:
            assert dx is None
            continue
        ref, mag = dl.double() @ Wd, dl.double().abs() @ Wd.abs()
        acc = (E + 8) * 2.0**-24 * mag
        bound = acc + HALF_ULP[dtype] * (ref.abs() + acc) + 2.0**-25
        assert bool(((dx.cpu().double() - ref).abs() <= bound).all())
    assert ext.router_linear_backward(xg, Wg, dlg, dag, True, False)[1] is None


@pytest.mark.parametrize("T,E", [(1, 1), (3, 2), (100, 64), (257, 65), (5000, 16), (30, 1024),
                                 (9000, 200)])
def test_router_stats(ext, T, E):
    g = torch.Generator().manual_seed(T + E)
    z = 3 * torch.randn(T, E, generator=g)
    counts = torch.randint(0, 50, (E,), generator=g, dtype=torch.int32)
    counts[0] = 1
    coef = 0.01 * E
    total, frac, mean, aux = ext.router_stats(z.cuda(), counts.cuda(), coef)
    zd = z.double().requires_grad_()
    mean_ref = zd.softmax(-1).mean(0)
    frac_ref = counts.double() / counts.sum()
    aux_ref = coef * (frac_ref * mean_ref).sum()
    assert total.dtype == torch.int64 and int(total) == int(counts.sum())
    torch.testing.assert_close(frac.cpu(), frac_ref.float(), rtol=2.0**-23, atol=0)
    # 2^-24 for each of exp's argument (|z - max| < 32: 2^-19), exp and division
    tol = dict(rtol=2.0**-18 + T * 2.0**-24, atol=0)
    torch.testing.assert_close(mean.cpu().double(), mean_ref.detach(), **tol)
    torch.testing.assert_close(aux.cpu().double(), aux_ref.detach(), **tol)
    dmean = torch.randn(E, generator=g)
    for da, dm in ((2.0, dmean), (2.0, None), (None, dmean)):
        out = ((da or 0.0) * aux_ref + (0.0 if dm is None else (dm.double() * mean_ref).sum()))
        (ref,) = torch.autograd.grad(out, zd, retain_graph=True)
        got = ext.router_stats_backward(z.cuda(), frac, None if da is None else torch.tensor(
            da, device="cuda"), None if dm is None else dm.cuda(), coef)
        # p (v - sum p v): absolute error of a few ulps of |v| p
        scale = float((2 * coef * frac_ref.max() + dmean.abs().max()) / T)
        torch.testing.assert_close(got.cpu().double(), ref, rtol=1e-5, atol=4e-6 * scale)


@pytest.mark.parametrize("E", [8, 40])  # one fused pass / two passes in training
def test_single_router_pass_matches_two_passes(ext, E):
    """A forward hook on the router makes the layer take the two-pass dataflow;
    values and gradients agree, with and without gradients, and the aux loss
    can be differentiated twice."""
    from nanotitan_amd.layer import MoE

    cfg = SimpleNamespace(d_model=48, num_experts=E, top_k=2, ffn_in=64, dtype=torch.float32,
                          moe_router_dtype=torch.float32, moe_backend="hip", router_alpha=0.01)
    torch.manual_seed(3)
    moe = MoE(cfg).cuda()
    for p in moe.experts.parameters():
        p.data.normal_(0, 0.1)
    x = torch.randn(2, 37, 48, device="cuda")
    names = ("tokens_per_expert", "probs_per_expert", "total_assignments", "ass_frac_per_expert",
             "aux_loss")

    def run(grad):
        with torch.set_grad_enabled(grad):
            xi = x.clone().requires_grad_(grad)
            y, st = moe(xi)
            outs = [y, *(getattr(st, n) for n in names)]
            assert st.num_tokens == 74
            if grad:
                outs += torch.autograd.grad(y.square().sum() + 5 * st.aux_loss
                                            + st.probs_per_expert.square().sum(),
                                            [xi, *moe.parameters()])
        return outs

    def second():
        _, st = moe(x.clone().requires_grad_())
        (g1,) = torch.autograd.grad(st.aux_loss, moe.router.weight, create_graph=True)
        return torch.autograd.grad(g1.square().sum(), moe.router.weight)

    fused = [run(True), run(False), second()]
    h = moe.router.register_forward_hook(lambda *a: None)
    plain = [run(True), run(False), second()]
    h.remove()
    for a, b in zip(fused, plain):
        for u, v in zip(a, b):
            assert u.dtype == v.dtype and u.shape == v.shape
            torch.testing.assert_close(u, v, rtol=2e-5, atol=2e-6)


def _moe(E, dtype=torch.float32, d=48):
    from nanotitan_amd.layer import MoE

    cfg = SimpleNamespace(d_model=d, num_experts=E, top_k=2, ffn_in=64, dtype=dtype,
                          moe_router_dtype=torch.float32, moe_backend="hip", router_alpha=0.01)
    torch.manual_seed(4)
    moe = MoE(cfg).cuda()
    for p in moe.experts.parameters():
        p.data.normal_(0, 0.1)
    return moe, torch.randn(2, 37, d, device="cuda").to(dtype)


@pytest.mark.parametrize("E", [8, 40])  # one pass / two passes in training
def test_loss_and_output_have_graphs_of_their_own(ext, E):
    moe, x = _moe(E)
    params = list(moe.parameters())
    y, st = moe(x.requires_grad_())
    together = torch.autograd.grad([y.square().sum() + st.aux_loss], [x, *params])
    for first in ("loss", "output"):
        y, st = moe(x)
        parts = [st.aux_loss, y.square().sum()]
        for p in (x, *params):
            p.grad = None
        for part in parts if first == "loss" else parts[::-1]:
            part.backward()  # without retain_graph
        for p, g in zip((x, *params), together):
            torch.testing.assert_close(p.grad, g, rtol=2e-5, atol=2e-6)
    # the loss reaches the router's weight alone
    _, st = moe(x)
    assert torch.autograd.grad(st.aux_loss, x, allow_unused=True, retain_graph=True)[0] is None
    moe.router.weight.requires_grad_(False)
    y, st = moe(x)
    assert y.requires_grad and not st.aux_loss.requires_grad
    assert not st.probs_per_expert.requires_grad


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_tokens_may_be_overwritten_after_the_forward(ext, dtype):
    """An in-place residual: the layer keeps the cast tokens, not x."""
    moe, x = _moe(8, dtype)
    params = list(moe.parameters())

    def step(in_place):
        leaf = x.clone().requires_grad_()
        h = leaf * 1
        y, st = moe(h)
        if in_place:
            h += y
        else:
            h = h + y
        return torch.autograd.grad(h.float().square().sum() + st.aux_loss, [leaf, *params])

    for a, b in zip(step(True), step(False)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,E,d,shift", [(5, 3, 7, 0), (65, 16, 130, 0), (130, 17, 64, 1)])
def test_router_linear_backward_from_float32(ext, dtype, T, E, d, shift):
    """x in float32, dx in the tokens' type: the bits of x in that type. Off
    8-byte alignment (shift) one column a thread divides the tokens otherwise,
    so dW is summed in another order: the bound of a sum of T products."""
    g = torch.Generator().manual_seed(T)
    x = torch.randn(T, d, generator=g).to(dtype)
    W, dl = torch.randn(E, d, generator=g).cuda(), torch.randn(T, E, generator=g).cuda()
    buf = torch.empty(T * d + shift, device="cuda")
    buf[shift:] = x.float().reshape(-1).cuda()
    got = ext.router_linear_backward(buf[shift:].view(T, d), W, dl, None, True, True, dtype)
    ref = ext.router_linear_backward(x.cuda(), W, dl, None, True, True)
    assert got[0].dtype == dtype
    assert torch.equal(got[0], ref[0])
    if shift == 0:
        assert torch.equal(got[1], ref[1])
    dld, xd = dl.cpu().double(), x.double()
    bound = (T + 8) * 2.0**-24 * (dld.abs().t() @ xd.abs())
    assert bool(((got[1].cpu().double() - dld.t() @ xd).abs() <= bound).all())
    with pytest.raises(RuntimeError):  # only float32 tokens may differ from their gradient
        ext.router_linear_backward(x.cuda(), W, dl, None, True, True, torch.float32)


class _Doubled(torch.nn.Linear):
    def forward(self, x):
        return 2 * super().forward(x)


@pytest.mark.parametrize("change", ["none", "bias", "subclass", "bf16", "pre_hook", "backward_hook",
                                    "backward_pre_hook", "global_hook", "instance_forward",
                                    "autocast", "tensor_weight"])
def test_only_a_plain_router_runs_once(ext, change):
    """Any other router is called, twice, and its statistics are torch's."""
    from nanotitan_amd.layer import _plain_router

    moe, x = _moe(8)
    r, handle, context = moe.router, None, torch.no_grad()
    if change == "bias":
        r.bias = torch.nn.Parameter(torch.randn(8, device="cuda"))
    elif change == "subclass":
        r.__class__ = _Doubled
    elif change == "bf16":
        r.to(torch.bfloat16)
    elif change == "pre_hook":
        handle = r.register_forward_pre_hook(lambda m, a: (a[0] * 3,))
    elif change == "backward_hook":
        handle = r.register_full_backward_hook(lambda *a: None)
    elif change == "backward_pre_hook":
        handle = r.register_full_backward_pre_hook(lambda *a: None)
    elif change == "global_hook":
        handle = torch.nn.modules.module.register_module_forward_hook(lambda *a: None)
    elif change == "instance_forward":
        r.forward = lambda t: torch.nn.functional.linear(t, r.weight) * 2
    elif change == "autocast":
        context = torch.autocast("cuda", dtype=torch.bfloat16)
    elif change == "tensor_weight":
        del r._parameters["weight"]
        r.weight = torch.randn(8, 48, device="cuda")
    try:
        flat = x.reshape(-1, 48)
        with context:
            assert _plain_router(r, flat) == (change == "none")
            _, st = moe(x)
            probs = r(flat.to(r.weight.dtype)).softmax(dim=-1).float().mean(dim=0)
        # the router's own logits: bf16 ones (and their mean) round to 8 bits
        low = change in ("bf16", "autocast")
        torch.testing.assert_close(st.probs_per_expert.float(), probs,
                                   rtol=2.0**-7 if low else 2e-5, atol=2.0**-9 if low else 1e-6)
        assert int(st.total_assignments) == 2 * flat.shape[0]
    finally:
        if handle is not None:
            handle.remove()
