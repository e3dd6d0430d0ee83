"""GPU parity of the dense parts of a training step: sdm_rt_weight_grad, sdm_rt_rms_norm_backward and
core.MixerFunction, against float64 on the same values and against the op-by-op training path.
"""
import math

import pytest
import torch

from sdmchat_amd import RunTimeSdm, TrainedSdm, core
from tests._gpu_util import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,n,k", [
    (1, 8, 8), (63, 136, 24), (64, 128, 128), (65, 40, 264),        # a step's edge, narrow tiles
    (255, 256, 256), (257, 264, 256), (12289, 264, 512),            # 256-wide tiles, their remainders, several splits
    (16384, 768, 768), (4000, 32, 768),
])
def test_weight_grad_matches_float64(rows, n, k):
    """Every output within the bound of a float32 sum of its products in any order: rows * 2^-24 times the sum of their
    magnitudes."""
    say(f"[weight grad] rows={rows} n={n} k={k}")
    g = torch.Generator(device="cuda").manual_seed(rows)
    wide = torch.randn(rows, n + 8, generator=g, device="cuda").bfloat16()   # a row stride of its own
    dy, x = wide[:, 8:], torch.randn(rows, k, generator=g, device="cuda").bfloat16()
    got = core.weight_grad(dy, x).double()
    ref = dy.double().t() @ x.double()
    bound = (rows + 1) * 2.0 ** -24 * (dy.double().abs().t() @ x.double().abs())
    assert bool(((got - ref).abs() <= bound).all())
    assert torch.equal(core.weight_grad(dy, x).double(), got)


def test_weight_grad_takes_unaligned_rows():
    g = torch.Generator(device="cuda").manual_seed(1)
    dy = torch.randn(70, 41, generator=g, device="cuda").bfloat16()[:, 1:]
    x = torch.randn(70, 24, generator=g, device="cuda").bfloat16()
    assert torch.equal(core.weight_grad(dy, x), core.weight_grad(dy.contiguous(), x))


@pytest.mark.parametrize("rows,d", [(1, 8), (7, 64), (9, 256), (33, 264), (4100, 768), (5, 1160), (3, 2048), (2, 2056)])
@pytest.mark.parametrize("xt,yt", [(torch.float32, torch.float32), (torch.float32, torch.bfloat16),
                                   (torch.bfloat16, torch.float32), (torch.bfloat16, torch.bfloat16)])
def test_rms_norm_backward_matches_float64(rows, d, xt, yt):
    """float32 arithmetic on up to 2,048 values a row: 1e-5 of the largest entry (d * 2^-24 = 1.2e-4 would be the worst
    case of every rounding alike), dx in bfloat16 plus half its ulp."""
    g = torch.Generator(device="cuda").manual_seed(d)
    x = torch.randn(rows, d, generator=g, device="cuda").to(xt)
    w = 1 + 0.3 * torch.randn(d, generator=g, device="cuda")
    dy = torch.randn(rows, d, generator=g, device="cuda").to(yt)
    dx, dw = core.rms_norm_backward(x, w, dy, 1e-6)
    x64, w64 = x.double().requires_grad_(True), w.double().requires_grad_(True)
    (x64 * torch.rsqrt(x64.square().mean(-1, keepdim=True) + 1e-6) * w64).backward(dy.double())
    tol = 1e-5 * x64.grad.abs().max() + (2.0 ** -8 * x64.grad.abs() if xt == torch.bfloat16 else 0.0)
    assert dx.dtype == xt and bool(((dx.double() - x64.grad).abs() <= tol).all())
    assert (dw.double() - w64.grad).abs().max() <= 1e-5 * w64.grad.abs().max()
    assert core.rms_norm_backward(x, w, dy, 1e-6, need_w=False)[1] is None
    assert torch.equal(core.rms_norm_backward(x, w, dy, 1e-6, need_x=False)[1], dw)


@pytest.mark.parametrize("amp,gate,reset,frozen", [
    (True, True, False, ()), (False, True, True, ()), (True, False, True, ("wk", "norm")), (False, False, False, ("wv",)),
])
def test_mixer_function_equals_the_op_by_op_path(amp, gate, reset, frozen):
    """The same forward bits; gradients within the compute type's rounding: each side rounds the projections' input
    gradient (and, op by op, each weight gradient) once or twice more, 2^-8 of a value in bfloat16, so 2e-2 of the
    largest entry there and 1e-5 in float32."""
    torch.manual_seed(3)
    B, T, d, H = 3, 130, 96, 4
    m = RunTimeSdm(d, heads=H, n_sub=8, d_a=16, k=8, decays=(0.6, 0.8, 0.95, 0.99), learn_decay=True, write_gate=gate,
                   addr_bias=0.2, mem_in_grad=0.5).to("cuda").train()
    for n, p in m.named_parameters():
        if n.split(".")[0] in frozen:
            p.requires_grad_(False)
    x = torch.randn(B, d, T, device="cuda").transpose(1, 2)   # not contiguous
    rs = torch.rand(B, T, device="cuda") < 0.05 if reset else None
    dy = torch.randn(B, T, d, device="cuda")

    def step(fits):
        keep, core.mixer_train_fits = core.mixer_train_fits, fits or core.mixer_train_fits
        try:
            xg = x.detach().clone().requires_grad_(True)
            with torch.autocast("cuda", dtype=torch.bfloat16, enabled=amp):
                y = m(xg, rs)
            ps = {n: p for n, p in m.named_parameters() if p.requires_grad}
            gs = torch.autograd.grad(y, [xg] + list(ps.values()), dy, allow_unused=True)
            return y, dict(zip(["x"] + list(ps), gs)), m.last_gate
        finally:
            core.mixer_train_fits = keep
    y1, g1, gate1 = step(None)
    y0, g0, gate0 = step(lambda *a: None)
    assert torch.equal(y1, y0) and torch.equal(gate1, gate0)
    for n in g0:
        assert (g0[n] is None) == (g1[n] is None), n
        if g0[n] is None:
            continue
        assert g1[n].dtype == g0[n].dtype and g1[n].shape == g0[n].shape, n
        err = (g1[n] - g0[n]).abs().max().item()
        scale = g0[n].abs().max().item()
        say(f"  d{n}: {err:.2e} of {scale:.2e}")
        assert err <= (2e-2 if amp else 1e-5) * max(scale, 1e-2), n


def test_hooks_on_the_output_map_still_run():
    m = RunTimeSdm(64, heads=2, n_sub=8, d_a=16, k=4, decays=(0.5, 0.9)).to("cuda").train()
    t = TrainedSdm(64, 8, heads=2, d_a=8, k=4).to("cuda").train()
    seen = []
    hooks = [mod.wo.register_forward_hook(lambda *a: seen.append(1)) for mod in (m, t)]
    x = torch.randn(2, 40, 64, device="cuda", requires_grad=True)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        (m(x) + t(x)).float().sum().backward()
    assert len(seen) == 2 and bool(torch.isfinite(x.grad).all())
    for h in hooks:
        h.remove()


def test_offloaded_saved_tensors_give_the_same_gradients():
    """Saved-tensor hooks see every tensor the mixer keeps: gradients from tensors offloaded to the host and back."""
    m = RunTimeSdm(64, heads=2, n_sub=8, d_a=16, k=4, decays=(0.5, 0.9)).to("cuda").train()
    x = torch.randn(2, 70, 64, device="cuda", requires_grad=True)
    torch.nn.init.xavier_uniform_(m.wo.weight)
    grads = []
    for off in (False, True):
        with torch.autograd.graph.saved_tensors_hooks(lambda v: v.cpu() if off else v, lambda v: v.cuda()):
            y = m(x)
        grads.append(torch.autograd.grad(y.square().sum(), [x] + list(m.parameters())))
    assert all(torch.equal(a, b) for a, b in zip(*grads)) and math.isfinite(grads[0][0].sum().item())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_norm_and_weight_gradients_of_broadcast_rows(dtype):
    """Gradients whose rows are one row repeated (stride 0, as a sum over tokens leaves them) equal those of the rows
    written out, as do inputs of such rows."""
    g = torch.Generator(device="cuda").manual_seed(4)
    x = torch.randn(3, 7, 64, generator=g, device="cuda").to(dtype).requires_grad_(True)
    w = torch.rand(64, generator=g, device="cuda").requires_grad_(True)
    v = torch.randn(64, generator=g, device="cuda").to(dtype)
    one = torch.randn(64, generator=g, device="cuda").to(dtype)
    for xi in (x, one.expand(3, 7, 64).requires_grad_(True)):
        y = core.RmsNormFunction.apply(xi, w, 1e-6, dtype)
        got = torch.autograd.grad(y, (xi, w), v.expand(3, 7, 64), retain_graph=True)
        want = torch.autograd.grad(y, (xi, w), v.expand(3, 7, 64).contiguous())
        assert all(torch.equal(a, b) for a, b in zip(got, want))
    if dtype == torch.bfloat16:
        x2 = x.detach().view(21, 64)
        for a, b in ((v.expand(21, 64), x2), (x2, one.expand(21, 64))):
            assert torch.equal(core.weight_grad(a, b), core.weight_grad(a.contiguous(), b.contiguous()))


@pytest.mark.parametrize("amp,dtype", [(True, torch.bfloat16), (True, torch.float32), (False, torch.float32)])
def test_training_steps_on_pooled_sums_and_broadcast_inputs(amp, dtype):
    """sum over tokens as the loss (its gradient has rows of stride 0), inputs of broadcast rows and inputs that start on
    no 16 bytes give what dense ones give."""
    torch.manual_seed(5)
    m = RunTimeSdm(64, heads=2, n_sub=8, d_a=16, k=4, decays=(0.5, 0.9)).to("cuda").train()
    t = TrainedSdm(64, 8, heads=2, d_a=8, k=4).to("cuda").train()
    torch.nn.init.xavier_uniform_(m.wo.weight)
    torch.nn.init.normal_(t.values)
    buf = torch.randn(2 * 70 * 64 + 1, device="cuda").to(dtype)
    inputs = [buf[1:].view(2, 70, 64), torch.randn(64, device="cuda").to(dtype).expand(2, 70, 64)]
    v = torch.randn(64, device="cuda").to(dtype)
    for mod in (m, t):
        for x in inputs:
            res = []
            for xi, dy in ((x, v.expand(2, 70, 64)), (x.clone(), v.expand(2, 70, 64).contiguous())):
                xi = xi.detach().requires_grad_(True)
                with torch.autocast("cuda", dtype=torch.bfloat16, enabled=amp):
                    y = mod(xi)
                res.append((y, *torch.autograd.grad(y, [xi, *mod.parameters()], dy, allow_unused=True)))
            for a, b in zip(*res):   # without autocast wo's gradients are the library's, in an order of its own by strides
                assert (a is None and b is None) or torch.equal(a, b) or (
                    not amp and (a - b).abs().max() <= 140 * 2.0 ** -24 * b.abs().max())


@pytest.mark.parametrize("d", [64, 768])
def test_the_norm_differentiates_twice(d):
    """The gradients of RmsNormFunction's gradients, against float64: sums of d float32 products in chains of four."""
    g = torch.Generator(device="cuda").manual_seed(d)
    x, dy, a = (torch.randn(3, 5, d, generator=g, device="cuda") for _ in range(3))
    w, b = torch.rand(d, generator=g, device="cuda") + 0.5, torch.randn(d, generator=g, device="cuda")

    def twice(norm, cast):
        xs, ws, ds = (cast(t).requires_grad_(True) for t in (x, w, dy))
        gx, gw = torch.autograd.grad(norm(xs, ws), (xs, ws), ds, create_graph=True)
        return torch.autograd.grad((gx * cast(a)).sum() + (gw * cast(b)).sum(), (xs, ws, ds))
    got = twice(lambda x, w: core.RmsNormFunction.apply(x, w, 1e-6, torch.float32), lambda t: t.clone())
    want = twice(lambda x, w: x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6) * w, lambda t: t.double())
    for p, q in zip(got, want):
        assert (p.double() - q).abs().max() <= 4 * d * 2.0 ** -24 * q.abs().max()


def test_the_output_map_differentiates_twice():
    """The gradients of an autocast map's gradients equal those of the module called op by op: the same products, the
    weight gradient not rounded to bfloat16 on its way (2^-8 of a value a rounding)."""
    g = torch.Generator(device="cuda").manual_seed(6)
    lin = torch.nn.Linear(64, 40, bias=False).cuda()
    x, dy = torch.randn(2, 30, 64, generator=g, device="cuda"), torch.randn(2, 30, 40, generator=g, device="cuda")
    a, b = torch.randn(40, 64, generator=g, device="cuda"), torch.randn(2, 30, 64, generator=g, device="cuda")
    for dtype in (torch.float32, torch.bfloat16):
        out = []
        for f in (lambda v: core.train_linear(lin, v, torch.float32), lambda v: lin(v).float()):
            xs, ds = x.to(dtype).requires_grad_(True), dy.clone().requires_grad_(True)
            with torch.autocast("cuda", dtype=torch.bfloat16):
                y = f(xs)
            gw, gx = torch.autograd.grad(y, (lin.weight, xs), ds, create_graph=True)
            out.append(torch.autograd.grad((gw * a).sum() + (gx.float() * b).sum(), (xs, lin.weight, ds)))
        for p, q in zip(*out):
            assert p.dtype == q.dtype
            assert (p.double() - q.double()).abs().max() <= 2e-2 * q.double().abs().max()


def test_hooks_and_replaced_forwards_of_the_table_layer_and_the_output_map_run():
    """A hook on the table layer's norm, and a forward that was put on a norm or a map itself, see every training call."""
    m = RunTimeSdm(64, heads=2, n_sub=8, d_a=16, k=4, decays=(0.5, 0.9)).to("cuda").train()
    t = TrainedSdm(64, 8, heads=2, d_a=8, k=4).to("cuda").train()
    x = torch.randn(2, 40, 64, device="cuda", requires_grad=True)
    seen = []

    def call(mod):
        with torch.autocast("cuda", dtype=torch.bfloat16):
            mod(x).float().sum().backward()
    hook = t.norm.register_forward_hook(lambda *a: seen.append("norm"))
    call(t)
    hook.remove()
    assert seen == ["norm"]
    for mod, sub in ((t, t.norm), (t, t.wq), (t, t.wo), (m, m.wo)):
        inner = sub.forward
        sub.forward = lambda *a, inner=inner: (seen.append(1), inner(*a))[1]
        call(mod)
        del sub.forward
    assert seen == ["norm", 1, 1, 1, 1]


def test_projections_and_norms_of_other_shapes_are_refused():
    """A projection or a norm replaced by one of another width raises, as the products and the norm raised op by op."""
    x = torch.randn(2, 40, 64, device="cuda", requires_grad=True)
    m = RunTimeSdm(64, heads=2, n_sub=8, d_a=16, k=4, decays=(0.5, 0.9)).to("cuda").train()
    m.wq = torch.nn.Linear(32, 32, bias=False).cuda()
    with pytest.raises(RuntimeError):
        m(x)
    t = TrainedSdm(64, 8, heads=2, d_a=8, k=4).to("cuda").train()
    t.norm = type(t.norm)(32).cuda()
    with pytest.raises(RuntimeError):
        t(x)


def test_the_table_layer_trains_past_the_norm_kernels_width():
    """Rows wider than the norm kernel holds go through the norm module, as those of a width it does not divide."""
    for d in (2056, 60):
        t = TrainedSdm(d, 8, heads=1, d_a=8, k=4).to("cuda").train()
        torch.nn.init.normal_(t.values)
        x = torch.randn(2, 9, d, device="cuda", requires_grad=True)
        y = t(x)
        y.square().sum().backward()
        q = t.wq(t.norm(x).float())
        r = core.TableSdmFunction.apply(q, t.keys1, t.keys2, t.log_scale, t.values, dict(k=4))
        assert torch.equal(y, t.wo(r)) and bool(torch.isfinite(x.grad).all())


def test_the_mixers_input_gradient_is_held_in_float32(monkeypatch):
    """Under autocast the norm's backward gets the projections' input gradient in float32: a product of bfloat16 operands
    within the bound of a float32 sum in any order, n 2^-24 of the sum of magnitudes, and not rounded to bfloat16."""
    torch.manual_seed(7)
    m = RunTimeSdm(96, heads=4, n_sub=8, d_a=16, k=8, decays=(0.6, 0.8, 0.95, 0.99)).to("cuda").train()
    torch.nn.init.xavier_uniform_(m.wo.weight)
    seen, prod = [], []
    norm_bwd, input_grad = core.rms_norm_backward, core._input_grad
    monkeypatch.setattr(core, "rms_norm_backward", lambda x, w, dy, *a: (seen.append(dy), norm_bwd(x, w, dy, *a))[1])
    monkeypatch.setattr(core, "_input_grad", lambda *a: (prod.append(a[:2]), input_grad(*a))[1])
    x = torch.randn(3, 130, 96, device="cuda", requires_grad=True)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        y = m(x)
    y.sum().backward()
    dhx, (dp, W) = seen[0], prod[0]
    assert dhx.dtype == torch.float32 and dp.dtype == W.dtype == torch.bfloat16
    assert not torch.equal(dhx, dhx.bfloat16().float())
    want = (dp.double() @ W.double()).view_as(dhx)
    bound = (dp.shape[1] + 1) * 2.0 ** -24 * (dp.double().abs() @ W.double().abs()).view_as(dhx)
    assert bool(((dhx.double() - want).abs() <= bound).all())
