"""MosAttention's training kernels (ssla_mos_train_fwd / _bwd, taken by
forward(fused=None) when a gradient is recorded) where tiles and dispatch can
go wrong: widths off the multiples of 4 and 16 and past one 64-channel scan
block, one kernel position, a single event, more events than one tile of
128, shared projections, frozen parameters or events, retained graphs --
against float64 CPU autograd of the layer on the same patch rows, at the
fp32 bar (rtol 1e-4) of the composed path's test."""
import pytest
import torch

from tests.conftest import assert_close
from tests.test_gpu_grad import _mos_t64, _random_grouped

pytestmark = pytest.mark.gpu


def _layer(dev, cin, hid, k, sp=True, gp=True):
    from ssla_amd.layers import MosAttention
    torch.manual_seed(cin * 10 + hid)
    return MosAttention(cin, hid, (12, 16), (k, k), scatter_proj=sp, gather_proj=gp).to(dev)


def _rows(layer, gr):
    from ssla_amd import events as E
    with torch.no_grad():
        layer(gr, fused=False)   # builds the lookup table
        src, _t, pos, _fi, f_len, _n = E._rf_scatter(gr, layer.frame_size, layer.patch2pixel_lut)
    return src.cpu(), pos.cpu(), f_len.cpu()


def _uses_train(y):
    f, seen = [y.grad_fn], set()
    while f:
        n = f.pop()
        if n is None or n in seen:
            continue
        seen.add(n)
        if "MosTrainFunction" in type(n).__name__:
            return True
        f += [m for m, _ in n.next_functions]
    return False


@pytest.mark.parametrize("cin,hid,k,sp,gp,n", [
    (8, 12, 3, True, True, 600),
    (10, 13, 3, True, True, 129),      # scalar loads throughout
    (24, 48, 3, True, True, 700),
    (48, 96, 3, True, True, 300),      # two scan blocks of 48 channels
    (96, 70, 3, True, True, 65),       # 35 + 35 channels, ragged tiles
    (2, 12, 1, True, True, 257),
    (16, 16, 5, False, True, 200),
    (12, 12, 3, True, False, 64),
    (128, 128, 3, True, True, 40),
    (6, 6, 3, True, True, 1),
])
def test_mos_train(dev, cin, hid, k, sp, gp, n):
    print(f"mos train cin={cin} hid={hid} k={k} sp={sp} gp={gp} n={n}", flush=True)
    gr = _random_grouped(dev, n=max(n, 3), C=cin, seed=cin + hid)
    if n == 1:   # one event on its own
        gr = {**{a: gr[a][:1] for a in ("events", "time", "batch_id", "h", "w")},
              "lengths": torch.ones(1, dtype=torch.int64, device=dev), "batch_size": 1}
    layer = _layer(dev, cin, hid, k, sp, gp)
    src, pos, f_len = _rows(layer, gr)
    ev = gr["events"].detach().requires_grad_()
    y = layer({**gr, "events": ev})["events"]
    assert _uses_train(y)
    w = torch.randn(y.shape, generator=torch.Generator().manual_seed(2), dtype=torch.float64)
    loss = (y * w.float().to(dev)).sum()
    prm = dict(layer.named_parameters())
    got = torch.autograd.grad(loss, [ev, *prm.values()], retain_graph=True)
    again = torch.autograd.grad(loss, [ev, *prm.values()])
    assert all(torch.equal(a, b) for a, b in zip(got[1:-2], again[1:-2])), "a second backward gives other gradients"
    p64 = {a: v.detach().cpu().double().requires_grad_() for a, v in prm.items()}
    e64 = gr["events"].detach().cpu().double().requires_grad_()
    y64 = _mos_t64(p64, e64, src, pos, f_len, hid, sp, gp)
    assert_close(y.detach().cpu().numpy(), y64.detach().numpy(), 1e-4, "forward")
    (y64 * w).sum().backward()
    assert_close(got[0].cpu().numpy(), e64.grad.numpy(), 1e-4, "d events")
    for (name, _), g in zip(prm.items(), got[1:]):
        assert_close(g.cpu().numpy(), p64[name].grad.numpy(), 1e-4, f"d {name}")


def test_mos_train_frozen(dev):
    """Frozen weights (gradients of the events only), events without a
    gradient (weights only), each equal to the full backward's."""
    gr = _random_grouped(dev, C=8, seed=3)
    layer = _layer(dev, 8, 12, 3)

    def grads(ev_grad, w_grad):
        layer.requires_grad_(w_grad)
        ev = gr["events"].detach().requires_grad_(ev_grad)
        y = layer({**gr, "events": ev})["events"]
        assert _uses_train(y)
        layer.zero_grad()
        y.square().sum().backward()
        return ev.grad, [p.grad for p in layer.parameters()]
    full = grads(True, True)
    assert torch.equal(grads(True, False)[0], full[0])
    assert all(torch.equal(a, b) for a, b in zip(grads(False, True)[1][:6], full[1][:6]))


def test_mos_train_keeps_the_composed_path(dev):
    """Calls the kernels do not stand for keep the composed path: a stride
    (most copies in no patch), autocast, a hooked or replaced projection."""
    from ssla_amd.layers import MosAttention
    gr = _random_grouped(dev, C=8, seed=4)
    gr["events"].requires_grad_()
    strided = MosAttention(8, 12, (12, 16), (3, 3), stride=(3, 3)).to(dev)
    assert not _uses_train(strided(gr)["events"])
    layer = _layer(dev, 8, 12, 3)
    assert not _uses_train(layer(gr, fused=False)["events"])
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert not _uses_train(layer(gr)["events"])
    layer.o_proj.register_forward_hook(lambda m, i, o: 2 * o)
    assert not _uses_train(layer(gr)["events"])


@pytest.mark.parametrize("H", [1, 3, 15, 16, 17, 33, 48, 70, 96, 128])
@pytest.mark.parametrize("n", [1, 17, 16 * 1024 + 1, 40000])
def test_row_norm(dev, H, n):
    """The LayerNorm kernels against float64, row counts about a workgroup's 16
    and the 16,384 of a full grid.  u = 2^-24: a row's mean and moment are sums
    of at most 8 + 4 terms in sequence, so y is within 16 u (|x| + |mean|) rstd
    |w| + 2 u |b| and dx within 32 u of its terms; a weight gradient sums at
    most 3 rows, 16 groups, 16 workgroups and 6 levels in sequence."""
    from ssla_amd.layers import RowNormFunction
    u, eps = 2.0 ** -24, 1e-5
    gen = torch.Generator().manual_seed(H * 7 + n)
    x = (torch.randn(n, H, generator=gen) * 2 + 1).to(dev).requires_grad_()
    w, b = (torch.randn(H, generator=gen).to(dev).requires_grad_() for _ in range(2))
    dy = torch.randn(n, H, generator=gen).to(dev)
    y = RowNormFunction.apply(x, w, b, eps)
    got = torch.autograd.grad(y, [x, w, b], dy, retain_graph=True)
    assert all(torch.equal(p, q) for p, q in zip(got, torch.autograd.grad(y, [x, w, b], dy)))
    X, W, Bi, D = (t.detach().double() for t in (x, w, b, dy))
    mean = X.mean(1, keepdim=True)
    rstd = ((X - mean).square().mean(1, keepdim=True) + eps).rsqrt()
    h, g = (X - mean) * rstd, D * W
    dh = 16 * u * (X.abs().amax(1, keepdim=True) + mean.abs()) * rstd * (1 + h.abs())   # bound on xhat's error
    assert ((y.double() - (h * W + Bi)).abs() <= dh * W.abs() + 2 * u * Bi.abs() + 1e-30).all()
    m1, m2 = g.mean(1, keepdim=True), (g * h).mean(1, keepdim=True)
    ga, gh = g.abs().mean(1, keepdim=True), (g * h).abs().mean(1, keepdim=True)
    bound = rstd * (32 * u * (g.abs() + ga + h.abs() * gh) + dh * gh + h.abs() * (g.abs() * dh).mean(1, keepdim=True))
    assert ((got[0].double() - rstd * (g - m1 - h * m2)).abs() <= bound + dh * rstd * (g.abs() + ga)).all()
    assert ((got[1].double() - (D * h).sum(0)).abs() <= 44 * u * (D * h).abs().sum(0) + (D.abs() * dh).sum(0)).all()
    assert ((got[2].double() - D.sum(0)).abs() <= 44 * u * D.abs().sum(0)).all()


def test_mos_train_hooked_norm(dev):
    """A norm with a hook or of another type is called as a module."""
    gr = _random_grouped(dev, C=8, seed=5)
    gr["events"].requires_grad_()
    layer = _layer(dev, 8, 12, 3)
    y = layer(gr)["events"]
    layer.norm.register_forward_hook(lambda m, i, o: 2 * o)
    assert torch.allclose(layer(gr)["events"], 2 * y, rtol=1e-5, atol=1e-5)
    layer.norm = torch.nn.Identity()
    out = layer(gr)["events"]
    assert _uses_train(out) and torch.allclose(torch.nn.functional.layer_norm(out, (12,)), y, rtol=1e-4, atol=1e-4)
