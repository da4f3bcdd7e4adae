"""The chunk-parallel fp32 GLA kernels (ssla_gla_chunk_f32_fwd_ws and
ssla_gla_chunk_f32_bwd) where their indexing can go wrong, against the fp64
recurrence at the fp32 bar of the other chunk tests (rtol 1e-4, atol 1e-4 of
the RMS): scalar loads (K or V not a multiple of 4), several value groups,
sequence counts that take one, two and three rounds of the 64-way slot
search, rows outside every sequence, and decays on both sides of the range
the matrix-core diagonal blocks take (40 binary orders within 16 rows)."""
import numpy as np
import pytest
import torch

import oracle
from tests.conftest import assert_close

pytestmark = pytest.mark.gpu


def _case(lens, lead, tail, H, K, V, gate, seed):
    gen = torch.Generator().manual_seed(seed)
    T = lead + sum(lens) + tail
    q, k, v = (torch.randn(T, H, d, generator=gen) for d in (K, K, V))
    g = -gate * torch.rand(T, H, K, generator=gen) if gate > 0 else torch.randn(T, H, K, generator=gen) * -gate
    cu = lead + np.concatenate([[0], np.cumsum(lens)])
    h0 = torch.randn(len(lens), H, K, V, generator=gen) * 0.1
    return q, k, v, g, torch.tensor(cu, dtype=torch.int64), h0


@pytest.mark.parametrize("lens,lead,tail,H,K,V,gate", [
    ([70, 64, 1], 3, 5, 2, 33, 30, 0.2),
    ([129], 0, 0, 1, 5, 130, 1.0),
    ([1] * 63 + [65] * 3, 2, 0, 1, 16, 16, 0.5),
    ([2] * 70 + [0, 0, 66], 0, 9, 1, 64, 64, 3.4),      # 15 steps of up to 4.9 bits: both sides of 40
    ([1] * 4100, 1, 1, 1, 4, 4, 0.1),
    ([200, 63], 0, 0, 2, 64, 64, 30.0),                 # far past it: every diagonal block term by term
    ([150], 0, 0, 2, 64, 48, -1.5),                     # growing gates: either sign
])
def test_f32_chunks(dev, lens, lead, tail, H, K, V, gate):
    from ssla_amd.gla import chunk_gla
    print(f"f32 chunks: {len(lens)} sequences K={K} V={V} gate={gate}", flush=True)
    q, k, v, g, cu, h0 = _case(lens, lead, tail, H, K, V, gate, seed=len(lens) + K)
    gen = torch.Generator().manual_seed(1)
    do, dht = torch.randn(v.shape, generator=gen), torch.randn(h0.shape, generator=gen) * 0.1
    lo, hi = int(cu[0]), int(cu[-1])
    leaf = [t.to(dev).requires_grad_() for t in (q, k, v, g, h0)]
    o, ht = chunk_gla(*leaf[:4], cu.to(dev), scale=0.3, initial_state=leaf[4], output_final_state=True)
    seq = lambda t: t[lo:hi].numpy()   # noqa: E731
    cz = cu.numpy() - lo
    ro, rht = oracle.gla_recurrent(seq(q), seq(k), seq(v), seq(g), cz, 0.3, h0.numpy(), True)
    assert_close(o.detach().cpu().numpy()[lo:hi], ro, 1e-4, "o")
    assert_close(ht.detach().cpu().numpy(), rht, 1e-4, "ht")
    if gate < 0:
        return   # sums of growing terms: the forward only
    # rows outside every sequence are unspecified: keep them out of the loss
    ((o[lo:hi] * do[lo:hi].to(dev)).sum() + (ht * dht.to(dev)).sum()).backward()
    ref = oracle.gla_recurrent_bwd(seq(q), seq(k), seq(v), seq(g), cz, seq(do), 0.3, h0.numpy(), dht.numpy())
    for nm, t, r in zip(("dq", "dk", "dv", "dg", "dh0"), leaf, ref):
        got = t.grad.cpu().numpy()
        assert_close(got if nm == "dh0" else got[lo:hi], r, 1e-4, nm)


def test_f32_chunk_forward_without_workspace(dev):
    """ssla_gla_chunk_f32_fwd (no workspace) on the same inputs."""
    from ssla_amd import _lib
    lib = _lib.load()
    q, k, v, g, cu, h0 = _case([70, 64, 1], 0, 0, 2, 32, 40, 0.3, seed=5)
    ro, rht = oracle.gla_recurrent(q.numpy(), k.numpy(), v.numpy(), g.numpy(), cu.numpy(), 0.3, h0.numpy(), True)
    d = [t.to(dev) for t in (q, k, v, g, cu, h0)]
    o, ht = torch.empty_like(d[2]), torch.empty_like(d[5])
    T, H, K = q.shape
    _lib.check(lib.ssla_gla_chunk_f32_fwd(*(_lib.ptr(t) for t in d[:5]), 3, T, H, K, 40, 0.3, _lib.ptr(d[5]), _lib.ptr(o),
                                          _lib.ptr(ht), _lib.stream_of(o)), "f32_fwd")
    assert_close(o.cpu().numpy(), ro, 1e-4, "o")
    assert_close(ht.cpu().numpy(), rht, 1e-4, "ht")


def test_f32_dg_cancellation(dev):
    """dg under logsigmoid gates, where it is small next to the q dq and k dk it
    is the difference of.  dq and dk hold each pair (i, j) with the same three
    factors, so what is left are the products' roundings: RMS within 16 u of
    dg's (u = 2^-24; measured 12.1 u, 20.6 u on like inputs when the exponent was split
    differently in dq and in dk)."""
    from ssla_amd.gla import chunk_gla
    q, k, v, _g, cu, h0 = _case([700, 300], 0, 0, 2, 64, 64, 1.0, seed=9)
    gen = torch.Generator().manual_seed(3)
    g = torch.nn.functional.logsigmoid(torch.randn(q.shape, generator=gen))
    do = torch.randn(v.shape, generator=gen)
    leaf = [t.to(dev).requires_grad_() for t in (q, k, v, g)]
    o, _ = chunk_gla(*leaf, cu.to(dev), scale=0.125, initial_state=h0.to(dev), output_final_state=True)
    o.backward(do.to(dev))
    ref = oracle.gla_recurrent_bwd(q.numpy(), k.numpy(), v.numpy(), g.numpy(), cu.numpy(), do.numpy(), 0.125, h0.numpy(),
                                   np.zeros(h0.shape, np.float32))[3]
    err = np.sqrt(np.square(leaf[3].grad.cpu().double().numpy() - ref).mean() / np.square(ref).mean())
    print(f"dg error {err:.2e}", flush=True)
    assert err <= 16 * 2.0 ** -24


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("name", ["q", "k", "v", "do"])
def test_f32_nonfinite_row_stays_causal(dev, name, bad):
    """An infinity or NaN in one row reaches no row that does not depend on
    it: with it in row t of v or k, o before t is finite and as without it,
    in q o at every other row; in dO, dv after t, and in q, k or v the
    gradients that no product with that row enters."""
    from ssla_amd.gla import chunk_gla
    n, t = 150, 64 + 21                       # inside the second chunk's second 16-row block
    q, k, v, g, cu, h0 = _case([n], 0, 0, 2, 64, 64, 0.2, seed=11)
    do = torch.randn(v.shape, generator=torch.Generator().manual_seed(12))
    print(f"f32 {bad} in {name}", flush=True)

    def run(poison):
        x = {"q": q.clone(), "k": k.clone(), "v": v.clone(), "do": do.clone()}
        if poison:
            x[name][t, :, 5] = bad
        leaf = [y.to(dev).requires_grad_() for y in (x["q"], x["k"], x["v"], g)]
        o, _ = chunk_gla(*leaf, cu.to(dev), scale=0.3, initial_state=h0.to(dev), output_final_state=True)
        return [y.detach().cpu().numpy() for y in (o, *torch.autograd.grad(o, leaf, x["do"].to(dev)))]
    clean, got = run(False), run(True)
    # rows of (o, dq, dk, dv) that the poisoned row has no part in
    rows = {"q": (np.r_[0:t, t + 1:n], np.r_[0:t, t + 1:n], np.r_[t + 1:n], np.r_[t + 1:n]),
            "k": (np.r_[0:t], np.r_[0:t], np.r_[0:t, t + 1:n], np.r_[0:t, t + 1:n]),
            "v": (np.r_[0:t], np.r_[0:t], np.r_[0:t, t + 1:n], np.r_[0:n]),
            "do": (np.r_[0:n], np.r_[0:t, t + 1:n], np.r_[t + 1:n], np.r_[t + 1:n])}[name]
    for nm, a, b, r in zip(("o", "dq", "dk", "dv"), got, clean, rows):
        assert_close(a[r], b[r], 1e-4, nm)
    assert not np.isfinite(got[0][t:] if name != "do" else got[3][:t + 1]).all()


@pytest.mark.parametrize("e", [-112, 112])
def test_f32_wide_exponents(dev, e):
    """q scaled by 2^e and k by 2^-e: where q~ or k~ would leave the normal
    range under the block's decay (some 30 bits here) the diagonal is summed
    term by term."""
    from ssla_amd.gla import chunk_gla
    q, k, v, g, cu, h0 = _case([130], 0, 0, 2, 64, 64, 2.0, seed=13)
    do = torch.randn(v.shape, generator=torch.Generator().manual_seed(14))
    ref = oracle.gla_recurrent_bwd(q.numpy(), k.numpy(), v.numpy(), g.numpy(), cu.numpy(), do.numpy(), 0.3)
    ro, _ = oracle.gla_recurrent(q.numpy(), k.numpy(), v.numpy(), g.numpy(), cu.numpy(), 0.3)
    print(f"f32 exponents {e}", flush=True)
    leaf = [y.to(dev).requires_grad_() for y in (q * 2.0 ** e, k * 2.0 ** -e, v, g)]
    o, _ = chunk_gla(*leaf, cu.to(dev), scale=0.3)
    o.backward(do.to(dev))
    assert_close(o.detach().cpu().numpy(), ro, 1e-4, "o")
    for nm, y, r, x in zip(("dq", "dk", "dv", "dg"), leaf, ref, (e, -e, 0, 0)):
        assert_close((y.grad.cpu().double() * 2.0 ** x).numpy(), r, 1e-4, nm)


def test_f32_forward_where_the_workspace_does_not_fit(dev, monkeypatch):
    """chunk_gla on a device without room for the chunks' states (16 KB per
    64 rows or sequence, and head) takes the entry that needs none."""
    from ssla_amd.gla import chunk_gla
    q, k, v, g, cu, h0 = _case([70, 64, 1], 0, 0, 2, 80, 40, 0.3, seed=6)
    ro, rht = oracle.gla_recurrent(q.numpy(), k.numpy(), v.numpy(), g.numpy(), cu.numpy(), 0.3, h0.numpy(), True)
    empty = torch.empty

    def full(*a, **kw):
        if kw.get("dtype") == torch.uint8:
            raise torch.OutOfMemoryError("no room")
        return empty(*a, **kw)
    monkeypatch.setattr(torch, "empty", full)
    with torch.no_grad():
        o, ht = chunk_gla(*(t.to(dev) for t in (q, k, v, g, cu)), scale=0.3, initial_state=h0.to(dev),
                          output_final_state=True)
    assert_close(o.cpu().numpy(), ro, 1e-4, "o")
    assert_close(ht.cpu().numpy(), rht, 1e-4, "ht")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_decreasing_offsets_stay_in_bounds(dev, dtype):
    """cu_seqlens that decrease break the contract, and what the overlapping
    sequences give is unspecified; but no chunk may start before its
    sequence (the slot search assumes increasing starts).  A correct call
    behind it is right."""
    from ssla_amd.gla import chunk_gla
    T, H, K = 640, 1, 64
    q, k, v, g, _cu, _h0 = _case([T], 0, 0, H, K, K, 0.2, seed=17)
    d = [x.to(dev) for x in (q.to(dtype), k.to(dtype), v.to(dtype), g)]
    cu = torch.tensor([0, 600] + [2 * i for i in range(150)] + [T], device=dev)
    print(f"decreasing offsets {dtype}", flush=True)
    with torch.no_grad():
        chunk_gla(*d, cu, scale=0.3, output_final_state=True)
        torch.cuda.synchronize()
        o, _ = chunk_gla(*d, torch.tensor([0, T], device=dev), scale=0.3)
    ro, _ = oracle.gla_recurrent(*(x.float().cpu().numpy() for x in d), np.array([0, T]), 0.3)
    assert_close(o.float().cpu().numpy(), ro, 1e-4 if dtype == torch.float32 else 2e-2, "o")
