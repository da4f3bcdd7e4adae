"""The 16-bit chunk forward's segments and key widths where their indexing
can go wrong, against the fp64 recurrence in the bands of test_gpu_gla.py
(twice the errors measured there; bf16 for both types): one long sequence
among short and empty ones (many segments of one chain, whose states fold
over more than one batch of 8), leading rows outside every sequence, more
sequences than one probe round of the slot search takes, key widths of one
partial group, two groups and two calls, and batches that fill the GPU with
whole sequences."""
import numpy as np
import pytest
import torch

from tests.conftest import assert_close
from tests.test_gpu_gla import HT_BANDS, O_BANDS, _inputs, _oracle, _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lens,H,K,V,dtype,g16", [
    ([5, 0, 2000, 64, 1, 0, 130], 2, 64, 64, torch.bfloat16, False),
    ([3000, 1, 63], 1, 64, 32, torch.float16, False),
    ([1] * 70 + [900] + [65] * 3, 2, 64, 48, torch.bfloat16, False),
    ([700, 0, 65, 7], 2, 16, 16, torch.bfloat16, False),
    ([700, 0, 65, 7], 3, 48, 64, torch.float16, True),
    ([1500, 64, 1], 2, 128, 128, torch.bfloat16, False),
    ([129, 700, 0], 3, 80, 16, torch.bfloat16, True),
    ([300, 65], 2, 112, 48, torch.float16, False),
    ([300, 65], 2, 144, 80, torch.bfloat16, False),
    ([200, 30], 1, 256, 64, torch.bfloat16, False),
])
def test_segments(dev, lens, H, K, V, dtype, g16):
    from ssla_amd.gla import chunk_gla
    print(f"segments lens={lens[:4]}.. H={H} K={K} V={V} {dtype} g16={g16}", flush=True)
    q, k, v, g, cu, s0 = _inputs(lens, H, K, V, dtype, seed=K + V)
    if g16:
        g = g.to(dtype)
    o, ht = _run(chunk_gla, q, k, v, g, cu, s0, K ** -0.5, dev)
    ro, rht = _oracle(q, k, v, g, cu, s0, K ** -0.5)
    assert_close(o, ro, 0.0, "o", band=O_BANDS["logsig"][0], ratio_max=O_BANDS["logsig"][1])
    assert_close(ht, rht, 0.0, "ht", band=HT_BANDS["logsig"][0], ratio_max=HT_BANDS["logsig"][1])
    # the same sequences after rows that belong to none
    pad = lambda t: torch.cat([torch.zeros(3, *t.shape[1:], dtype=t.dtype), t])   # noqa: E731
    o2, ht2 = _run(chunk_gla, pad(q), pad(k), pad(v), pad(g), cu + 3, s0, K ** -0.5, dev)
    assert_close(o2[3:], ro, 0.0, "o, led", band=O_BANDS["logsig"][0], ratio_max=O_BANDS["logsig"][1])
    assert_close(ht2, rht, 0.0, "ht, led", band=HT_BANDS["logsig"][0], ratio_max=HT_BANDS["logsig"][1])


@pytest.mark.parametrize("lens,H,K", [
    ([256, 256, 100, 412], 2, 64),             # two sequences where equal lengths would put them, two not
    ([0, 512, 256, 256], 3, 64),
    ([100, 668, 256], 1, 64),
    ([256] * 5, 3, 128),
    ([2048, 1, 2047, 4096], 1, 64),
    ([384, 384, 1, 767, 384], 9, 48),
])
def test_totals_of_equal_lengths(dev, lens, H, K):
    """Batches whose total is a whole number of segments per sequence, so that
    workgroups are dealt as for equal lengths, with equal and other lengths."""
    from ssla_amd.gla import chunk_gla
    print(f"even totals lens={lens} H={H} K={K}", flush=True)
    q, k, v, g, cu, s0 = _inputs(lens, H, K, 32, torch.bfloat16, seed=K + H)
    o, ht = _run(chunk_gla, q, k, v, g, cu, s0, K ** -0.5, dev)
    ro, rht = _oracle(q, k, v, g, cu, s0, K ** -0.5)
    assert_close(o, ro, 0.0, "o", band=O_BANDS["logsig"][0], ratio_max=O_BANDS["logsig"][1])
    assert_close(ht, rht, 0.0, "ht", band=HT_BANDS["logsig"][0], ratio_max=HT_BANDS["logsig"][1])


def test_many_ragged_sequences(dev):
    """64 sequences x 8 heads of 1,024 rows on average (one segment each
    fills the GPU), one of them 9,000 rows: every sequence in one walk."""
    from ssla_amd.gla import chunk_gla
    rng = np.random.default_rng(0)
    lens = rng.integers(600, 1150, 63).tolist()
    lens = lens + [64 * 1024 - sum(lens)]
    q, k, v, g, cu, s0 = _inputs(lens, 8, 64, 16, torch.bfloat16, seed=9)
    print("many ragged sequences", flush=True)
    o, ht = _run(chunk_gla, q, k, v, g, cu, s0, 0.125, dev)
    ro, rht = _oracle(q, k, v, g, cu, s0, 0.125)
    for nm, a, b, bands in (("o", o, ro, O_BANDS), ("ht", ht, rht, HT_BANDS)):
        assert_close(a, b, 0.0, nm, band=bands["logsig"][0], ratio_max=bands["logsig"][1])


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_full_batches_carry_the_state_in_fp32(dev, dtype):
    """A ragged batch whose sequences and heads fill the GPU uncut: each
    sequence's bits are those of a call of its own, which is one walk with the
    state in fp32 (a cut would enter its segments from 16-bit states), and
    the allocation-free entry's are the same."""
    from ssla_amd import _lib
    from ssla_amd.gla import chunk_gla
    lens, H, V = [2500, 0, 300], 512, 16
    gen = torch.Generator(device=dev).manual_seed(3)
    T = sum(lens)
    q, k = (torch.randn(T, H, 64, generator=gen, device=dev).to(dtype) for _ in range(2))
    v = torch.randn(T, H, V, generator=gen, device=dev).to(dtype)
    g = torch.nn.functional.logsigmoid(torch.randn(T, H, 64, generator=gen, device=dev)) / 16
    cu = torch.tensor(np.concatenate([[0], np.cumsum(lens)]), dtype=torch.int64, device=dev)
    print(f"full batch {dtype}", flush=True)
    with torch.no_grad():
        o, ht = chunk_gla(q, k, v, g, cu, output_final_state=True)
        for n, (a, b) in enumerate(zip(cu.tolist(), cu.tolist()[1:])):
            if b > a:
                on, hn = chunk_gla(q[a:b], k[a:b], v[a:b], g[a:b], torch.tensor([0, b - a], device=dev),
                                   output_final_state=True)
                assert torch.equal(o[a:b], on) and torch.equal(ht[n], hn[0]), f"sequence {n}"
    lib, P = _lib.load(), _lib.ptr
    o2, ht2 = torch.empty_like(o), torch.empty_like(ht)
    _lib.check(lib.ssla_gla_chunk_fwd_noalloc(P(q), P(k), P(v), P(g), _lib.SSLA_F32, P(cu), 3, T, H, 64, V, 64 ** -0.5,
                                              None, P(o2), P(ht2), _lib.DTYPE_CODE[dtype], _lib.stream_of(o2)), "noalloc")
    assert torch.equal(o2, o) and torch.equal(ht2, ht)


@pytest.mark.parametrize("K", [16, 32, 48, 80, 128, 144])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_unaligned_views(dev, K, dtype):
    """q, k and g that start one element off a 16-byte boundary (slices of a
    flat buffer) give the aligned tensors' bits at key widths other than 64."""
    from ssla_amd.gla import chunk_gla
    q, k, v, g, cu, s0 = (t.to(dev) for t in _inputs([130, 7], 1, K, 16, dtype, seed=K))
    off = lambda t: torch.cat([t.flatten()[:1], t.flatten()])[1:].view(t.shape)   # noqa: E731
    print(f"unaligned K={K} {dtype}", flush=True)
    with torch.no_grad():
        for gg in (g, g.to(dtype)):
            a = chunk_gla(q, k, v, gg, cu, initial_state=s0, output_final_state=True)
            b = chunk_gla(off(q), off(k), v, off(gg), cu, initial_state=off(s0), output_final_state=True)
            assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])


def test_long_sequence_of_wide_keys(dev):
    """One sequence past 2^31 bytes of 128 fp32 gates, which 64 keys a call still take."""
    from ssla_amd.gla import chunk_gla
    T, K, V = (1 << 22) + 70, 128, 16
    gen = torch.Generator(device=dev).manual_seed(2)
    q, k, v = (torch.randn(T, 1, d, generator=gen, device=dev, dtype=torch.bfloat16) for d in (K, K, V))
    g = torch.randn(T, 1, K, generator=gen, device=dev).abs_().mul_(-0.1)
    print("long sequence of 128 keys", flush=True)
    with torch.no_grad():
        o, ht = chunk_gla(q, k, v, g, torch.tensor([0, T], device=dev), output_final_state=True)
        t0 = T - 2000   # gates of 0.1 a step on average: the state forgets within a few hundred rows
        last = [x[t0:].contiguous() for x in (q, k, v, g)]
        on, hn = chunk_gla(*last, torch.tensor([0, T - t0], device=dev), output_final_state=True)
    err = lambda a, b: float((a.double() - b.double()).norm() / b.double().norm())   # noqa: E731
    assert err(o[-1000:], on[-1000:]) < 6e-3 and err(ht, hn) < 6e-3   # two bf16 roundings of o, and the state's
    assert bool(torch.isfinite(o).all())
