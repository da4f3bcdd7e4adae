"""The 16-lane field fill and count (rf_merge_fields, rf_count16) against the
radix-sort fill, bit for bit: fields below, at and past the rows a field's
LDS area holds (96), 2 to 16 kernel positions, many timestamp ties, strided
and overlapping fields, several samples."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kh,kw,sh,sw", [(1, 2, 1, 1), (2, 3, 1, 2), (3, 3, 1, 1), (3, 4, 1, 1), (4, 4, 1, 1), (5, 3, 2, 1),
                                         (3, 3, 3, 3)])
@pytest.mark.parametrize("hot", [8, 95, 96, 97, 400])
def test_field_fill_equals_sort(dev, kh, kw, sh, sw, hot):
    from ssla_amd import events as E
    H, W, B = 9, 11, 2
    rng = np.random.default_rng(kh * 100 + kw * 10 + hot)
    ev = []
    for b in range(B):   # `hot` events spread over one 2 x 2 patch of pixels, 60 elsewhere
        xy = np.concatenate([np.stack([4 + rng.integers(0, 2, hot), 3 + rng.integers(0, 2, hot)], 1),
                             np.stack([rng.integers(0, W, 60), rng.integers(0, H, 60)], 1)])
        t = np.sort(rng.integers(0, 40, hot + 60))
        ev.append(np.concatenate([xy[rng.permutation(hot + 60)], t[:, None], np.ones((hot + 60, 1))], 1))
    ev = torch.from_numpy(np.stack(ev).astype(np.float32)).to(dev)
    gr = E.group_events((ev, torch.full((B,), hot + 60, dtype=torch.int64, device=dev)), (H, W))
    lut, _ = E.compute_rf2pixels((H, W), (kh, kw), (sh, sw), device=dev)
    print(f"field fill {kh}x{kw}/{sh},{sw} hot={hot}", flush=True)
    a = E._rf_scatter(gr, (H, W), lut, dst_map=True)
    b = E._rf_scatter(gr, (H, W), lut, force_sort=True)
    for name, x, y in zip(("src", "time", "pos", "f_index", "f_len"), a[:5], b[:5]):
        assert torch.equal(x, y), name
    src, pos, dst = (t.cpu().numpy() for t in (a[0], a[2], a[6]))
    assert np.array_equal(dst[src * kh * kw + pos], np.arange(src.size)) and int((dst >= 0).sum()) == src.size


def test_field_fill_late_times(dev):
    """Timestamps past the 56 bits a row's key holds are placed by search."""
    from ssla_amd import events as E
    n = 40
    t = (1 << 57) + torch.arange(n, device=dev) // 3
    gr = {"time": torch.cat([t[0::2], t[1::2]]), "batch_id": torch.zeros(2, dtype=torch.int64, device=dev),
          "h": torch.zeros(2, dtype=torch.int64, device=dev), "w": torch.tensor([0, 1], device=dev),
          "lengths": torch.tensor([n // 2, n // 2], device=dev), "batch_size": 1}
    lut, _ = E.compute_rf2pixels((2, 3), (1, 3), (1, 1), device=dev)
    src, tim, pos, _fi, f_len, _n = E._rf_scatter(gr, (2, 3), lut)
    at = 0
    for m in f_len.tolist():   # rows in (time, position, event) order
        rows = list(zip(tim[at:at + m].tolist(), pos[at:at + m].tolist(), src[at:at + m].tolist()))
        assert rows == sorted(rows) and torch.equal(tim[at:at + m], gr["time"][src[at:at + m]])
        at += m
    assert at == src.numel() > 2 * n


@pytest.mark.parametrize("kh,kw", [(1, 2), (2, 2), (1, 5), (3, 3), (4, 4)])
@pytest.mark.parametrize("late", [0, 1 << 57])
def test_large_fields(dev, kh, kw, late):
    """Pixels of 1 to 5,000 events without a cap: fields of one to hundreds
    of 64-row pieces, about the edges of a piece, beside small ones, two runs
    of the same workspace; also with timestamps past a key's 56 bits."""
    from ssla_amd import events as E
    H, W = 12, 17
    gen = torch.Generator().manual_seed(kh * 10 + kw)
    cnt = torch.randint(0, 3, (H * W,), generator=gen)
    for p, n in ((20, 97), (40, 128), (60, 129), (80, 191), (100, 192), (120, 193), (140, 5000), (141, 700), (158, 64)):
        cnt[p] = n
    pix = torch.nonzero(cnt).flatten()
    ln = cnt[pix]
    t = torch.randint(0, 300, (int(ln.sum()),), generator=gen)
    gid = torch.repeat_interleave(torch.arange(pix.numel()), ln)
    t = t[torch.argsort(gid * 300 + t, stable=True)] + late
    gr = {"time": t.to(dev), "batch_id": torch.zeros_like(pix).to(dev), "h": (pix // W).to(dev), "w": (pix % W).to(dev),
          "lengths": ln.to(dev), "batch_size": 1}
    lut, _ = E.compute_rf2pixels((H, W), (kh, kw), (1, 1), device=dev)
    print(f"large fields {kh}x{kw} late={late}", flush=True)
    a = E._rf_scatter(gr, (H, W), lut, dst_map=True)
    if late == 0:
        b = E._rf_scatter(gr, (H, W), lut, force_sort=True)
        for name, x, y in zip(("src", "time", "pos", "f_index", "f_len"), a[:5], b[:5]):
            assert torch.equal(x, y), name
        return
    # (the radix keys do not hold such times with the field beside them)
    src, tim, pos, f_len = (x.cpu() for x in (a[0], a[1], a[2], a[4]))
    assert torch.equal(tim, t[src])
    field = torch.repeat_interleave(torch.arange(f_len.numel()), f_len)
    key = torch.stack([field, tim - late, pos, src])   # strictly increasing
    d = key[:, 1:] - key[:, :-1]
    first = (d != 0).int().argmax(0)
    assert (d.gather(0, first[None]) > 0).all()
    dst = a[6].cpu()
    assert torch.equal(dst[src * kh * kw + pos], torch.arange(src.numel(), dtype=torch.int32))
    assert int((dst >= 0).sum()) == src.numel()
