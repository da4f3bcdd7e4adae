"""Answers read back while the work behind them runs: the scatter functions'
index check (ssla_scatter_*_checked) at the edges of its blocks and in every
path, and the recurrent GLA's row bounds, against the plain calls."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E,n_out", [(1, 3), (256, 40), (1025, 300), (70000, 9000), (300000, 400000)])
@pytest.mark.parametrize("srt", [True, False])
def test_bad_index_is_reported(dev, E, n_out, srt):
    from ssla_amd.scatter import scatter_max, scatter_mean
    print(f"checked scatter E={E} n_out={n_out} sorted={srt}", flush=True)
    gen = torch.Generator().manual_seed(E)
    src = torch.randn(E, 5, generator=gen).to(dev)
    idx = torch.randint(0, n_out, (E,), generator=gen)
    idx = (torch.sort(idx).values if srt else idx).to(dev)
    for fn in (scatter_max, scatter_mean):
        good, plain = (fn(src, idx, dim=0, dim_size=n_out, sorted_index=srt, check=c) for c in (True, False))
        if fn is scatter_max or srt:   # (a shuffled mean adds in the order its atomics land)
            for a, b in zip(good if fn is scatter_max else [good], plain if fn is scatter_max else [plain]):
                assert torch.equal(a, b)
        places = {0, E - 1, E // 2, min(E - 1, 255), min(E - 1, 256), min(E - 1, 1023), min(E - 1, 1024)}
        for i in sorted(places):
            for v in (-1, n_out):
                bad = idx.clone()
                bad[i] = v
                with pytest.raises(ValueError, match="out of range"):
                    fn(src, bad, dim=0, dim_size=n_out, sorted_index=srt)
            if srt and i > 0 and int(idx[i - 1]) > 0:
                bad = idx.clone()
                bad[i] = int(idx[i - 1]) - 1
                with pytest.raises(ValueError, match="not sorted"):
                    fn(src, bad, dim=0, dim_size=n_out, sorted_index=True)
        again = fn(src, idx, dim=0, dim_size=n_out, sorted_index=srt)
        if fn is scatter_max:
            assert all(torch.equal(a, b) for a, b in zip(again, good))


def test_checked_scatter_of_nothing(dev):
    from ssla_amd.scatter import scatter_max, scatter_mean
    e = torch.zeros(0, dtype=torch.int64, device=dev)
    for srt in (True, False):
        out, arg = scatter_max(torch.zeros(0, 4, device=dev), e, dim=0, dim_size=3, sorted_index=srt)
        assert not out.any() and bool((arg == 0).all())
        assert scatter_mean(torch.zeros(0, 4, device=dev), e, dim=0, dim_size=0, sorted_index=srt).shape == (0, 4)


def test_recurrent_bounds(dev):
    """o covers cu_seqlens[0]:cu_seqlens[-1] wherever the bounds come from,
    also with calls of other bounds in flight on two streams."""
    from ssla_amd.gla import fused_recurrent_gla, fused_recurrent_gla_rows
    gen = torch.Generator().manual_seed(0)
    q, k, v, g = (torch.randn(300, 2, 16, generator=gen).to(dev) for _ in range(4))
    g = -g.abs()
    other = torch.cuda.Stream()
    other.wait_stream(torch.cuda.current_stream())
    with torch.no_grad():
        for lo, hi in ((0, 300), (3, 290), (17, 17), (0, 1)):
            cu = torch.tensor([lo, (lo + hi) // 2, hi])
            rows, ht = fused_recurrent_gla_rows(q, k, v, g, cu.to(dev), output_final_state=True)
            for c in (cu.to(dev), cu, cu.to(dev).int()):
                o, h = fused_recurrent_gla(q, k, v, g, c, output_final_state=True)
                with torch.cuda.stream(other):
                    full, _ = fused_recurrent_gla(q, k, v, g, torch.tensor([0, 300], device=dev))
                assert o.shape == (hi - lo, 2, 16) and full.shape[0] == 300
                assert torch.equal(o, rows[lo:hi]) and torch.equal(h, ht)
    torch.cuda.synchronize()
