"""The scans at the ends of their tiles (1024 items) and on both sides of the
number of tiles (2048) up to which the writing pass sums the tiles before its own:
kept-sample compaction, cell lists and sample ends, exact."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,cap", [(0, 5), (1, 1), (1023, 1024), (1024, 1024), (1025, 4096),
                                   (5000, 300000), (2097152, 2097152), (2097153, 2097153),
                                   (2100000, 2300000)])
def test_scans_at_tile_ends(n, cap, dev):
    from supernormal_amd import _lib
    from supernormal_amd._lib import call, ptr, stream_of
    lib, s = _lib.lib(), stream_of(dev)
    g = torch.Generator().manual_seed(n + cap)
    keep = (torch.rand(cap, generator=g) < 0.6).to(torch.uint8).to(dev)
    ri = torch.randint(0, 50, (cap,), generator=g).sort().values.to(dev)
    t0 = torch.rand(cap, generator=g).to(dev)
    t1 = torch.where(torch.rand(cap, generator=g).to(dev) < 0.7, t0.roll(-1), t0 + 1)
    nd = torch.tensor([n], dtype=torch.int32, device=dev)
    i64 = lambda k: torch.full((k,), -7, dtype=torch.int64, device=dev)
    f32 = lambda k: torch.full((k,), -7.0, device=dev)
    one = lambda: torch.full((1,), -7, dtype=torch.int32, device=dev)
    o_ri, o_t0, o_t1, n_out = i64(cap), f32(cap), f32(cap), one()
    ws = torch.empty(lib.sn_compact_workspace_bytes(cap), dtype=torch.uint8, device=dev)
    call("sn_compact_samples_dev", ptr(keep), cap, ptr(nd), ptr(ri), ptr(t0), ptr(t1), ptr(o_ri),
         ptr(o_t0), ptr(o_t1), ptr(n_out), None, 0, None, ptr(ws), ws.numel(), s)
    k = keep[:n].bool()
    m = int(k.sum())
    assert int(n_out) == m
    for got, src in ((o_ri, ri), (o_t0, t0), (o_t1, t1)):
        assert torch.equal(got[:m], src[:n][k]) and bool((got[m:] == -7).all())
    cells, cnt = i64(cap), one()
    call("sn_occ_nonzero", ptr(keep), cap, ptr(cells), ptr(cnt), ptr(ws), ws.numel(), s)
    assert torch.equal(cells[:int(cnt)], keep.nonzero()[:, 0])
    oc, dc = torch.zeros(50, 3, device=dev), torch.ones(50, 3, device=dev)
    di = torch.full((cap,), -7, dtype=torch.int32, device=dev)
    n_diff, n_eval, pts = one(), one(), f32(6 * cap)
    ws = torch.empty(lib.sn_step_workspace_bytes(cap), dtype=torch.uint8, device=dev)
    call("sn_centre_points", ptr(ri), ptr(t0), ptr(t1), cap, ptr(nd), ptr(oc), ptr(dc), 3, ptr(di),
         ptr(n_diff), ptr(pts), ptr(n_eval), ptr(ws), ws.numel(), s)
    own = torch.ones(n, dtype=torch.bool, device=dev)
    own[:-1] = ~((ri[1:n] == ri[:n - 1]) & (t1[:n - 1] == t0[1:n])) if n > 1 else own[:-1]
    ref = torch.where(own, torch.cumsum(own.int(), 0) - 1, torch.full_like(di[:n], -1))
    assert torch.equal(di[:n], ref.int()) and int(n_diff) == int(own.sum())
    assert int(n_eval) == n + int(own.sum())
