"""The hash-grid backward's bucket records (x pairs of table rows) where a pair
can go wrong: rows in two buckets (x cell -1 of a hashed level, a dense level's
bucket boundary), more than 64 and 256 buckets per level, one feature per
level, ends of a workgroup's 512 points, an unaligned workspace, positions that
are not finite.  Reference: the atomic path (no workspace), which the oracle
pins elsewhere.

Tolerance: both paths round each of the <= n terms of a row to fp32 and add
them in another order: n = 1537 roundings of one sign are 9e-5 of the sum of
magnitudes, so 1e-4 |ref| + 1e-5 max|ref|."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _both(dev, F, log2_T, n, ad, kind, shift=0):
    from supernormal_amd import _lib
    from supernormal_amd._lib import call, ptr, stream_of
    from supernormal_amd.tcnn import Encoding
    gargs = (16, F, log2_T, 16, 1.38, 16)
    e = Encoding(3, {"otype": "HashGrid", "n_levels": 16, "n_features_per_level": F,
                     "log2_hashmap_size": log2_T, "base_resolution": 16,
                     "per_level_scale": 1.38}).to(dev)
    g = torch.Generator().manual_seed(1000 * F + log2_T + n)
    x = torch.rand(n, 3, generator=g) * 1.8 - 0.9
    if kind == "edge":  # x cells -1 and 0 of every level, groups of near points
        x[:, 0] = (torch.rand(n, generator=g) - 0.5) * 10 ** (-4 * torch.rand(n, generator=g))
        x[n // 2:] = x[n // 2:n // 2 + 1] + 1e-4 * torch.randn(n - n // 2, 3, generator=g)
    elif kind == "dense":  # whole cells of the dense levels in order
        i = torch.arange(n)
        x = torch.stack([(i % 29) / 29.0, (i // 29 % 29) / 29.0, (i // 841) / 29.0], 1)
    elif kind == "nan":
        x[3, 0], x[700 % n, 2], x[5, 1] = float("nan"), float("inf"), -float("inf")
    x = x.float().contiguous().to(dev)
    r = lambda *s: torch.randn(*s, generator=g).to(dev)
    genc, g2, v = r(n, 16 * F), r(n, 16 * F), r(n, 3)
    nb = _lib.lib().sn_hashgrid_bwd_workspace_bytes(*gargs[:5], 4096)
    ws = torch.zeros(nb + 16, dtype=torch.uint8, device=dev)
    out = []
    for w in (None, ws, ws):
        gp = torch.zeros_like(e.params)
        wp, wb = (None, 0) if w is None else (w.data_ptr() + shift, nb)
        if ad:
            call("sn_hashgrid_bwd_ad_ws_dev", ptr(x), n, None, ptr(e.params), *gargs, None,
                 ptr(genc), ptr(v), ptr(g2), ptr(gp), wp, wb, stream_of(dev))
        else:
            call("sn_hashgrid_bwd_ws_dev", ptr(x), n, None, ptr(e.params), *gargs, None,
                 ptr(genc), ptr(gp), None, wp, wb, stream_of(dev))
        torch.cuda.synchronize()
        out.append(gp)
    return out


@pytest.mark.parametrize("F,log2_T,n,ad,kind,shift", [
    (2, 19, 1537, False, "edge", 0), (2, 19, 513, True, "edge", 0), (1, 19, 512, False, "edge", 0),
    (2, 20, 1025, False, "edge", 0), (2, 22, 1025, True, "edge", 0), (1, 21, 511, True, "edge", 0),
    (2, 19, 1537, False, "dense", 0), (1, 20, 1, True, "any", 0), (2, 22, 1537, False, "any", 0),
    (2, 19, 1024, False, "edge", 4), (2, 15, 1537, False, "edge", 8)])
def test_pair_records(F, log2_T, n, ad, kind, shift, dev):
    ref, a, b = _both(dev, F, log2_T, n, ad, kind, shift)
    scale = float(ref.abs().max())
    for got in (a, b):
        torch.testing.assert_close(got, ref, rtol=1e-4, atol=1e-5 * scale)


@pytest.mark.parametrize("ad", [False, True])
def test_positions_not_finite(ad, dev):
    ref, a, _ = _both(dev, 2, 19, 1025, ad, "nan")
    assert int(torch.isnan(ref).sum()) > 0
    assert torch.equal(torch.isnan(a), torch.isnan(ref))
    fin = ~torch.isnan(ref)
    scale = float(ref[fin].abs().max())
    torch.testing.assert_close(a[fin], ref[fin], rtol=1e-4, atol=1e-5 * scale)
