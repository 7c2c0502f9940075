"""The encoding by levels: the same bits as the encoding by rows, for both tables
and for counts at the ends of a workgroup's points; and the MLP kernels on it:
the same bits as on rows (exact: the same sums in the same order)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("L,log2_T,n_cap,n,active", [
    (16, 19, 1, 1, 16), (16, 15, 257, 255, 5), (2, 19, 1025, 1023, 2), (14, 19, 3000, 3000, 14),
    (16, 20, 70001, 66001, 16), (16, 19, 640, 0, 16)])
def test_levels_equal_rows(L, log2_T, n_cap, n, active, half, dev):
    from supernormal_amd import _lib
    from supernormal_amd._lib import call, ptr, stream_of
    g = torch.Generator().manual_seed(L + n_cap)
    r = lambda *s: torch.randn(*s, generator=g).to(dev)
    tot = _lib.lib().sn_hashgrid_layout(L, log2_T, 16, 1.38, None)
    tab = r(tot * 2)
    t16 = tab.half() if half else None
    x = (torch.rand(n_cap, 3, generator=g) * 2 - 0.5).to(dev)
    x[n_cap // 2, 0] = 1e-9  # x cells -1 and 0
    nd = torch.tensor([n], dtype=torch.int32, device=dev)
    la = torch.tensor([active], dtype=torch.int32, device=dev)
    s, E, H, NH = stream_of(dev), 2 * L, 64, 2
    rows, lev = torch.zeros(n_cap, E, device=dev), torch.zeros(L, n_cap, 2, device=dev)
    if half:
        call("sn_hashgrid_fwd16_dev", ptr(x), n_cap, ptr(nd), ptr(t16), L, 2, log2_T, 16, 1.38, L,
             ptr(la), ptr(rows), s)
    else:
        call("sn_hashgrid_fwd_dev", ptr(x), n_cap, ptr(nd), ptr(tab), L, 2, log2_T, 16, 1.38, L,
             ptr(la), ptr(rows), s)
    call("sn_hashgrid_fwd_levels_dev", ptr(x), n_cap, ptr(nd), ptr(tab), ptr(t16), L, log2_T, 16,
         1.38, L, ptr(la), ptr(lev), s)
    assert torch.equal(lev.permute(1, 0, 2).reshape(n_cap, E), rows)

    lib = _lib.lib()
    np_ = lib.sn_mlp_n_params(3 + E, H, NH)
    mlp, gs = r(np_) * 0.2, r(n_cap)
    name = "sn_mlp16" if half else "sn_mlp"
    out = []
    for sfx, enc in (("", rows), ("_levels", lev)):
        sdf, ge = torch.zeros(n_cap, device=dev), torch.zeros(n_cap, E, device=dev)
        gm = torch.zeros(np_, device=dev)
        call(name + "_fwd" + sfx, ptr(x), ptr(enc), E, n_cap, ptr(nd), ptr(mlp), H, NH, 100.0,
             ptr(sdf), *(() if half else (None,)), s)
        ws = torch.empty(lib.sn_mlp16_bwd_workspace_bytes(n_cap, E, H, NH) if half else
                         lib.sn_mlp_bwd_workspace_bytes(n_cap, E, H, NH, 0), dtype=torch.uint8,
                         device=dev)
        call(name + "_bwd" + sfx, ptr(x), ptr(enc), E, n_cap, ptr(nd), ptr(mlp), H, NH, 100.0,
             ptr(gs), ptr(ge), None, ptr(gm), 0, ptr(ws), ws.numel(), s)
        out.append((sdf, ge, gm))
    for a, b in zip(*out):
        assert torch.equal(a, b)
