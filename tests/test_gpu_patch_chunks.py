"""Patch weights, transmittance, their backward, accumulation and packing where
their kernels' chunks end: 1024 values of a patch at a time in LDS (P <= 64), 16
samples ahead per ray (P > 64), 64 sorted indices per wavefront.  Forward: the
bits of the sequential loop in fp32 (numpy); backward: autograd in fp64, whose
sums of at most 2100 terms an fp32 recurrence follows within 2100 * 2^-24 =
1.3e-4 of the largest value."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P,counts", [
    (9, [0, 1, 112, 113, 114, 227, 2]), (1, [1023, 1024, 1025, 2049, 0]), (64, [15, 16, 17, 33]),
    (65, [15, 16, 17, 1, 0, 40]), (7, [146, 147, 300])])
@pytest.mark.parametrize("outs", ["w", "T", "wT"])
def test_patch_weights_at_chunk_ends(P, counts, outs, dev):
    from supernormal_amd._lib import call, ptr, stream_of
    g = torch.Generator().manual_seed(P)
    S, B = sum(counts), len(counts)
    # (a patch's largest opacities are 1: nothing behind them, finite backward)
    al = (torch.rand(S, P, generator=g) ** 6 * 0.2).float()
    al[::50] = 1.0
    cn = torch.tensor(counts)
    pk = torch.stack([torch.cumsum(cn, 0) - cn, cn], -1).int()
    gw = torch.randn(S, P, generator=g) if "w" in outs else None
    gT = torch.randn(S, P, generator=g) if "T" in outs else None
    w = np.zeros((S, P), np.float32)
    T = np.zeros((S, P), np.float32)
    a = al.numpy()
    for b, c in pk.tolist():
        t = np.ones(P, np.float32)
        for s in range(b, b + c):
            T[s], w[s] = t, a[s] * t
            t = t * (np.float32(1) - a[s])
    D = lambda t: None if t is None else t.contiguous().to(dev)
    ald, pkd = D(al), D(pk)
    wd, Td = (torch.zeros(S, P, device=dev) if k in outs else None for k in "wT")
    call("sn_patch_weight_fwd", ptr(pkd), B, P, S, ptr(ald), ptr(wd), ptr(Td), stream_of(dev))
    for got, ref in ((wd, w), (Td, T)):
        if got is not None:
            np.testing.assert_array_equal(got.cpu().numpy(), ref)
    x = al.double().requires_grad_(True)
    J = 0.0
    for b, c in pk.tolist():
        if c:
            t = torch.cumprod(torch.cat([torch.ones(1, P, dtype=torch.float64),
                                         1 - x[b:b + c]]), 0)[:-1]
            J = J + ((gw[b:b + c].double() * x[b:b + c] * t).sum() if gw is not None else 0)
            J = J + ((gT[b:b + c].double() * t).sum() if gT is not None else 0)
    J.backward()
    gwd, gTd, ga = D(gw), D(gT), torch.zeros(S, P, device=dev)
    call("sn_patch_weight_bwd", ptr(pkd), B, P, S, ptr(ald), ptr(gwd), ptr(gTd), ptr(ga),
         stream_of(dev))
    assert float((ga.cpu().double() - x.grad).abs().max()) <= 1.3e-4 * float(x.grad.abs().max())


@pytest.mark.parametrize("n,row,kind", [(1, 1, "sorted"), (63, 27, "sorted"), (65, 3, "random"),
                                        (4097, 27, "sorted"), (40000, 27, "random"),
                                        (300000, 1, "one"), (129, 9, "bad")])
def test_sorted_runs(n, row, kind, dev):
    """Accumulation by index and packed counts, indices in runs or not, some out
    of range; whole numbers as values: every sum is exact in fp32."""
    from supernormal_amd import _lib
    from supernormal_amd._lib import call, ptr, stream_of
    g = torch.Generator().manual_seed(n)
    m = 50
    idx = torch.randint(0, m, (n,), generator=g)
    if kind == "sorted":
        idx = idx.sort().values
    elif kind == "one":
        idx[:] = 7
    elif kind == "bad":
        idx[::5] = -3
        idx[1::7] = m
    v = torch.randint(-8, 9, (n, row), generator=g).float()
    ok = (idx >= 0) & (idx < m)
    ref = torch.zeros(m, row).index_add_(0, idx[ok], v[ok])
    out = torch.zeros(m, row, device=dev)
    di, dv = idx.to(dev), v.to(dev)
    call("sn_scatter_add_rows", ptr(di), n, row, ptr(dv), ptr(out), m, stream_of(dev))
    assert torch.equal(out.cpu(), ref)
    pk = torch.zeros(m, 2, dtype=torch.int32, device=dev)
    bad = torch.zeros(1, dtype=torch.int32, device=dev)
    nb = _lib.lib().sn_pack_info_workspace_bytes(m)
    ws = torch.zeros(max(int(nb), 1), dtype=torch.uint8, device=dev)
    call("sn_pack_info", ptr(di), n, m, ptr(pk), ptr(bad), ptr(ws), ws.numel(), stream_of(dev))
    cnt = torch.bincount(idx[ok], minlength=m)
    assert torch.equal(pk[:, 1].cpu().long(), cnt) and int(bad) == int((~ok).sum())
