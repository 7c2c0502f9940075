"""The fp32 MLP kernels (sn_mlp_fwd, sn_mlp_bwd, sn_mlp_bwd_ad) against fp64
autograd at the edges of their tiles: 16 points per wavefront, 64 per
workgroup step, inputs padded to blocks of 16, rows of the encoding that
allow 16-byte loads or not.

Tolerance: a value is a chain of at most three dot products of <= 64 terms
(and for weight gradients a sum over the points), each fp32 operation off by
2^-24 relative to the largest partial sum; 64 roundings in a row of one sign
are 4e-6, so 1e-5 of the largest reference value."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

RTOL = 1e-5


def _close(got, ref, name):
    err = (got.double().cpu() - ref.cpu()).abs().max().item()
    assert err <= RTOL * max(ref.abs().max().item(), 1e-30), f"{name}: {err}"


def _reference(x, enc, layers, a, v, vd):
    """sdf, dsdf/dh0, and for J = sum a sdf (+ the tangent of sdf along
    (v, vd)) the gradients to every weight, to h0 and to the tangent input."""
    h0 = torch.cat([x, enc], 1).requires_grad_(True)
    t0 = torch.cat([v, vd], 1).requires_grad_(True)
    ws = [(W.clone().requires_grad_(True), b.clone().requires_grad_(True)) for W, b in layers]

    def field(h):
        for i, (W, b) in enumerate(ws):
            h = F.linear(h, W, b)
            if i < len(ws) - 1:
                h = F.softplus(h, beta=100)
        return h[:, 0]

    f = field(h0)
    g, = torch.autograd.grad(f.sum(), h0, create_graph=True)
    flat = [t for p in ws for t in p]
    plain = torch.autograd.grad((a * f).sum(), [h0] + flat, retain_graph=True)
    J = (a * f).sum() + (g * t0).sum()
    both = torch.autograd.grad(J, [h0, t0] + flat, allow_unused=True)
    both = [torch.zeros_like(t) if q is None else q for q, t in zip(both, [h0, t0] + flat)]
    cat = lambda ts: torch.cat([t.reshape(-1) for t in ts])
    return f.detach(), g.detach(), plain[0], cat(plain[1:]), both[0], both[1], cat(both[2:])


@pytest.mark.parametrize("E", [5, 13, 16, 29, 32, 45, 60, 61])
@pytest.mark.parametrize("H,NH", [(32, 1), (64, 2)])
@pytest.mark.parametrize("n", [1, 63, 257, 40001])
def test_mlp32_vs_fp64(n, H, NH, E, dev):
    from supernormal_amd import _lib
    from supernormal_amd._lib import call, ptr, stream_of
    g = torch.Generator().manual_seed(n * 100 + E)
    rn = lambda *s: torch.randn(*s, generator=g, dtype=torch.float32)
    x, enc, v, vd, a = rn(n, 3) * 0.5, rn(n, E) * 0.1, rn(n, 3), rn(n, E), rn(n)
    dims = [3 + E] + [H] * NH + [1]
    layers = [(rn(dims[i + 1], dims[i]) / dims[i] ** 0.5, 0.1 * rn(dims[i + 1]))
              for i in range(NH + 1)]
    d64 = lambda t: t.double()
    f, gr, p_h0, p_w, b_h0, b_t0, b_w = _reference(
        d64(x), d64(enc), [(d64(W), d64(b)) for W, b in layers], d64(a), d64(v), d64(vd))
    x, enc, v, vd, a = (t.to(dev) for t in (x, enc, v, vd, a))
    mlp = torch.cat([t.reshape(-1) for p in layers for t in p]).to(dev)
    s = stream_of(dev)
    sdf, sdf2, dh0 = torch.empty(n, device=dev), torch.empty(n, device=dev), \
        torch.empty(n, 3 + E, device=dev)
    call("sn_mlp_fwd", ptr(x), ptr(enc), E, n, None, ptr(mlp), H, NH, 100.0, ptr(sdf), None, s)
    call("sn_mlp_fwd", ptr(x), ptr(enc), E, n, None, ptr(mlp), H, NH, 100.0, ptr(sdf2), ptr(dh0), s)
    _close(sdf, f, "sdf")
    assert torch.equal(sdf, sdf2)
    _close(dh0, gr, "dsdf/dh0")
    lib = _lib.lib()
    ws = torch.empty(lib.sn_mlp_bwd_workspace_bytes(n, E, H, NH, 0), dtype=torch.uint8, device=dev)
    ge, gx, gw = torch.empty_like(enc), torch.empty_like(x), torch.empty_like(mlp)
    call("sn_mlp_bwd", ptr(x), ptr(enc), E, n, None, ptr(mlp), H, NH, 100.0, ptr(a), ptr(ge),
         ptr(gx), ptr(gw), 0, ptr(ws), ws.numel(), s)
    _close(gx, p_h0[:, :3], "dL/dx")
    _close(ge, p_h0[:, 3:], "dL/denc")
    _close(gw, p_w, "dL/dW")
    ws = torch.empty(lib.sn_mlp_bwd_workspace_bytes(n, E, H, NH, 1), dtype=torch.uint8, device=dev)
    o1, o2 = torch.empty(n, 3 + E, device=dev), torch.empty(n, 3 + E, device=dev)
    call("sn_mlp_bwd_ad", ptr(x), ptr(enc), ptr(v), ptr(vd), E, n, None, ptr(mlp), H, NH, 100.0,
         ptr(a), ptr(o1), ptr(o2), ptr(gw), 0, ptr(ws), ws.numel(), s)
    _close(o1, b_h0, "dJ/dh0")
    _close(o2, b_t0, "dJ/dhd0")
    _close(gw, b_w, "dJ/dW")
    e1, e2 = torch.empty_like(enc), torch.empty_like(enc)
    call("sn_mlp_bwd_ad_enc", ptr(x), ptr(enc), ptr(v), ptr(vd), E, n, None, ptr(mlp), H, NH,
         100.0, ptr(a), ptr(e1), ptr(e2), ptr(gw), 0, ptr(ws), ws.numel(), s)
    assert torch.equal(e1, o1[:, 3:].contiguous()) and torch.equal(e2, o2[:, 3:].contiguous())
