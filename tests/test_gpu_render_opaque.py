"""The fused rendering step's fine form: its mask loss on opaque and grazing rays, where 1 - sum
of the weights is far below 1 and the loss's gradient is at its largest.

Tolerance: 1 - sum w is the product of up to 128 factors e / (c + 1e-5), each
with a relative error of a few roundings (exponentials of arguments up to 12
rounded at 6e-8 relative, hardware reciprocals): 128 * 1.5e-6 = 2e-4 in norm
if all err alike.  Formed as 1 - sum w it would be 1e-3 to 1e-2 off."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("impl", [1, 0])
@pytest.mark.parametrize("Ph,Pw,cnt", [(3, 3, 1), (3, 3, 64), (3, 3, 65), (2, 4, 63), (2, 4, 128)])
def test_mask_loss_of_opaque_rays(Ph, Pw, cnt, impl, dev):
    from supernormal_amd import _lib
    from supernormal_amd._lib import call, ptr, stream_of
    B, P, inv_s = 5, Ph * Pw, 60.0
    g = torch.Generator().manual_seed(Ph * 100 + cnt)
    S = B * cnt
    # a ray passes the surface once and ends at sigma(s f) = 2e-5 .. 1e-3
    lo = -(6.9 + 3.9 * torch.rand(B, 1, P, generator=g)) / inv_s
    f = 0.1 + (lo - 0.1) * (torch.arange(cnt + 1) / cnt)[None, :, None]
    f = f.float()
    ss, se = f[:, :-1].reshape(S, P).contiguous(), f[:, -1].contiguous()
    di = torch.full((S,), -1, dtype=torch.int32)
    di[cnt - 1::cnt] = torch.arange(B, dtype=torch.int32)
    # fp64: weights, mask loss, gradient
    a, z = ss.double().requires_grad_(True), se.double().requires_grad_(True)
    full = torch.cat([a.view(B, cnt, P), z[:, None]], 1)
    sg = torch.sigmoid(full * inv_s)
    alpha = ((sg[:, :-1] - sg[:, 1:] + 1e-5) / (sg[:, :-1] + 1e-5)).clip(0, 1)
    T = torch.cumprod(torch.cat([torch.ones(B, 1, P, dtype=torch.float64), 1 - alpha], 1), 1)
    ws = (alpha * T[:, :-1]).sum(1).clip(1e-5, 1 - 1e-5)
    torch.nn.functional.binary_cross_entropy(ws, torch.zeros_like(ws)).backward()
    D = lambda t: t.float().contiguous().to(dev)
    o = torch.zeros(B, P, 3)
    d = torch.randn(B, P, 3, generator=g) * 0.01 + torch.tensor([0.0, 0.0, 1.0])
    buf = dict(o=D(o), d=D(d), n=D(torch.tensor([[0.0, 0.0, 1.0]]).expand(B, 3)),
               nt=D(torch.ones(B, P, 3)), m=D(torch.zeros(B, P)),
               pk=torch.stack([torch.arange(B) * cnt, torch.full((B,), cnt)], -1).int().to(dev),
               t=D(torch.arange(S)), t1=D(torch.arange(S) + 1.0), di=di.to(dev), ss=D(ss), se=D(se),
               gs=D(torch.ones(S, P, 3)), inv=D(torch.tensor([inv_s])),
               ms=D(torch.tensor([1.0])), ns=torch.tensor([S], dtype=torch.int32, device=dev))
    g_ss, g_se = torch.empty(S, P, device=dev), torch.empty(B, P, device=dev)
    g_gs, losses = torch.empty(S, P, 3, device=dev), torch.empty(4, device=dev)
    part = torch.empty(4 * _lib.lib().sn_render_step_waves(B, P), device=dev)
    _lib.lib().sn_render_step_set_impl(impl)
    try:
        call("sn_render_step_fine", B, Ph, Pw, ptr(buf["o"]), ptr(buf["d"]), ptr(buf["n"]), None,
             ptr(buf["nt"]), ptr(buf["m"]), ptr(buf["pk"]), ptr(buf["t"]), ptr(buf["t1"]),
             ptr(buf["di"]), ptr(buf["ss"]), ptr(buf["se"]), ptr(buf["gs"]), ptr(buf["inv"]),
             ptr(buf["ms"]), ptr(buf["ns"]), 0.0, 0.0, 1.0, 0, ptr(g_ss), ptr(g_se), ptr(g_gs),
             ptr(losses), ptr(part), None, None, stream_of(dev))
        torch.cuda.synchronize()
    finally:
        _lib.lib().sn_render_step_set_impl(1)
    for got, ref in ((g_ss, a.grad), (g_se, z.grad)):
        assert float((got.cpu().double() - ref).norm()) <= 2e-4 * float(ref.norm())
