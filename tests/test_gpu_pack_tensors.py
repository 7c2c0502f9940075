"""pack_weight_norm (one launch each way on the layers' own tensors) against fp64
autograd of torch.nn.utils.weight_norm's formula; tolerance as the flat form's
(fp32 row sums of at most 64 squares against fp64: 1e-5).  Under create_graph
the gradient has a graph of its own, as the torch form's."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shapes,has_g", [(((64, 35), (64, 64), (1, 64)), True),
                                          (((32, 3), (1, 32)), True), (((5, 67), (1, 5)), False)])
def test_pack_tensors_vs_fp64(shapes, has_g, dev):
    from supernormal_amd.sdf import _PackFn, fold_weight_norm, pack_mlp, pack_weight_norm
    g = torch.Generator().manual_seed(len(shapes))
    r = lambda *s: torch.randn(*s, generator=g)
    cpu = [(r(o, i), r(o, 1) if has_g else None, r(o)) for o, i in shapes]
    leaf = lambda t, **k: None if t is None else t.to(**k).requires_grad_(True)
    a = [tuple(leaf(t, device=dev) for t in lay) for lay in cpu]
    b = [tuple(leaf(t, dtype=torch.float64) for t in lay) for lay in cpu]
    pa = pack_weight_norm(a)
    assert type(pa.grad_fn).__name__ == _PackFn.__name__ + "Backward"
    pb = pack_mlp([(fold_weight_norm(v, s), c) for v, s, c in b])
    w = r(pb.numel())
    la = [t for lay in a for t in lay if t is not None]
    lb = [t for lay in b for t in lay if t is not None]
    ga = torch.autograd.grad(pa, la, w.to(dev), retain_graph=True)
    gb = torch.autograd.grad(pb, lb, w.double(), retain_graph=True)
    for x, y in ((pa, pb), *zip(ga, gb)):
        torch.testing.assert_close(x.cpu().double(), y, rtol=1e-5, atol=1e-5)
    if has_g:
        sa = sum((t * t).sum() for t in torch.autograd.grad(pa, la, w.to(dev), create_graph=True))
        sb = sum((t * t).sum() for t in torch.autograd.grad(pb, lb, w.double(), create_graph=True))
        for x, y in zip(torch.autograd.grad(sa, la[:2]), torch.autograd.grad(sb, lb[:2])):
            torch.testing.assert_close(x.cpu().double(), y, rtol=1e-4,
                                       atol=1e-4 * float(y.abs().max()))


def test_pack_on_cpu_and_other_types_takes_torch():
    from supernormal_amd.sdf import pack_weight_norm
    v = torch.randn(4, 3, dtype=torch.float64, requires_grad=True)
    s, b = torch.randn(4, 1, dtype=torch.float64), torch.randn(4, dtype=torch.float64)
    p = pack_weight_norm([(v, s, b)])
    torch.testing.assert_close(p[:12].view(4, 3), s * v / v.norm(dim=1, keepdim=True))
