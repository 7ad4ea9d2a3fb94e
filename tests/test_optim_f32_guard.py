"""Which fp32 parameters SRSgd hands to its kernel by address: the others take torch's ops."""
import pytest
import torch

from haste_amd import optim_sr
from haste_amd.optim_sr import SRSgd

CPU = torch.device("cpu")


class Sub(torch.Tensor):
    pass


def triple(n=6):
    return torch.nn.Parameter(torch.ones(n)), torch.ones(n), torch.zeros(n)


def test_plain_tensors_on_the_device():
    p, g, m = triple()
    assert optim_sr._fusable_f32(p, g, m, CPU) and optim_sr._fusable_f32(p, g, None, CPU)
    assert not optim_sr._fusable_f32(p, g, m, torch.device("cuda", 0))


@pytest.mark.parametrize("other", [
    lambda t: t.to("meta"), lambda t: t.double(), lambda t: t.half(), lambda t: t.as_subclass(Sub),
    lambda t: t[:-1], lambda t: t.view(2, 3), lambda t: t.repeat(2)[::2], lambda t: t.to_sparse(),
    torch._neg_view,
], ids=["device", "wider", "narrower", "subclass", "shorter", "shape", "strided", "sparse", "neg"])
def test_any_other_tensor(other):
    p, g, m = triple()
    assert not optim_sr._fusable_f32(p, other(g), m, CPU)
    assert not optim_sr._fusable_f32(p, g, other(m), CPU)


@pytest.mark.parametrize("data", [
    torch.ones(6, device="meta"), torch.ones(6).double(), torch.ones(6).as_subclass(Sub),
    torch.ones(12)[::2], torch._neg_view(torch.ones(6))],
    ids=["device", "wider", "subclass", "strided", "neg"])
def test_any_other_parameter(data):
    p = torch.nn.Parameter(data)
    assert not optim_sr._fusable_f32(p, torch.ones(6), None, CPU)


def overlapping(triples):
    return optim_sr._overlapping([(*optim_sr._span(t), t is not g) for p, g, m in triples
                                  for t in (p, g, m) if t is not None and optim_sr._span(t)])


def test_overlapping():
    flat = torch.zeros(12)
    a, b, c = (torch.nn.Parameter(flat[i:j]) for i, j in ((0, 6), (6, 12), (5, 7)))
    g, h = torch.ones(6), torch.ones(2)
    assert not overlapping([(a, g, None), (b, g, None)])   # a shared grad is only read
    assert overlapping([(a, g, None), (c, h, None)])
    assert overlapping([(a, g, None), (a, g, None)])
    assert overlapping([(a, b.data, None), (b, g, None)])            # one's grad is the other
    assert overlapping([(a, g, torch.zeros(6)), (b, g, flat[:6])])
    t = torch.nn.Parameter(flat.view(3, 4).t())
    assert overlapping([(b, g, None), (t, torch.ones(4, 3), None)])
    assert not overlapping([(torch.nn.Parameter(torch.zeros(0)), torch.zeros(0), None)])


@pytest.mark.gpu
def test_momentum_left_on_the_host_is_refused(dev):
    p = torch.nn.Parameter(torch.ones(5))
    opt = SRSgd([p], lr=0.1, momentum=0.9)
    p.data = p.data.to(dev)
    p.grad = torch.ones(5, device=dev)
    with pytest.raises(RuntimeError, match="same device"):
        opt.step()


@pytest.mark.gpu
@pytest.mark.parametrize("momentum", [0.0, 0.9])
def test_shared_storage_is_stepped_in_order(dev, momentum):
    w = torch.randn(70001, device=dev)
    ref = w.clone()
    ps = [torch.nn.Parameter(w), torch.nn.Parameter(w[1:].view(1, -1))]
    views = [ref, ref[1:].view(1, -1)]
    bufs = [torch.zeros_like(r) for r in views]
    opt = SRSgd(ps, lr=0.1, weight_decay=0.01, momentum=momentum)
    for _ in range(2):
        for p, r, m in zip(ps, views, bufs):
            p.grad = torch.randn_like(p)
            u = p.grad.add(r, alpha=0.01)
            if momentum:
                u = m.mul_(momentum).add_(u)
            r.add_(u, alpha=-0.1)
        opt.step()
    assert torch.equal(w, ref)


@pytest.mark.gpu
def test_kernel_and_torch_ops_in_one_group(dev):
    """Parameters for the kernel and one that is not contiguous, apart and sharing memory."""
    for shared in (False, True):
        w = torch.randn(40, 30, device=dev)
        ts = [torch.randn(7, device=dev), w.t() if shared else torch.randn(30, 40, device=dev).t(),
              w, torch.zeros(0, device=dev)]
        ref = [t.clone() for t in ts]
        if shared:
            ref[1] = ref[2].t()
        ps = [torch.nn.Parameter(t) for t in ts]
        v = [p._version for p in ps]
        for p, r in zip(ps, ref):
            p.grad = torch.randn(p.shape, device=dev)
            r.add_(p.grad, alpha=-0.5)
        SRSgd(ps, lr=0.5).step()
        assert all(torch.equal(p, r) for p, r in zip(ps, ref))
        assert all(p._version > a for p, a in zip(ps, v))
