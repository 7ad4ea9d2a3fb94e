"""The fp32 layer's own passes against the torch ops they replace, bit for bit."""
import pytest
import torch

from haste_amd import _C
from haste_amd.optim_sr import SRSgd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wd", [0.0, 1e-3])
@pytest.mark.parametrize("mu", [0.0, 0.9])
def test_sgd_f32(dev, wd, mu):
    g = torch.Generator(device=dev).manual_seed(1)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev)
    # one element, around a vector and a block, more tensors than a launch takes,
    # one off 16-byte boundaries, one not contiguous
    ts = [rnd(n) for n in (1, 3, 4, 1023, 1024, 1025, 70001, 5, 6, 7)]
    ts += [rnd(1001)[1:], rnd(33, 20).t()]
    ts[2][:2] = torch.tensor([float("inf"), float("nan")], device=dev)
    ps = [torch.nn.Parameter(t) for t in ts]
    opt = SRSgd(ps, lr=0.05, weight_decay=wd, momentum=mu)
    ref = [p.detach().clone() for p in ps]
    buf = [torch.zeros_like(r) for r in ref]
    for _ in range(3):
        for p, r, m in zip(ps, ref, buf):
            p.grad = rnd(*p.shape)
            upd = p.grad.add(r, alpha=wd) if wd else p.grad
            if mu:
                m.mul_(mu).add_(upd)
                upd = m
            r.add_(upd, alpha=-0.05)
        v = [p._version for p in ps]
        opt.step()
        assert all(p._version > a for p, a in zip(ps, v))
    for p, r, m in zip(ps, ref, buf):
        assert torch.equal(p.detach().nan_to_num(7.0), r.nan_to_num(7.0))
        if mu:
            assert torch.equal(opt.state[p]["momentum_buf"].nan_to_num(7.0), m.nan_to_num(7.0))


@pytest.mark.parametrize("B,O,ld,off", [(1, 2, 2, 0), (3, 7, 7, 0), (5, 8, 8, 0), (4, 2049, 2049, 0),
                                        (7, 131, 140, 3), (64, 4096, 4096, 0),
                                        # rows sharing a workgroup: its last one partly filled,
                                        # widths around a power of two of pieces
                                        (600, 20, 20, 0), (257, 9, 9, 0), (33, 64, 67, 1),
                                        (5, 1025, 1025, 0), (3, 2047, 2047, 2)])
def test_compute_rows(dev, B, O, ld, off):
    buf = torch.randn(B * ld + 16, device=dev) * 100
    buf[off:off + 2] = torch.tensor([1e6, float("nan")], device=dev)
    t = torch.as_strided(buf, (B, O), (ld, 1), off)
    rows, ldo = _C.compute_rows(t)
    assert ldo % 64 == 0 and rows.data_ptr() % 16 == 0 and rows.stride() == (ldo, 1)
    assert torch.equal(rows.nan_to_num(7.0), t.to(torch.float16).nan_to_num(7.0))


def test_compute_rows_of_a_negated_view(dev):
    t = torch._neg_view(torch.randn(5, 37, device=dev))
    rows, _ = _C.compute_rows(t)
    assert torch.equal(rows, (-torch._neg_view(t)).to(torch.float16))
