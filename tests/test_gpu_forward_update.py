"""The weight update that also computes the logits (FFITrainStep.step,
haste_ffi_forward_bwd_weights_sgd_dx) against the calls it joins, bit for bit."""
import pytest
import torch

from haste_amd import _lib
from haste_amd.step import FFITrainStep

pytestmark = pytest.mark.gpu


def case(dev, B, D, O, G, F, seed=0):
    g = torch.Generator(device=dev).manual_seed(seed)
    Gc = -(-O // G)
    x = torch.randn(B, D, generator=g, device=dev).bfloat16()
    W = (torch.rand(O, F, generator=g, device=dev) - 0.5).bfloat16()
    bias = torch.randn(O, generator=g, device=dev).bfloat16()
    idx = torch.randint(D, (Gc, F), generator=g, device=dev, dtype=torch.int32)
    dY = (torch.randn(B, O + 24, generator=g, device=dev) * 0.1).bfloat16()
    return x, W, bias, idx, dY


def both(dev, x, W, bias, idx, G, dYs, device_seed=False):
    """(fused, separate) steps on copies, two steps each."""
    out = []
    for fused in (True, False):
        b = None if bias is None else bias.clone()
        st = FFITrainStep(W.clone(), b, idx, x.shape[0], x.shape[1], G, 0.01, 1e-4, seed=5,
                          device_seed=device_seed)
        st.logits_buf.fill_(7.0)
        for dY, ld in dYs:
            if fused:
                st.step(x, dY, ld)
            else:
                st.forward(x)
                st.backward_features(dY, ld, defer_dx=True)
                st.backward_weights_sgd(dY, ld)
        out.append(st)
    return out


# one chunk of 64 (32) batch rows, one more row, odd and even chunk counts; a last
# group of one label and of all but one; fan-ins between the kernel's sizes
@pytest.mark.parametrize("G", [16, 32, 64, 128])
@pytest.mark.parametrize("B,D,F,extra", [(1, 40, 16, 1), (64, 300, 32, 0), (65, 300, 48, 1),
                                         (130, 500, 64, -1), (33, 700, 96, 5), (200, 768, 128, 1),
                                         (97, 700, 176, -1), (160, 1024, 256, 1)])
def test_step_is_its_parts(dev, G, B, D, F, extra):
    O = 5 * G + extra
    x, W, bias, idx, dY = case(dev, B, D, O, G, F, seed=B + F)
    ld = (O + 7) // 8 * 8
    dYs = [(dY[:, :ld].contiguous(), ld), (dY[:, 8:8 + ld].contiguous(), ld)]
    a, b = both(dev, x, W, bias, idx, G, dYs)
    assert torch.equal(a.logits, b.logits)
    assert torch.equal(a.dX, b.dX)
    assert torch.equal(a.W, b.W)
    assert torch.equal(a.bias, b.bias)
    pad = a.logits_buf[:, (O + 7) // 8 * 8:]
    assert torch.all(pad == 7.0)


def test_without_bias_and_with_device_seed(dev):
    x, W, _, idx, dY = case(dev, 100, 300, 321, 64, 64)
    dYs = [(dY[:, :328].contiguous(), 328)] * 2
    a, b = both(dev, x, W, None, idx, 64, dYs, device_seed=True)
    assert torch.equal(a.logits, b.logits) and torch.equal(a.W, b.W) and torch.equal(a.dX, b.dX)
    assert a.current_seed() == b.current_seed() == 7


def test_rows_off_16_bytes_and_dY_in_the_logits(dev):
    x, W, bias, idx, dY = case(dev, 70, 300, 321, 32, 64)
    odd = dY[:, :321].contiguous()
    a, b = both(dev, x, W, bias, idx, 32, [(odd, 321)] * 2)
    assert torch.equal(a.logits, b.logits) and torch.equal(a.W, b.W) and torch.equal(a.dX, b.dX)
    # dY in the logits buffer: the step reads the logits it has just written
    for st in (a, b):
        st.logits_buf.zero_()
    a.step(x, a.logits_buf, a.ldo)
    b.forward(x)
    b.backward_features(b.logits_buf, b.ldo, defer_dx=True)
    b.backward_weights_sgd(b.logits_buf, b.ldo)
    assert torch.equal(a.logits, b.logits) and torch.equal(a.W, b.W) and torch.equal(a.dX, b.dX)


@pytest.mark.parametrize("G,F", [(16, 32), (64, 64), (128, 128)])
def test_step_is_its_parts_with_streamed_dY(dev, G, F):
    """dY just above the size from which the launch loads it without keeping it in the caches."""
    B, D, O = 512, 300, 270001
    x, W, bias, idx, dY = case(dev, B, D, O, G, F)
    ld = (O + 7) // 8 * 8
    dY = dY[:, :ld].contiguous()
    assert (256 << 20) < dY.numel() * 2 < (272 << 20)
    a, b = both(dev, x, W, bias, idx, G, [(dY, ld)] * 2)
    assert _lib.lib().haste_ffi_forward_bwd_weights_joined(dY.data_ptr(), ld, a.ldo, B, F, O, G) == 1
    assert torch.equal(a.logits, b.logits) and torch.equal(a.dX, b.dX)
    assert torch.equal(a.W, b.W) and torch.equal(a.bias, b.bias)
