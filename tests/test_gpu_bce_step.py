"""FFITrainStep.step_bce, whose label and loss work rides in other launches, against
the separate calls, bit for bit."""
import pytest
import torch

from haste_amd.step import FFITrainStep

pytestmark = pytest.mark.gpu


# no labels, one, a workgroup's 256 and one more, more label workgroups than the
# transpose has columns; repeated pairs and pairs out of range; steps in turn with
# other labels (the bits are cleared)
@pytest.mark.parametrize("device_seed", [False, True])
@pytest.mark.parametrize("nnz", [0, 1, 256, 257, 3000])
@pytest.mark.parametrize("B,D,O,G,F", [(1, 40, 70, 16, 16), (64, 300, 2049, 64, 64),
                                       (130, 500, 1300, 128, 48)])
def test_step_bce_is_its_parts(dev, B, D, O, G, F, nnz, device_seed):
    g = torch.Generator(device=dev).manual_seed(nnz + B)
    x = torch.randn(B, D, generator=g, device=dev).bfloat16()
    W = (torch.rand(O, F, generator=g, device=dev) - 0.5).bfloat16()
    bias = torch.randn(O, generator=g, device=dev).bfloat16()
    idx = torch.randint(D, (-(-O // G), F), generator=g, device=dev, dtype=torch.int32)
    mk = lambda: FFITrainStep(W.clone(), bias.clone(), idx, B, D, G, 0.01, 1e-4, seed=3,
                              device_seed=device_seed)
    a, b = mk(), mk()
    for k in range(3):
        lab = torch.stack([torch.randint(-1, B + 1, (nnz,), generator=g, device=dev),
                           torch.randint(-1, O + 1, (nnz,), generator=g, device=dev)], 1).int()
        la = a.step_bce(x, lab).clone()
        lb = b.forward_bce(x, lab).clone()
        b.backward_features(b.dY_buf, b.ldo, defer_dx=True)
        b.backward_weights_sgd(b.dY_buf, b.ldo)
        assert torch.equal(la, lb)
        assert torch.equal(a.dY_buf, b.dY_buf) and torch.equal(a.dX, b.dX)
        assert torch.equal(a.W, b.W) and torch.equal(a.bias, b.bias)
        nb = a.B * (-(-(-(-O // G) * G) // 32)) * 4
        assert not a.bce_ws[:nb].any()
    assert a.current_seed() == b.current_seed()
