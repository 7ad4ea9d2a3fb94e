"""dX of fp16 and fp32 layers finished in the weight-gradient launch: the fp32 dX^T of
backward_features transposed and converted, bit for bit."""
import pytest
import torch

import haste_amd
from haste_amd import ops
from test_gpu_ffi import make_case

pytestmark = pytest.mark.gpu


# one row and column of the 32 x 32 tiles, whole tiles, one more; several slices
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("B,D,O,G,F", [(1, 33, 40, 16, 16), (32, 64, 3000, 32, 32),
                                       (33, 300, 9001, 64, 64), (70, 1000, 5000, 16, 48)])
def test_dx_is_dxt_converted(dev, B, D, O, G, F, dtype):
    x, W, bias, idx, dY = (t.to(dev) for t in make_case(B, D, O, G, F, idx_mode="random"))
    x, W, bias, dY = (t.to(dtype) for t in (x, W, bias, dY))
    xr, Wr, br = (t.clone().requires_grad_(True) for t in (x, W, bias))
    ops.group_ffi_mul(xr, Wr, idx, br, G).backward(dY)
    xT = x.t().contiguous()
    dxt = haste_amd.backward_features(xT, W, idx, dY, G)
    assert xr.grad.dtype == dtype and torch.equal(xr.grad, dxt.t().to(dtype))
    assert torch.equal(Wr.grad, haste_amd.backward_weights(xT, W, idx, dY, G))
    # dX with the bias gradient only, and alone
    xb, bb = x.clone().requires_grad_(True), bias.clone().requires_grad_(True)
    ops.group_ffi_mul(xb, W, idx, bb, G).backward(dY)
    assert torch.equal(xb.grad, xr.grad) and torch.equal(bb.grad, br.grad)
    xa = x.clone().requires_grad_(True)
    ops.group_ffi_mul(xa, W, idx, None, G).backward(dY)
    assert torch.equal(xa.grad, xr.grad)
