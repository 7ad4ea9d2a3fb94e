"""The staged backward to features with two waves to a tile (ranges of at most four
tiles) against the oracle (fp32 sums in another order)."""
import pytest
import torch

import oracle
from bwdf_cases import HALF_CASES
from haste_amd import _C, _lib
from test_gpu_ffi import TOL32, make_case

pytestmark = pytest.mark.gpu


# (B, D, O, G, F): four tiles in one range at 32 and 64 batch columns,
# two ranges of three tiles; a partial last group; O odd, so that dY's rows are off 16-byte
# boundaries; batches of one row, of a tile and one row more
@pytest.mark.parametrize("mode", ["perm", "dups", "shared"])
@pytest.mark.parametrize("B,D,O,G,F", [(1, 768, 2000, 32, 64), (33, 768, 2001, 64, 64),
                                       (64, 300, 3000, 64, 64), (65, 300, 2999, 32, 64),
                                       (97, 600, 2500, 128, 64), (40, 1500, 3001, 64, 96),
                                       (70, 1700, 2000, 32, 80)])
def test_two_waves_to_a_tile(dev, B, D, O, G, F, mode):
    x, W, bias, idx, dY = make_case(B, D, O, G, F, idx_mode=mode, seed=B + F)
    # one group with every feature in the first range: more tiles than the pipeline's
    idx[-2] = torch.arange(F, dtype=torch.int32)
    dXT = _C.ffi_backward_features_cuda(x.t().contiguous().to(dev), W.to(dev), idx.to(dev),
                                        dY.to(dev), B, D, F, O, G)
    ref = oracle.ffi_backward_features(idx, W, dY, G, D)
    torch.testing.assert_close(dXT.cpu(), ref, **TOL32)


# front: in some windows of groups a range holds every feature, more tiles than the
# plan's window layout tracks
@pytest.mark.parametrize("mode", ["random", "dups", "front"])
@pytest.mark.parametrize("B,D,O,G,F", HALF_CASES)
def test_every_build_with_two_waves_to_a_tile(dev, B, D, O, G, F, mode):
    """One shape per build (tests/test_abi.py checks the coverage), whatever the default is."""
    x, W, bias, idx, dY = make_case(B, D, O, G, F, seed=D,
                                    idx_mode="random" if mode == "front" else mode)
    if mode == "front":
        idx[1::4] = torch.randperm(F).to(torch.int32)
        idx[2::4] = torch.randperm(F).to(torch.int32)
    prev = _lib.lib().haste_ffi_bwd_features_set_build(3)
    try:
        dXT = _C.ffi_backward_features_cuda(x.t().contiguous().to(dev), W.to(dev), idx.to(dev),
                                            dY.to(dev), B, D, F, O, G)
    finally:
        _lib.lib().haste_ffi_bwd_features_set_build(prev)
    ref = oracle.ffi_backward_features(idx, W, dY, G, D)
    torch.testing.assert_close(dXT.cpu(), ref, **TOL32)
