"""haste_rewire_select (the k-th smallest (score, slot) key of a layer) and the prune
pass that takes given scores."""
import math

import numpy as np
import pytest
import torch

import oracle
from haste_amd import _C, _lib


def test_select_rejects_bad_arguments():
    L = _lib.lib()
    n = L.haste_rewire_select_workspace_size()
    assert n > 0 and n % 4 == 0
    assert L.haste_rewire_select(None, 10, 1, 16, 32, n, None) == _lib.HASTE_ERR_INVALID_ARG
    assert L.haste_rewire_select(16, 10, 0, 16, 32, n, None) == _lib.HASTE_ERR_INVALID_ARG
    assert L.haste_rewire_select(16, 10, 11, 16, 32, n, None) == _lib.HASTE_ERR_INVALID_ARG
    assert L.haste_rewire_select(16, 1 << 32, 1, 16, 32, n, None) == _lib.HASTE_ERR_INVALID_ARG
    assert L.haste_rewire_select(16, 10, 1, 16, 32, n - 4, None) == _lib.HASTE_ERR_INVALID_ARG


# sizes around one workgroup, one pass of the grid and the 1024 chunks of the ties
@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 255, 257, 1024, 3 * 1024 + 1, 300007])
@pytest.mark.parametrize("kind", ["distinct", "few_values", "equal", "zeros", "nan"])
def test_select(dev, n, kind):
    rng = np.random.default_rng(n)
    s = (0.05 + 0.01 * rng.random(n)).astype(np.float32)
    if kind == "few_values":
        s = np.round(s, 3)
    elif kind == "equal":
        s[:] = 0.125
    elif kind == "zeros":
        s[rng.random(n) < 0.4] = 0.0
    elif kind == "nan":
        s[rng.random(n) < 0.2] = np.nan
        s[rng.random(n) < 0.2] = -np.inf
        s[rng.random(n) < 0.2] = np.inf
    keys = np.sort((s.view(np.int32).astype(np.int64) << 32) | np.arange(n, dtype=np.int64))
    sd = torch.from_numpy(s).to(dev)
    nb = _lib.lib().haste_rewire_select_workspace_size()
    for k in sorted({1, n, max(1, n // 2), max(1, int(n * 0.15))}):
        ws = torch.zeros(nb, dtype=torch.uint8, device=dev)
        key = torch.empty(1, dtype=torch.int64, device=dev)
        _lib.call("haste_rewire_select", sd.data_ptr(), n, k, key.data_ptr(), ws.data_ptr(), nb,
                  _C.stream_of(sd))
        assert int(key.item()) == keys[k - 1], k


# more groups than resident workgroups, a partial last group, and groups whose
# rows are off 16-byte boundaries (the general kernel)
@pytest.mark.gpu
@pytest.mark.parametrize("O,F,G,D,init", [(150001, 64, 32, 768, "random"), (40000, 16, 16, 99, "zero"),
                                          (1001, 13, 7, 50, "random")])
def test_given_scores_prune(dev, O, F, G, D, init):
    rng = np.random.default_rng(O)
    bound = 1.0 / math.sqrt(F)
    w = oracle.f32_to_bf16_bits(rng.uniform(-bound, bound, (O, F)).astype(np.float32))
    Gc = (O + G - 1) // G
    idx = rng.integers(0, D, (Gc, F)).astype(np.int32)
    k = int(Gc * F * 0.15)
    im = oracle.INIT_RANDOM if init == "random" else oracle.INIT_ZERO
    ref_w, ref_idx, ref_n, _, _ = oracle.rewire_ex(
        w, idx, G, D, prune_mode=oracle.PRUNE_GLOBAL_FRACTION, score_mode=oracle.SCORE_MEAN, k=k,
        regrow_mode=oracle.REGROW_RANDOM, init_mode=im, bound=bound, seed=77)
    Wd = torch.from_numpy(w.view(np.int16)).to(dev)
    idxd = torch.from_numpy(idx).to(dev)
    st = _C.stream_of(Wd)
    scores = torch.empty(Gc, F, device=dev)
    key = torch.empty(1, dtype=torch.int64, device=dev)
    cnt = torch.zeros(1, dtype=torch.int32, device=dev)
    nb = _lib.lib().haste_rewire_select_workspace_size()
    ws = torch.zeros(nb, dtype=torch.uint8, device=dev)
    _lib.call("haste_rewire_scores", Wd.data_ptr(), _lib.DTYPE_BF16, None, 0, _lib.SCORE_MEAN,
              scores.data_ptr(), O, F, G, st)
    _lib.call("haste_rewire_select", scores.data_ptr(), Gc * F, k, key.data_ptr(), ws.data_ptr(),
              nb, st)
    _lib.call("haste_rewire_ex", Wd.data_ptr(), _lib.DTYPE_BF16, idxd.data_ptr(), None, 0,
              _lib.SCORE_MEAN, scores.data_ptr(), key.data_ptr(), None, cnt.data_ptr(), O, F, G, D,
              _lib.PRUNE_GLOBAL_FRACTION, 0.0, k, _lib.REGROW_RANDOM, im, bound, 77, st)
    assert int(cnt.item()) == ref_n == k
    assert np.array_equal(idxd.cpu().numpy(), ref_idx)
    assert np.array_equal(Wd.cpu().numpy().view(np.uint16), ref_w)
