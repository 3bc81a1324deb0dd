"""GPU: nxg_upload_words and the offsets and scales that go by it: sizes around a launch's 896
words, past the largest (which takes torch's copy), and calls in a row whose host arrays are
changed right after the call."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as t
    assert t.cuda.is_available(), "no GPU"
    return t


@pytest.mark.parametrize("n", [1, 255, 257, 895, 896, 897, 3584, 3585])
def test_words_arrive(nxg, torch, n):
    print(f"upload {n} words", flush=True)
    nxg.init()
    a = np.random.default_rng(n).integers(-2**31, 2**31, n).astype(np.int32)
    f = np.random.default_rng(n).standard_normal(n).astype(np.float32)
    ta, tf = nxg._uploaded(a, torch.device("cuda")), nxg._uploaded(f, torch.device("cuda"))
    ref_a, ref_f = a.copy(), f.copy()
    a[:], f[:] = 0, 0                     # read before the call returned
    assert (ta.cpu().numpy() == ref_a).all() and (tf.cpu().numpy() == ref_f).all()
    assert ta.dtype == torch.int32 and tf.dtype == torch.float32


def test_refused(nxg, torch):
    nxg.init()
    L = nxg.load_library()
    d = torch.empty(16, dtype=torch.int32, device="cuda")
    a = np.zeros(16, np.int32)
    assert L.nxg_upload_words(a.ctypes.data, 3585, d.data_ptr(), None) == nxg.NXG_EINVAL
    assert L.nxg_upload_words(a.ctypes.data, -1, d.data_ptr(), None) == nxg.NXG_EINVAL
    assert L.nxg_upload_words(None, 4, d.data_ptr(), None) == nxg.NXG_EINVAL
    assert L.nxg_upload_words(a.ctypes.data, 4, d.data_ptr() + 2, None) == nxg.NXG_EINVAL
    assert L.nxg_upload_words(None, 0, None, None) == nxg.NXG_OK
