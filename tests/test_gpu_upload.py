"""GPU: nxg_upload_words and the offsets and scales that go by it: sizes around a launch's 896
words, past the largest (which takes torch's copy), calls in a row whose host arrays are
changed right after the call, and calls recorded in a graph."""
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


def test_captured_calls_keep_the_words_of_capture_time(nxg, torch):
    """Host offsets and scales of calls under graph capture: every replay uses those of capture time,
    whatever happens to the arrays afterwards, with eager work of the same calls in between."""
    nxg.init()
    g = torch.Generator("cuda").manual_seed(4)
    T, H, G = 150, 4, 2
    new = lambda *shape: torch.randn(*shape, device="cuda", generator=g)
    q, k, v, a, x, b, taps = new(T, H * 64), new(G, T, 64), new(G, T, 64), *(new(T, 64) for _ in range(3)), new(5, 64)
    cu, scale = np.array([0, 40, 41, T], np.int32), np.array([0.1, 0.2, 0.3], np.float32)

    def calls(cu, scale):
        return nxg.attention(q, k, v, cu, scale, H, G), nxg.lily_state_quantize_rows(a, x, b, taps, cu)

    def same(y, ref):
        return torch.equal(y[0], ref[0]) and torch.equal(y[1].q, ref[1].q) and torch.equal(y[1].sx, ref[1].sx)
    other = calls([0, T], np.array([0.4], np.float32))
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        calls(cu, scale)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = calls(cu, scale)
    kept = cu.copy(), scale.copy()
    cu[1:3], scale[:] = (7, 90), 9.0
    for rep in range(3):
        q.normal_(generator=g)
        graph.replay()
        torch.cuda.synchronize()
        print(f"captured offsets: replay {rep}", flush=True)
        ref = calls(*kept)
        assert same(y, ref) and not torch.equal(ref[0], other[0])
        calls(cu, scale)
