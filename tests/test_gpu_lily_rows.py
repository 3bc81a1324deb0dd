"""GPU: SnowLily's state over enough rows for the kernel that forms the a * x products in LDS
(a, x and b more than 256 MiB together) and over fewer, bit for bit against the oracle: documents
that begin and end inside a 16-row group, even and odd kernels, inputs that are no multiple of
256, non-finite values beside the documents' edges."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as t
    assert t.cuda.is_available(), "no GPU"
    return t


@pytest.fixture(scope="module")
def dev(torch, nxg):
    nxg.init()
    return torch.device("cuda:0")


@pytest.mark.parametrize("C,k,lengths", [
    (1024, 5, [1, 2, 3, 15, 16, 17, 33, 5000, 11405]),
    (1024, 2, [16390]),
    (288, 3, [30000, 7, 1, 2762]),
    (96, 1, [65500, 9, 30]),
    (1024, 5, [1, 2, 3, 15, 16, 17, 33, 5000, 16758]),      # 21,845 rows: just below 256 MiB
    (1024, 5, [1, 2, 3, 15, 16, 17, 33, 5000, 16759]),      # just past, as all that follow
    (1024, 2, [22001]),
    (288, 3, [75000, 7, 1, 2762]),
    (96, 1, [233000, 9, 30]),
])
def test_lily_state_many_rows(nxg, orc, torch, dev, C, k, lengths):
    print(f"lily state C={C} k={k} lengths={lengths}", flush=True)
    rng = np.random.default_rng(C + k)
    cu = nxg.cu_offsets_of(lengths)
    T = int(cu[-1])
    assert ((T + 15) // 16) * ((C + 255) // 256) >= 4096
    a, x, b = (rng.standard_normal((T, C)).astype(np.float32) for _ in range(3))
    for row, v in ((0, np.inf), (T - 1, np.nan), (int(cu[1]) - 1, -np.inf), (min(int(cu[1]), T - 1), 1e38)):
        x[row, rng.integers(0, C, 4)] = v
    taps = rng.standard_normal((k, C)).astype(np.float32)
    c = lambda t: torch.from_numpy(t).cuda()
    ref = orc.lily_state(a, x, b, taps, cu)
    for act_max in (127, 63):
        qa = nxg.lily_state_quantize_rows(c(a), c(x), c(b), c(taps), cu, act_max=act_max)
        u8, sx = nxg.export_qact(qa)
        q_ref, sx_ref = orc.quantize_rows(ref, act_max)
        assert (u8.cpu().numpy() == q_ref).all()
        assert (sx.cpu().numpy().view(np.uint32) == np.asarray(sx_ref).view(np.uint32)).all()
