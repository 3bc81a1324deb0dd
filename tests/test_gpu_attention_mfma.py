"""GPU: attention on the matrix cores bit for bit against the oracle where its tiling can go
wrong: key counts around the 16-key tile and the 8-key group, every head ratio that divides 16,
bands narrower and wider than a tile, workgroups whose queries lie in several documents (also
where those documents' scores do not fit together), scores split between LDS and a workspace of
any size and alignment, non-finite queries, keys and values, and sums that underflow to -0."""
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


def bits(a):
    return np.ascontiguousarray(a, dtype=np.float32).view(np.uint32)


def check(nxg, orc, torch, lengths, half, H, G, workspaces=(None,), seed=0, spoil=None):
    rng = np.random.default_rng(seed)
    cu = nxg.cu_offsets_of(lengths)
    T = int(cu[-1])
    q = rng.standard_normal((T, H * 64)).astype(np.float32)
    k, v = (rng.standard_normal((G, T, 64)).astype(np.float32) for _ in range(2))
    scale = rng.uniform(0.05, 0.3, len(lengths)).astype(np.float32)
    if spoil:
        spoil(q, k, v)
    ref = orc.attention(q, k, v, cu, scale, H, G, half)
    dev = [torch.from_numpy(a).cuda() for a in (q, k, v)]
    for ws in workspaces:
        size = ws if ws is None or isinstance(ws, str) else ws.numel()
        print(f"attention lengths={lengths} half={half} H={H} G={G} workspace={size}", flush=True)
        y = nxg.attention(*dev, cu, scale, H, G, half, workspace=ws).cpu().numpy()
        assert ((bits(y) == bits(ref)) | (np.isnan(y) & np.isnan(ref))).all()
    return ref


@pytest.mark.parametrize("H,G", [(4, 4), (4, 2), (4, 1), (8, 1), (16, 1)])
@pytest.mark.parametrize("half", [-1, 0, 3, 8, 20])
def test_tile_edges(nxg, orc, torch, dev, H, G, half):
    check(nxg, orc, torch, [15, 16, 17, 1, 23, 24, 25, 33, 64, 7, 113], half, H, G, seed=H + half)


@pytest.mark.parametrize("lengths,half,H,G", [
    ([700, 900, 5, 820], -1, 4, 2),       # neighbours span more keys than the tiles hold
    ([1290, 1283, 1296], -1, 2, 1),
    ([1401, 1500], 640, 4, 4),
    ([3100, 3, 2900], -1, 2, 1),
    ([2700, 40], 1300, 16, 1),
])
def test_scores_in_lds_and_workspace(nxg, orc, torch, dev, lengths, half, H, G):
    T, most = sum(lengths), max(lengths) if half < 0 else min(max(lengths), 2 * half + 1)
    slot = 16 * most * 4
    odd = torch.empty(5 * slot + 16, dtype=torch.uint8, device="cuda")[4:]    # 4-byte aligned only
    one = torch.empty(slot, dtype=torch.uint8, device="cuda")
    check(nxg, orc, torch, lengths, half, H, G, workspaces=(None, "auto", odd, one), seed=T)


@pytest.mark.parametrize("n", [1536, 3000])
def test_workspace_of_less_than_a_slot_is_not_used(nxg, orc, torch, dev, n):
    """16 * max_keys floats are the least that is used; with less the launch is the one without a
    workspace, its scores in LDS (1,536 keys) or recomputed (3,000), on the whole device."""
    slot = 16 * n * 4
    ws = [torch.full((b,), 0xA5, dtype=torch.uint8, device="cuda") for b in (1024, 4096, slot // 2, slot - 4, slot)]
    check(nxg, orc, torch, [n], -1, 2, 1, workspaces=[None] + ws, seed=n)
    for w in ws[:-1]:
        assert bool((w == 0xA5).all()), f"{w.numel()} bytes were written"
    if n == 3000:                         # (a workgroup by itself keeps 1,536 keys in LDS)
        assert not bool((ws[-1] == 0xA5).all())


def test_half_a_workspace_is_no_slower_than_less(nxg, torch, dev):
    """Half the workspace holds slots for a workgroup on every CU and a few more, which would share
    theirs and have all others wait: 1.3 times the time of 3/8 of the workspace."""
    n = 8192
    g = torch.Generator("cuda").manual_seed(n)
    q = torch.randn(n, 1024, device="cuda", generator=g)
    k, v = (torch.randn(8, n, 64, device="cuda", generator=g) for _ in range(2))
    full = nxg.attention_workspace_bytes(n, 16, 8, n)

    def ms(size):
        ws, best = torch.empty(size, dtype=torch.uint8, device="cuda"), float("inf")
        for _ in range(6):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            y = nxg.attention(q, k, v, [0, n], np.array([0.1], np.float32), 16, 8, workspace=ws)
            b.record()
            b.synchronize()
            best = min(best, a.elapsed_time(b))
        return best, y

    (half, y_half), (less, y_less) = ms(full // 2), ms(full * 3 // 8)
    print(f"{n} keys: half the workspace {half:.2f} ms, 3/8 {less:.2f}", flush=True)
    assert torch.equal(y_half.view(torch.int32), y_less.view(torch.int32))
    assert half < 1.1 * less


def test_workspace_asked_for_is_one_that_is_used(nxg, orc, torch, dev):
    """Past 2^23 keys the scores are recomputed whatever the workspace: none is asked for (a slot for
    every workgroup would be 550 GB), and a call under such a bound runs without one."""
    at, past = 1 << 23, (1 << 23) + 1
    full = nxg.attention_workspace_bytes(past, 16, 8, at)
    assert full > 0 and full % (64 * at) == 0
    assert nxg.attention_workspace_bytes(past, 16, 8, past) == 0
    H, G, T = 2, 1, 40
    rng = np.random.default_rng(2)
    q = rng.standard_normal((T, H * 64)).astype(np.float32)
    k, v = (rng.standard_normal((G, T, 64)).astype(np.float32) for _ in range(2))
    d = [torch.from_numpy(a).cuda() for a in (q, k, v)]
    cu, sc = torch.tensor([0, T], dtype=torch.int32, device="cuda"), torch.full((1,), 0.125, device="cuda")
    ws, out = torch.full((4096,), 0xA5, dtype=torch.uint8, device="cuda"), torch.empty_like(d[0])
    L = nxg.load_library()
    args = [t.data_ptr() for t in (*d, cu)] + [1, sc.data_ptr(), T, H, G, -1, past, out.data_ptr()]
    assert L.nxg_attention_ws(*args, ws.data_ptr(), ws.numel(), None) == 0
    torch.cuda.synchronize()
    assert bool((ws == 0xA5).all())
    assert (bits(out.cpu().numpy()) == bits(orc.attention(q, k, v, [0, T], np.float32([0.125]), H, G))).all()


@pytest.mark.parametrize("half", [-1, 9])
def test_non_finite_queries_keys_values(nxg, orc, torch, dev, half):
    n = [40, 70, 21]

    def nan_first_key(q, k, v):
        k[0, 0, 3] = np.nan               # the first score of document 0: the maximum is NaN
        k[1, 55, 60] = np.nan             # a later one: never the maximum
    check(nxg, orc, torch, n, half, 8, 2, seed=1, spoil=nan_first_key)

    def inf_key_and_query(q, k, v):
        k[0, 12, 1] = np.inf
        k[1, 90, 2] = -np.inf
        q[44, 5] = np.inf
        q[129, 7] = np.nan
    check(nxg, orc, torch, n, half, 8, 2, seed=2, spoil=inf_key_and_query)

    def values(q, k, v):
        v[0, 0, 0], v[0, 39, 1], v[1, 40, 2], v[1, 130, 63] = np.inf, np.nan, -np.inf, np.nan
    check(nxg, orc, torch, n, half, 8, 2, seed=3, spoil=values)

    def tiny(q, k, v):
        v *= np.float32(1e-38)            # sums among the subnormals
    check(nxg, orc, torch, n, half, 8, 2, seed=4, spoil=tiny)


@pytest.mark.parametrize("lengths,half,workspace", [
    ([5, 40, 24, 2, 300], -1, None),      # documents that share a workgroup, padding after the last
    ([5, 40, 24, 2, 300], 9, None),       # keys past the band
    ([100, 2900, 60], -1, "auto"),
    ([2900], 1300, "auto"),
    ([100, 2900, 60], -1, None),          # attention_long_kernel
    ([2900], 1300, None),
])
def test_sums_that_underflow_keep_their_sign(nxg, orc, torch, dev, lengths, half, workspace):
    """Products of the smallest subnormal with weights under one half round to -0 or +0 by the
    value's sign: a sum of -0 stays -0 whatever the values of the keys that follow it outside the
    pair's range, and +0 stays +0."""
    def spoil(q, k, v):
        rng = np.random.default_rng(5)
        v[:] = np.float32(-1e-45)
        v[:, :, 1] = np.float32(1e-45)
        v[:, :, 2] = rng.choice(np.array([-1e-45, 1e-45, -0.0, 0.0], np.float32), v.shape[:2])
        v[:, :, 3] = 0.0
        v[:, :, 4] = -0.0
        v[:, ::3, 5:20] = rng.standard_normal(v[:, ::3, 5:20].shape)
        q *= np.float32(0.01)             # weights near 1 / n
    ref = check(nxg, orc, torch, lengths, half, 4, 2, workspaces=(workspace,), seed=7, spoil=spoil)
    assert (bits(ref) == 0x80000000).mean() > 0.3 and (bits(ref) == 0).any()


@pytest.mark.parametrize("lengths,half,workspaces", [
    ([500, 70], -1, (None,)),
    ([700], 200, (None,)),
    ([40, 2900, 25], -1, ("auto", 16 * 2900 * 4)),
    ([3000], 1300, ("auto", 16 * 2601 * 4)),
])
def test_non_finite_values_in_whole_and_partial_tiles(nxg, orc, torch, dev, lengths, half, workspaces):
    """Inf and NaN values in tiles that every pair attends to and in the first, last and masked
    ones: sums taken again give the oracle's bits, also those of the dimensions beside them."""
    def spoil(q, k, v):
        T = v.shape[1]
        for j, x in ((0, np.inf), (17, np.nan), (T // 2, -np.inf), (T // 2 + 40, np.inf), (T - 1, np.nan)):
            v[:, j, [j % 64, (j + 1) % 64]] = x
        v[:, T // 3] = 3e38               # sums that overflow
    ws = [w if isinstance(w, (str, type(None))) else torch.empty(w, dtype=torch.uint8, device="cuda") for w in workspaces]
    ref = check(nxg, orc, torch, lengths, half, 2, 1, workspaces=ws, seed=11, spoil=spoil)
    assert np.isfinite(ref).any() and not np.isfinite(ref).all()


@pytest.mark.parametrize("n", [1024, 4096])
def test_non_finite_values_cost_little(nxg, torch, dev, n):
    """One NaN row makes every output NaN and every sum is taken again: about a third of the work,
    not key by key (5 and 13 times the whole)."""
    g = torch.Generator("cuda").manual_seed(n)
    q = torch.randn(n, 1024, device="cuda", generator=g)
    k, v = (torch.randn(8, n, 64, device="cuda", generator=g) for _ in range(2))
    bad = v.clone()
    bad[:, n // 3] = float("nan")
    cu, scale = [0, n], np.array([0.1], np.float32)

    def us(values):
        best = float("inf")
        for _ in range(5):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(10):
                y = nxg.attention(q, k, values, cu, scale, 16, 8, workspace="auto")
            b.record()
            b.synchronize()
            best = min(best, a.elapsed_time(b) * 100)
        return best, y

    (fine, y), (nan, y_nan) = us(v), us(bad)
    print(f"{n} keys: {fine:.0f} us, with a NaN row {nan:.0f}", flush=True)
    assert torch.isfinite(y).all() and torch.isnan(y_nan).all()
    assert nan < 3 * fine


@pytest.mark.parametrize("workspace", ["auto", "slot"])
@pytest.mark.parametrize("lengths,half", [([40, 2900, 21], -1), ([3100], 1400)])
def test_non_finite_and_extreme_scores_in_the_workspace(nxg, orc, torch, dev, lengths, half, workspace):
    """Scores that live in a workspace slot: the maximum and the sums of the slot's exponentials are
    code of their own. NaN and Inf keys and queries in tiles kept in LDS, in the slot and among a
    pair's last n % 8 keys, a NaN first key, and scores over +-400."""
    T, most = sum(lengths), max(lengths) if half < 0 else min(max(lengths), 2 * half + 1)
    start = lengths[0] if len(lengths) > 1 else 0             # of the long document
    ws = (torch.empty(16 * most * 4, dtype=torch.uint8, device="cuda") if workspace == "slot" else "auto",)

    def spoil_keys(rows):
        def spoil(q, k, v):
            for j, x in rows:
                k[0, start + j, j % 64] = x
            q[start + 1500, 5], q[start + 77, 70] = np.inf, np.nan
        return spoil
    end = lengths[1] if len(lengths) > 1 else lengths[0]
    for rows in ([(0, np.nan)],                               # the first score of every pair, or of the first rows
                 [(30, np.nan), (1000, np.inf), (2500, np.nan), (2600, -np.inf)],
                 [(end - 1, np.nan), (end - 2, np.inf)]):     # the last keys
        ref = check(nxg, orc, torch, lengths, half, 2, 1, workspaces=ws, seed=end, spoil=spoil_keys(rows))
        assert np.isfinite(ref).any()

    def extreme(q, k, v):
        q *= 50
    check(nxg, orc, torch, lengths, half, 2, 1, workspaces=ws, seed=3, spoil=extreme)
