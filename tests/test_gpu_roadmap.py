"""The rank selection and the edge rows at the edges of their passes, against
numpy: arrays up to, at and past the sample, ranks at both ends, ties, signed
zeros and infinities, unaligned starts, an array that the sample misjudges, a
workspace without room for the bracket; rows shorter than a vector to rows of
several rounds."""
import ctypes

import numpy as np
import pytest

import pump_amd as P

from test_gpu_parity import dev, host, ptr

pytestmark = pytest.mark.gpu

BASE_WS = 280 + 2048 * 8  # no room for the bracket's keys


def select(g, at, n, k, ws):
    rn = ctypes.c_float()
    P.check("select", P.lib.pump_select_rn(ctypes.c_void_p(g.ptr + 4 * at), n, k, ctypes.byref(rn), ws.p,
                                           ws.nbytes, None))
    return np.float32(rn.value)


@pytest.mark.parametrize("n", [1, 2, 63, 1025, 16383, 16384, 16385, 70001, 262147, 6000003])
@pytest.mark.parametrize("kind", ["lognormal", "mixed", "ties", "misjudged"])
def test_select_at_the_edges(n, kind):
    rng = np.random.default_rng(n)
    x = rng.lognormal(1.0, 0.7, n + 3).astype(np.float32)
    if kind == "mixed":
        x = rng.choice(np.array([0.0, -0.0, 1e-40, -1.5, 3.0, 1e30, np.inf, -np.inf], np.float32),
                       n + 3) + np.where(rng.uniform(size=n + 3) < 0.5, 0, x).astype(np.float32)
    elif kind == "ties":
        x = np.round(x)
    elif kind == "misjudged" and n > 16384:
        # the keys that the sample reads are far below all others
        step = n // 1024
        j = np.arange(1024, dtype=np.uint32)
        at = j.astype(np.int64) * step + ((j * np.uint32(2654435769)) >> np.uint32(7)).astype(
            np.int64) % (step - 15)
        x[(at[:, None] + np.arange(16)).ravel()] *= np.float32(1e-6)
    g = dev(x)
    ws_n = P.lib.pump_select_rn_workspace(n)
    full = P.DeviceArray(shape=(ws_n,), dtype=np.uint8, fill=0x5b)
    small = P.DeviceArray(shape=(BASE_WS,), dtype=np.uint8, fill=0x5b)
    for at in (0, 1, 3):
        s = np.sort(x[at: at + n])
        for k in sorted({0, min(1, n - 1), n // 160, n // 5, n // 2, n - 1}):
            print("select", n, kind, at, k, flush=True)
            for ws in (full, small):
                assert select(g, at, n, k, ws) == s[k], (at, k, ws.nbytes)


@pytest.mark.parametrize("n,kind", [(n, k) for n in (16385, 70001, 6000003) for k in (
    "ordered", "equal", "two", "crowded")] + [((1 << 25) + 3, "ordered")])
def test_select_where_the_regions_may_not_do(n, kind):
    """Keys of the bracket that lie together, that are all equal, or that fall
    to one workgroup (it reads every r-th stretch of 1024 keys): the regions
    overflow and the passes go over the array, inside the bracket."""
    rng = np.random.default_rng(n)
    x = rng.lognormal(1.0, 0.7, n).astype(np.float32)
    if kind == "ordered":
        x = np.sort(x)
    elif kind == "equal":
        x[:] = np.float32(2.5)
    elif kind == "two":
        x = np.where(x < np.float32(3), np.float32(1), np.float32(2))
    else:
        regions = min((n + 8191) // 8192, 1024)
        one = (np.arange(n) // 1024) % regions == 0  # with vectors from keys[0] on
        x[one] = np.median(x) * rng.uniform(0.9999, 1.0001, one.sum()).astype(np.float32)
    g = dev(x)
    s = np.sort(x)
    ws_n = P.lib.pump_select_rn_workspace(n)
    ws = P.DeviceArray(shape=(ws_n,), dtype=np.uint8, fill=0x5b)
    below = int((x < np.float32(2)).sum())
    for k in sorted({0, n // 5000, n // 160, n // 2, below - 1, below, n - 1} & set(range(n))):
        print("select", n, kind, k, flush=True)
        assert select(g, 0, n, k, ws) == s[k], k


@pytest.mark.parametrize("num", [2, 3, 5, 6, 257, 1025, 1026, 8192, 8194, 8201])
def test_edge_rows_at_the_edges(num):
    rng = np.random.default_rng(num)
    n = num * (num - 1)
    rows = min(num, 40)  # rows past these hold nothing below the threshold
    c = np.full((num, num - 1), np.float32(np.inf))
    c[:rows] = rng.uniform(0, 1, (rows, num - 1))
    c[rng.integers(0, rows)] = 0.0  # a row that is kept whole
    c[0, 0], c[0, -1], c[rows - 1, -1] = np.nan, 0.1, 0.2
    t = np.arange(n, dtype=np.float32).reshape(c.shape)
    rn = np.float32(0.3)
    keep = c < rn
    src, k = np.nonzero(keep)
    g, gt = dev(c), dev(t)
    row_start = dev(np.zeros(num + 1, np.int64))
    ws_n = P.lib.pump_scan_workspace(num + 1)
    ws = P.DeviceArray(shape=(ws_n,), dtype=np.uint8)
    ne = ctypes.c_int64()
    print("rows", num, flush=True)
    P.check("count", P.lib.pump_count_edges(ptr(g), num, rn, ptr(row_start), ctypes.byref(ne),
                                            ws.p, ws_n, None))
    assert ne.value == len(src)
    assert np.array_equal(host(row_start), np.concatenate([[0], np.cumsum(keep.sum(1))]))
    e = [dev(np.full(len(src) + 1, -9, d)) for d in (np.int32, np.int32, np.float32, np.float32)]
    P.check("fill", P.lib.pump_fill_edges(ptr(g), ptr(gt), num, rn, ptr(row_start),
                                          *(ptr(a) for a in e), None))
    want = (src, k + (k >= src), c[keep], t[keep])
    for a, w in zip(e, want):
        assert host(a)[-1] == -9 and np.array_equal(host(a)[:-1], w.astype(host(a).dtype))
