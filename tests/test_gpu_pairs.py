"""The pair pass's launch shapes (sets of 64 pairs dealt out to the waves,
chunks claimed from the counter) and its special pairs against the oracle and
the library's plain host bisection."""
import numpy as np
import pytest

import oracle
import pump_amd as P

from test_gpu_parity import assert_close_f32, dev, host

pytestmark = pytest.mark.gpu

O = oracle.load()


def gpu_tables(s, tmax):
    n = s.shape[0]
    g = dev(s)
    c = P.DeviceArray(shape=(n * (n - 1),), dtype=np.float32, fill=0xff)
    t = P.DeviceArray(shape=(n * (n - 1),), dtype=np.float32, fill=0xff)
    h = P.DeviceArray(shape=(n,), dtype=np.float32, fill=0xff)
    P.check("pump_fill_copts_topts",
            P.lib.pump_fill_copts_topts(g.p, n, tmax, c.p, t.p, None))
    P.check("pump_heuristic", P.lib.pump_heuristic(g.p, n, P.fp(s[-1].copy()), tmax, h.p, None))
    return host(c), host(t), host(h)


def states(n, seed):
    rng = np.random.default_rng(seed)
    return np.concatenate([rng.uniform(0, 1, (n, 3)),
                           rng.uniform(-0.5, 0.5, (n, 3))], 1).astype(np.float32)


# one pair, a part of a set, whole sets and one more, the last launch of one
# workgroup (16 for the pairs, 256 to the goal), one set per wave, several per
# wave, and (from 4.2 million pairs) claimed chunks
@pytest.mark.parametrize("n", [2, 8, 9, 16, 17, 64, 65, 256, 257, 513, 1100, 2200])
def test_pair_tables_over_launch_shapes(n):
    s = states(n, n)
    print("pairs", n, flush=True)
    c, t, h = gpu_tables(s, 5.0)
    rc, rt = np.zeros_like(c), np.zeros_like(t)
    O.po_fill_copts_topts(oracle.fp(s), n, 5.0, oracle.fp(rc), oracle.fp(rt), 8)
    assert_close_f32(t, rt, max_mismatch_frac=max(1e-5, 1.5 / t.size))
    assert_close_f32(c, rc, max_mismatch_frac=max(1e-5, 1.5 / t.size))
    # to the goal: the cost of the pair (i, n - 1), the last of row i
    assert h[-1] == 0 and np.array_equal(h[:-1], c.reshape(n, n - 1)[:-1, -1])


@pytest.mark.parametrize("tmax", [5.0, 0.3, 40.0, 200.0])
def test_pair_tables_of_special_states(tmax):
    """Repeated, nearly equal, distant and resting states, and brackets whose
    ends leave the range of the shortcuts: bit for bit the plain bisection."""
    s = states(60, 3)
    s[10:20] = s[0]
    s[20:30, :3] = s[0, :3] + np.float32(1e-3) * s[20:30, :3]
    s[30:35] *= np.float32(40)
    s[35:45, 3:] = 0
    print("special", tmax, flush=True)
    c, t, h = gpu_tables(s, tmax)
    assert np.array_equal(h[:-1], c.reshape(60, 59)[:-1, -1], equal_nan=True)
    k = 0
    for i in range(60):
        for j in range(60):
            if i == j:
                continue
            rt = np.float32(P.lib.pump_host_topt(P.fp(s[i].copy()), P.fp(s[j].copy()), tmax))
            rc = np.float32(P.lib.pump_host_cost(rt, P.fp(s[i].copy()), P.fp(s[j].copy())))
            assert t[k].tobytes() == rt.tobytes(), (i, j, t[k], rt)
            assert c[k].tobytes() == rc.tobytes() or (np.isnan(c[k]) and np.isnan(rc))
            k += 1
