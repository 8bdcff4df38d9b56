"""A roadmap's device memory: searches whose buffers grow within and past the
blocks they are cut from give the results of a fresh roadmap, roadmaps of two
threads do not meet, and what a roadmap takes goes back with it."""
import ctypes
import threading

import numpy as np
import pytest

import pump_amd as P

pytestmark = pytest.mark.gpu


def problem(num, seed):
    rng = np.random.default_rng(seed)
    s = np.concatenate([rng.uniform(0, 1, (num, 3)), rng.uniform(-0.3, 0.3, (num, 3))], 1)
    s[0], s[-1] = (0.1, 0.1, 0.1, 0, 0, 0), (0.9, 0.9, 0.9, 0, 0, 0)
    lo = rng.uniform(0.2, 0.7, (6, 3))
    o = np.concatenate([lo, np.full((6, 3), -3.1), lo + 0.1, np.full((6, 3), 3.1)], 1)
    return s.astype(np.float32), o.astype(np.float32).reshape(-1, 12)


def prm(num, n_p, **over):
    return P.params(rn_perc=float(np.float32(30 / (num - 1))), w_fixed=0, wp_dt=0.05, w_cap=64,
                    offset_mult=0.02, n_p=n_p, max_hs=5, cp_target=0.01, cp_factor=2.0, **over)


def free_bytes():
    """hipMemGetInfo of the runtime that the library is linked to."""
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert P.lib.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


@pytest.fixture(scope="module")
def noise():
    ot, xc, _, _ = P.make_noise_device(P.noise_spec(n_mc=2048, tmax_steps=200))
    return ot, xc


def outcome(rm, p):
    r = rm.search(p)
    d = {k: v for k, v in P.search_result_dict(r).items() if not k.startswith("ms")}
    return d, rm.paths(int(r.num_paths))


def same(a, b):
    assert {k: v for k, v in a[0].items() if "time_ms" not in k} == {
        k: v for k, v in b[0].items() if "time_ms" not in k}
    for k in a[1]:
        assert np.array_equal(a[1][k], b[1][k]), k


@pytest.mark.parametrize("num,keep", [(40, 1), (600, 0), (2300, 1)])
def test_growing_searches_match_fresh_ones(num, keep, noise):
    # 2300 samples: pair tables of 21 MB, past the largest cut range
    s, o = problem(num, num)
    sizes = [(64, 1), (2048, 0), (128, 1), (2000, 1)]
    print("memory", num, keep, flush=True)
    kept = P.Roadmap(s, o, s[-1], *noise, prm(num, 64, keep_pairs=keep))
    for n_p, bits in sizes:
        p = prm(num, n_p, keep_pairs=keep, validity_bits=bits)
        fresh = P.Roadmap(s, o, s[-1], *noise, p)
        same(outcome(kept, p), outcome(fresh, p))
        fresh.close()
    kept.close()


def test_two_threads_and_return(noise):
    s, o = problem(500, 3)
    p = prm(500, 512, validity_bits=1)
    rm = P.Roadmap(s, o, s[-1], *noise, p)
    want = outcome(rm, p)
    rm.close()
    P.sync()
    before = free_bytes()
    bad = []

    def work():
        try:
            for _ in range(4):
                r = P.Roadmap(s, o, s[-1], *noise, p)
                same(outcome(r, p), want)
                r.close()
        except BaseException as e:  # reported by the main thread
            bad.append(e)
    th = [threading.Thread(target=work) for _ in range(2)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad, bad
    P.sync()
    # eight roadmaps came and went; the runtime may keep a block or two
    assert before - free_bytes() < 256 << 20
