"""A roadmap's device memory: searches whose buffers grow within and past the
blocks they are cut from give the results of a fresh roadmap, roadmaps of two
threads do not meet, what a roadmap takes goes back with it, and the pair
tables that it does not keep go back with the build."""
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
    # 2300 samples: pair tables of 21 MB, past what shared blocks give
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


@pytest.mark.parametrize("num", [700, 1500, 2500])  # tables below, at and past a cut range's size
def test_pair_tables_go_back(num, noise):
    s, o = problem(num, 7)
    table = num * (num - 1) * 4
    held = {}
    for keep in (0, 1, 0, 1):  # the second time without the runtime's own first allocations
        P.sync()
        before = free_bytes()
        rm = P.Roadmap(s, o, s[-1], *noise, prm(num, 64, keep_pairs=keep))
        P.sync()
        held[keep] = before - free_bytes()
        print("pair tables", num, keep, held[keep] >> 20, flush=True)
        d = rm.device()
        assert bool(d.copts) == bool(d.topts) == bool(keep)
        rm.close()
    # 4 MiB: the granularity of two allocations
    assert held[1] - held[0] >= 2 * table - (4 << 20)


def test_batch_holds_what_its_problems_need(noise):
    """No more than a quarter above the arrays of the problems (and 2 MiB, the
    granularity of an allocation, for each array that stands alone)."""
    num, n = 1200, 12
    problems, need = [], 0
    for j in range(n):
        s, o = problem(num, 50 + j)
        problems.append((s, o, s[-1], prm(num, 64)))
    P.Batch(problems, *noise).close()  # the runtime's own first allocations
    P.sync()
    before = free_bytes()
    b = P.Batch(problems, *noise)
    P.sync()
    held = before - free_bytes()
    for j in range(n):
        i = b.roadmap(j).info
        E, W, hs = int(i.n_edges), int(i.n_waypoints), int(i.max_hs)
        need += 45 * num + 33 * E + W * (24 + 16 * hs + 4)
    noise_bytes = 200 * 2048 * 3 * 4 * 2 + P.lib.pump_split_offsets_bytes(200, 2048)
    print("batch", held >> 20, (need + noise_bytes) >> 20, flush=True)
    assert held <= 1.25 * (need + noise_bytes) + n * 6 * (2 << 20)
    b.close()
