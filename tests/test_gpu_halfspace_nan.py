"""The half-space cache at waypoints that are not finite, among finite ones of
the same wave, against the oracle: a NaN on any axis makes every box's distance
NaN, which the reference's d2 > maxd2 does not skip (hsmc.cu:69), so the first
max_hs boxes are stored; an infinite one is past every finite box."""
import numpy as np
import pytest

import oracle
import pump_amd as P

from test_gpu_parity import dev, edge_mask_host, host, ptr

pytestmark = pytest.mark.gpu

O = oracle.load()


@pytest.mark.parametrize("n_obs,max_hs", [(3, 3), (70, 5), (600, 5), (70, 40)])
@pytest.mark.parametrize("odd", ["nan", "-nan", "inf", "mixed"])
def test_waypoints_that_are_not_finite(n_obs, max_hs, odd):
    rng = np.random.default_rng(n_obs + max_hs)
    c = rng.uniform(0, 1, (n_obs, 3))
    h = rng.uniform(0.005, 0.04, (n_obs, 3))
    obs = np.zeros((n_obs, 12), np.float32)
    obs[:, :3], obs[:, 6:9] = c - h, c + h
    W = rng.integers(2, 40, 60)
    off = np.concatenate([[0], np.cumsum(W)]).astype(np.int64)
    n_wp, E = int(off[-1]), len(W)
    # the finite waypoints of a wave are close together, boxes all around them
    disc = rng.uniform(0.45, 0.55, (n_wp, 6)).astype(np.float32)
    nan = np.float32(np.nan)
    values = {"nan": [nan], "-nan": [np.copysign(nan, np.float32(-1))],
              "inf": [np.float32(np.inf), np.float32(-np.inf)]}
    pick = values.get(odd) or sum(values.values(), [])
    at = rng.choice(n_wp, n_wp // 20, replace=False)
    for j, g in enumerate(at):  # single waypoints, on one axis or on all
        disc[g, j % 4 if j % 4 < 3 else slice(0, 3)] = pick[j % len(pick)]
    free = (rng.uniform(size=E) < 0.8).astype(np.uint8)
    md2 = np.float32(0.01)
    hs = n_wp * max_hs
    ref_as, ref_bs = np.zeros((hs, 3), np.float32), np.zeros(hs, np.float32)
    ref_cnt = np.zeros(n_wp, np.int32)
    O.po_setup_as_bs(hs, oracle.fp(ref_bs), oracle.fp(ref_as))
    O.po_cache_halfspaces(E, oracle.fp(disc), oracle.lp(off), oracle.bp(free), n_obs, max_hs,
                          oracle.fp(obs), oracle.fp(ref_as), oracle.fp(ref_bs),
                          oracle.ip(ref_cnt), md2, 4)
    as_, bs = dev(np.zeros((hs, 3), np.float32)), dev(np.zeros(hs, np.float32))
    cnt, emask = dev(np.full(n_wp, -7, np.int32)), dev(np.zeros(E, np.uint64))
    gdisc, gfree, gobs, goff = dev(disc), dev(free), dev(obs), dev(off)
    print("halfspaces", n_obs, max_hs, odd, flush=True)
    P.check("cache_hs", P.lib.pump_cache_halfspaces(
        E, ptr(gdisc), ptr(gfree), n_obs, max_hs, ptr(gobs), 0, ptr(goff),
        ptr(as_), ptr(bs), ptr(cnt), md2, 1, ptr(emask), None))
    assert np.array_equal(host(cnt), ref_cnt)
    assert np.array_equal(host(bs), ref_bs, equal_nan=True)
    assert np.array_equal(host(as_), ref_as, equal_nan=True)
    assert np.array_equal(host(emask), edge_mask_host(off, ref_bs, max_hs))
    if odd != "inf":
        assert np.isnan(ref_bs).any()
