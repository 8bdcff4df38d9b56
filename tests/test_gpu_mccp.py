"""Full Monte Carlo CP against the oracle's hit counts at the edges of the
kernel's work split: particles around the groups of 64, few and many segments
per wave, box counts around the 64 held per register set and past them, launch
sizes on either side of each rule of its dispatch."""
import numpy as np
import pytest

import oracle
import pump_amd as P

from test_gpu_parity import dev, host, ptr

pytestmark = pytest.mark.gpu

O = oracle.load()


@pytest.mark.parametrize("n_mc,n_obs,n_paths,om", [
    (1, 1, 1, 0.5), (63, 0, 3, 1.0), (64, 64, 3, 0.2), (65, 65, 3, 0.2), (300, 128, 5, 0.3),
    (200, 129, 9, 0.3), (130, 256, 4, 2.0), (130, 257, 4, 0.1), (700, 600, 2, 0.1),
    (1000, 30, 300, 0.05)])
def test_mccp_hits_against_oracle(n_mc, n_obs, n_paths, om):
    compare(n_mc, n_obs, n_paths, om, 90, 120)  # paths longer than the noise table stop at its end


@pytest.mark.parametrize("n_mc,n_obs,n_paths", [
    # four lanes per particle: groups of 16, up to 128 groups of 64
    (15, 70, 1), (16, 5, 2), (17, 64, 3), (63, 300, 40), (2048, 40, 4),
    # past them: boxes in a loop, up to 64 in registers
    (2049, 40, 4), (130, 90, 60), (130, 200, 60), (70, 300, 100),
    # four waves and fewer to a workgroup: up to 256 boxes in registers
    (64, 100, 4100), (64, 200, 4100), (64, 260, 4100)])
def test_mccp_hits_of_short_paths(n_mc, n_obs, n_paths):
    compare(n_mc, n_obs, n_paths, 0.3, 12, 14)


def compare(n_mc, n_obs, n_paths, om, tsteps, cap):
    rng = np.random.default_rng(n_mc + n_obs)
    obs = np.zeros((max(n_obs, 1), 12), np.float32)
    c = rng.uniform(0, 1, (len(obs), 3))
    sd = rng.uniform(0.01, 0.1, (len(obs), 3)) * (30 / (n_obs + 10)) ** 0.33
    obs[:, :3], obs[:, 6:9] = c - sd / 2, c + sd / 2
    obs[:, 3:6], obs[:, 9:12] = -3.1, 3.1
    xc = rng.normal(0, 0.05, (n_mc, tsteps, 3)).astype(np.float32)
    paths = np.zeros((n_paths, cap, 6), np.float32)
    Ts = rng.integers(2, cap, n_paths).astype(np.int32)
    Ts[: 6] = [cap, 3, 2, 4, 1, 0][: min(6, n_paths)]
    a, b = rng.uniform(0, 1, (2, n_paths, 1, 3))
    a[0], b[0] = c[0] - 0.3, c[0] + 0.3  # through the first box
    paths[:, :, :3] = a + np.linspace(0, 1, cap)[None, :, None] * (b - a)
    om = np.float32(om)
    ref = []
    for k in range(n_paths):
        T = min(int(Ts[k]), tsteps + 1)
        ref.append(O.po_mccp_hits(oracle.fp(obs), n_obs, oracle.fp(xc), tsteps, n_mc, om,
                                  oracle.fp(np.ascontiguousarray(paths[k])), T, None)
                   if T > 2 else 0)
    g = [dev(x) for x in (obs, xc, paths, Ts)]
    hits = dev(np.full(n_paths, 77, np.int32))
    print("mccp", n_mc, n_obs, n_paths, flush=True)
    for zero in (1, 0):  # into cleared counters, then onto the caller's
        P.check("mccp_many", P.lib.pump_collision_probability_many(
            ptr(g[0]) if n_obs else None, n_obs, ptr(g[1]), tsteps, n_mc, om, ptr(g[2]), cap,
            ptr(g[3]), n_paths, ptr(hits), zero, None))
    assert host(hits).tolist() == [2 * r for r in ref]
    assert n_obs == 0 or n_mc == 1 or ref[0] > 0
