"""The workgroup-per-path form of the HSMC step (small wavefronts) against the
oracle at the edges of its loops: particle counts around the groups of 64 and
the waves' share, edges longer than a 64-bit summary, slot counts that need
several passes of the half-space list, rows with and without half-spaces."""
import numpy as np
import pytest

import pump_amd as P

from test_gpu_parity import (dev, edge_mask_host, host, oracle_propagate, pack_bits, ptr,
                             random_hsmc_inputs, unpack_bits)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_p,w_range,max_hs,n_new", [
    (1, (2, 6), 1, 40), (63, (2, 40), 5, 40), (64, (2, 40), 5, 40), (65, (2, 40), 5, 40),
    (1024, (2, 20), 5, 40), (1025, (2, 20), 5, 300), (2000, (60, 70), 5, 40),
    (130, (64, 65), 3, 40), (320, (200, 230), 5, 20), (96, (2, 9), 700, 12),
    (96, (2, 9), 1024, 12), (272, (3, 4), 5, 4095),
    # to the 64-paths-per-wave form with few slots and particles
    (96, (2, 9), 1, 20479), (96, (2, 9), 1, 20480), (1000, (2, 3), 4, 24576)])
def test_path_form_against_oracle(n_p, w_range, max_hs, n_new):
    d = random_hsmc_inputs(n_p + max_hs, n_edges=80, max_hs=max_hs, n_p=n_p, n_mc=n_p + 3, T=70,
                           n_new=n_new, n_parent=9, variable=True, w_range=w_range)
    # a third of the edges store nothing, some only in their last waypoint
    for e in range(0, 80, 3):
        lo, hi = d["off"][e] * max_hs, d["off"][e + 1] * max_hs
        d["bs"][lo: hi - (max_hs if e % 2 else 0)] = 1111
    # a NaN slot is a stored half-space that no particle passes; the oracle's
    # clamp (b < 1000) leaves it out, so its edge is kept inside the table
    d["bs"][5] = np.nan
    nan_edge = int(np.searchsorted(d["off"] * max_hs, 5, side="right")) - 1
    d["wf_edge"][0] = nan_edge
    d["times"][0] = 0.5
    d["wf_prev"][d["wf_edge"] == nan_edge] = 0
    ref_v, ref_cp, ref_cl = oracle_propagate(d)
    npar = d["n_parent"]
    g = {k: dev(d[k]) for k in ("off", "as_", "bs", "offs", "topts", "times", "wf_edge",
                                 "wf_prev")}
    g_mask = dev(edge_mask_host(d["off"], d["bs"], max_hs))
    edges = (n_new, 0, ptr(g["off"]), ptr(g["wf_edge"]), ptr(g["wf_prev"]))
    table = (ptr(g["times"]), ptr(g["topts"]), d["dt"], max_hs, ptr(g["offs"]), d["T"], d["om"],
             d["n_mc"])
    print("path form", n_p, w_range, max_hs, n_new, flush=True)
    # the drop-in call, children after their parents in one array
    valid, clamp = dev(d["valid"]), dev(np.zeros(1, np.uint64))
    P.check("propagate", P.lib.pump_propagate_valid_particles(
        *edges, npar, ptr(g["as_"]), ptr(g["bs"]), None, *table, ptr(valid), n_p, ptr(clamp),
        None))
    assert np.array_equal(host(valid), ref_v) and int(host(clamp)[0]) == ref_cl
    for bits in (0, 1):
        width = (n_p + 63) // 64 * 8 if bits else n_p
        src = dev(pack_bits(d["valid"][:npar], n_p) if bits else d["valid"][:npar])
        for mask in (None, g_mask.p):
            dst = dev(np.full((n_new + 1, width), 0x5a, np.uint8))
            cp, clamp = dev(np.zeros(n_new + 2, np.float32)), dev(np.zeros(1, np.uint64))
            row_src, pcp = dev(np.full(n_new, -7, np.int32)), dev(np.zeros(npar, np.float32))
            P.check("propagate_cp_cow", P.lib.pump_propagate_cp_cow(
                bits, *edges, ptr(g["as_"]), ptr(g["bs"]), mask, *table, ptr(src), ptr(pcp),
                ptr(dst), 1, ptr(row_src), n_p, ptr(cp), 2, 0, None, None, ptr(clamp), None, 0,
                None))
            rows = host(dst)
            assert (rows[0] == 0x5a).all() and int(host(clamp)[0]) == ref_cl
            got = unpack_bits(rows[1:].copy().view(np.uint64), n_p) if bits else rows[1:]
            assert np.array_equal(got, ref_v[npar:]), (bits, mask is None)
            assert np.array_equal(host(cp)[2:], ref_cp[npar:])
            assert np.array_equal(host(row_src), np.arange(n_new))


@pytest.mark.parametrize("w_range,max_hs,n_p,n_new", [
    ((2, 4), 1, 64, 4096), ((2, 9), 5, 120, 4097), ((2, 17), 5, 200, 5000),
    ((30, 33), 8, 72, 4100), ((33, 64), 9, 68, 4096), ((60, 70), 5, 333, 4200),
    ((2, 20), 3, 24, 20500)])
def test_batched_form_without_summaries(w_range, max_hs, n_p, n_new):
    """The batched form finds the waypoints that store a half-space from the
    slots themselves: groups of 4 to 64 lanes per path, more slots than one
    round of loads, edges past 64 waypoints among them; byte rows of 8-, 4-
    and 1-byte units; the drop-in call in place at its batched sizes."""
    d = random_hsmc_inputs(max_hs + n_p, n_edges=700, max_hs=max_hs, n_p=n_p, n_mc=n_p + 1, T=90,
                           n_new=n_new, n_parent=33, variable=True, w_range=w_range)
    drop = np.random.default_rng(1).uniform(size=700) < 0.7
    for e in np.nonzero(drop)[0]:
        d["bs"][d["off"][e] * max_hs: d["off"][e + 1] * max_hs] = 1111
    ref_v, ref_cp, ref_cl = oracle_propagate(d)
    npar = d["n_parent"]
    g = {k: dev(d[k]) for k in ("off", "as_", "bs", "offs", "topts", "times", "wf_edge",
                                 "wf_prev")}
    edges = (n_new, 0, ptr(g["off"]), ptr(g["wf_edge"]), ptr(g["wf_prev"]))
    table = (ptr(g["times"]), ptr(g["topts"]), d["dt"], max_hs, ptr(g["offs"]), d["T"], d["om"],
             d["n_mc"])
    print("batched", w_range, max_hs, n_p, n_new, flush=True)
    ws_bytes = P.lib.pump_propagate_workspace(n_new, d["T"])
    ws = P.DeviceArray(shape=(ws_bytes,), dtype=np.uint8, fill=0x77)
    src, dst = dev(d["valid"][:npar]), dev(np.full((n_new, n_p), 9, np.uint8))
    cp, clamp = dev(np.zeros(n_new, np.float32)), dev(np.zeros(1, np.uint64))
    P.check("propagate_cp", P.lib.pump_propagate_cp(
        *edges, ptr(g["as_"]), ptr(g["bs"]), None, *table, ptr(src), ptr(dst), 0, n_p, ptr(cp), 0,
        ptr(clamp), ws.p, ws_bytes, None))
    assert np.array_equal(host(dst), ref_v[npar:]) and np.array_equal(host(cp), ref_cp[npar:])
    assert int(host(clamp)[0]) == ref_cl
    valid, clamp = dev(d["valid"]), dev(np.zeros(1, np.uint64))
    P.check("propagate", P.lib.pump_propagate_valid_particles(
        *edges, npar, ptr(g["as_"]), ptr(g["bs"]), None, *table, ptr(valid), n_p, ptr(clamp),
        None))
    assert np.array_equal(host(valid), ref_v) and int(host(clamp)[0]) == ref_cl
    allcp = dev(np.zeros(npar + n_new, np.float32))
    P.check("cp", P.lib.pump_calculate_cp_hsmc(n_new, npar, ptr(allcp), ptr(valid), n_p, None))
    assert np.array_equal(host(allcp)[npar:], ref_cp[npar:])


@pytest.mark.parametrize("n_p,max_hs,scale", [(64, 1, 1.0), (300, 5, 1.0), (520, 9, 1.0),
                                              (300, 5, 1e-14), (300, 5, 1e12)])
def test_batched_tests_at_the_reach_of_the_particles(n_p, max_hs, scale):
    """The batched tests leave out a half-space that no particle reaches.
    Normals along a group's farthest particle with offsets a float above, at
    and below that particle's product, and values that the bound cannot judge
    (zero, tiny, infinite and NaN normals, offsets at and below zero)."""
    n_new = 4100
    d = random_hsmc_inputs(n_p, n_edges=300, max_hs=max_hs, n_p=n_p, n_mc=n_p, T=50, n_new=n_new,
                           n_parent=9, variable=True, w_range=(2, 9))
    rng = np.random.default_rng(n_p)
    f = np.float32
    # the same particles at every time: the products do not depend on the path
    o = d["offs"][0] * f(scale)
    o[: n_p // 2] *= f(0.25)  # groups of different reach
    o[1] = 0.0
    d["offs"][:] = o
    far = o[np.argmax((o * o).sum(1))]
    hs = d["bs"].size
    d["as_"][:] = far * f(1.0 / scale) * rng.choice(np.array([0.5, 1, 2], f), (hs, 1))
    lhs = d["as_"][:, 0] * far[0]
    lhs = lhs + d["as_"][:, 1] * far[1]
    lhs = (lhs + d["as_"][:, 2] * far[2]) * d["om"]
    d["bs"][:] = lhs * rng.choice(np.array([0.9, 0.9999, 1, 1, 1.00001, 1.0001, 1.1], f), hs)
    up = rng.integers(-1, 2, hs)
    d["bs"][:] = np.where(up == 0, d["bs"], np.nextafter(d["bs"], np.where(up < 0, f(-np.inf), f(np.inf))))
    d["bs"][d["bs"] >= 1000] = 999
    odd = rng.uniform(size=hs) < 0.1
    values = np.array([0, -0.0, 1e-45, 1e-25, 1e-8, -1e-3, 900], f)
    d["bs"][odd] = rng.choice(values, odd.sum())
    # a normal that fails a particle for good is kept rare
    odd = rng.uniform(size=hs) < 0.02
    d["as_"][odd] = rng.choice(np.array([0, 1e-38, 1e-24, 1e20, np.inf, np.nan], f),
                               (odd.sum(), 3))
    d["bs"][rng.uniform(size=hs) < 0.5] = 1111
    ref_v, ref_cp, ref_cl = oracle_propagate(d)
    npar = d["n_parent"]
    assert 0.02 < ref_v[npar:].mean() < 0.84
    g = {k: dev(d[k]) for k in ("off", "as_", "bs", "offs", "topts", "times", "wf_edge",
                                 "wf_prev")}
    g_mask = dev(edge_mask_host(d["off"], d["bs"], max_hs))
    ws_bytes = P.lib.pump_propagate_workspace(n_new, d["T"])
    ws = P.DeviceArray(shape=(ws_bytes,), dtype=np.uint8)
    print("reach", n_p, max_hs, scale, flush=True)
    for bits in (0, 1):
        width = (n_p + 63) // 64 * 8 if bits else n_p
        src = dev(pack_bits(d["valid"][:npar], n_p) if bits else d["valid"][:npar])
        dst = dev(np.zeros((n_new, width), np.uint8))
        cp, clamp = dev(np.zeros(n_new, np.float32)), dev(np.zeros(1, np.uint64))
        fn = P.lib.pump_propagate_cp_bits if bits else P.lib.pump_propagate_cp
        P.check("propagate_cp", fn(
            n_new, 0, ptr(g["off"]), ptr(g["wf_edge"]), ptr(g["wf_prev"]), ptr(g["as_"]),
            ptr(g["bs"]), g_mask.p, ptr(g["times"]), ptr(g["topts"]), d["dt"], max_hs,
            ptr(g["offs"]), d["T"], d["om"], d["n_mc"], ptr(src), ptr(dst), 0, n_p, ptr(cp), 0,
            *((0, None, None) if bits else ()), ptr(clamp), ws.p, ws_bytes, None))
        rows = host(dst)
        got = unpack_bits(rows.view(np.uint64), n_p) if bits else rows
        assert np.array_equal(got, ref_v[npar:]), bits
        assert np.array_equal(host(cp), ref_cp[npar:])


@pytest.mark.parametrize("T", [1, 1025, 4096, 4097, 5200])
def test_batched_chunks_of_many_times(T):
    """The chunks of tables around the scan's LDS capacity of 4096 times, most
    of the pairs in few times and the others spread over all of them."""
    n_new, n_p, max_hs = 6000, 64, 3
    d = random_hsmc_inputs(T, n_edges=300, max_hs=max_hs, n_p=n_p, n_mc=n_p, T=T, n_new=n_new,
                           n_parent=40, variable=True, w_range=(2, 9))
    d["dt"] = np.float32(4.0 / 5200)
    d["wf_prev"][: n_new // 2] = 0
    d["wf_edge"][: n_new // 2] = 5
    ref_v, ref_cp, ref_cl = oracle_propagate(d)
    npar = d["n_parent"]
    g = {k: dev(d[k]) for k in ("off", "as_", "bs", "offs", "topts", "times", "wf_edge",
                                 "wf_prev")}
    g_mask = dev(edge_mask_host(d["off"], d["bs"], max_hs))
    ws_bytes = P.lib.pump_propagate_workspace(n_new, T)
    ws = P.DeviceArray(shape=(ws_bytes,), dtype=np.uint8)
    src = dev(pack_bits(d["valid"][:npar], n_p))
    dst = dev(np.zeros((n_new, 8), np.uint8))
    cp, clamp = dev(np.zeros(n_new, np.float32)), dev(np.zeros(1, np.uint64))
    row_src = dev(np.zeros(n_new, np.int32))
    pcp = dev(1 - d["valid"][:npar].mean(1, dtype=np.float32))
    print("times", T, flush=True)
    P.check("cow", P.lib.pump_propagate_cp_cow(
        1, n_new, 0, ptr(g["off"]), ptr(g["wf_edge"]), ptr(g["wf_prev"]), ptr(g["as_"]),
        ptr(g["bs"]), g_mask.p, ptr(g["times"]), ptr(g["topts"]), d["dt"], max_hs, ptr(g["offs"]),
        T, d["om"], d["n_mc"], ptr(src), ptr(pcp), ptr(dst), 0, ptr(row_src), n_p, ptr(cp), 0, 0,
        None, None, ptr(clamp), ws.p, ws_bytes, None))
    own = host(row_src) >= 0
    assert own.mean() > 0.5 and int(host(clamp)[0]) == ref_cl
    got = unpack_bits(host(dst).view(np.uint64), n_p)
    assert np.array_equal(got[own], ref_v[npar:][own])
    assert np.array_equal(ref_v[npar:][~own], d["valid"][d["wf_prev"][~own]])
    assert np.array_equal(host(cp)[own], ref_cp[npar:][own])
