"""The workloads whose speed matters, and how to run each once.

A planning program calls the library stage by stage: all-pairs 2pBVP solve,
neighbour selection, edge waypoints and collision flags, the half-space cache,
then per search iteration one half-space Monte Carlo (HSMC) step, and for the
candidate solutions the full Monte Carlo collision probability.  There is one
family of cases per stage, driven through the C ABI on device buffers as
bench.py and a C++ host drive it, one for a whole plan (roadmap and search of
one problem) and one for the captured graphs of a batch of problems.  Sizes
are those of pump_amd.configs (NUM 4000/16000/32000, 30 to 200 boxes, 1000 to
4096 particles) and of the small problems of the tests.

listed() and draw() give cases, prepare() what a program holds before the
call, run() one pass, exact() the same outputs in 64 bits by plain torch,
work() the bytes and operations a pass cannot do without.
"""
import ctypes
import functools
import math

import numpy as np
import torch

import pump_amd as P

DEV = "cuda"
DT = 0.05          # time step of the noise tables and of sampled paths
TMAX = 5.0         # upper bracket of the arrival time
G = -9.81
MAX_HS = 5
NOISE_STEPS = 2001
_PATH_ROWS = 256   # rows a program allots for a candidate path


def listed():
    return [
        # a toy problem's pair table: one short launch, latency is all of it
        dict(name="pairs_256", kind="pairs", num=256),
        # the pair table of the NUM=16000 problem: 256 million arrival times,
        # the longest pass of a plan
        dict(name="pairs_16000", kind="pairs", num=16000),
        # from the pair tables to the numbered edges and their waypoint
        # counts, at the largest problem of the 256-problem workload
        dict(name="neighbours_8000", kind="neighbours", num=8000, k=50, w_fixed=0),
        # the reference's shape: 20 waypoints on every edge, ten boxes
        dict(name="edges_w20_4000", kind="edges", num=4000, k=50, n_obs=10, walls=False,
             w_fixed=20, form="fused"),
        # ceil(tau/dt) waypoints per edge, thirty boxes, 1.28 million edges
        dict(name="edges_16000", kind="edges", num=16000, k=80, n_obs=30, walls=False,
             w_fixed=0, form="fused"),
        # the cluttered corridor world through the FP32-waypoint form
        dict(name="edges_walls_fp32", kind="edges", num=32000, k=50, n_obs=200, walls=True,
             w_fixed=0, form="fp32"),
        # half-spaces of the same 1.28 million edges
        dict(name="halfspaces_16000", kind="halfspaces", num=16000, k=80, n_obs=30, walls=False,
             w_fixed=0, offset_mult=0.03),
        # the reference's call pair on byte rows: an ordinary wavefront
        dict(name="hsmc_bytes_4000", kind="hsmc", num=4000, k=50, n_obs=10, w_fixed=20,
             offset_mult=0.02, n_new=60000, n_parents=1500, n_p=1000, form="dropin"),
        # the search's step on bit rows at the NUM=16000 problem's largest
        # wavefronts, with the survivors' rows gathered
        dict(name="hsmc_cow_16000", kind="hsmc", num=16000, k=80, n_obs=30, w_fixed=0,
             offset_mult=0.03, n_new=1000000, n_parents=16000, n_p=2000, form="cow"),
        # full Monte Carlo of the 64 candidate paths of one query in the
        # corridor world
        dict(name="mccp_walls_64", kind="mccp", n_paths=64, n_mc=4096, n_obs=200, walls=True,
             offset_mult=0.02),
        # one small problem from host arrays to its path: build and search
        dict(name="plan_1000", kind="plan", num=1000, k=50, n_obs=10, offset_mult=0.02,
             n_p=500),
        # eight uneven problems: the captured pair, edge and Monte Carlo stages
        dict(name="batch_8", kind="batch", n_inst=8, num_lo=1000, num_hi=4000),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["pairs", "neighbours", "edges", "edges", "halfspaces", "hsmc", "hsmc",
                       "mccp", "plan", "batch"])
    walls = rng.random() < 0.3
    n_obs = _log_int(rng, 1, 200)
    w_fixed = rng.choice([0, 0, 9, 20])
    om = round(rng.uniform(0.01, 0.05), 4)
    k = rng.randint(20, 80)
    if kind == "pairs":
        return dict(kind=kind, num=_log_int(rng, 64, 12000))
    if kind == "neighbours":
        return dict(kind=kind, num=_log_int(rng, 300, 12000), k=k, w_fixed=w_fixed)
    if kind == "edges":
        return dict(kind=kind, num=_log_int(rng, 300, 16000), k=k, n_obs=n_obs, walls=walls,
                    w_fixed=w_fixed, form=rng.choice(["fused", "fused", "fp32", "plain"]))
    if kind == "halfspaces":
        return dict(kind=kind, num=_log_int(rng, 300, 16000), k=k, n_obs=n_obs, walls=walls,
                    w_fixed=w_fixed, offset_mult=om)
    if kind == "hsmc":
        n_new = _log_int(rng, 200, 400000)
        return dict(kind=kind, num=_log_int(rng, 1000, 8000), k=k, n_obs=n_obs,
                    w_fixed=w_fixed, offset_mult=om, n_new=n_new,
                    n_parents=max(1, n_new // rng.randint(10, 60)),
                    n_p=rng.choice([128, 500, 1000, 2000, 4096, rng.randint(100, 2047)]),
                    form=rng.choice(["dropin", "cow", "cow", "bits", "split"]))
    if kind == "mccp":
        return dict(kind=kind, n_paths=_log_int(rng, 1, 64), n_mc=_log_int(rng, 256, 8192),
                    n_obs=n_obs, walls=walls, offset_mult=om)
    if kind == "plan":
        return dict(kind=kind, num=_log_int(rng, 300, 3000), k=k, n_obs=rng.randint(5, 50),
                    offset_mult=om, n_p=rng.choice([128, 500, 1000]))
    lo = _log_int(rng, 500, 1500)
    return dict(kind=kind, n_inst=rng.randint(2, 8), num_lo=lo, num_hi=lo + rng.randint(0, 2500))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _problem(num, seed, n_obs, walls=False, start=None, goal=None, side=(0.03, 0.15)):
    """Samples and boxes of pump_amd.configs' distributions."""
    s = P.ProblemSpec()
    s.num, s.seed, s.n_obs = num, seed, n_obs
    s.lo[:] = [0, 0, 0, -0.5, -0.5, -0.5]
    s.hi[:] = [1, 1, 1, 0.5, 0.5, 0.5]
    s.start[:] = list(start) if start else [0.1, 0.1, 0.1, 0, 0, 0]
    s.goal[:] = list(goal) if goal else [0.9, 0.9, 0.9, 0, 0, 0]
    s.obstacle_kind = 1 if walls else 0
    s.centre_lo, s.centre_hi = (0.0, 1.0) if walls else (0.2, 0.8)
    s.side_lo, s.side_hi = side
    s.wall_thickness = 0.02
    s.wall_long_lo, s.wall_long_hi = 0.3, 0.8
    s.wall_short_lo, s.wall_short_hi = 0.05, 0.3
    s.vel_span = 3.1
    return P.gen_problem(s)


def _params(c, **over):
    return P.params(rn_perc=float(np.float32(c["k"] / (c["num"] - 1))),
                    w_fixed=c.get("w_fixed", 0), wp_dt=DT, w_cap=64,
                    offset_mult=c.get("offset_mult", 0.02), n_p=c.get("n_p", 128),
                    max_hs=MAX_HS, **over)


@functools.lru_cache(maxsize=3)
def _noise(n_mc):
    """One noise table, as a program keeps it: (offsets_time, xcomb) on the host."""
    ot, xc, _, _ = P.make_noise_device(P.noise_spec(n_mc=n_mc, tmax_steps=NOISE_STEPS))
    return ot, xc


def _up(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


class _Raw:
    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = dict(data=(ptr, False), shape=tuple(shape),
                                             typestr=typestr, version=2)


def _view(owner, ptr, shape, typestr):
    """Device memory of the library as a tensor (no copy).  The tensor holds
    its owner (the roadmap or batch), which frees the memory when it goes."""
    t = torch.as_tensor(_Raw(owner, ptr, shape, typestr), device=DEV)
    assert t.data_ptr() == ptr
    return t


def _edge_cap(c):
    """Edges at most: the pairs cheaper than the rn_perc-th."""
    num = c["num"]
    return int(P.lib.pump_rn_index(num, float(np.float32(c["k"] / (num - 1)))))


def _waypoint_cap(c):
    """Rows a program allots for the waypoints of _edge_cap(c) edges."""
    w = c.get("w_fixed", 0)
    return _edge_cap(c) * w if w else int(2.2 * _edge_cap(c) * _waypoints(c)) + 64


def _pad(a, rows):
    """a in the first rows of a zeroed array of a size the case fixes."""
    assert len(a) <= rows
    out = np.zeros((rows,) + a.shape[1:], a.dtype)
    out[: len(a)] = a
    return out


def _roadmap(c, seed):
    """A built roadmap's edges (and half-spaces) as tensors of their own."""
    samples, obstacles = _problem(c["num"], seed, c["n_obs"], c.get("walls", False))
    rm = P.Roadmap(samples, obstacles, samples[-1], None, None, _params(c))
    i, d = rm.info, rm.device()
    E, n_wp, hs = int(i.n_edges), int(i.n_waypoints), int(i.max_hs)
    P.sync()
    assert E <= _edge_cap(c) and n_wp <= _waypoint_cap(c)
    m = dict(
        samples=_view(rm, d.samples, (c["num"], 6), "<f4").clone(),
        obstacles=_view(rm, d.obstacles, (c["n_obs"], 12), "<f4").clone(),
        src=_view(rm, d.edge_src, (E,), "<i4").clone(), dst=_view(rm, d.edge_dst, (E,), "<i4").clone(),
        tau=_view(rm, d.topts_edge, (E,), "<f4").clone(),
        off=_view(rm, d.wp_offsets, (E + 1,), "<i8").clone(),
        row_start=_view(rm, d.row_start, (c["num"] + 1,), "<i8").clone(),
        free=_view(rm, d.is_free_edges, (E,), "|u1").clone(), E=E, n_wp=n_wp, max_hs=hs)
    if c["kind"] == "halfspaces":
        m["disc"] = _view(rm, d.disc, (n_wp, 6), "<f4").clone()
    if c["kind"] == "hsmc":
        m["as"] = _view(rm, d.as_, (n_wp, hs, 3), "<f4").clone()
        m["bs"] = _view(rm, d.bs, (n_wp, hs), "<f4").clone()
        m["mask"] = _view(rm, d.edge_hs_mask, (E,), "<i8").clone()
    torch.cuda.synchronize()
    rm.close()
    return m


def _wavefront(m, c, gen):
    """Open paths at random nodes, each followed by its node's free out-edges."""
    rs = m["row_start"].cpu().numpy()
    free = m["free"].cpu().numpy().astype(bool)
    rng = np.random.default_rng(gen)
    nodes = rng.integers(0, c["num"], c["n_parents"])
    edges, prev, n = [], [], 0
    p = 0
    while n < c["n_new"] and p < 64 * c["n_parents"]:
        i = nodes[p % c["n_parents"]] if p < c["n_parents"] else rng.integers(0, c["num"])
        e = np.arange(rs[i], rs[i + 1])
        e = e[free[e]][: c["n_new"] - n]
        edges.append(e)
        prev.append(np.full(len(e), p % c["n_parents"]))
        n += len(e)
        p += 1
    prev, edges = np.concatenate(prev), np.concatenate(edges)
    order = np.argsort(prev, kind="stable")
    return _up(edges[order].astype(np.int32)), _up(prev[order].astype(np.int32)), rng


def _pack(valid):
    """bool [rows, n_p] to 64-bit words, bit p % 64 of word p // 64."""
    rows, n_p = valid.shape
    words = (n_p + 63) // 64
    v = torch.zeros((rows, words * 64), dtype=torch.int64, device=DEV)
    v[:, :n_p] = valid
    return (v.view(rows, words, 64) << torch.arange(64, device=DEV)).sum(2)


def _candidate_paths(c, seed):
    """Paths along free edges of a small roadmap, sampled at DT: what a search
    hands to the full Monte Carlo."""
    rng = np.random.default_rng(seed)
    num, k = 2000, 40
    samples, obstacles = _problem(num, seed, c["n_obs"], c["walls"])
    rm = P.Roadmap(samples, obstacles, samples[-1], None, None,
                   _params(dict(num=num, k=k, w_fixed=20)))
    e, f = rm.edges(), rm.flags()
    rm.close()
    rs, free = e["row_start"], f["is_free_edges"].astype(bool)
    paths, tries = [], 0
    while len(paths) < c["n_paths"]:
        hops, tries = int(rng.integers(4, 8)), tries + 1
        node = int(rng.integers(num))
        nodes = [node]
        while len(nodes) <= hops:
            out = e["edge_dst"][rs[node]:rs[node + 1]][free[rs[node]:rs[node + 1]]]
            out = out[~np.isin(out, nodes)]
            if len(out) == 0:
                break
            node = int(rng.choice(out))
            nodes.append(node)
        if len(nodes) > hops or (tries > 100 * c["n_paths"] and len(nodes) > 1):
            paths.append(P.find_optimal_path(samples[nodes], DT, _PATH_ROWS)[0])
    return obstacles, paths


# ---------------------------------------------------------------------------
def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed)


def run(state):
    return _RUN[state["kind"]](state)


def exact(case, seed):
    f = _EXACT.get(case["kind"])
    return f(case, seed) if f else None


def _p(t):
    return t.data_ptr()


# ---- all-pairs 2pBVP ------------------------------------------------------
def _prepare_pairs(c, seed):
    samples, _ = _problem(c["num"], seed, 1)
    n = c["num"] * (c["num"] - 1)
    return dict(kind="pairs", num=c["num"], samples=_up(samples),
                copts=torch.empty(n, device=DEV), topts=torch.empty(n, device=DEV))


def _run_pairs(s):
    P.check("pump_fill_copts_topts", P.lib.pump_fill_copts_topts(
        _p(s["samples"]), s["num"], TMAX, _p(s["copts"]), _p(s["topts"]), None))
    return dict(copts=s["copts"], topts=s["topts"])


def _cost64(t, D, S, R, vz):
    return 12 * D / t**3 - 12 * S / t**2 + 4 * R / t + 2 * G * vz + (1 + G * G) * t


def _exact_pairs(c, seed):
    """Arrival time by 60 bisection steps on the cost's derivative, in FP64."""
    x = _prepare_pairs(c, seed)["samples"].double()
    n = c["num"]
    cost = torch.empty(n * (n - 1), dtype=torch.float64, device=DEV)
    time = torch.empty_like(cost)
    step = max(1, (1 << 22) // n)
    for i0 in range(0, n, step):
        a = x[i0:i0 + step, None]
        dp, v0, v1 = x[None, :, :3] - a[..., :3], a[..., 3:], x[None, :, 3:]
        D, S, R = (dp * dp).sum(2), (dp * (v0 + v1)).sum(2), (v0 * v0 + v0 * v1 + v1 * v1).sum(2)
        lo, hi = torch.full_like(D, 1e-6), torch.full_like(D, TMAX)
        for _ in range(60):
            t = 0.5 * (lo + hi)
            up = ((1 + G * G) * t * t - 4 * R) * t * t + 24 * S * t - 36 * D > 0
            hi, lo = torch.where(up, t, hi), torch.where(up, lo, t)
        t = 0.5 * (lo + hi)
        cst = _cost64(t, D, S, R, a[..., 5] - x[None, :, 5])
        keep = torch.ones_like(D, dtype=torch.bool)
        keep[torch.arange(len(a), device=DEV), torch.arange(i0, i0 + len(a), device=DEV)] = False
        o = i0 * (n - 1)
        cost[o:o + len(a) * (n - 1)] = cst[keep]
        time[o:o + len(a) * (n - 1)] = t[keep]
    return dict(copts=cost, topts=time)


# ---- neighbour selection --------------------------------------------------
def _prepare_neighbours(c, seed):
    s = _prepare_pairs(c, seed)
    _run_pairs(s)
    num, n = c["num"], c["num"] * (c["num"] - 1)
    idx = cap = _edge_cap(c)
    ws = max(P.lib.pump_select_rn_workspace(n), P.lib.pump_scan_workspace(max(num, cap) + 1))
    return dict(kind="neighbours", num=num, n=n, idx=idx, w_fixed=c["w_fixed"],
                samples=s["samples"], copts=s["copts"], topts=s["topts"],
                goal=np.ascontiguousarray(s["samples"][-1].cpu().numpy()),
                ws=torch.empty(ws, dtype=torch.uint8, device=DEV), ws_bytes=ws,
                row_start=torch.zeros(num + 1, dtype=torch.int64, device=DEV),
                src=torch.zeros(cap, dtype=torch.int32, device=DEV),
                dst=torch.zeros(cap, dtype=torch.int32, device=DEV),
                ce=torch.zeros(cap, device=DEV), te=torch.zeros(cap, device=DEV),
                deg=torch.zeros(num, dtype=torch.int32, device=DEV),
                h=torch.zeros(num, device=DEV),
                off=torch.zeros(cap + 1, dtype=torch.int64, device=DEV))


def _run_neighbours(s):
    rn, ne = ctypes.c_float(), ctypes.c_int64()
    nn, total = ctypes.c_int(), ctypes.c_int64()
    lib, num = P.lib, s["num"]
    P.check("pump_select_rn", lib.pump_select_rn(
        _p(s["copts"]), s["n"], s["idx"], ctypes.byref(rn), _p(s["ws"]), s["ws_bytes"], None))
    P.check("pump_count_edges", lib.pump_count_edges(
        _p(s["copts"]), num, rn.value, _p(s["row_start"]), ctypes.byref(ne), _p(s["ws"]),
        s["ws_bytes"], None))
    E = ne.value  # at most idx: the costs strictly below the idx-th smallest
    P.check("pump_fill_edges", lib.pump_fill_edges(
        _p(s["copts"]), _p(s["topts"]), num, rn.value, _p(s["row_start"]), _p(s["src"]),
        _p(s["dst"]), _p(s["ce"]), _p(s["te"]), None))
    P.check("pump_max_nn_size", lib.pump_max_nn_size(
        _p(s["row_start"]), _p(s["dst"]), E, num, _p(s["deg"]), ctypes.byref(nn), None))
    P.check("pump_heuristic", lib.pump_heuristic(
        _p(s["samples"]), num, P.fp(s["goal"]), TMAX, _p(s["h"]), None))
    P.check("pump_waypoint_offsets", lib.pump_waypoint_offsets(
        _p(s["te"]), E, s["w_fixed"], DT, 64, _p(s["off"]), ctypes.byref(total), _p(s["ws"]),
        s["ws_bytes"], None))
    return dict(rn=rn.value, n_edges=E, max_nn=nn.value, n_waypoints=total.value,
                row_start=s["row_start"], src=s["src"], dst=s["dst"], copts=s["ce"], topts=s["te"],
                in_degree=s["deg"], h=s["h"], offsets=s["off"])


def _exact_neighbours(c, seed):
    s = _prepare_neighbours(c, seed)
    keys, _ = torch.sort(s["copts"])
    rn = keys[s["idx"]]
    at = torch.nonzero(s["copts"] < rn).view(-1)
    x = s["samples"].double()
    a, g = x, x[-1]
    dp, v0, v1 = g[:3] - a[:, :3], a[:, 3:], g[3:]
    D, S, R = (dp * dp).sum(1), (dp * (v0 + v1)).sum(1), (v0 * v0 + v0 * v1 + v1 * v1).sum(1)
    lo, hi = torch.full_like(D, 1e-6), torch.full_like(D, TMAX)
    for _ in range(60):
        t = 0.5 * (lo + hi)
        up = ((1 + G * G) * t * t - 4 * R) * t * t + 24 * S * t - 36 * D > 0
        hi, lo = torch.where(up, t, hi), torch.where(up, lo, t)
    h = _cost64(0.5 * (lo + hi), D, S, R, a[:, 5] - g[5])
    h[-1] = 0
    ce, te = s["ce"].double(), s["te"].double()
    ce[: len(at)], te[: len(at)] = s["copts"][at].double(), s["topts"][at].double()
    return dict(rn=float(rn), n_edges=None, max_nn=None, n_waypoints=None, row_start=None,
                src=None, dst=None, copts=ce, topts=te, in_degree=None, h=h, offsets=None)


# ---- edge waypoints and flags ---------------------------------------------
def _prepare_edges(c, seed):
    m = _roadmap(c, seed)
    return dict(kind="edges", form=c["form"], n_obs=c["n_obs"], **m,
                disc=torch.zeros((_waypoint_cap(c), 6), device=DEV),
                flags=torch.zeros(_edge_cap(c), dtype=torch.uint8, device=DEV))


def _run_edges(s):
    lib = P.lib
    edges = (_p(s["samples"]), _p(s["src"]), _p(s["dst"]), _p(s["tau"]), s["E"], _p(s["off"]), 0)
    if s["form"] == "plain":
        P.check("pump_discretize_edges", lib.pump_discretize_edges(*edges, _p(s["disc"]), None))
        P.check("pump_free_edges_var", lib.pump_free_edges_var(
            _p(s["obstacles"]), s["n_obs"], _p(s["off"]), _p(s["disc"]), _p(s["flags"]), s["E"],
            None))
    elif s["form"] == "fp32":
        P.check("pump_edges_discretize_check_fp32", lib.pump_edges_discretize_check_fp32(
            *edges, _p(s["obstacles"]), s["n_obs"], _p(s["disc"]), _p(s["flags"]), None, None))
    else:
        P.check("pump_edges_discretize_check", lib.pump_edges_discretize_check(
            *edges, _p(s["obstacles"]), s["n_obs"], _p(s["disc"]), _p(s["flags"]), None))
    return dict(waypoints=s["disc"], free=s["flags"])


def _exact_edges(c, seed):
    """The cubic Hermite segment through both end states."""
    m = _roadmap(c, seed)
    x = m["samples"].double()
    whole = torch.zeros((_waypoint_cap(c), 6), dtype=torch.float64, device=DEV)
    out = whole[: m["n_wp"]]
    W = m["off"][1:] - m["off"][:-1]
    e = torch.repeat_interleave(torch.arange(m["E"], device=DEV), W)
    k = torch.arange(m["n_wp"], device=DEV) - m["off"][e]
    tau = m["tau"].double()[e]
    dt = m["tau"][e] / (W[e] - 1).float()
    t = (dt * k.float()).double()  # the sampled times are part of the inputs
    first, last = k == 0, k == W[e] - 1
    a, b = x[m["src"].long()[e]], x[m["dst"].long()[e]]
    for d in range(3):
        p0, v0, p1, v1 = a[:, d], a[:, d + 3], b[:, d], b[:, d + 3]
        c2 = 3 * (p1 - p0) / tau**2 - (2 * v0 + v1) / tau
        c3 = 2 * (p0 - p1) / tau**3 + (v0 + v1) / tau**2
        out[:, d] = torch.where(last, p1, torch.where(first, p0, p0 + t * (v0 + t * (c2 + t * c3))))
        out[:, d + 3] = torch.where(last, v1, torch.where(first, v0, v0 + t * (2 * c2 + t * 3 * c3)))
    return dict(waypoints=whole, free=None)


# ---- half-space cache -----------------------------------------------------
def _prepare_halfspaces(c, seed):
    m = _roadmap(c, seed)
    hs, rows = m["max_hs"], _waypoint_cap(c)
    return dict(kind="halfspaces", n_obs=c["n_obs"], **m,
                maxd2=float(P.lib.pump_maxd2(c["offset_mult"])),
                as_=torch.zeros((rows, hs, 3), device=DEV),
                bs=torch.zeros((rows, hs), device=DEV),
                count=torch.zeros(rows, dtype=torch.int32, device=DEV),
                mask=torch.zeros(_edge_cap(c), dtype=torch.int64, device=DEV))


def _run_halfspaces(s):
    P.check("pump_cache_halfspaces", P.lib.pump_cache_halfspaces(
        s["E"], _p(s["disc"]), _p(s["free"]), s["n_obs"], s["max_hs"], _p(s["obstacles"]), 0,
        _p(s["off"]), _p(s["as_"]), _p(s["bs"]), _p(s["count"]), s["maxd2"], 1, _p(s["mask"]),
        None))
    return dict(normals=s["as_"], offsets=s["bs"], count=s["count"], mask=s["mask"])


def _exact_halfspaces(c, seed):
    """The closest point of each near box, its velocity component removed."""
    s = _prepare_halfspaces(c, seed)
    hs, n_wp = s["max_hs"], s["n_wp"]
    W = s["off"][1:] - s["off"][:-1]
    free = torch.repeat_interleave(s["free"].bool(), W)
    normals, offsets = s["as_"].double(), s["bs"].double()  # zero past the waypoints
    normals[:n_wp], offsets[:n_wp] = -1.0, 1111.0
    stored = torch.zeros(n_wp, dtype=torch.int64, device=DEV)
    pos, vel = s["disc"][:, :3].double(), s["disc"][:, 3:].double()
    vv = (vel * vel).sum(1)
    vv = torch.where(vv == 0, torch.full_like(vv, 1e-5), vv)
    for box in s["obstacles"].double():
        v = torch.minimum(torch.maximum(pos, box[0:3]), box[6:9]) - pos
        # whether a box is near is decided on the 32-bit distance, as stored
        near = free & ((v * v).sum(1).float() <= s["maxd2"]) & (stored < hs)
        at = torch.nonzero(near).view(-1)
        u = v[at] - ((v[at] * vel[at]).sum(1) / vv[at])[:, None] * vel[at]
        normals[at, stored[at]] = u
        offsets[at, stored[at]] = (u * u).sum(1)
        stored[at] += 1
    return dict(normals=normals, offsets=offsets, count=None, mask=None)


# ---- half-space Monte Carlo step ------------------------------------------
def _prepare_hsmc(c, seed):
    m = _roadmap(c, seed)
    edge, prev, rng = _wavefront(m, c, seed)
    n_new, n_par, n_p = len(edge), c["n_parents"], c["n_p"]
    n_mc = max(2048, n_p)
    # open paths have lost up to two particles in a hundred, at times up to 2 s
    alive = _up((1.0 - 0.02 * rng.random(n_par)).astype(np.float32))
    gen = torch.Generator(device=DEV).manual_seed(seed)
    valid = torch.rand((n_par, n_p), generator=gen, device=DEV) < alive[:, None]
    form = c["form"]
    s = dict(kind="hsmc", form=form, n_new=n_new, n_par=n_par, n_p=n_p, n_mc=n_mc,
             om=c["offset_mult"], **m, edge=edge, prev=prev,
             times=_up(rng.uniform(0, 2, n_par).astype(np.float32)),
             offsets=_up(_noise(n_mc)[0]), parents=valid)
    par_cp = (n_p - valid.sum(1)).float() / float(n_p)
    if form == "dropin":
        s["valid"] = torch.zeros((n_par + n_new, n_p), dtype=torch.uint8, device=DEV)
        s["valid"][:n_par] = valid
        s["cp"] = torch.zeros(n_par + n_new, device=DEV)
        s["cp"][:n_par] = par_cp
        return s
    words = (n_p + 63) // 64
    ws = P.lib.pump_propagate_workspace(n_new, NOISE_STEPS)
    s.update(src_rows=_pack(valid), par_cp=par_cp, words=words,
             rows=torch.zeros((n_new, words), dtype=torch.int64, device=DEV),
             cp=torch.zeros(n_new, device=DEV),
             ws=torch.empty(ws, dtype=torch.uint8, device=DEV), ws_bytes=ws)
    if form == "split":
        n_split = P.lib.pump_split_offsets_bytes(NOISE_STEPS, n_mc)
        s["split"] = torch.empty(n_split, dtype=torch.uint8, device=DEV)
        P.check("pump_split_offsets", P.lib.pump_split_offsets(
            _p(s["offsets"]), NOISE_STEPS, n_mc, _p(s["split"]), None))
    if form == "cow":
        sel = np.sort(rng.permutation(n_new)[: max(1, n_new // 8)]).astype(np.int32)
        s.update(row_src=torch.zeros(n_new, dtype=torch.int32, device=DEV), sel=_up(sel),
                 kept=torch.zeros((len(sel), words), dtype=torch.int64, device=DEV))
    return s


def _run_hsmc(s):
    lib, form = P.lib, s["form"]
    wave = (s["n_new"], 0, _p(s["off"]), _p(s["edge"]), _p(s["prev"]))
    if form == "dropin":
        # the reference's two calls: children after their parents, in place
        P.check("pump_propagate_valid_particles", lib.pump_propagate_valid_particles(
            *wave, s["n_par"], _p(s["as"]), _p(s["bs"]), None, _p(s["times"]), _p(s["tau"]), DT,
            s["max_hs"], _p(s["offsets"]), NOISE_STEPS, s["om"], s["n_mc"], _p(s["valid"]),
            s["n_p"], None, None))
        P.check("pump_calculate_cp_hsmc", lib.pump_calculate_cp_hsmc(
            s["n_new"], s["n_par"], _p(s["cp"]), _p(s["valid"]), s["n_p"], None))
        return dict(rows=s["valid"], cp=s["cp"])
    step = (_p(s["as"]), _p(s["bs"]), _p(s["mask"]), _p(s["times"]), _p(s["tau"]), DT,
            s["max_hs"], _p(s["offsets"]), NOISE_STEPS, s["om"], s["n_mc"], _p(s["src_rows"]))
    if form == "cow":
        # the search's step: children that meet no half-space share their
        # parent's row, then the survivors' rows are gathered
        P.check("pump_propagate_cp_cow", lib.pump_propagate_cp_cow(
            1, *wave, *step, _p(s["par_cp"]), _p(s["rows"]), 0, _p(s["row_src"]), s["n_p"],
            _p(s["cp"]), 0, 0, None, None, None, _p(s["ws"]), s["ws_bytes"], None))
        P.check("pump_gather_rows_cow", lib.pump_gather_rows_cow(
            _p(s["rows"]), _p(s["src_rows"]), _p(s["row_src"]), _p(s["sel"]), len(s["sel"]),
            _p(s["kept"]), 0, s["words"] * 8, 1, None))
        return dict(rows=s["kept"], cp=s["cp"])
    split = form == "split"
    P.check("pump_propagate_cp_bits", lib.pump_propagate_cp_bits(
        *wave, *step, _p(s["rows"]), 0, s["n_p"], _p(s["cp"]), 0, 1 if split else 0,
        _p(s["split"]) if split else None, None, None, _p(s["ws"]), s["ws_bytes"], None))
    return dict(rows=s["rows"], cp=s["cp"])


def _exact_hsmc(c, seed):
    """Every (waypoint, half-space) pair of every child, particle by particle."""
    s = _prepare_hsmc(c, seed)
    e, prev, n_p = s["edge"].long(), s["prev"].long(), s["n_p"]
    g0, W = s["off"][e], s["off"][e + 1] - s["off"][e]
    live = (s["bs"] < 1000).any(1)
    above = torch.zeros(s["n_wp"] + 1, dtype=torch.int64, device=DEV)
    above[1:] = live.cumsum(0)
    hit = torch.nonzero(above[g0 + W] > above[g0]).view(-1)
    inv = (n_p - s["parents"].sum(1)).double()[prev]
    dtl = s["tau"][e] / (W - 1).float()
    offs = s["offsets"][:, :n_p].double()
    for q0 in range(0, len(hit), 20000):
        w = hit[q0:q0 + 20000]
        ok = s["parents"][prev[w]]
        for i in range(int(W[w].max())):
            for h in range(s["max_hs"]):
                wp = torch.minimum(g0[w] + i, g0[w] + W[w] - 1)
                use = torch.nonzero((i < W[w]) & (s["bs"][wp, h] < 1000)).view(-1)
                if len(use) == 0:
                    continue
                time = s["times"][prev[w[use]]] + torch.tensor(float(i), device=DEV) * dtl[w[use]]
                ti = (time / np.float32(DT)).to(torch.int64).clamp(0, NOISE_STEPS - 1)
                a, b = s["as"][wp[use], h].double(), s["bs"][wp[use], h].double()
                for u0 in range(0, len(use), 4000):
                    u = slice(u0, u0 + 4000)
                    lhs = (offs[ti[u]] * a[u, None]).sum(2) * float(np.float32(s["om"]))
                    ok[use[u]] &= lhs < b[u, None]
        inv[w] = (n_p - ok.sum(1)).double()
    cp = inv / n_p
    if c["form"] == "dropin":
        cp = torch.cat([s["cp"][: s["n_par"]].double(), cp])
    return dict(rows=None, cp=cp)


# ---- full Monte Carlo -----------------------------------------------------
def _prepare_mccp(c, seed):
    obstacles, paths = _candidate_paths(c, seed)
    rows = np.stack([_pad(p, _PATH_ROWS) for p in paths])
    n_mc = c["n_mc"]
    return dict(kind="mccp", n_obs=c["n_obs"], n_mc=n_mc, n_paths=len(paths), stride=_PATH_ROWS,
                om=c["offset_mult"], obstacles=_up(obstacles), xcomb=_up(_noise(n_mc)[1]),
                paths=_up(rows), rows=len(paths[0]), T=_up(np.array([len(p) for p in paths], np.int32)),
                hits=torch.zeros(len(paths), dtype=torch.int32, device=DEV))


def _run_mccp(s):
    if s["n_paths"] == 1:
        # a single candidate through the reference's own call
        cp = ctypes.c_float()
        P.check("pump_collision_probability", P.lib.pump_collision_probability(
            _p(s["obstacles"]), s["n_obs"], _p(s["xcomb"]), NOISE_STEPS, s["n_mc"], s["om"],
            _p(s["paths"]), s["rows"], ctypes.byref(cp), None))
        return dict(cp=cp.value)
    P.check("pump_collision_probability_many", P.lib.pump_collision_probability_many(
        _p(s["obstacles"]), s["n_obs"], _p(s["xcomb"]), NOISE_STEPS, s["n_mc"], s["om"],
        _p(s["paths"]), s["stride"], _p(s["T"]), s["n_paths"], _p(s["hits"]), 1, None))
    return dict(hits=s["hits"])


# ---- a whole plan ---------------------------------------------------------
def _prepare_plan(c, seed):
    samples, obstacles = _problem(c["num"], seed, c["n_obs"], side=(0.05, 0.2))
    ot, xc = _noise(1024)
    return dict(kind="plan", samples=samples, obstacles=obstacles, ot=ot, xc=xc,
                edge_cap=_edge_cap(c), path_cap=int(2 * c["num"] * math.sqrt(c["num"])),
                prm=_params(c, cp_target=0.01, cp_factor=2.0, validity_bits=1))


def _run_plan(s):
    rm = P.Roadmap(s["samples"], s["obstacles"], s["samples"][-1], s["ot"], s["xc"], s["prm"])
    r = rm.search()
    table, flags = rm.paths(int(r.num_paths)), rm.flags()
    rm.close()
    nodes = np.array(list(r.soln_nodes)[: r.soln_len], np.int64)
    return dict(status=r.status, itrs=r.itrs, num_paths=r.num_paths, considered=r.num_considered,
                cost=r.soln_cost, cp=r.soln_cp, time=r.soln_time, nodes=_pad(nodes, 256),
                paths={k: _pad(v, s["path_cap"]) for k, v in table.items()},
                free_samples=flags["is_free_samples"],
                free_edges=_pad(flags["is_free_edges"], s["edge_cap"]),
                wp_offsets=_pad(flags["wp_offsets"], s["edge_cap"] + 1))


# ---- a batch of problems --------------------------------------------------
def _prepare_batch(c, seed):
    rng = np.random.default_rng(seed)
    problems, cases = [], []
    for j in range(c["n_inst"]):
        # sizes spread evenly over the logarithm of the range
        at = (j + 0.5) / c["n_inst"]
        num = int(round(c["num_lo"] ** (1 - at) * c["num_hi"] ** at))
        start = tuple(rng.uniform(0, 0.2, 3)) + (0.0, 0.0, 0.0)
        goal = tuple(rng.uniform(0.8, 1.0, 3)) + (0.0, 0.0, 0.0)
        smp, obs = _problem(num, int(rng.integers(1 << 31)), 5 + (j * 29) % 46,
                            start=start, goal=goal, side=(0.03, 0.2))
        cases.append(dict(num=num, k=50, offset_mult=float(rng.uniform(0.01, 0.05)),
                          n_p=(500, 1000, 2000)[j % 3]))
        problems.append((smp, obs, smp[-1], _params(cases[-1], keep_pairs=1)))
    ot, xc = _noise(2048)
    b = P.Batch(problems, ot, xc)
    b.mc_build(n_parents=1024, seed=int(rng.integers(1 << 31)))
    views, out = [], []
    for j, cj in enumerate(cases):
        rm = b.roadmap(j)
        i, d = rm.info, rm.device()
        E, n_wp, hs = int(i.n_edges), int(i.n_waypoints), int(i.max_hs)
        views.append(dict(waypoints=_view(rm, d.disc, (n_wp, 6), "<f4"),
                          free=_view(rm, d.is_free_edges, (E,), "|u1"),
                          normals=_view(rm, d.as_, (n_wp, hs, 3), "<f4"),
                          offsets=_view(rm, d.bs, (n_wp, hs), "<f4")))
        rows = _waypoint_cap(cj)
        out.append(dict(copts=_view(rm, d.copts, (int(i.n_pairs),), "<f4"),
                        topts=_view(rm, d.topts, (int(i.n_pairs),), "<f4"),
                        waypoints=torch.zeros((rows, 6), device=DEV),
                        free=torch.zeros(_edge_cap(cj), dtype=torch.uint8, device=DEV),
                        normals=torch.zeros((rows, hs, 3), device=DEV),
                        offsets=torch.zeros((rows, hs), device=DEV)))
    return dict(kind="batch", batch=b, views=views, out=out)


def _run_batch(s):
    b = s["batch"]
    for stage in (0, 1, 2):
        b.replay(stage)
    for k, (v, o) in enumerate(zip(s["views"], s["out"])):
        # into the program's own arrays, which outlive the batch
        for name, t in v.items():
            o[name][: len(t)].copy_(t)
        o["cp"] = _pad(b.mc_get(k)["cp"], len(o["free"]))
    return s["out"]


# ---------------------------------------------------------------------------
_PREPARE = dict(pairs=_prepare_pairs, neighbours=_prepare_neighbours, edges=_prepare_edges,
                halfspaces=_prepare_halfspaces, hsmc=_prepare_hsmc, mccp=_prepare_mccp,
                plan=_prepare_plan, batch=_prepare_batch)
_RUN = dict(pairs=_run_pairs, neighbours=_run_neighbours, edges=_run_edges,
            halfspaces=_run_halfspaces, hsmc=_run_hsmc, mccp=_run_mccp, plan=_run_plan,
            batch=_run_batch)
_EXACT = dict(pairs=_exact_pairs, neighbours=_exact_neighbours, edges=_exact_edges,
              halfspaces=_exact_halfspaces, hsmc=_exact_hsmc)


def _waypoints(c):
    """Waypoints per edge: fixed, or the mean of ceil(tau/dt) (5.7 at 80
    neighbours of 16000, growing slowly with the neighbours' share)."""
    return c.get("w_fixed") or 5.7 * (c["k"] / c["num"] / 0.005) ** 0.1


def work(case):
    """What a pass cannot do without: inputs read once, outputs written once;
    a pair's root of the quartic and one cost, a waypoint's two cubics, a
    segment against the few boxes near it, three products per half-space test."""
    c, kind = case, case["kind"]
    if kind == "pairs":
        n = c["num"] * (c["num"] - 1)
        return dict(bytes=8 * n + 24 * c["num"], flops=200 * n)
    if kind == "neighbours":
        n, E = c["num"] * (c["num"] - 1), c["num"] * c["k"]
        # the costs are read once and the arrival times of the edges
        return dict(bytes=4 * n + 28 * E + 44 * c["num"], flops=n)
    if kind in ("edges", "halfspaces"):
        E = c["num"] * c["k"]
        wp = E * _waypoints(c)
        if kind == "edges":
            return dict(bytes=24 * wp + 33 * E + 24 * c["n_obs"], flops=60 * wp)
        hs = min(MAX_HS, c["n_obs"])
        return dict(bytes=(24 + 16 * hs + 4) * wp + 17 * E, flops=20 * wp)
    if kind == "hsmc":
        row = c["n_p"] if c["form"] == "dropin" else (c["n_p"] + 63) // 64 * 8
        # copy-on-write: one child in thirty gets a row, one in eight is kept
        rows = c["n_new"] * (1 / 30 + 1 / 8) if c["form"] == "cow" else c["n_new"]
        return dict(bytes=row * (rows + c["n_parents"]) + 20 * c["n_new"],
                    flops=6 * c["n_p"] * c["n_new"] / 25)
    if kind == "mccp":
        T = 45  # rows of a candidate path
        return dict(bytes=12 * T * c["n_mc"] + 24 * T * c["n_paths"],
                    flops=40 * T * c["n_mc"] * c["n_paths"])
    num = c["num"] if kind == "plan" else 0.5 * (c["num_lo"] + c["num_hi"])
    inst = 1 if kind == "plan" else c["n_inst"]
    n, E = num * num, num * 50
    per = 8 * n + E * 6.4 * (24 + 24 + 16 * MAX_HS + 4)
    tables = 24 * 1024 * NOISE_STEPS if kind == "plan" else 0
    return dict(bytes=inst * per + tables, flops=inst * 200 * n)


def tolerance(case):
    """The tables are defined value by value (flags, indices and counts are
    whole numbers and equal); arrival times and costs hold 1e-5, what 32-bit
    evaluation of a waypoint or half-space leaves is below 1e-6."""
    kind = case["kind"]
    if kind == "neighbours":
        return {"rel": 1e-6}
    if kind in ("edges", "halfspaces", "hsmc"):
        return {"rel": 1e-6, "max": 1e-4}
    if kind == "mccp":
        return {"rel": 1e-6}
    return {"rel": 1e-5, "max": 1e-3}
