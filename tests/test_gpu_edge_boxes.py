"""The edge pass with more than 64 boxes (their slab table) against the oracle:
box counts around the table's words and the staged 256; extents that cannot be
cut into slabs (one point, infinite, overflowing); boxes with a NaN, infinite
or inverted bound, without thickness, with faces on end states, and far outside
the extent.  Flags bit-exact, both waypoint forms."""
import numpy as np
import pytest

from test_gpu_edges import edge_set, gpu_pass, gpu_pass32, oracle_pass
from test_gpu_parity import assert_close_f32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("extent", ["unit", "point", "infinite", "overflow", "nan"])
@pytest.mark.parametrize("n_obs", [65, 128, 129, 192, 256, 257])
def test_many_boxes(n_obs, extent):
    d = edge_set(n_obs, 90, 11, n_obs, 2, 24, side=(0.01, 0.05))
    rng = np.random.default_rng(n_obs)
    lo, hi = d["obs"][:, 0:3], d["obs"][:, 6:9]
    # the first 64 boxes give the extent and are left as they are in the others
    odd = np.arange(64 if extent != "unit" else 0, n_obs)
    odd = odd[rng.uniform(size=len(odd)) < 0.3]
    for i, b in enumerate(odd):
        ax = i % 3
        f = np.float32
        if i % 8 == 0:
            lo[b, ax] = np.nan
        elif i % 8 == 1:
            hi[b, ax] = np.nan
        elif i % 8 == 2:
            lo[b, ax] = -np.inf
        elif i % 8 == 3:
            hi[b, ax] = np.inf
        elif i % 8 == 4:
            hi[b, ax] = lo[b, ax]
        elif i % 8 == 5:
            lo[b, ax], hi[b, ax] = hi[b, ax], lo[b, ax]
        elif i % 8 == 6:
            lo[b, ax] = d["s"][b % len(d["s"]), ax]
            hi[b, ax] = lo[b, ax] + f(0.02)
        else:
            lo[b, ax], hi[b, ax] = f(40), f(41)
    if extent == "point":
        lo[:64] = hi[:64] = np.float32(0.5)
    elif extent == "infinite":
        lo[:64, 0], hi[:64, 0] = -np.inf, -np.inf
        lo[:64, 1] = -np.inf
        hi[:64, 1] = np.float32(-5)
    elif extent == "overflow":
        lo[0], hi[0] = np.float32(-3e38), np.float32(-3e38)
        lo[1], hi[1] = np.float32(3e38), np.float32(3.1e38)
    elif extent == "nan":
        lo[:64, 2] = hi[:64, 2] = np.nan
        hi[:64, 0] = lo[:64, 0]
    print("boxes", n_obs, extent, flush=True)
    disc_ref, free_ref = oracle_pass(d)
    assert 0.02 < free_ref.mean() < 0.995
    disc, flags, flags2 = gpu_pass(d)
    assert np.array_equal(flags, free_ref) and np.array_equal(flags2, free_ref)
    assert_close_f32(disc, disc_ref)
    for write in (True, False):
        assert np.array_equal(gpu_pass32(d, write=write)[1], free_ref), write
