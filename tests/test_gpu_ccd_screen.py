"""The CCD's screening pass and the quotients of its root search.

The step's CCD screens its candidates one per thread and searches the rest one
per wavefront; the earliest TOI of every outer iteration decides where the step
rolls back to, so a candidate dropped wrongly shows as another TOI.  Against
the oracle replaying the step: a sheet with a handful of candidates (less than
one wavefront) and one with several thousand (many workgroups, the last one
ragged).

The search divides box widths by tolerances with a reciprocal while every
tolerance is at least 2^-44, and by division below; the queries here lie on
both sides of that line and on it."""
import numpy as np
import pytest

import oracle as O
from helpers import gpu_world, lockstep_step
from test_gpu_collision import MS, TOL, _pair_worlds, _queries

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,subdiv,steps", [(2, 0, 8), (24, 2, 6)])
def test_step_toi_matches_oracle(n, subdiv, steps):
    kw = dict(acceleration_z=-9.81, dt=1 / 60, max_inner_iteration=20,
              linear_solver_rel_tol_min=1e-6, linear_solver_rel_tol_max=1e-6,
              initial_linear_rel_tol=1e-6)
    V, F, SV, SF, w, h, ho, ow, perm = _pair_worlds(n, subdiv, 0.315, kw)
    dt = float(np.float32(1 / 60))
    x_prev = V.astype(np.float64).reshape(-1)
    v_prev = np.zeros_like(x_prev)
    cands = []
    for _ in range(steps):
        xg, _, e_rep, _, missing = lockstep_step(w, h, ow, V.size, x_prev, v_prev)
        assert missing == 0
        # The replayed step, each TOI included, within the lockstep bound.
        assert e_rep <= 1e-4
        cands.append(w.last_stats.ccd_candidates)
        v_prev = (xg - x_prev) / dt
        x_prev = xg
    assert min(cands) > 0 and (min(cands) < 64) == (n == 2)


@pytest.mark.parametrize("scale", [1.0, 2.0 ** 22, 2.0 ** 24])
def test_root_search_bit_exact_at_every_tolerance(scale):
    """Coordinates scaled by powers of two (exact), so the parameter
    tolerances TOL / (3 extent) cross 2^-44 with extents of about 1e6 to 1e7;
    minimum separation and filters scale along.  Same bits as the oracle."""
    w = gpu_world()
    vf, p0, p1, err = _queries(400, seed=11)
    p0, p1, err = p0 * scale, p1 * scale, err * scale
    hit, toi = w.debug_ccd(vf, p0, p1, err, MS * scale, TOL)
    ohit = np.zeros_like(hit)
    otoi = np.zeros_like(toi)
    for i in range(vf.size):
        h, t = O.ccd(bool(vf[i]), p0[i].reshape(4, 3), p1[i].reshape(4, 3), MS * scale,
                     TOL, err[i], stack_cap=64)
        ohit[i], otoi[i] = h, (t if h else 0.0)
    assert ohit.sum() > vf.size // 8
    np.testing.assert_array_equal(hit, ohit)
    np.testing.assert_array_equal(toi, otoi)
