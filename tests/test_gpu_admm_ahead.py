"""The ADMM loop enqueued a few iterations ahead of the device, against the
same loop enqueued whole (as a graph): same bits and counts for limits below,
at and just above the lead, and for one that the loop stops long before."""
import numpy as np
import pytest

import silk_physics_amd as sp
from silk_physics_amd import scenes

from helpers import gpu_world

pytestmark = pytest.mark.gpu


def _run(n, inner, graph):
    V, F = scenes.grid_sheet(n)
    w = gpu_world(acceleration_z=-9.81, dt=1 / 60, max_inner_iteration=inner, admm_graph=graph)
    r, h = w.add_cloth(sp.ClothConfig(), sp.CollisionConfig(), V, F, np.array([0], np.int32))
    assert r, r.to_string()
    out = []
    for _ in range(4):
        r = w.solver_step()
        assert r, r.to_string()
        _, x = w.get_cloth_position(h, n=V.size)
        st = w.last_stats
        out.append((x, st.admm_iterations, st.pcg_solves, st.pcg_iterations))
    return out


@pytest.mark.parametrize("n,inner", [(9, 1), (9, 3), (9, 4), (9, 5), (9, 100), (33, 100)])
def test_same_steps_as_the_loop_enqueued_whole(n, inner):
    whole = _run(n, inner, sp.GRAPH_ON)
    ahead = _run(n, inner, sp.GRAPH_OFF)
    for k, (a, b) in enumerate(zip(whole, ahead)):
        assert np.array_equal(a[0], b[0]), f"step {k}: {np.abs(a[0] - b[0]).max():.3e}"
        assert a[1:] == b[1:]
        assert 1 <= a[1] <= inner
    if inner == 100:
        assert max(a[1] for a in whole) < inner - 10
