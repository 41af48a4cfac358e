"""Every form of the contact update (one, two or four contacts per thread; a
vertex as four or three words of LDS; normals in LDS or in registers) against
the one that keeps everything in global memory and branches: the same
operations in the same order, so the same bits.  A sheet lying on a coarse
one, at contact counts on both sides of the thread limits, and a sheet under
spikes that each touch three vertices of their own, so that many vertices
meet few contacts (too many for four words each)."""
import numpy as np
import pytest

import silk_physics_amd as sp
from silk_physics_amd import scenes

from helpers import gpu_world

pytestmark = pytest.mark.gpu


def _flat(n, m):
    V, F = scenes.grid_sheet(n, z=0.004)
    SV, SF = scenes.grid_sheet(m, z=0.0)
    return V, F, SV * 1.1 - [0.05, 0.05, 0.0], SF


def _spikes():
    V, F = scenes.grid_sheet(101, z=0.0)
    lo, hi = V.min(0), V.max(0)
    h = (hi[0] - lo[0]) / 100
    SV, SF = [], []
    for i in range(0, 100, 2):
        for j in range(0, 100, 2):
            # Near the middle of one of the cell's triangles, base far above.
            x, y = lo[0] + (i + 0.3) * h, lo[1] + (j + 0.35) * h
            b = len(SV)
            SV += [[x, y, 2e-4], [x - 1e-3, y, 0.05], [x + 1e-3, y, 0.05]]
            SF.append([b, b + 1, b + 2])
    return V, F, np.array(SV), np.array(SF, np.int32)


def _run(scene, gravity, variant, monkeypatch, steps):
    if variant is not None:
        monkeypatch.setenv("SILK_HIP_CONTACT_VARIANT", str(variant))
    else:
        monkeypatch.delenv("SILK_HIP_CONTACT_VARIANT", raising=False)
    V, F, SV, SF = scene
    w = gpu_world(acceleration_z=gravity, dt=1 / 60, max_inner_iteration=12)
    cc = sp.CollisionConfig()
    r, h = w.add_cloth(sp.ClothConfig(), cc, V, F, [])
    assert r, r.to_string()
    r, _ = w.add_obstacle(cc, np.ascontiguousarray(SV, V.dtype), SF)
    assert r, r.to_string()
    xs, counts = [], []
    for _ in range(steps):
        r = w.solver_step()
        assert r, r.to_string()
        r, x = w.get_cloth_position(h, n=V.size)
        xs.append(x)
        counts.append(w.last_stats.contacts)
    return xs, counts


@pytest.mark.parametrize("name,lo,hi", [("one", 1, 1024), ("two", 1025, 2048),
                                        ("four", 2049, 4096), ("narrow", 2049, 4096)])
def test_forms_of_the_update_give_the_same_bits(name, lo, hi, monkeypatch):
    scene = {"one": lambda: _flat(8, 3), "two": lambda: _flat(20, 6),
             "four": lambda: _flat(30, 8), "narrow": _spikes}[name]()
    gravity = 9.81 if name == "narrow" else -9.81
    ref, counts = _run(scene, gravity, 3, monkeypatch, 3)
    print(name, "contacts per step", counts)
    assert any(lo <= c <= hi for c in counts)
    for variant in (None, 1):
        got, _ = _run(scene, gravity, variant, monkeypatch, 3)
        for k, (a, b) in enumerate(zip(ref, got)):
            assert np.array_equal(a, b), (variant, k, np.abs(a - b).max())
