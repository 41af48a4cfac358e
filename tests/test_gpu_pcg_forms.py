"""Forms of the persistent PCG that grids of ordinary size do not reach: rows too
wide for the registers, and the two-exchange kernel (SILK_HIP_PCG=two; by
itself it serves sheets of more than 20 coarse banks) under the residual
replacement, in batches of systems and in the autotuner's comparison of its one-
and two-workgroups-per-CU variants.  Two worlds of different sizes on one
kernel instance, stepped in turn."""
import numpy as np
import pytest

import oracle as O
import silk_physics_amd as sp
from silk_physics_amd import scenes

from helpers import f32, gpu_world

pytestmark = pytest.mark.gpu

OFF = sp.CollisionConfig(is_collision_on=False, is_self_collision_on=False)
STEP = dict(acceleration_z=-9.81, dt=1 / 60, max_inner_iteration=10,
            linear_solver_rel_tol_min=1e-6, linear_solver_rel_tol_max=1e-6,
            initial_linear_rel_tol=1e-6)


def _fan(spokes, rings):
    """A disc of `rings` rings of `spokes` vertices around one vertex."""
    a = 2 * np.pi * np.arange(spokes) / spokes
    r = np.linspace(0, 0.5, rings + 1)[1:]
    V = np.concatenate([[[0.0, 0.0, 0.0]]] + [
        np.stack([x * np.cos(a), x * np.sin(a), 0.03 * np.sin(9 * x + a)], 1) for x in r])
    nxt = (np.arange(spokes) + 1) % spokes
    F = [np.stack([np.zeros(spokes, int), 1 + np.arange(spokes), 1 + nxt], 1)]
    for k in range(rings - 1):
        p, q = 1 + k * spokes, 1 + (k + 1) * spokes
        F += [np.stack([p + np.arange(spokes), q + np.arange(spokes), q + nxt], 1),
              np.stack([p + np.arange(spokes), q + nxt, p + nxt], 1)]
    return V.astype(np.float32), np.concatenate(F).astype(np.int32)


@pytest.mark.parametrize("kernel", ["one", "two"])
@pytest.mark.parametrize("rings", [2, 14])
def test_rows_wider_than_the_registers(rings, kernel, monkeypatch):
    """The middle of a fan of 48 has more neighbours than the 32 a thread keeps
    (the bending operator joins second neighbours, so its ring has too): a
    solve against the oracle, and steps under the true-residual criterion whose
    FP64 residuals are recomputed by a kernel of their own."""
    monkeypatch.setenv("SILK_HIP_PCG", kernel)
    V, F = _fan(48, rings)
    nv = V.shape[0]
    w = gpu_world(pcg_criterion=sp.PCG_RHS, linear_solver_abs_tol=1e-30)
    r, h = w.add_cloth(sp.ClothConfig(), OFF, V, F, [])
    assert r, r.to_string()
    assert w.scene_info()["pcg_exchanges"] == (1 if kernel == "one" else 2)
    _, perm, offs = w.get_partition(h, nv)
    Vp, Fp = np.zeros_like(V), perm[F]
    Vp[perm] = V
    mass = 0.1 * O.mass_area(Vp.astype(np.float64), Fp)[0]
    d = (mass / f32(1 / 60) ** 2).astype(np.float32)
    b = (np.random.default_rng(5).normal(size=(nv, 3)) * 300 * mass[:, None])
    b = b.astype(np.float32).reshape(-1)
    x, it = w.debug_pcg(d, b, 1e-6)
    xo, oi = O.pcg(Vp.astype(np.float64), Fp, f32(100.0), f32(1e-4), offs,
                   np.repeat(d.astype(np.float64), 3), b.astype(np.float64),
                   np.zeros(b.size), 1e-6, 1e-30, 3000, criterion=1)
    assert oi["status"] == 1
    e = np.abs(x - xo).max() / np.abs(xo).max()
    print(f"{rings} rings, {kernel}: {it} / {oi['iters']} iterations, error {e:.2e}")
    # As for the grids: the error |r| <= 1e-6 |b| leaves is the oracle's own.
    assert e <= 2e-5
    assert abs(it - oi["iters"]) <= 2 + oi["iters"] // 10

    w = gpu_world(**STEP, pcg_criterion=sp.PCG_TRUE, true_residual_stats=1)
    edge = np.array([nv - 48, nv - 24], np.int32)
    r, h = w.add_cloth(sp.ClothConfig(), OFF, V, F, edge)
    assert r, r.to_string()
    for _ in range(4):
        assert w.solver_step()
        st = w.last_stats
        assert st.pcg_unverified_solves == 0 and st.pcg_stalled_solves == 0
        assert st.max_true_rel_residual <= 1e-6


def test_two_exchange_replacements(monkeypatch):
    """Steps of the 80x80 sheet meeting the sphere: some solves pass the
    recurrence test and not the FP64 one, are continued from the replaced
    residual, and all pass it in the end."""
    monkeypatch.setenv("SILK_HIP_PCG", "two")
    s = scenes.c2_scene(80, z=0.305)
    w = gpu_world(**STEP, max_outer_iteration=4, pcg_criterion=sp.PCG_TRUE,
                  true_residual_stats=1)
    cc = sp.CollisionConfig()
    assert w.add_cloth(sp.ClothConfig(), cc, s["V"], s["F"], s["pins"])[0]
    assert w.add_obstacle(cc, s["SV"], s["SF"])[0]
    assert w.scene_info()["pcg_exchanges"] == 2
    restarts = 0
    for _ in range(8):
        assert w.solver_step()
        st = w.last_stats
        assert st.pcg_unverified_solves == 0 and st.pcg_stalled_solves == 0
        assert st.max_true_rel_residual <= 1e-6
        restarts += st.pcg_restarts
    assert restarts > 0


def test_two_exchange_batches_match_one_launch(monkeypatch):
    """Sheets of uneven size in one launch of the two-exchange kernel, in
    batches and each alone: the same bits."""
    monkeypatch.setenv("SILK_HIP_PCG", "two")
    sizes = [3, 40, 21, 97]

    def run(ns):
        w = gpu_world(**STEP, admm_abs_tol=1e-9, admm_rel_tol=1e-9, pcg_criterion=sp.PCG_TRUE)
        hs = []
        for n in ns:
            V, F = scenes.grid_sheet(n)
            r, h = w.add_cloth(sp.ClothConfig(), OFF, V, F, scenes.top_corner_pins(n))
            assert r
            hs.append((h, V.size))
        for _ in range(3):
            assert w.solver_step()
            assert w.last_stats.pcg_unverified_solves == 0
        return [w.get_cloth_position(h, n=n)[1] for h, n in hs], w.scene_info()

    together, info = run(sizes)
    monkeypatch.setenv("SILK_HIP_PCG_BATCH_WG", "50")
    batched, info_b = run(sizes)
    monkeypatch.delenv("SILK_HIP_PCG_BATCH_WG")
    assert info["pcg_exchanges"] == info_b["pcg_exchanges"] == 2
    assert info_b["pcg_launches"] > info["pcg_launches"] == 1
    for n, xt, xb in zip(sizes, together, batched):
        alone, _ = run([n])
        np.testing.assert_array_equal(xt, alone[0])
        np.testing.assert_array_equal(xb, alone[0])


def test_autotune_compares_the_two_exchange_variants(monkeypatch):
    """A sheet whose solve fits the device both ways: the autotuner times one and
    two workgroups per CU, finds the same solution (it fails otherwise), keeps
    the faster, and the steps that follow are those of a world left alone."""
    monkeypatch.setenv("SILK_HIP_PCG", "two")
    V, F = scenes.grid_sheet(48)

    def world():
        w = gpu_world(**STEP)
        r, h = w.add_cloth(sp.ClothConfig(), OFF, V, F, scenes.top_corner_pins(48))
        assert r
        assert w.solver_step()
        return w, h

    (plain, hp), (tuned, ht) = world(), world()
    r, rep = tuned.autotune()
    assert r, r.to_string()
    assert rep["pcg_us"][0] > 0 and rep["pcg_us"][1] > 0
    assert rep["pcg_us"][rep["pcg_variant"]] == min(rep["pcg_us"].values())
    assert tuned.scene_info()["pcg_dense"] == rep["pcg_variant"]
    for _ in range(3):
        assert plain.solver_step() and tuned.solver_step()
    np.testing.assert_array_equal(plain.get_cloth_position(hp, n=V.size)[1],
                                  tuned.get_cloth_position(ht, n=V.size)[1])


def test_worlds_of_different_size_in_turn(monkeypatch):
    """A large and a small sheet on the same kernel instance, stepped in turn:
    the same bits as each by itself."""
    monkeypatch.delenv("SILK_HIP_PCG", raising=False)

    def world(n):
        V, F = scenes.grid_sheet(n)
        w = gpu_world(**STEP)
        r, h = w.add_cloth(sp.ClothConfig(), OFF, V, F, scenes.top_corner_pins(n))
        assert r
        return w, h, V.size

    def step(ws):
        for _ in range(3):
            for w, _, _ in ws:
                assert w.solver_step()
        return [w.get_cloth_position(h, n=n)[1] for w, h, n in ws]

    alone = [step([world(n)])[0] for n in (120, 100)]
    large, small = world(120), world(100)
    info = [w.scene_info() for w in (large[0], small[0])]
    assert info[0]["pcg_lds_bytes"] > info[1]["pcg_lds_bytes"]
    assert all(12 < i["coarse_banks"] <= 20 for i in info)  # one instance
    for a, b in zip(alone, step([large, small])):
        np.testing.assert_array_equal(a, b)
