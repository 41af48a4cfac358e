"""The traversal (64 queries per wavefront against chunks of 64 primitives)
where it can go wrong: trees of one chunk and less, ragged last chunks, one
wavefront's worth of queries and one more, and a crowd in which every box
overlaps every other, so that the stage of hits fills and empties many times.
Exact sets against the oracle, at the default split and after tuning it."""
import numpy as np
import pytest

from test_gpu_collision import _f32, _pair_worlds

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,subdiv,spread", [(2, 0, 0.02), (5, 0, 0.02), (8, 1, 0.02),
                                             (9, 2, 0.05), (33, 3, 0.01), (9, 1, None)])
def test_candidate_sets_equal_oracle(n, subdiv, spread):
    V, F, SV, SF, w, h, ho, ow, perm = _pair_worlds(n, subdiv)
    rng = np.random.default_rng(n)
    base = np.zeros((V.shape[0] + SV.shape[0], 3))
    base[perm] = V
    base[V.shape[0]:] = SV
    if spread is None:  # a crowd
        base = rng.uniform(-0.01, 0.01, base.shape)
        spread = 0.05
    a = _f32(base + rng.uniform(-spread, spread, base.shape))
    b = _f32(a + rng.uniform(-spread, spread, base.shape))
    opt, oee = ow.candidates(a.reshape(-1), b.reshape(-1))
    assert w.solver_step()  # (the tuning below needs one)
    for tuned in (False, True):
        if tuned:
            r, _ = w.autotune()
            assert r, r.to_string()
        gpt, gee = w.debug_candidates(a, b)
        assert sorted(map(tuple, gpt.tolist())) == sorted(map(tuple, opt.tolist()))
        assert sorted(map(tuple, gee.tolist())) == sorted(map(tuple, oee.tolist()))
    print(f"n={n}: PT {len(opt)} EE {len(oee)}")
    assert len(opt) + len(oee) > 0
