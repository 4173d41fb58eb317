"""GPU test of the gather-mode adjoint's membership words (kept modulo 8 cells
and clamped): particles thrown up to 12 cells between the frame's grid and a
pass's positions, in both directions of every axis and against the walls, so
that pairs occur of which both, one or neither are each other's candidates.
The scatter mode decides them by comparing whole cells.
"""
import numpy as np
import pytest

from pbf import params as P
from pbf import scenes
from test_gpu_adjoint import _target, gpu_grad, rel

pytestmark = pytest.mark.gpu


# (9, 9, 9): a team of lanes a target; 90,113 and more particles: one lane a
# target
@pytest.mark.parametrize("counts,box", [((9, 9, 9), (1.2, 1.2, 1.2)),
                                        ((46, 46, 46), (3.0, 3.0, 3.0))])
def test_members_of_fast_particles_match_scatter(pbf_mod, counts, box):
    p = P.reference_defaults()
    sc = scenes.block(counts, box, seed=3, vel_sigma=0.5)
    rng = np.random.default_rng(4)
    k = rng.choice(sc.n, sc.n // 6, replace=False)
    sc.vel[k] = rng.uniform(-12.0, 12.0, (k.size, 3)) * p.h / p.dt
    print(f"members n {sc.n}", flush=True)
    g = [gpu_grad(pbf_mod, sc, p, 1, _target(sc), adjoint=a) for a in ("scatter", "gather")]
    assert np.isfinite(g[1][0]).all() and np.isfinite(g[1][1]).all()
    # the same terms in another order: a few hundred float additions a component
    assert rel(g[1][0], g[0][0]) < 2e-5 and rel(g[1][1], g[0][1]) < 2e-5
