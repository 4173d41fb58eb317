"""GPU test of the gather-mode adjoint on large sets (query grids by counting up
to 2^20 particles and by the radix sort beyond, the XSPH pass on screening
coordinates) against the scatter mode, which has neither: fast particles whose
candidate relations are one-sided, and a compressed region whose targets go to
the work lists.
"""
import numpy as np
import pytest

from pbf import params as P
from pbf import scenes
from test_gpu_adjoint import _target, gpu_grad, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,layout", [((1 << 19) + 77, 4), (1 << 20, 3), ((1 << 20) + 1, 4)])
def test_large_gather_gradients_match_scatter(pbf_mod, n, layout):
    p = P.reference_defaults().replace(niter=2)
    full = scenes.block((102, 102, 102), (6.0, 5.6, 5.2), seed=31, vel_sigma=0.5)
    x, v = full.pos[:n].copy(), full.vel[:n].copy()
    assert len(x) == n
    mid = np.array([1.2, 2.5, 2.5])
    near = np.abs(x - mid).max(1) < 0.6
    x[near] = (mid + 0.7 * (x[near] - mid)).astype(np.float32)  # ~600 candidates a target
    rng = np.random.default_rng(4)
    k = rng.choice(n, n // 50, replace=False)
    v[k] = rng.uniform(-3.0, 3.0, (k.size, 3)) * p.h / p.dt
    sc = scenes.Scene(x, v, np.arange(n, dtype=np.uint32), full.ulim, full.llim)
    print(f"large gather n {n} layout {layout}", flush=True)
    g = [gpu_grad(pbf_mod, sc, p, 1, _target(sc), layout=layout, adjoint=a)
         for a in ("scatter", "gather")]
    assert np.isfinite(g[1][0]).all() and np.isfinite(g[1][1]).all()
    # the same terms in another order: a few hundred float additions a component
    assert rel(g[1][0], g[0][0]) < 2e-5 and rel(g[1][1], g[0][1]) < 2e-5
    assert g[1][2] == pytest.approx(g[0][2], rel=2e-5)
