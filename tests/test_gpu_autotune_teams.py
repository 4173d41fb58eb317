"""GPU test of the autotuner where a step uses no launch shape (a team of lanes
per target, up to 90,112 particles): the shapes in force stay, also such as are
no candidates; one particle more, or a fixed heavy threshold, chooses again.
"""
import pytest

from pbf import params as P
from pbf import scenes
from test_gpu_parity import Run

pytestmark = pytest.mark.gpu

CANDIDATES = [(b, g) for b in (64, 128, 256) for g in (512, 1024, 2048, 4096)]
OWN = (128, 700)


@pytest.mark.parametrize("n,threshold,kept", [(1000, 0, True), (90112, 0, True),
                                              (90113, 0, False), (90112, 256, False)])
def test_shapes_stay_where_no_kernel_has_them(pbf_mod, device, n, threshold, kept):
    full = scenes.block((46, 45, 46), (5.0, 5.0, 5.0), seed=7, vel_sigma=0.3)
    sc = scenes.Scene(full.pos[:n], full.vel[:n], full.iid[:n], full.ulim, full.llim)
    assert sc.n == n
    print(f"autotune n {n} threshold {threshold}", flush=True)
    run = Run(pbf_mod, sc, P.reference_defaults())
    run.sim.set_heavy_threshold(threshold)
    run.sim.set_shapes(*OWN)
    best, ms = run.sim.autotune(run.a[0], run.a[1], run.iid, n, reps=1)
    assert ms > 0
    assert run.sim.get_shapes() == best
    assert best == OWN if kept else best in CANDIDATES
