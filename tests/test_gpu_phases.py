"""GPU test of the phase timing: every phase of a step records its intervals,
whichever way the step orders its particles (counted up to 2^19, radix sort
beyond); the velocity update is part of the last delta-p launch.
"""
import pytest

from pbf import params as P
from pbf import scenes
from test_gpu_parity import Run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("counts", [(16, 16, 16), (81, 81, 80)])
def test_every_phase_is_recorded(pbf_mod, device, counts):
    p = P.reference_defaults().replace(niter=2)
    sc = scenes.block(counts, tuple(0.055 * c for c in counts), seed=4, vel_sigma=0.2)
    print(f"phases n {sc.n}", flush=True)
    run = Run(pbf_mod, sc, p)
    run.sim.set_timing(True)
    for _ in range(3):
        run.step()
    t = run.sim.get_timing()
    want = dict(predict=3, sort=3, grid=3, lam=6, delta=6, velocity=0, xsph=3, step=3)
    want["lambda"] = want.pop("lam")
    assert {k: c for k, (_, c) in t.items()} == want
    assert all(ms > 0.0 for k, (ms, c) in t.items() if c)
    assert sum(ms for k, (ms, _) in t.items() if k != "step") <= t["step"][0] * 1.001
