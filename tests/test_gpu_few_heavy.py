"""GPU test of the adaptive heavy threshold where few targets may be heavy
though they are more than 1 in 25 (a crowded quarter of a small scene): steps
with it equal steps with the threshold fixed at its largest, bit for bit."""
import numpy as np
import pytest

from pbf import params as P
from pbf import scenes
from test_gpu_parity import Run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("counts,crowd", [((46, 44, 46), 20000), ((46, 44, 46), 33000),
                                          ((64, 64, 64), 32000)])
def test_few_heavy_targets_change_no_bit(pbf_mod, device, counts, crowd):
    p = P.dam_params(niter=2)
    sc = scenes.block(counts, tuple(0.07 * c for c in counts), seed=31, vel_sigma=0.5)
    rng = np.random.default_rng(crowd)
    k = rng.choice(sc.n, crowd, replace=False)
    side = (crowd / 2600.0) ** (1.0 / 3.0)  # about 70 candidates each
    sc.pos[k] = rng.uniform(0.1, 0.1 + side, (crowd, 3)).astype(np.float32)
    print(f"few heavy n {sc.n} crowd {crowd}", flush=True)
    adaptive, fixed = Run(pbf_mod, sc, p, 4), Run(pbf_mod, sc, p, 4)
    fixed.sim.set_heavy_threshold(256)
    for _ in range(2):
        a, b = adaptive.step(), fixed.step()
        for key in ("npos", "nvel", "iid"):
            np.testing.assert_array_equal(a[key], b[key])
