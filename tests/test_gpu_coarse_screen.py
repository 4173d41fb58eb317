"""GPU test of the passes that screen on 16-bit coordinates modulo 16 h (the
steps of more than 2^19 particles) against the oracle's FP32 mirror, bit for
bit: boxes many periods wide, with negative and with large coordinates (where
neighbouring floats are half a percent of h apart), particles outside the box,
on its walls, in piles and exactly h apart.
"""
import numpy as np
import pytest

from pbf import params as P
from pbf import scenes
from test_gpu_parity import Run, assert_bitexact, mirror

pytestmark = pytest.mark.gpu

N = (1 << 19) + 77


@pytest.mark.parametrize("shift,layout", [((-7.3, -2.55, -11.0), 4), ((4096.0, -4096.0, 0.0), 3)])
def test_coarse_screened_step_bitexact(pbf_mod, orc, device, shift, layout):
    p = P.dam_params(niter=2)
    sc = scenes.block((82, 80, 80), (9.0, 4.5, 4.5), seed=17, vel_sigma=1.0)
    x, v = sc.pos[:N].astype(np.float64), sc.vel[:N].copy()
    rng = np.random.default_rng(5)
    x[:400] = rng.uniform(-3.0, 12.0, (400, 3))  # in and outside the box
    x[400:1000] = [0.05, 0.05, 0.05]  # a pile
    x[1000:1400:2] = x[1001:1400:2] + [0.1, 0.0, 0.0]  # pairs h apart
    x[1400:1500, 0] = 0.0
    x = (x + np.array(shift)).astype(np.float32)
    ul = tuple(float(np.float32(a + b)) for a, b in zip((9.0, 4.5, 4.5), shift))
    ll = tuple(float(np.float32(s)) for s in shift)
    sc = scenes.Scene(x, v, np.arange(N, dtype=np.uint32), ul, ll)
    pos, vel = sc.as_layout(layout)
    print(f"coarse screen shift {shift}", flush=True)
    assert_bitexact(Run(pbf_mod, sc, p, layout).step(), mirror(orc, p, sc, pos, vel, sc.iid),
                    f"shift {shift}")
