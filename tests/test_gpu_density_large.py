"""GPU test of the density statistic on large sets against the oracle's FP32
mirror: the counted grid with screening coordinates (from 2^19 particles to
2^21) and the radix sort (beyond), with piles, crowded and empty regions,
particles in the last cell, on the walls and outside the box, boxes many
screening periods from the origin, in input and in random order.
"""
import numpy as np
import pytest

from conftest import to_dev
from pbf import params as P
from pbf import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,layout,shift,shuffle", [
    ((1 << 19) + 77, 4, (-7.3, -2.55, -11.0), True),
    ((1 << 19) + 77, 3, (4096.0, -4096.0, 0.0), False),
    (1 << 21, 4, (0.0, 0.0, 0.0), False),
    (1 << 21, 3, (-7.3, -2.55, -11.0), True),
    ((1 << 21) + 1, 3, (0.0, 0.0, 0.0), True),
    ((1 << 21) + 1, 4, (4096.0, -4096.0, 0.0), False)])
def test_density_error_matches_oracle(pbf_mod, orc, device, n, layout, shift, shuffle):
    p = P.dam_params().replace(k_boundaryDensity=0.5)
    box = (8.0, 7.0, 7.0)
    x = scenes.block((129, 128, 128), box, seed=23).pos[:n].astype(np.float64)
    assert len(x) == n
    rng = np.random.default_rng(9)
    k = rng.permutation(n)[:7000]  # taken from all over the block
    x[k[:600]] = [0.05, 0.05, 0.05]
    x[k[600:3600]] = rng.uniform(0.31, 0.39, (3000, 3))
    x[k[3600:4600]] = rng.uniform(-0.5, 8.5, (1000, 3))
    x[k[4600:5600]] = np.array(box) - rng.uniform(0.0, 0.25, (1000, 3))  # the last cells
    x[k[5600:6000], 2] = 0.0
    x[k[6000:7000:2]] = x[k[6001:7000:2]] + [0.1, 0.0, 0.0]  # pairs h apart
    if shuffle:
        x = x[rng.permutation(n)]
    x = (x + np.array(shift)).astype(np.float32)
    ul = tuple(float(np.float32(a + b)) for a, b in zip(box, shift))
    ll = tuple(float(np.float32(s)) for s in shift)
    pos = np.zeros((n, layout), np.float32)
    pos[:, :3] = x
    print(f"density error n {n} layout {layout} shift {shift}", flush=True)
    sim = pbf_mod.Simulator(p, ul, ll, capacity=n, layout=layout)
    dev = to_dev(pos, device)
    mean_o, max_o, _ = orc.density_error_f32(p, ul, ll, x)
    for _ in range(2):  # the second call finds the counts the first one cleared
        mean_g, max_g = sim.density_error(dev, n)
        assert mean_g == pytest.approx(mean_o, rel=1e-12)
        assert max_g == pytest.approx(max_o, rel=1e-15)
