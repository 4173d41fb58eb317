"""GPU test of the radix path's ranking at the edges of its tiles (2048 pairs,
a quarter a wavefront): steps of more than 2^19 particles whose last tile ends
in the first, a middle and the last quarter, with runs of equal cells longer
than a tile, bit for bit against the oracle's FP32 mirror (whose sort is
stable: the identities' order shows every misplaced pair)."""
import numpy as np
import pytest

from pbf import params as P
from pbf import scenes
from test_gpu_parity import Run, assert_bitexact, mirror

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rest", [1, 1087, 2048])
def test_last_tile_of_the_radix_sort(pbf_mod, orc, device, rest):
    n = (1 << 19) + rest
    p = P.dam_params(niter=1)
    sc = scenes.block((82, 80, 81), (9.0, 4.5, 4.5), seed=29, vel_sigma=1.0)
    x, v = sc.pos[:n].copy(), sc.vel[:n].copy()
    k = np.random.default_rng(rest).permutation(n)
    x, v = x[k], v[k]  # input order unrelated to the cells
    x[:2600] = np.float32([4.05, 2.05, 1.05])  # one cell, more than a tile
    v[:2600] = 0.0
    sc = scenes.Scene(x, v, np.arange(n, dtype=np.uint32), sc.ulim, sc.llim)
    pos, vel = sc.as_layout(4)
    print(f"radix tiles n {n}", flush=True)
    assert_bitexact(Run(pbf_mod, sc, p, 4).step(), mirror(orc, p, sc, pos, vel, sc.iid), f"{rest}")
