"""GPU tests of the counted grid build (cells numbered with atomics, ranked by
input index) against the oracle's FP32 mirror and its stable order: cells on
both sides of the size where a whole wavefront ranks them, piles whose
particles are scattered over the input, every grid size class of the scan, and
the largest counts that build their grid this way, with one more.
"""
import numpy as np
import pytest

from pbf import params as P
from pbf import scenes
from test_gpu_parity import Run, assert_bitexact, mirror

pytestmark = pytest.mark.gpu


def _cells(sizes, box, seed=11, extra=500):
    """Cells of the given particle counts along the floor, the particles of all
    of them (and of a sparse rest) in random input order."""
    rng = np.random.default_rng(seed)
    parts = [rng.uniform(0.0, 1.0, (extra, 3)) * np.array(box)]
    for k, m in enumerate(sizes):
        parts.append(np.array([0.3 * k, 0.0, 0.0]) + rng.uniform(0.02, 0.08, (m, 3)))
    x = np.concatenate(parts).astype(np.float32)
    x = x[rng.permutation(len(x))]
    return scenes.Scene(x, np.zeros_like(x), np.arange(len(x), dtype=np.uint32), box,
                        (0.0, 0.0, 0.0))


@pytest.mark.parametrize("layout", [4, 3])
@pytest.mark.parametrize("box", [(3.2, 1.0, 1.0), (6.4, 3.2, 1.6), (6.4, 6.4, 6.4),
                                 (12.0, 10.0, 40.0)])
def test_ranked_cells_bitexact(pbf_mod, orc, device, box, layout):
    """Grids of 3,200 to 4.8M cells: one, several and more than 2,048 scan tiles."""
    p = P.reference_defaults()
    sc = _cells([1, 7, 8, 9, 63, 64, 65, 128, 129, 700], box)
    print(f"counted grid box {box} layout {layout}", flush=True)
    run = Run(pbf_mod, sc, p, layout)
    pos, vel = sc.as_layout(layout)
    state = (pos, vel, sc.iid)
    for frame in range(2):
        g = run.step()
        m = mirror(orc, p, sc, *state)
        assert_bitexact(g, m, f"box {box} frame {frame}")
        state = (m["npos"], m["nvel"], m["iid"])


@pytest.mark.parametrize("n", [(1 << 19), (1 << 19) + 1])
def test_largest_counted_steps_bitexact(pbf_mod, orc, device, n):
    full = scenes.block((81, 81, 80), (9.0, 4.5, 4.5), seed=5, vel_sigma=2.0)
    assert full.n > n
    order = np.random.default_rng(3).permutation(full.n)[:n]
    sc = scenes.Scene(full.pos[order], full.vel[order], np.arange(n, dtype=np.uint32), full.ulim,
                      full.llim)
    p = P.reference_defaults().replace(niter=1)
    pos, vel = sc.as_layout(4)
    assert_bitexact(Run(pbf_mod, sc, p).step(), mirror(orc, p, sc, pos, vel, sc.iid), f"n={n}")
