"""GPU test of the counted grid's ranks in piles: cells of a few loads of entries,
up to a few thousand, in input order and in random order, against the oracle's
FP32 mirror and its stable order.
"""
import numpy as np
import pytest

from pbf import params as P
from pbf import scenes
from test_gpu_parity import Run, assert_bitexact, mirror

pytestmark = pytest.mark.gpu


# 64 entries a load, four loads in flight
@pytest.mark.parametrize("order", ["input", "random", "interleaved"])
@pytest.mark.parametrize("sizes", [(255, 256, 257), (319, 320, 321, 513), (4001, 777)])
def test_pile_ranks_bitexact(pbf_mod, orc, device, sizes, order):
    p = P.reference_defaults().replace(niter=1)
    rng = np.random.default_rng(21)
    parts = [rng.uniform(0.0, 2.0, (3000, 3))]
    parts += [np.array([0.3 * k, 0.0, 0.0]) + rng.uniform(0.02, 0.08, (m, 3))
              for k, m in enumerate(sizes)]
    x = np.concatenate(parts).astype(np.float32)
    if order == "random":
        x = x[rng.permutation(len(x))]
    elif order == "interleaved":  # every second particle from the other end
        x[1::2] = x[1::2][::-1].copy()
    sc = scenes.Scene(x, np.zeros_like(x), np.arange(len(x), dtype=np.uint32), (2.0, 2.0, 2.0),
                      (0.0, 0.0, 0.0))
    print(f"pile ranks {sizes} {order}", flush=True)
    run = Run(pbf_mod, sc, p)
    pos, vel = sc.as_layout(4)
    assert_bitexact(run.step(), mirror(orc, p, sc, pos, vel, sc.iid), f"{sizes} {order}")
