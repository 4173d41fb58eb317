"""GPU test of backward passes run in a row on a stored tape, without a step of
the solver in between, where targets are on the work lists: every pass gives the
gradients of the first.
"""
import numpy as np
import pytest
import torch

from conftest import from_dev, to_dev
from pbf import params as P
from pbf import scenes
from test_gpu_adjoint import rel

pytestmark = pytest.mark.gpu


# one and three frames: an odd number of neighbour passes; the small scene with
# every target on the lists, the large one with a pile
@pytest.mark.parametrize("adjoint", ["gather", "scatter"])
@pytest.mark.parametrize("counts,frames,threshold", [((12, 12, 12), 1, 64), ((12, 12, 12), 3, 64),
                                                     ((46, 44, 46), 1, 0)])
def test_backward_repeats(pbf_mod, device, counts, frames, threshold, adjoint):
    p = P.reference_defaults()
    sc = scenes.block(counts, tuple(0.07 * c for c in counts), seed=5, vel_sigma=0.5)
    rng = np.random.default_rng(8)
    if threshold == 0:
        sc.pos[:1500] = rng.uniform(0.12, 0.18, (1500, 3)).astype(np.float32)
    n = sc.n
    print(f"backward repeats n {n} frames {frames} {adjoint}", flush=True)
    sim = pbf_mod.Simulator(p, sc.ulim, sc.llim, capacity=n)
    sim.set_heavy_threshold(threshold)
    tape = pbf_mod.Tape(sim, n, frames, store=True, adjoint=adjoint)
    pos, vel = sc.as_layout(4)
    tape.forward(to_dev(pos, device), to_dev(vel, device), to_dev(sc.iid, device))
    g = to_dev(rng.normal(0.0, 1.0, (n, 4)).astype(np.float32), device)
    first = None
    for rep in range(4):
        out = [torch.zeros(n * 4, device=device) for _ in range(2)]
        grho = tape.backward(g, g, out[0], out[1])
        got = [from_dev(x) for x in out]
        assert all(np.isfinite(x).all() for x in got) and np.isfinite(grho)
        if first is None:
            first = got, grho
            continue
        for a, b in zip(got, first[0]):
            if adjoint == "gather":
                np.testing.assert_array_equal(a, b)
            else:  # atomics add in any order: a few float roundings a component
                assert rel(a, b) < 1e-4
        if adjoint == "gather":
            assert grho == first[1]
