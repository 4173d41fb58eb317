"""GPU test of rescaling tapes with padded (float4) seeds: what stands in the
padding changes neither the scale nor a bit of the gradients.
"""
import numpy as np
import pytest
import torch

from conftest import from_dev, to_dev
from pbf import params as P
from pbf import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pad", [1e30, -3e38, np.inf, np.nan])
def test_padding_does_not_choose_the_scale(pbf_mod, device, pad):
    p = P.reference_defaults()
    sc = scenes.block((8, 8, 8), (1.0, 1.0, 1.0), seed=5, vel_sigma=0.5)
    n = sc.n
    print(f"rescale padding {pad}", flush=True)
    sim = pbf_mod.Simulator(p, sc.ulim, sc.llim, capacity=n)
    tape = pbf_mod.Tape(sim, n, 1, adjoint="gather", rescale=True)
    pos, vel = sc.as_layout(4)
    tape.forward(to_dev(pos, device), to_dev(vel, device), to_dev(sc.iid, device))
    seed = np.random.default_rng(2).normal(0.0, 1.0, (n, 4)).astype(np.float32)
    got = []
    for w in (0.0, pad):
        seed[:, 3] = w
        out = [torch.zeros(n * 4, device=device) for _ in range(2)]
        grho = tape.backward(to_dev(seed, device), to_dev(seed, device), out[0], out[1])
        got.append([tape.gradient_log2_scale(), grho] + [from_dev(t) for t in out])
    assert got[0][:2] == got[1][:2]
    for a, b in zip(got[0][2:], got[1][2:]):
        assert np.isfinite(a).all()
        np.testing.assert_array_equal(a, b)
