"""GPU test of the adjoint where a particle's adjoint has overflowed and another
particle lies just beyond h of it, inside the padded screening radius: there is
no term between the two, so the other's gradient stays exactly its own.
"""
import numpy as np
import pytest
import torch

from conftest import from_dev, to_dev
from pbf import params as P
from pbf import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("threshold", [0, 256])  # a team of lanes, one lane a target
@pytest.mark.parametrize("adjoint", ["scatter", "gather"])
def test_overflowed_adjoint_stays_within_h(pbf_mod, device, adjoint, threshold):
    p = P.reference_defaults().replace(g=0.0, niter=1)
    x = np.array([[0.95, 1.0, 1.0], [1.0, 1.0, 1.0], [1.100002, 1.0, 1.0]], np.float32)
    r2 = np.float32(x[2, 0] - x[1, 0]) ** 2
    h2 = np.float32(p.h) * np.float32(p.h)
    assert h2 <= r2 < h2 * np.float32(1.0001)
    sc = scenes.Scene(x, np.zeros_like(x), np.arange(3, dtype=np.uint32), (2.0, 2.0, 2.0),
                      (0.0, 0.0, 0.0))
    print(f"overflowed adjoint {adjoint} threshold {threshold}", flush=True)
    sim = pbf_mod.Simulator(p, sc.ulim, sc.llim, capacity=3)
    sim.set_heavy_threshold(threshold)
    tape = pbf_mod.Tape(sim, 3, 1, adjoint=adjoint)
    pos, vel = sc.as_layout(4)
    tape.forward(to_dev(pos, device), to_dev(vel, device), to_dev(sc.iid, device))
    xf = torch.zeros(12, device=device)
    iid = torch.zeros(3, dtype=torch.int32, device=device)
    tape.read(1, pos=xf, iid=iid)
    order = from_dev(iid)
    seed = np.zeros((3, 4), np.float32)
    seed[order == 1, 0] = 3e38  # the particle in the middle
    seed[order == 2, :3] = [1.0, -2.0, 0.5]  # the one beyond h of it
    out = [torch.zeros(12, device=device) for _ in range(2)]
    tape.backward(to_dev(seed, device), None, out[0], out[1])
    gx, gv = (from_dev(t).reshape(3, 4)[:, :3] for t in out)
    assert not np.isfinite(gx[1]).all()  # the overflow did reach its adjoint
    # x1 = x0 + dt v with no neighbour inside h
    np.testing.assert_array_equal(gx[2], np.float32([1.0, -2.0, 0.5]))
    np.testing.assert_array_equal(gv[2], np.float32(p.dt) * np.float32([1.0, -2.0, 0.5]))
