"""GPU tests of the team kernels (a team of lanes per target, the neighbour
passes of small steps) against the lane kernels, which a fixed heavy threshold
selects at every size: the same bits after every frame of a step, at sizes
around the workgroups and around the sizes where the team width changes, with
piles of several hundred coincident and near-coincident particles, empty
columns and a batch; gradients within the spread of a reordered FP32 sum.
"""
import numpy as np
import pytest
import torch

from pbf import params as P
from pbf import scenes
from test_gpu_adjoint import _scene, _target, gpu_grad, rel
from test_gpu_batched import BatchRun, _small_batch
from test_gpu_parity import Run

pytestmark = pytest.mark.gpu

KEYS = ("pos", "vel", "npos", "nvel", "iid")


def _piled(n, seed=31):
    """The first n sites of a moving lattice; a tenth of them, up to 700, pile
    up in one corner (half of these at one point)."""
    full = scenes.block((46, 45, 44), (5.0, 3.0, 4.0), seed=seed, vel_sigma=0.6)
    pos, vel = full.pos[:n].copy(), full.vel[:n].copy()
    k = min(n // 10, 700)
    pos[:k] = 0.03 * (pos[:k] / 5.0)
    pos[: k // 2] = 0.01
    vel[:k] = 0.0
    return scenes.Scene(pos, vel, full.iid[:n].copy(), full.ulim, full.llim)


def _same(a, b, what):
    for k in KEYS:
        assert np.array_equal(a[k].view(np.uint32), b[k].view(np.uint32)), f"{what}: {k}"


@pytest.mark.parametrize("layout", [4, 3])
@pytest.mark.parametrize("n", [1, 15, 17, 33, 1000, 20480, 20481, 90112, 90113])
def test_team_steps_equal_lane_steps(pbf_mod, device, n, layout):
    p = P.dam_params().replace(k_boundaryDensity=0.5)
    sc = _piled(n)
    print(f"team n={n} layout={layout}", flush=True)
    team, lane = Run(pbf_mod, sc, p, layout), Run(pbf_mod, sc, p, layout)
    lane.sim.set_heavy_threshold(256)
    for frame in range(3):
        _same(team.step(), lane.step(), f"n {n} frame {frame}")


def test_team_batch_equals_lane_batch(pbf_mod, device):
    p = P.dam_params()
    team, lane = (BatchRun(pbf_mod, _small_batch(), p, 4) for _ in range(2))
    lane.sim.set_heavy_threshold(64)
    for frame in range(3):
        _same(team.step(), lane.step(), f"frame {frame}")


def test_team_density_error_equals_lane(pbf_mod, device):
    sc = _piled(3000)
    r = Run(pbf_mod, sc, P.dam_params())
    a = r.sim.density_error(r.a[0], sc.n)
    r.sim.set_heavy_threshold(64)
    assert r.sim.density_error(r.a[0], sc.n) == a


@pytest.mark.parametrize("adjoint", ["scatter", "gather"])
def test_team_gradients_match_lane_gradients(pbf_mod, device, adjoint, monkeypatch):
    """The adjoint's terms are added in another order (whole terms instead of
    their parts): FP32 sums of ~33 terms differ by ~33 * 2^-24 = 2e-6 of their
    terms per pass; nine passes of two frames stay within 1e-4."""
    p = P.reference_defaults()
    sc = _scene((12, 9, 11), (1.0, 1.0, 1.0))
    tgt = _target(sc)
    a = gpu_grad(pbf_mod, sc, p, 2, tgt, adjoint=adjoint)
    make = pbf_mod.Simulator

    def fixed(*args, **kw):
        sim = make(*args, **kw)
        sim.set_heavy_threshold(256)
        return sim

    monkeypatch.setattr(pbf_mod, "Simulator", fixed)
    b = gpu_grad(pbf_mod, sc, p, 2, tgt, adjoint=adjoint)
    np.testing.assert_array_equal(a[3], b[3])
    assert rel(a[0], b[0]) < 1e-4 and rel(a[1], b[1]) < 1e-4
    assert abs(a[2] - b[2]) <= 1e-4 * abs(b[2])


def test_sizes_mix_on_one_solver(pbf_mod, device):
    """One solver steps a large count (lane kernels), a small one (team) and the
    large one again: the lane kernels' work lists are clean each time."""
    p = P.dam_params()
    big, small = _piled(90113), _piled(5000)
    r = Run(pbf_mod, big, p)
    ref = [Run(pbf_mod, big, p).step(), Run(pbf_mod, small, p).step()]
    for k, sc in enumerate((big, small, big, small)):
        pos, vel = sc.as_layout(4)
        for t, a in ((r.a[0], pos), (r.a[1], vel)):
            t[: a.size].copy_(torch.from_numpy(a.ravel()))
        r.iid[: sc.n].copy_(torch.from_numpy(sc.iid.astype(np.int32)))
        r.n = sc.n
        r.sim.step(r.a[0], r.b[0], r.a[1], r.b[1], r.iid, sc.n)
        _same(r.state(), ref[k % 2], f"step {k}")
