"""GPU test of a tape used with another solver than the one it was made for: what
fits gives the same gradients, what does not is refused before anything is
written.
"""
import numpy as np
import pytest
import torch

from conftest import from_dev, to_dev
from pbf import params as P
from pbf import scenes

pytestmark = pytest.mark.gpu

CAPACITY, STATE = 2, 5


def _state(sc, device):
    pos, vel = sc.as_layout(4)
    return to_dev(pos, device), to_dev(vel, device), to_dev(sc.iid, device)


def _sim(pbf_mod, p, ulim, n, cells):
    return pbf_mod.Simulator(p, ulim, (0.0, 0.0, 0.0), capacity=n, max_cells=cells)


@pytest.mark.parametrize("store", [True, False])
def test_tape_checks_the_solver_it_is_used_with(pbf_mod, device, store):
    p = P.reference_defaults()
    sc = scenes.block((8, 8, 8), (1.0, 1.0, 1.0), seed=3, vel_sigma=0.5)
    n = sc.n
    x, v, i = _state(sc, device)
    g = to_dev(np.random.default_rng(1).normal(0.0, 1.0, (n, 4)).astype(np.float32), device)
    own = _sim(pbf_mod, p, sc.ulim, n, 1000)
    tape = pbf_mod.Tape(own, n, 2, store=store, adjoint="gather")
    print(f"tape with other solvers, store {store}", flush=True)

    def backward():
        out = [torch.zeros(n * 4, device=device) for _ in range(2)]
        tape.backward(g, None, out[0], out[1])
        return [from_dev(t) for t in out]

    tape.forward(x, v, i)
    want = backward()
    # room for more particles and cells, the box the tape was made for
    tape.sim = _sim(pbf_mod, p, sc.ulim, 2 * n, 8000)
    tape.forward(x, v, i)
    for a, b in zip(backward(), want):
        np.testing.assert_array_equal(a, b)
    # a box of more cells than the stored tables hold
    tape.sim = _sim(pbf_mod, p, (2.0, 2.0, 2.0), n, 8000)
    if store:
        with pytest.raises(pbf_mod.PBFError) as e:
            tape.forward(x, v, i)
        assert e.value.code == CAPACITY
        with pytest.raises(pbf_mod.PBFError) as e:
            backward()
        assert e.value.code == STATE
    else:
        tape.forward(x, v, i)
        backward()
    # fewer particles than the tape's
    tape.sim = own
    tape.forward(x, v, i)
    tape.sim = _sim(pbf_mod, p, sc.ulim, n - 1, 1000)
    for call in (backward, lambda: tape.forward(x, v, i)):
        with pytest.raises(pbf_mod.PBFError) as e:
            call()
        assert e.value.code == CAPACITY
    # a batch of scenes
    tape.sim = pbf_mod.BatchedSimulator(p, [sc.ulim], [(0.0, 0.0, 0.0)], [n])
    with pytest.raises(pbf_mod.PBFError) as e:
        backward()
    assert e.value.code == STATE
    tape.sim = own
    tape.forward(x, v, i)
    for a, b in zip(backward(), want):
        np.testing.assert_array_equal(a, b)
