"""GPU test of a tape that steps its checkpoints and stored frames in place and
reads the seeds where they are: inputs and seeds stay untouched, every
checkpoint is the state before its frame, also when steps are replayed from
recorded graphs, the gradients do not depend on the seeds' padding.
"""
import numpy as np
import pytest
import torch

from conftest import from_dev, to_dev
from pbf import params as P
from pbf import scenes
from test_gpu_parity import Run

pytestmark = pytest.mark.gpu

FRAMES = 3


@pytest.mark.parametrize("store,graph,rescale", [(False, False, False), (False, True, False),
                                                 (True, False, False), (True, False, True)])
def test_tape_leaves_inputs_and_seeds(pbf_mod, device, store, graph, rescale):
    p = P.dam_params()
    sc = scenes.block((8, 8, 8), (1.0, 1.0, 1.0), seed=5, vel_sigma=0.5)
    print(f"tape arrays store {store} graph {graph} rescale {rescale}", flush=True)
    run = Run(pbf_mod, sc, p, 4)
    steps = [run.step() for _ in range(FRAMES)]
    sim = pbf_mod.Simulator(p, sc.ulim, sc.llim, capacity=sc.n)
    sim.set_graph(graph)
    tape = pbf_mod.Tape(sim, sc.n, FRAMES, store=store, rescale=rescale)
    stream = torch.cuda.Stream()
    pos, vel = sc.as_layout(4)
    with torch.cuda.stream(stream):
        dp, dv, di = to_dev(pos, device), to_dev(vel, device), to_dev(sc.iid, device)
        rng = np.random.default_rng(2)
        seed = rng.normal(0.0, 1.0, (sc.n, 4)).astype(np.float32)
        grads = []
        for rep in range(2):  # the second time over recorded graphs
            tape.forward(dp, dv, di)
            np.testing.assert_array_equal(from_dev(dp).reshape(-1, 4), pos.reshape(-1, 4))
            np.testing.assert_array_equal(from_dev(dv).reshape(-1, 4), vel.reshape(-1, 4))
            np.testing.assert_array_equal(from_dev(di).astype(np.uint32), sc.iid)
            for f in range(FRAMES + 1):
                a = [torch.zeros(sc.n * 4, device=device) for _ in range(2)]
                i = torch.zeros(sc.n, dtype=torch.int32, device=device)
                tape.read(f, a[0], a[1], i)
                want = (pos, vel, sc.iid) if f == 0 else tuple(
                    steps[f - 1][k] for k in ("npos", "nvel", "iid"))
                np.testing.assert_array_equal(from_dev(a[0]).reshape(-1, 4)[:, :3],
                                              want[0].reshape(-1, 4)[:, :3])
                np.testing.assert_array_equal(from_dev(a[1]).reshape(-1, 4)[:, :3],
                                              want[1].reshape(-1, 4)[:, :3])
                np.testing.assert_array_equal(from_dev(i).astype(np.uint32), want[2])
            if rescale:
                seed[:, 3] = 0.0
            else:
                seed[:, 3] = np.nan if rep else 0.0
            g = [to_dev(seed, device), to_dev(seed[::-1].copy(), device)]
            before = [from_dev(x).copy() for x in g]
            out = [torch.zeros(sc.n * 4, device=device) for _ in range(2)]
            tape.backward(g[0], g[1], out[0], out[1])
            for x, b in zip(g, before):
                np.testing.assert_array_equal(from_dev(x), b)
            grads.append([from_dev(x).reshape(-1, 4)[:, :3].copy() for x in out])
        for a, b in zip(*grads):
            assert np.isfinite(a).all()
            # scatter mode's atomics add in any order: a few float roundings of
            # sums of up to a few hundred terms, through FRAMES frames
            assert np.linalg.norm(a - b) <= 1e-4 * np.linalg.norm(a)
