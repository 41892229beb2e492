"""GPU: the neighbour passes with four lanes per particle (launches of few
slots) against those with one: a small scene alone and the same scene in a
batch beside a large one, every bit of the state, at counts around the edges
of a quad's wave and workgroup and for lists of every kind."""
import numpy as np
import pytest

from libfluid_amd import _lib as L
from libfluid_amd import configs

pytestmark = pytest.mark.gpu

FILLER = 120_000  # particles of the other scene: past every four-lane limit


def scene(kind, n):
    if kind == "block":
        cfg = configs.block_scene(n, (1.6, 1.7, 1.8), (0.3, -1.0, 0.2), seed=n)
    elif kind == "spray":       # near-isolated particles
        cfg = configs.spray_only(n, seed=n)
    else:                       # cloud of n particles a cell: long rows and lists
        cfg = configs.cloud(float(n), 0.1, seed=n)
    return cfg


@pytest.mark.parametrize("full", [False, True])
@pytest.mark.parametrize("kind,n,speed", [("block", 1, 0.1), ("block", 2, 0.1), ("block", 15, 0.1), ("block", 17, 0.1),
                                          ("block", 63, 0.1), ("block", 65, 0.1), ("block", 513, 0.1),
                                          ("block", 4097, 0.1), ("spray", 20_011, 0.1), ("cloud", 8, 2.0),
                                          ("cloud", 30, 0.1), ("cloud", 45, 2.0), ("cloud", 140, 0.1)])
def test_four_lanes_equal_one(gpu, kind, n, speed, full):
    cfg = scene(kind, n)
    if full:
        cfg.params.viscosity, cfg.params.surface_tension, cfg.params.adhesion = 0.2, 1.0, 0.1
    vel = np.random.Generator(np.random.PCG64(n)).normal(0, speed, cfg.pos.shape).astype(np.float32)
    dt, steps = (1e-3 if speed > 1 else 1e-4), 4
    with gpu.Scene(cfg.params, cfg.n) as sc:
        sc.upload(cfg.pos, vel)
        sc.step(dt * steps, steps)
        got = sc.download(L.LF_ORDER_CELL)
    big = configs.block_scene(FILLER, (1.2, 1.2, 1.2), (0.0, -1.0, 0.0), seed=5)
    with gpu.Batch(cfg.n + FILLER + 1024, cfg.params.ncells + big.params.ncells + 2, 2) as b:
        b.upload(b.add(big.params, big.n, 1e-4), big.pos)
        i = b.add(cfg.params, cfg.n, float(np.float32(np.float32(dt * steps) / np.float32(steps))))
        b.upload(i, cfg.pos, vel)
        b.step(steps)
        want = b.download(i, L.LF_ORDER_CELL)
    for k in want:
        assert np.array_equal(got[k], want[k]), k
