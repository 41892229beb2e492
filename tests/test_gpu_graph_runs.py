"""GPU: substeps replayed in runs of captured ones against kernels launched one
by one, bit for bit: calls of fewer, as many and more substeps than a run,
starting from either pairing of the state buffers, repeated with downloads,
parameter changes and a paused scene between the replays."""
import numpy as np
import pytest

from libfluid_amd import _lib as L
from libfluid_amd import configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("counts", [(8, 8, 8), (1, 8, 9, 7), (17, 1, 16, 3), (24, 5, 24)])
def test_runs_equal_single_launches(gpu, counts):
    cfg = configs.scaled_c1(16, 12, 14)
    vel = np.random.Generator(np.random.PCG64(sum(counts))).normal(0, 0.2, cfg.pos.shape).astype(np.float32)
    outs = []
    for graphs in (False, True):
        got = []
        with gpu.Scene(cfg.params, cfg.n) as sc:
            sc.set_graphs(graphs)
            sc.upload(cfg.pos, vel)
            for r, k in enumerate(counts):
                if r == 2:
                    p = L.LfParams.from_buffer_copy(cfg.params)
                    p.viscosity, p.surface_tension = 0.2, 1.0
                    sc.set_params(p)
                sc.step(1e-4 * k, k)
                got.append(sc.download(L.LF_ORDER_CELL))
            assert sc.step_count() == sum(counts)
        outs.append(got)
    for a, b in zip(*outs):
        for k in a:
            assert np.array_equal(a[k], b[k]), k


def test_runs_with_a_paused_scene(gpu):
    scenes = [configs.block_scene(n, (1.6, 1.7, 1.8), (0.1, -1.0, 0.3), seed=n) for n in (700, 1500, 2300)]
    outs = []
    for graphs in (False, True):
        with gpu.Batch(3 * 4096, sum(c.params.ncells + 1 for c in scenes), 3) as b:
            b.set_graphs(graphs)
            ids = [b.add(c.params, c.n, 1e-4) for c in scenes]
            for i, c in zip(ids, scenes):
                b.upload(i, c.pos)
            b.step(9)
            b.set_active(ids[1], False)
            b.step(16)
            b.step(3)
            b.set_active(ids[1], True)
            b.step(8)
            outs.append([b.download(i) for i in ids])
    for a, b in zip(*outs):
        for k in a:
            assert np.array_equal(a[k], b[k]), k
