"""GPU: the neighbour kernels with one lane per particle.  Block sizes and walk
modes that are set are taken at every size, so small scenes reach these kernels
with every one of them: rows of every length and far moves against the full
scan of every stencil slot, bit for bit, and every force term against the
oracle."""
import ctypes as C
import types

import numpy as np
import pytest

from libfluid_amd import _lib as L
from libfluid_amd import configs
from tests.test_gpu_parity import compare_substep, gpu_substep, oracle_substep

pytestmark = pytest.mark.gpu

DEFAULT = ((256, 256, 256, 256), (1, 1, 2))
# (block sizes, walk modes): every size with every mode
SHAPES = [((b,) * 4, (w,) * 3) for b in (128, 256, 512) for w in (0, 1, 2)]


def lanes(h, batch=False):
    k = C.c_int(0)
    fn = L.lib.lf_batch_debug_lanes if batch else L.lib.lf_debug_lanes
    L.check(fn(h._h, C.byref(k)), "lanes")
    return k.value


@pytest.mark.parametrize("batch", [False, True])
def test_shapes_that_are_set_are_taken(gpu, batch):
    cfg = configs.cloud(30.0, 0.1, seed=4)  # long rows, every term: four lanes take half the time of one
    cfg.params.viscosity, cfg.params.surface_tension = 0.2, 1.0
    h = gpu.Batch(cfg.n + 512, cfg.params.ncells + 1, 1) if batch else gpu.Scene(cfg.params, cfg.n)
    with h:
        if batch:
            h.upload(h.add(cfg.params, cfg.n, cfg.dt), cfg.pos)
        else:
            h.upload(cfg.pos)
        assert lanes(h, batch) == 4
        for sizes, walks in SHAPES + [((256, 128, 256, 256), DEFAULT[1]), (DEFAULT[0], (1, 1, 1))]:
            h.set_tuning(sizes)
            h.set_walks(walks)
            assert lanes(h, batch) == 1
        h.set_tuning(DEFAULT[0])
        h.set_walks(DEFAULT[1])
        assert lanes(h, batch) == 4
        h.step(1) if batch else h.step(cfg.dt, 1)
        assert np.all(h.autotune(5) > 0)
        assert lanes(h, batch) == 4


def stepped(gpu, cfg, vel, dt, shape, scan=False):
    p = L.LfParams.from_buffer_copy(cfg.params)
    p.viscosity, p.surface_tension, p.adhesion = 0.2, 1.0, 0.1
    with gpu.Scene(p, cfg.n) as sc:
        sc.upload(cfg.pos, vel)
        sc.set_debug(forces=True, scan=scan, normals_pass=True)
        sc.set_tuning(shape[0])
        sc.set_walks(shape[1])
        assert lanes(sc) == (4 if shape == DEFAULT else 1)
        sc.step(3 * dt, 3)
        out = sc.download(L.LF_ORDER_ID)
        out["normal"] = sc.field(L.FIELD_NORMAL)
        out["forces"] = sc.field(L.FIELD_FORCES)
        return out


# (particles per cell, speed): rows below and above one mask word, above two
# and three words, of more words than a walk's table has entries; slow and far moves
@pytest.mark.parametrize("ppc,speed", [(6, 0.2), (18, 0.2), (30, 0.2), (70, 0.2), (190, 0.2), (6, 2.0), (30, 2.0),
                                       (70, 2.0)])
def test_walks_equal_the_full_scan(gpu, ppc, speed):
    cfg = configs.cloud(float(ppc), 0.1, seed=5 + ppc)
    vel = np.random.Generator(np.random.PCG64(ppc)).normal(0, speed, cfg.pos.shape).astype(np.float32)
    dt = 1e-3 if speed > 1 else 1e-5
    want = stepped(gpu, cfg, vel, dt, SHAPES[3], scan=True)
    for shape in SHAPES + [DEFAULT]:
        got = stepped(gpu, cfg, vel, dt, shape)
        for k in want:
            assert np.array_equal(got[k], want[k]), (shape, k)


@pytest.mark.parametrize("walks", [0, 1, 2])
@pytest.mark.parametrize("case", ["double_dam", "dense"])
def test_every_term_against_the_oracle(gpu, oracle_omp, case, walks):
    cfg = configs.double_dam(4096, 16) if case == "double_dam" else configs.dense_block(16, 15, 14)
    cfg.params.viscosity, cfg.params.surface_tension, cfg.params.adhesion = 0.2, 1.0, 0.1

    def scene(params, n):
        sc = gpu.Scene(params, n)
        sc.set_walks((walks,) * 3)
        assert lanes(sc) == 1
        return sc

    vel = np.random.Generator(np.random.PCG64(3)).normal(0, 0.1, cfg.pos.shape).astype(np.float32)
    acc = np.zeros_like(vel)
    g = gpu_substep(types.SimpleNamespace(Scene=scene), cfg, cfg.pos, vel, acc)
    o = oracle_substep(oracle_omp, cfg, cfg.pos, vel, acc)
    compare_substep(g, o, float(np.float32(cfg.params.particle_size)), f"{case} walks {walks}", orc=oracle_omp,
                    cfg=cfg, state=(cfg.pos, vel, acc))
