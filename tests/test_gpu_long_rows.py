"""GPU: stencil rows of more than 64 slots (mask words kept up to slot 95,
tested again from there on, walked in batches of table entries) and far-moving
scenes (every word tested on the integrated positions), against the full scan
of every stencil slot (LF_DEBUG_SCAN): every bit of the state and of the
normals and force components is the same."""
import numpy as np
import pytest

from libfluid_amd import _lib as L
from libfluid_amd import configs

pytestmark = pytest.mark.gpu


def stepped(gpu, cfg, vel, dt, full, scan):
    p = L.LfParams.from_buffer_copy(cfg.params)
    if full:
        p.viscosity, p.surface_tension, p.adhesion = 0.2, 1.0, 0.1
    with gpu.Scene(p, cfg.n) as sc:
        sc.upload(cfg.pos, vel)
        sc.set_debug(forces=True, scan=scan, normals_pass=True)
        sc.step(3 * dt, 3)
        out = sc.download(L.LF_ORDER_ID)
        out["normal"] = sc.field(L.FIELD_NORMAL)
        out["forces"] = sc.field(L.FIELD_FORCES)
        start = sc.field(L.FIELD_START).astype(np.int64)
        return out, start


def longest_row(cfg, start):
    gx, gy, gz = (int(g) for g in cfg.params.grid)
    count = np.diff(start)[: gx * gy * gz].reshape(-1, gx)
    pad = np.pad(count, ((0, 0), (1, 1)))
    return int((pad[:, :-2] + pad[:, 1:-1] + pad[:, 2:]).max())


# (particles per cell, longest row at least, at most): rows ending below, at
# and above the edges at 64 and 96 slots, rows of several tested words, and
# rows of more words than the walk's table has entries (512 slots)
@pytest.mark.parametrize("ppc,lo,hi", [(21, 65, 96), (30, 97, 160), (70, 200, 300), (190, 513, 800)])
@pytest.mark.parametrize("full", [False, True])
def test_long_rows_equal_the_full_scan(gpu, ppc, lo, hi, full):
    cfg = configs.cloud(float(ppc), 0.1, seed=17 + ppc)
    vel = np.random.Generator(np.random.PCG64(ppc)).normal(0, 0.2, cfg.pos.shape).astype(np.float32)
    want, start = stepped(gpu, cfg, vel, 1e-5, full, True)
    got, _ = stepped(gpu, cfg, vel, 1e-5, full, False)
    rows = longest_row(cfg, start)
    assert lo <= rows <= hi, rows
    for k in want:
        assert np.array_equal(got[k], want[k]), k


@pytest.mark.parametrize("ppc,scene", [(6, "short rows"), (30, "long rows")])
def test_far_moves_equal_the_full_scan(gpu, ppc, scene):
    cfg = configs.cloud(float(ppc), 0.1, seed=3 + ppc)
    vel = np.random.Generator(np.random.PCG64(ppc)).normal(0, 2.0, cfg.pos.shape).astype(np.float32)
    want, _ = stepped(gpu, cfg, vel, 1e-3, True, True)   # moves of up to a quarter of h
    got, _ = stepped(gpu, cfg, vel, 1e-3, True, False)
    for k in want:
        assert np.array_equal(got[k], want[k]), k
