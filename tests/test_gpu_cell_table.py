"""GPU: the cell table and the (cell key, id) order at the edges of the scan's
tiles and of its one-launch range, and a crowded bucket whose segment sort
takes three passes over many tiles, against the oracle bit for bit; two
substeps, so that the counts cleared by the first are used by the second."""
import numpy as np
import pytest

from libfluid_amd import _lib as L
from libfluid_amd import configs

pytestmark = pytest.mark.gpu


def check(gpu, oracle, p, pos, dt):
    with gpu.Scene(p, len(pos)) as sc:
        sc.upload(pos)
        for _ in range(2):
            before = sc.download(L.LF_ORDER_ID)["pos"]
            order0 = sc.download(L.LF_ORDER_CELL)["ids"]  # the state's order: keys are reported in it
            sc.step(dt, 1)
            okeys, _ = oracle.hash(p, before)
            assert np.array_equal(sc.field(L.FIELD_KEYS), okeys[order0])
            assert np.array_equal(sc.field(L.FIELD_START), oracle.cell_start(p, okeys))
            assert np.array_equal(sc.field(L.FIELD_SORTED_IDS), oracle.sort(okeys))


# grid cells: with the out-of-grid bucket one below, at and above one tile
# (4,096), the most tiles scanned in one launch (16) and beyond it
@pytest.mark.parametrize("grid", [(1, 1, 1), (1, 63, 65), (15, 13, 21), (16, 16, 16), (1, 1, 12287), (3, 53, 412),
                                  (5, 107, 121), (1, 65535, 1), (4, 128, 128), (97, 101, 103)])
def test_cell_table_at_tile_edges(gpu, oracle, grid):
    p = configs.scaled_c1(2, 2, 2).params
    for a in range(3):
        p.grid[a] = grid[a]
        p.box[a] = np.float32(grid[a] / np.float64(p.inv_cell[a]) * (1 - 1e-6))
    rng = np.random.Generator(np.random.PCG64(sum(grid)))
    box = np.array([p.box[a] for a in range(3)], np.float64)
    pos = (rng.uniform(0.01, 0.99, (1500, 3)) * box).astype(np.float32)
    check(gpu, oracle, p, pos, 1e-6)


@pytest.mark.parametrize("crowd", [1023, 1025, 70_000])
def test_crowded_buckets(gpu, oracle, crowd):
    cfg = configs.scaled_c1(10, 10, 10)
    rng = np.random.Generator(np.random.PCG64(crowd))
    h = float(np.float32(cfg.params.h))
    outside = rng.uniform(0.05, 0.4, (crowd, 3))
    outside[:, 0] = -rng.uniform(0.001, 0.05, crowd)
    inside = (np.array([30, 5, 5]) + rng.uniform(0.05, 0.95, (900, 3))) * h
    pos = np.concatenate([cfg.pos, outside, inside]).astype(np.float32)
    pos = pos[rng.permutation(len(pos))]
    check(gpu, oracle, cfg.params, pos, 1e-6)
