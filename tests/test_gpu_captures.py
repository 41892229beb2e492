"""GPU: when substeps are captured into graphs: only what is needed a second time
with the same parameters, launch shapes and active scenes."""
import ctypes as C

import numpy as np
import pytest

from libfluid_amd import _lib as L
from libfluid_amd import configs
from libfluid_amd.serve import Server

pytestmark = pytest.mark.gpu


def captures():
    k = C.c_int64(0)
    L.check(L.lib.lf_debug_captures(C.byref(k)), "lf_debug_captures")
    return k.value


def test_nothing_is_captured_before_its_second_use(gpu):
    """A scene whose parameters change before every call captures no graph;
    one that does not captures each run and single substep once, when it is
    needed again."""
    cfg = configs.scaled_c1(12, 10, 8)
    with gpu.Scene(cfg.params, cfg.n) as sc:
        sc.upload(cfg.pos)
        at = captures()
        p = L.LfParams.from_buffer_copy(cfg.params)
        for k in (10, 8, 1, 15, 7):
            p.gravity[0] += 0.25
            sc.set_params(p)
            sc.step(1e-4 * k, k)
            assert captures() == at, k
        sc.step(1e-4 * 8, 8)   # after 7 single ones: the other pairing's first run
        assert captures() == at
        sc.step(1e-4 * 24, 24)
        assert captures() == at + 1
        sc.step(1e-4 * 2, 2)   # singles of both pairings, for the second call
        assert captures() == at + 3
        for k in (2, 8, 10):
            sc.step(1e-4 * k, k)
        assert captures() == at + 3
    with gpu.Scene(cfg.params, cfg.n) as sc:
        sc.upload(cfg.pos)
        sc.step(1e-4 * 16, 16)
        assert captures() == at + 4


def test_paused_and_resumed_scenes_capture_nothing(gpu):
    scenes = [configs.block_scene(n, (1.6, 1.7, 1.8), (0.1, -1.0, 0.3), seed=n) for n in (700, 1500)]
    with gpu.Batch(2 * 4096, sum(c.params.ncells + 1 for c in scenes), 2) as b:
        ids = [b.add(c.params, c.n, 1e-4) for c in scenes]
        for i, c in zip(ids, scenes):
            b.upload(i, c.pos)
        at = captures()
        for k in range(6):
            b.set_active(ids[1], k % 2 == 0)
            b.step(9)
        assert captures() == at


@pytest.mark.parametrize("run_ahead,graphs,want", [(0, True, 2), (0, False, 0), (2, True, 0), (2, False, 0)])
def test_server_ticks_replay_graphs_where_they_wait(gpu, run_ahead, graphs, want):
    cfg = configs.scaled_c1(12, 10, 8)
    with Server(2048, cfg.params.ncells + 1, 2) as srv:
        srv.configure(run_ahead, graphs)
        at = captures()
        job = srv.submit(cfg.params, cfg.pos, None, cfg.dt, 9)
        while not srv.tick():
            pass
        assert captures() == at + want
        got = srv.result(job)
    with gpu.Scene(cfg.params, cfg.n) as sc:
        sc.upload(cfg.pos)
        sc.run(cfg.dt, 9)
        ref = sc.download(L.LF_ORDER_ID)
    for k in ("pos", "vel", "acc"):
        assert np.array_equal(got[k], ref[k]), k
