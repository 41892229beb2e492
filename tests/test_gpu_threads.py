"""GPU: one scene used by several threads.  Downloads share the pool's scratch
arrays and pinned staging, so each must find them free: concurrent downloads in
either order, small (one staging buffer) and large (several), and downloads
beside a thread that steps, each of which must see the whole state of one
step."""
import threading

import numpy as np
import pytest

from libfluid_amd import _lib as L
from libfluid_amd import configs

pytestmark = pytest.mark.gpu

STATE = ("pos", "vel", "acc", "colour", "ids")


def run(*bodies):
    errors = []

    def guarded(body):
        try:
            body()
        except BaseException as e:  # reported by the test's own thread
            errors.append(e)

    threads = [threading.Thread(target=guarded, args=(b,)) for b in bodies]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    if errors:
        raise errors[0]


@pytest.mark.parametrize("n", [3001, 90_007])  # 156 KB and 4.7 MB a download
def test_concurrent_downloads(gpu, n):
    cfg = configs.block_scene(n, (1.6, 1.7, 1.8), (0.3, -1.0, 0.2), seed=n)
    vel = np.random.Generator(np.random.PCG64(n)).normal(0, 0.2, cfg.pos.shape).astype(np.float32)
    with gpu.Scene(cfg.params, cfg.n) as sc:
        sc.upload(cfg.pos, vel)
        sc.step(4e-4, 4)
        want = {o: sc.download(o) for o in (L.LF_ORDER_CELL, L.LF_ORDER_ID)}

        def body(order):
            for _ in range(40):
                got = sc.download(order)
                for k in STATE:
                    assert np.array_equal(got[k], want[order][k]), k

        run(*[lambda o=o: body(o) for o in (L.LF_ORDER_CELL, L.LF_ORDER_ID) * 2])


@pytest.mark.parametrize("n", [3001, 90_007])
def test_downloads_beside_steps(gpu, n):
    cfg = configs.block_scene(n, (1.6, 1.7, 1.8), (0.3, -1.0, 0.2), seed=n)
    vel = np.random.Generator(np.random.PCG64(n)).normal(0, 0.2, cfg.pos.shape).astype(np.float32)
    calls = (1, 8, 3, 9, 1, 16, 2, 8)
    with gpu.Scene(cfg.params, cfg.n) as sc:  # the state after each call
        sc.upload(cfg.pos, vel)
        seen = [sc.download()]
        for k in calls:
            sc.step(1e-4 * k, k)
            seen.append(sc.download())
    with gpu.Scene(cfg.params, cfg.n) as sc:
        sc.upload(cfg.pos, vel)
        done = threading.Event()

        def stepping():
            try:
                for k in calls:
                    sc.step(1e-4 * k, k)
                    done.wait(2e-3)
            finally:
                done.set()

        def reading():
            while not done.is_set():
                got = sc.download()
                at = [k for k, s in enumerate(seen) if np.array_equal(got["pos"], s["pos"])]
                assert at, "positions of no step"
                for k in STATE:
                    assert any(np.array_equal(got[k], seen[a][k]) for a in at), k

        run(stepping, reading)
        got = sc.download()
        for k in STATE:
            assert np.array_equal(got[k], seen[-1][k]), k


def test_steps_of_two_threads_keep_their_lengths(gpu):
    """A lone particle stepped by two threads with different step lengths falls
    for the sum of them: each call's length belongs to its own substeps."""
    p = configs.scaled_c1(2, 2, 2).params
    k, d1, d2 = 300, 1e-4, 3e-4
    with gpu.Scene(p, 1) as sc:
        sc.upload(np.array([[0.5, 0.45, 0.25]], np.float32))

        def body(dt):
            for _ in range(k):
                sc.step(dt, 1)

        run(lambda: body(d1), lambda: body(d2))
        v = sc.download()["vel"][0]
    # one step's half is integrated with the acceleration before it (zero at first)
    assert abs(float(v[1]) + 9.8 * k * (d1 + d2)) <= 0.5 * 9.8 * d2 + 1e-4
    assert v[0] == 0.0 and v[2] == 0.0
