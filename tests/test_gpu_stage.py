"""The planes' way in and out of a world: the same bits back, below and above the sizes from which several host threads
copy through pinned chunks (8 MiB down, 24 MiB up: 14 planes are 8.26 MB at 384^2, 24.7 at 664^2 and 25.3 at 672^2), at
sizes that end inside a chunk, and from several threads at once, each with its own world."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [(8, 8), (384, 384), (392, 392), (1024, 200), (664, 664), (672, 672), (1304, 728)]


def planes(w, h, seed):
    p = np.random.default_rng(seed).uniform(0.5, 1.5, (14, h, w)).astype(np.float32)
    p[4:] /= p[4:].sum(axis=0)
    return p


def round_trip(w, h, seeds, bad):
    import sandbox_reactions_amd as sr
    world = sr.World(w, h, gravity=False, hydro=True, heat=False)
    for seed in seeds:
        p = planes(w, h, seed)
        q = p.copy()
        world.upload(q)
        q[:] = -1.0  # the caller's array is its own again once upload returns
        if not np.array_equal(world.readback().view(np.uint32), p.view(np.uint32)):
            bad.append((w, h, seed))
    world.close()


@pytest.mark.parametrize("w,h", SIZES)
def test_planes_come_back_bit_for_bit(gpu_lib, w, h):
    print(f"transfer {w}x{h}", flush=True)
    bad = []
    round_trip(w, h, (1, 2, 3), bad)
    assert not bad


def test_worlds_transfer_from_several_threads(gpu_lib):
    print("transfers from four threads", flush=True)
    bad = []
    ts = [threading.Thread(target=round_trip, args=(w, h, (k, k + 10), bad)) for k, (w, h) in enumerate(SIZES[1:])]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
