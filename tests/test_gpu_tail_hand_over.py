"""Small bounces handed to the tail launch ahead of its own bounce.

A bounce from 1 on with at most 16384 rays is left by the stages to the tail
launch. Views around that many paths must render bit for bit the film of the
stages alone, and count the same rays, hits, misses and connections up to the
tail's own bounce.
"""

from __future__ import annotations

import numpy as np
import pytest

import cenote_amd as cn
from cenote_amd import workloads

pytestmark = pytest.mark.gpu

TAIL_BOUNCE = 6


@pytest.fixture(scope="module", params=["cornell", "chart"])
def scene(ctx, request):
    s = cn.Scene(ctx, workloads.build(request.param))
    yield s
    s.close()


def wave(ctx, scene, size, tail, counting=False, bvh_width=4):
    r = cn.Renderer(ctx, max_bounces=9)
    r.shape = {"tail_bounce": tail, "bvh_width": bvh_width}
    r.set_counters(counting)
    film = cn.Film(ctx, *size)
    sums = None
    for _ in range(3):  # eager, captured, replayed
        film.reset()
        r.accumulate(scene, film, count=1)
        sums = film.sums()
    counts = r.wave_counts()
    film.close()
    r.close()
    return sums, counts


@pytest.mark.parametrize("bvh_width", [4, 8])
@pytest.mark.parametrize("size", [(1, 1), (7, 9), (128, 127), (128, 128), (129, 127), (160, 128), (321, 200)])
def test_handed_over_bounces_render_and_count_the_same(ctx, scene, size, bvh_width):
    print(f"hand over: {size} width {bvh_width}", flush=True)
    want, _ = wave(ctx, scene, size, 0, bvh_width=bvh_width)
    got, counts = wave(ctx, scene, size, TAIL_BOUNCE, bvh_width=bvh_width)
    for k, (g, w) in enumerate(zip(got, want)):
        assert np.array_equal(g, w, equal_nan=True), k
    _, whole = wave(ctx, scene, size, TAIL_BOUNCE, counting=True, bvh_width=bvh_width)
    for key, last in (("rays", TAIL_BOUNCE), ("hits", TAIL_BOUNCE), ("misses", TAIL_BOUNCE),
                      ("shadows", TAIL_BOUNCE - 1)):
        assert np.array_equal(counts[key][: last + 1], whole[key][: last + 1]), key
