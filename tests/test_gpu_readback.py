"""Results on their way to the host: one staged copy, many pieces over
several workers, last pieces that are not full, bands of fewer than eight rows
and bands wider than a staging slot. Whole values, compared bit for bit."""

import numpy as np
import pytest

import cenote_amd as cn
from cenote_amd import workloads

pytestmark = pytest.mark.gpu


def by_pixel(sample, width, height):
    """A sample as the film folds it: its values lie in band order (8-row
    bands top to bottom, each walked column by column)."""
    y, x = np.divmod(np.arange(width * height), width)
    rows = np.minimum(8, height - y // 8 * 8)
    index = y // 8 * (width * 8) + x * rows + y % 8
    return sample.reshape(width * height, -1)[index].reshape(sample.shape)


@pytest.mark.parametrize("width,height", [(1, 1), (37, 29), (512, 128), (513, 129), (701, 503), (1280, 721)])
def test_sums_and_averages_arrive_whole(ctx, width, height):
    print(f"film {width}x{height}", flush=True)
    rng = np.random.default_rng(width * 10007 + height)
    films = [rng.standard_normal((height, width, 4)).astype(np.float32) for _ in range(3)]
    depth = rng.uniform(0.0, 100.0, (height, width)).astype(np.float32)
    film = cn.Film(ctx, width, height)
    r = cn.Renderer(ctx)
    want = [np.zeros_like(a) for a in (*films, depth)]
    for k in range(3):
        sample = [np.roll(a, k, axis=0) for a in (*films, depth)]
        film.set_sample(*sample)
        r.accumulate_sample(film)
        sample = [by_pixel(a, width, height) for a in sample]
        want = [w + a if k else a for a, w in zip(sample, want)]
    for got, w in zip(film.sums(), want):
        assert np.array_equal(got, w)
    for result in (film.averages(), r.resolve(film)):
        for got, w in zip(result, want):
            assert np.array_equal(got, w / np.float32(3.0))
    r.close()
    film.close()


@pytest.mark.parametrize("width,height", [(1, 1), (5, 9), (64, 64), (333, 217), (1000, 700), (9001, 11)])
def test_traced_images_arrive_row_major(ctx, width, height):
    print(f"trace {width}x{height}", flush=True)
    scene = cn.Scene(ctx, workloads.cornell())
    r = cn.Renderer(ctx, max_bounces=2)
    film = cn.Film(ctx, width, height)
    r.accumulate(scene, film)  # sample 0, folded on the device by pixel
    for got, want in zip(r.trace(scene, width, height, 0, aov=True), film.sums()):
        assert np.array_equal(got, want)
    assert np.array_equal(r.trace(scene, width, height, 0), film.sums()[0])
    film.close()
    r.close()
    scene.close()
