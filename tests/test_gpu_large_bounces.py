"""The tail launch, the launch shapes and fractional opacity on views whose
bounces hold more rays than the stages hand over early (TAIL_PATHS, 16384), so
that the stages run up to the bounce that each test names. Every test counts
the rays of those bounces first."""

from __future__ import annotations

import numpy as np
import pytest

import cenote_amd as cn
from cenote_amd import _abi, workloads
from oracle import oracle as orc

from reference_scenes import translucent_scene

pytestmark = pytest.mark.gpu

TAIL_PATHS = 16384  # cn_stages.hip


@pytest.fixture(scope="module")
def scenes(ctx):
    made = {"cornell": workloads.cornell(), "chart": workloads.chart(), "translucent": translucent_scene()}
    out = {name: (data, cn.Scene(ctx, data)) for name, data in made.items()}
    yield out
    for _, scene in out.values():
        scene.close()


def film(ctx, scene, view, depth, counting=False, shape=None, capacity=0, mode=cn.LightSampling.MIS, graphs=True):
    """The sums of a wave of `view` (width, height, samples) twice over, the
    second folded into the first, and with `counting` the rays by bounce."""
    r = cn.Renderer(ctx, capacity=capacity, max_bounces=depth, light_sampling=mode)
    r.shape = shape or {}
    r.set_graphs(graphs)
    r.set_counters(counting)
    f = cn.Film(ctx, *view[:2])
    for _ in range(2):
        r.accumulate(scene, f, count=view[2])
    rays = r.wave_counts()["rays"] if counting else None
    sums = f.sums()
    f.close()
    r.close()
    return sums, rays


def assert_same(got, want, label):
    for k, (g, w) in enumerate(zip(got, want)):
        assert np.array_equal(g, w, equal_nan=True), (label, k, int(np.sum(g != w)))


def assert_large(rays, last, label, ranges=1):
    """Bounces 1..last of a wave stay with the stages in each of `ranges`
    pool ranges of like content (twice the threshold, where there are several)."""
    print(label, "rays", rays[: last + 1].tolist(), flush=True)
    assert rays[1: last + 1].min() > TAIL_PATHS * (1 if ranges == 1 else 2 * ranges), label


@pytest.mark.parametrize("bvh_width", [4, 8])
@pytest.mark.parametrize("name,view,depth,tails", [
    ("cornell", (256, 256, 8), 8, (1, 2, 3, 5)),
    ("chart", (640, 360, 6), 12, (1, 2, 3)),
    ("translucent", (320, 240, 6), 9, (1, 2, 3)),
])
def test_the_tail_starts_at_its_own_bounce(ctx, scenes, name, view, depth, tails, bvh_width):
    _, scene = scenes[name]
    _, rays = film(ctx, scene, view, depth, counting=True)
    assert_large(rays, max(tails), name)
    want, _ = film(ctx, scene, view, depth, shape={"tail_bounce": 0})
    for tail in tails:
        print(f"{name} tail {tail} width {bvh_width}", flush=True)
        got, _ = film(ctx, scene, view, depth, shape={"tail_bounce": tail, "bvh_width": bvh_width})
        assert_same(got, want, (name, tail))


@pytest.mark.parametrize("mode", [cn.LightSampling.BSDF_ONLY, cn.LightSampling.NEE_ONLY])
def test_the_tail_keeps_every_light_sampling_mode(ctx, scenes, mode):
    _, scene = scenes["cornell"]
    view = (256, 256, 3)
    _, rays = film(ctx, scene, view, 8, counting=True, mode=mode)
    assert_large(rays, 3, f"mode {int(mode)}")
    want, _ = film(ctx, scene, view, 8, shape={"tail_bounce": 0}, mode=mode)
    got, _ = film(ctx, scene, view, 8, shape={"tail_bounce": 3}, mode=mode, graphs=False)
    assert_same(got, want, mode)


def test_the_tail_over_several_pool_ranges(ctx, scenes):
    _, scene = scenes["cornell"]
    view = (384, 512, 2)
    capacity = view[0] * view[1] // 3  # a wave of one sample walks three ranges of pixels
    _, rays = film(ctx, scene, view, 8, counting=True, capacity=capacity)
    assert rays[0] == 3 * capacity
    assert_large(rays, 2, "three ranges", ranges=3)
    want, _ = film(ctx, scene, view, 8, shape={"tail_bounce": 0})
    for tail in (1, 2):
        print("ranges, tail", tail, flush=True)
        got, _ = film(ctx, scene, view, 8, shape={"tail_bounce": tail}, capacity=capacity)
        assert_same(got, want, tail)


@pytest.mark.parametrize("variant", [_abi.SHADE_1024_LDS, _abi.SHADE_512_LDS, _abi.SHADE_256_LDS,
                                     _abi.SHADE_256_GLOBAL, _abi.SHADE_512_LDS_SORTED,
                                     _abi.SHADE_256_LDS_SORTED, _abi.SHADE_256_GLOBAL_SORTED])
@pytest.mark.parametrize("blocks", [(7, 3, 5), (2048, 512, 1024)])
def test_launch_shapes_over_large_bounces(ctx, scenes, variant, blocks):
    _, scene = scenes["cornell"]
    view = (256, 256, 8)
    _, rays = film(ctx, scene, view, 8, counting=True)
    assert_large(rays, 5, "shapes")
    want, _ = film(ctx, scene, view, 8)
    print(f"variant {variant} blocks {blocks}", flush=True)
    got, _ = film(ctx, scene, view, 8, shape={"trace_blocks": blocks[0], "shade_variant": variant,
                                              "shade_blocks": blocks[1], "light_blocks": blocks[2]})
    assert_same(got, want, (variant, blocks))


def test_fractional_opacity_over_large_bounces_matches_the_oracle(ctx, scenes):
    data, scene = scenes["translucent"]
    width, height = 480, 360
    r = cn.Renderer(ctx, max_bounces=8)
    r.set_counters(True)
    r.trace(scene, width, height, 0)
    assert_large(r.wave_counts()["rays"], 2, "opacity")
    r.set_counters(False)
    ref = orc.OracleScene(data)
    for sample in range(2):
        print(f"opacity sample {sample}", flush=True)
        img = r.trace(scene, width, height, sample)
        want = ref.trace(width, height, sample)
        # the other parity tests' bound: paths differ by their transcendentals' last bits
        close = np.isclose(img, want, rtol=1e-4, atol=1e-6).all(axis=-1)
        assert close.mean() >= 0.99, (sample, close.mean())
    r.close()
