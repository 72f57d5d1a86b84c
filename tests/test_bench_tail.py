"""bench.py's byte model and launch counts where the tail launch starts ahead
of its own bounce: a wave's small bounces are the tail's, not the stages'."""

import sys
from pathlib import Path
from types import SimpleNamespace

import numpy as np

sys.path.insert(0, str(Path(__file__).resolve().parents[1]))
import bench  # noqa: E402

INFO = SimpleNamespace(bvh_node_bytes=64, bvh_triangle_bytes=48)


def wave(rays):
    rays = np.array(rays, np.int64)
    counts = {"rays": rays, "hits": rays // 2, "misses": rays - rays // 2, "shadows": rays // 4}
    return counts, np.stack([rays * 10, rays * 3, rays * 5, rays], axis=1)


def bytes_of(waves, tail, ranges=1):
    out, totals = bench.algorithmic_bytes(waves, INFO, 1000, True, 4, tail, 0, ranges)
    return {k: v for k, v in out.items()}, totals


def test_the_tail_starts_at_the_first_small_bounce():
    assert bench.tail_start([10**6, 50000, 16385, 16384, 9000, 100, 5], 6) == 3
    assert bench.tail_start([10**6, 50000, 30000, 20000, 18000, 17000, 16900], 5) == 5
    assert bench.tail_start([4096, 4000, 3000, 10], 3) == 1
    assert bench.tail_start([4096, 4000, 3000, 10], 0) == 4  # no tail
    assert bench.tail_start([4096, 4000, 3000, 10], 6) == 4  # too few bounces for one
    assert bench.tail_start([200000, 30000, 20000, 10], 3, ranges=2) == 1


def test_bytes_follow_the_hand_over_wave_by_wave():
    large, small = wave([500000, 400000, 300000, 200000, 100000]), wave([5000, 4000, 3000, 2000, 1000])
    # Each wave alone against a tail set to the bounce where it starts.
    for w, starts in ((large, 3), (small, 1)):
        want, _ = bytes_of([w], starts)
        got, totals = bytes_of([w], 3)
        assert got == want
        assert totals["rays"] == int(w[0]["rays"].sum())
    both, totals = bytes_of([large, small], 3)
    alone = [bytes_of([w], 3)[0] for w in (large, small)]
    for k in ("shade_surface", "shade_miss", "tail"):
        assert both[k] == sum(a[k] for a in alone)
    assert both["trace"] == sum(a["trace"] for a in alone) - 1000 * 72  # the frame's camera paths, once
    # The stages and the tail share out the same work wherever the tail starts.
    work = {k: bytes_of([large, small], t)[0] for k, t in (("none", 0), ("tail", 3))}
    parts = ("trace", "shade_surface", "shade_miss", "tail")
    assert sum(work["none"].get(k, 0) for k in parts) == sum(work["tail"].get(k, 0) for k in parts)


def test_small_ranges_launch_the_tail_after_bounce_1():
    whole = bench.timed_launches("cornell", 2, 1 << 22, 6)
    assert whole["trace"] == whole["raygen"] * 7
    # 16 waves of a sample each a frame, of 8 ranges each
    small = bench.timed_launches("cornell", 2, 8192, 6)
    assert small == {"raygen": 256, "trace": 512, "shade_miss": 0, "shade_surface": 256, "accumulate": 32,
                     "tail": 256}
