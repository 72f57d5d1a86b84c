"""What a scene keeps on the device is what its renders read: the records of
its trees, triangles and tables. The full-precision nodes that cn_scene_bvh
hands out are made when it is called, the same each time."""

from __future__ import annotations

import ctypes as C
import dataclasses

import numpy as np
import pytest

import cenote_amd as cn
from cenote_amd import _abi
from cenote_amd.scene import Material, MeshData, SceneData, identity

pytestmark = pytest.mark.gpu

COUNT = 1_000_000


def soup():
    rng = np.random.default_rng(5)
    p = rng.uniform(-1, 1, (COUNT, 1, 3)) + rng.normal(scale=1e-3, size=(COUNT, 3, 3))
    data = SceneData()
    mesh = data.add_mesh(MeshData(np.ascontiguousarray(p.reshape(-1, 3), np.float32),
                                  np.tile(np.array([0.0, 0.0, 1.0], np.float32), (3 * COUNT, 1)),
                                  np.arange(3 * COUNT, dtype=np.uint32).reshape(-1, 3)))
    data.add_instance(mesh, identity(), Material.matte((0.5, 0.5, 0.5)))
    data.env_texels = np.ones((1, 1, 4), np.float32)
    return data


def free_bytes():
    free, total = C.c_size_t(), C.c_size_t()
    assert _abi.library().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("builder", [_abi.BVH_DEVICE, _abi.BVH_HOST])
def test_a_scene_holds_the_records_its_renders_read(ctx, builder):
    print(f"builder {builder}", flush=True)
    data = soup()
    cn.Scene(ctx, data, bvh_builder=builder).close()  # the runtime's own first allocations
    before = free_bytes()
    scene = cn.Scene(ctx, data, bvh_builder=builder)
    held = before - free_bytes()
    info = scene.info()
    nodes = info.bvh_node_count
    assert nodes * 128 > 40 << 20  # the full-precision nodes would show
    # 64- and 128-byte nodes of the per-ray and packet walks, 128-byte 8-wide
    # ones, 48- and 80-byte triangles; 24 MiB for the small arrays and the
    # allocator's rounding.
    records = nodes * (64 + 128) + info.bvh8_node_count * 128 + COUNT * (48 + 80)
    print(f"held {held} of {records} bytes of records", flush=True)
    assert held <= records + (24 << 20)
    first, tris = scene.bvh()
    assert free_bytes() >= before - held - (8 << 20)  # nothing stays behind
    edited = dataclasses.replace(data)
    edited.instances = [dataclasses.replace(i, material=Material.matte((0.1, 0.2, 0.3))) for i in data.instances]
    scene.update(edited, _abi.DIRTY_MATERIALS)
    again, tris_again = scene.bvh()
    assert np.array_equal(first, again) and np.array_equal(tris, tris_again)
    scene.close()
