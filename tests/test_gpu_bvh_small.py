"""The device builder against the host builder, at the edges of its steps.

Ranges of at most 64 triangles are built by one wave, a triangle a lane;
larger ones come to it through a workgroup's splits. Both builders must grow
the same nodes and leaf order, bit for bit.
"""

from __future__ import annotations

import numpy as np
import pytest

import cenote_amd as cn
from cenote_amd import _abi
from cenote_amd.scene import Material, MeshData, SceneData, identity

pytestmark = pytest.mark.gpu


def corners(kind: str, count: int) -> np.ndarray:
    rng = np.random.default_rng(count)
    if kind == "soup":
        return rng.uniform(-1, 1, (count, 1, 3)) + rng.normal(scale=0.05, size=(count, 3, 3))
    if kind == "coincident":  # no axis has an extent: ranges split at their middle
        return np.tile(np.array([[[0, 0, 0], [1, 0, 0], [0, 1, 0]]], np.float64), (count, 1, 1))
    # Powers of two along one axis: splits of one triangle against the rest.
    base = np.array([[0, 0, 0], [0, 1, 0], [0, 0, 1]], np.float64)
    return base[None] + np.array([1.0, 0, 0]) * np.exp2(-(np.arange(count) % 30.0))[:, None, None]


@pytest.mark.parametrize("kind", ["soup", "coincident", "chain"])
@pytest.mark.parametrize("count", [1, 2, 3, 5, 63, 64, 65, 127, 129, 1000])
def test_small_ranges_match_the_host_builder(ctx, kind, count):
    p = np.ascontiguousarray(corners(kind, count).reshape(-1, 3), dtype=np.float32)
    n = np.tile(np.array([0.0, 0.0, 1.0], np.float32), (3 * count, 1))
    data = SceneData()
    mesh = data.add_mesh(MeshData(p, n, np.arange(3 * count, dtype=np.uint32).reshape(-1, 3)))
    data.add_instance(mesh, identity(), Material.matte((0.5, 0.5, 0.5)))
    data.env_texels = np.ones((1, 1, 4), np.float32)
    trees = []
    for builder in (_abi.BVH_HOST, _abi.BVH_DEVICE):
        scene = cn.Scene(ctx, data, bvh_builder=builder)
        trees.append((*scene.bvh(), scene.bvh8()))
        scene.close()
    for host, device in zip(*trees):
        assert np.asarray(host).tobytes() == np.asarray(device).tobytes()


@pytest.mark.parametrize("counts", [(7,), (0, 5, 0, 0, 70, 0), (1, 1, 300, 1)])
def test_instances_reach_the_world_as_the_host_takes_them(ctx, counts):
    data = SceneData()
    rng = np.random.default_rng(len(counts))
    meshes = []
    for count in counts:
        p = rng.uniform(-1, 1, (3 * count, 3)).astype(np.float32)
        n = np.tile(np.array([0.0, 0.0, 1.0], np.float32), (3 * count, 1))
        meshes.append(data.add_mesh(MeshData(p, n, np.arange(3 * count, dtype=np.uint32).reshape(-1, 3))))
    for k, mesh in enumerate(meshes + meshes[::-1]):
        t = np.asarray(identity(), np.float32).reshape(3, 4) + rng.normal(scale=0.3, size=(3, 4)).astype(np.float32)
        data.add_instance(mesh, t.reshape(np.shape(identity())), Material.matte((0.1 * k, 0.5, 0.5)))
    data.env_texels = np.ones((1, 1, 4), np.float32)
    trees = []
    for builder in (_abi.BVH_HOST, _abi.BVH_DEVICE):
        scene = cn.Scene(ctx, data, bvh_builder=builder)
        trees.append((*scene.bvh(), scene.bvh8()))
        assert scene.info().triangle_count == 2 * sum(counts)
        scene.close()
    for host, device in zip(*trees):
        assert np.asarray(host).tobytes() == np.asarray(device).tobytes()
