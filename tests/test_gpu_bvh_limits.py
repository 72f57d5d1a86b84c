"""The device builder at the tree's limits: it gives way to the coarser rules,
and refuses, exactly where the host builder does, with the same nodes."""

from __future__ import annotations

import bvh_host
import numpy as np
import pytest

import cenote_amd as cn
from cenote_amd import _abi
from cenote_amd.scene import Material, MeshData, SceneData, identity

pytestmark = pytest.mark.gpu


def scene_of(corners):
    count = len(corners)
    normals = np.tile(np.array([0.0, 0.0, 1.0], np.float32), (3 * count, 1))
    data = SceneData()
    mesh = data.add_mesh(MeshData(np.ascontiguousarray(corners.reshape(-1, 3)), normals,
                                  np.arange(3 * count, dtype=np.uint32).reshape(-1, 3)))
    data.add_instance(mesh, identity(), Material.matte((0.5, 0.5, 0.5)))
    data.env_texels = np.ones((1, 1, 4), np.float32)
    return data


@pytest.mark.parametrize("levels", [64, 65, 70])
def test_deep_scenes_match_the_host_builder(ctx, levels):
    print(f"chain of {levels} clusters", flush=True)
    data = scene_of(bvh_host.chain(levels, 7))
    trees = []
    for builder in (_abi.BVH_HOST, _abi.BVH_DEVICE):
        scene = cn.Scene(ctx, data, bvh_builder=builder)
        trees.append((*scene.bvh(), scene.bvh8()))
        assert 3 * scene.info().bvh_max_depth <= bvh_host.STACK_MAX
        scene.close()
    for host, device in zip(*trees):
        assert np.asarray(host).tobytes() == np.asarray(device).tobytes()


def test_scenes_too_deep_by_both_rules_are_refused(ctx):
    print("chain of 66 clusters", flush=True)
    data = scene_of(bvh_host.chain(66, 7))
    for builder in (_abi.BVH_HOST, _abi.BVH_DEVICE):
        with pytest.raises(cn.CenoteError, match="too deep"):
            cn.Scene(ctx, data, bvh_builder=builder)
