"""Scenes whose trees come near the builder's limits (host builder, CPU): a
tree by the usual rules that is too deep for the traversal stack gives way to
the coarser one, and only a scene that is too deep by both is refused."""

import bvh_host
import pytest


@pytest.mark.parametrize("levels,cluster,depth", [(64, 7, 40), (65, 7, 41), (70, 7, 42)])
def test_deep_scenes_are_built(levels, cluster, depth):
    # (64, 7) fits by the usual rules; those would take the others to depth 43.
    tree, error = bvh_host.build(bvh_host.chain(levels, cluster))
    assert error == ""
    assert tree["depth4"] == depth and 3 * depth <= bvh_host.STACK_MAX


def test_the_coarse_rules_are_kept_for_trees_that_need_them():
    corners = bvh_host.chain(64, 7)
    usual, _ = bvh_host.build(corners)
    coarse, error = bvh_host.build(corners, max_stack=3 * 39)
    assert error == ""
    assert coarse["depth4"] < usual["depth4"] and coarse["nodes4"] < usual["nodes4"]


def test_a_scene_too_deep_by_both_rules_is_refused():
    _, error = bvh_host.build(bvh_host.chain(66, 7))
    assert "too deep for the traversal stack" in error
