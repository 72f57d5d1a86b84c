"""Scenes whose trees come near the builder's limits (host builder, CPU): a
tree by the usual rules that is too deep for the traversal stack, or has more
nodes than the traversal addresses, gives way to the coarser one, and only a
scene that is past the limits by both is refused."""

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


@pytest.mark.parametrize("side", [16, 32])
def test_nodes_stay_within_their_addresses(side):
    # The limit stands to the triangles as 2^26 does to the 2^27 a scene may
    # have. Of 32^3 single triangles two thirds would be nodes by the usual rules.
    corners = bvh_host.lattice(side)
    limit = len(corners) // 2
    tree, error = bvh_host.build(corners, nodes4=limit)
    assert error == "" and tree["nodes4"] <= limit
    assert bvh_host.build(corners, nodes4=len(corners))[0]["nodes4"] >= tree["nodes4"]


def test_an_eight_wide_tree_past_its_addresses_is_left_out():
    corners = bvh_host.lattice(16)
    whole, _ = bvh_host.build(corners)
    assert whole["nodes8"] > 0
    tree, error = bvh_host.build(corners, nodes8=whole["nodes8"] - 1)
    assert error == "" and tree["nodes8"] == 0 and tree["nodes4"] == whole["nodes4"]


def test_too_many_nodes_by_both_rules_are_refused():
    _, error = bvh_host.build(bvh_host.lattice(16), nodes4=100)
    assert "more nodes than the traversal addresses" in error
