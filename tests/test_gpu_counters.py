"""Work counters of TN_ISECT_COUNT launches.  The cooperative traversal visits the
nodes, leaves and triangles that the schedule of a leaf per lane does, so all counts
but [6] are equal: whole numbers, no tolerance.  [6] counts the records read whole:
every one in launches of at most a ray per lane on the reference tree (which read
both halves at once), else those whose first half did not decide."""
import numpy as np
import pytest

import turner_amd as T
from turner_amd import scenes
from turner_amd._lib import TN_ISECT_COUNT, TN_ISECT_EXHAUSTIVE, TN_ISECT_LEAF, TN_ISECT_REFINED
from tests import helpers as H

pytestmark = pytest.mark.gpu


def _counts(tree, n, flags, seed=3):
    import torch
    o, d = scenes.random_rays(n, seed=seed)
    cnt = np.zeros(8, np.uint64)
    T.check(T.lib().tn_get_counters(tree.handle, cnt.ctypes.data, 1))
    T.KDTreeIntersection(tree).intersect_batch(torch.from_numpy(o).cuda(), torch.from_numpy(d).cuda(),
                                               flags | TN_ISECT_COUNT)
    T.check(T.lib().tn_get_counters(tree.handle, cnt.ctypes.data, 1))
    return [int(x) for x in cnt]


SCENES = {"one": lambda: H.tri((0, 0, 1), (0, 1, 1), (1, 0, 1))[None], "cube": H.cube12,
          "sphere": lambda: scenes.intersect_scene(level=3)["verts"]}


@pytest.mark.parametrize("name", sorted(SCENES))
@pytest.mark.parametrize("exhaustive", [0, TN_ISECT_EXHAUSTIVE])
def test_counts_equal_the_per_lane_schedule(gpu, name, exhaustive):
    for kind in ({}, {"empty_leaves": True}):
        tree = T.KDTree(SCENES[name](), **kind)
        for n in (1, 63, 1000, 500001):
            coop, leaf = _counts(tree, n, exhaustive), _counts(tree, n, exhaustive | TN_ISECT_LEAF)
            assert coop[:6] + coop[7:] == leaf[:6] + leaf[7:], f"{n} rays, {kind}"


def test_longest_traversal_of_a_refined_tree(gpu):
    tree = T.KDTree(SCENES["one"](), refined=True)
    c = _counts(tree, 64, TN_ISECT_REFINED)
    assert c[1] > 0 and c[7] == 1  # the only leaf


def test_whole_records(gpu):
    tree = T.KDTree(SCENES["sphere"](), refined=True)
    _, cus = T.device_info()
    lanes = cus * 28 * 64  # resident lanes
    for n in (1, 1000, lanes):
        c = _counts(tree, n, 0)
        assert c[6] == c[3] > 0, f"{n} rays"
    c = _counts(tree, lanes + 1, 0)
    assert 0 < c[6] < c[3]
    c = _counts(tree, 1000, TN_ISECT_REFINED)
    assert 0 < c[6] < c[3]
