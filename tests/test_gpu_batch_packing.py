"""A batch packs its scenes' trees on the device, child indices and leaf offsets
rebased: trees of a lone leaf, of one and two levels and of many, in an order that
puts each after smaller and larger ones, twice.  Every scene renders as by itself (bars of
test_gpu_batch.py: 1e-5 relative, 1e-6 absolute; equal ray counts)."""
import numpy as np
import pytest

import turner_amd as T
from turner_amd import scenes
from turner_amd._lib import TN_RENDER_COSINE
from tests import helpers as H
from tests.test_gpu_batch import MASK, STEP, _single

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", [{}, {"empty_leaves": True}])
def test_every_tree_is_rebased(gpu, kind):
    from turner_amd.batch import Batch
    wall = H.tri((-4, -4, 2), (0, 6, 2), (4, -4, 2)).astype(np.float32)
    soups = [wall[None], np.stack([wall, wall + np.float32(0.5)]), H.cube12(), H.grid_mesh(3),
             H.random_soup(300, np.random.default_rng(3), spread=2.0), scenes.intersect_scene(level=3)["verts"]]
    trees = [T.KDTree(np.ascontiguousarray(np.asarray(v, np.float32).reshape(-1, 9)), **kind) for v in soups]
    order = [0, 5, 1, 4, 0, 2, 3, 5, 1]
    light = [((0.2, 0.5, -3.0), (1.0, 0.5, 0.25, 1.0))]
    views = [scenes.camera((0.1, 0.2, z), 60.0) for z in (-4.0, 4.0)]
    for cam in views:
        sc = {"camera": cam, "lights": light}
        jobs = [{**sc, "width": 20 + k, "height": 17, "spp": 3, "bg": (0.1, 0.2, 0.3, 1.0)} for k in range(len(order))]
        b = Batch([trees[k] for k in order])
        imgs, st, _ = b.render(jobs, max_depth=2, mc_samples=1, flags=TN_RENDER_COSINE, seed=7)
        rays = 0
        for s, k in enumerate(order):
            ref, one = _single(trees[k], sc, jobs[s], 2, 1, TN_RENDER_COSINE, (7 + s * STEP) & MASK)
            np.testing.assert_allclose(imgs[s].cpu().numpy() * 3, ref, rtol=1e-5, atol=1e-6, err_msg=f"scene {s}")
            rays += one["rays"]
        assert st["rays"] == rays
        b.close()
