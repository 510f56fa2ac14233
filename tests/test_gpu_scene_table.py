"""The scene table of a batch passes through pinned memory up to 1 MiB and by a copy of
its own beyond: one-pixel images of scenes that the camera does not see, each with a
background of its own, on both sides of the line (160 bytes a scene).  A missed ray
returns its scene's background exactly."""
import numpy as np
import pytest

import turner_amd as T
from turner_amd import batch, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [5, 5000, 7000])
def test_every_scene_keeps_its_entry(gpu, n):
    tree = T.KDTree(np.array([[0, 0, -9, 0, 1, -9, 1, 0, -9]], np.float32))
    cam = scenes.camera((0.0, 0.0, 0.0), 40.0)
    probe = T.TracerConfig(width=1, max_recursion_depth=1, num_pixel_samples=1, bg_color=(1.0, 1.0, 1.0, 1.0))
    seen, _ = T.render(tree, cam, [], probe)
    if not np.array_equal(seen[0, 0], np.ones(4, np.float32)):  # the camera looks the other way
        tree = T.KDTree(np.array([[0, 0, 9, 0, 1, 9, 1, 0, 9]], np.float32))
    b = batch.Batch([tree] * n)
    bg = np.arange(4 * n, dtype=np.float32).reshape(n, 4) + 1
    jobs = [{"camera": cam, "lights": [], "width": 1, "height": 1, "spp": 1, "bg": bg[k]} for k in range(n)]
    _, st, acc = b.render(jobs, max_depth=0, mc_samples=0, seed=1)
    assert st["rays"] == n and np.array_equal(acc.cpu().numpy().reshape(n, 4), bg)
    b.close()
