"""The shade kernels reserve queue slots per block: path counts around a wave,
a block and a grid's worth of blocks, with none to several children and shadow
rays per segment.  The segment and shadow-ray counts of a closed scene are
known exactly, and every path draws its own stream, so the image does not
depend on how the samples are cut into chunks (pixels within FP32 summation
order: at most 100 contributions, 1e-5 relative)."""
import numpy as np
import pytest

import turner_amd as T
from turner_amd import guide, scenes
from turner_amd._lib import TN_RENDER_AREA_LIGHTS, TN_RENDER_COSINE

pytestmark = pytest.mark.gpu
FLAGS = TN_RENDER_COSINE | TN_RENDER_AREA_LIGHTS


@pytest.fixture(scope="module")
def closed(gpu):
    sc = scenes.furnace(level=1)
    sc["lights"] = [((0.0, 3.0, -3.0), (1.0, 1.0, 1.0, 1.0))]
    return sc, T.KDTree(sc["verts"], sc["normals"], sc["albedo"], sc["emission"])


def _render(sc, tree, w, h, spp, m, depth, chunk=0, net=None):
    import torch
    conf = T.TracerConfig(width=w, aspect=w / h, max_recursion_depth=depth, num_pixel_samples=spp,
                          num_monte_carlo_samples=m, flags=FLAGS, seed=5, chunk_paths=chunk)
    assert conf.height() == h
    acc = torch.zeros((h, w, 4), device="cuda")
    if net is None:
        st = T.render_accumulate(tree, sc["camera"], sc["lights"], conf, acc)
    else:
        st = guide.render_guided(tree, sc["camera"], sc["lights"], conf, net, acc)
    return acc.cpu().numpy(), st


@pytest.mark.parametrize("w,h,spp", [(1, 1, 1), (1, 1, 63), (8, 8, 1), (13, 5, 1), (51, 5, 1), (16, 16, 1),
                                     (257, 1, 1), (128, 64, 1), (100, 41, 2), (320, 41, 5), (512, 512, 2)])
@pytest.mark.parametrize("m", [0, 1, 3])
def test_counts_and_chunks(closed, w, h, spp, m):
    sc, tree = closed
    depth = 2
    a, st = _render(sc, tree, w, h, spp, m, depth)
    assert st["rays"] == w * h * spp * sum(m ** k for k in range(depth + 1))  # every segment hits
    assert st["shadow_rays"] >= st["rays"]  # one point-light ray per hit, an emitter ray for some
    n = w * h * spp
    b, sb = _render(sc, tree, w, h, spp, m, depth, chunk=max(1, n // 3))
    assert (sb["rays"], sb["shadow_rays"]) == (st["rays"], st["shadow_rays"])
    assert np.allclose(a, b, rtol=1e-5, atol=1e-6)


@pytest.mark.parametrize("w,h,spp", [(1, 1, 1), (13, 5, 1), (127, 1, 1), (16, 8, 1), (43, 3, 1), (100, 41, 2)])
@pytest.mark.parametrize("m", [1, 2])
def test_guided_counts_and_chunks(closed, w, h, spp, m):
    sc, tree = closed
    net = guide.Guide.for_tree(tree)
    a, st = _render(sc, tree, w, h, spp, m, 2, net=net)
    b, sb = _render(sc, tree, w, h, spp, m, 2, chunk=max(1, w * h * spp // 3), net=net)
    assert (sb["rays"], sb["shadow_rays"]) == (st["rays"], st["shadow_rays"])
    assert w * h * spp <= st["rays"] <= w * h * spp * (1 + m + m * m)
    assert np.allclose(a, b, rtol=1e-5, atol=1e-6)
