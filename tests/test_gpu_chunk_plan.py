"""Chunks of a render around the lines of their plan (m 4, depth 3: 64 segments at
the deepest level per sample): split over two pipelines from 2^23 such segments
on, at most 2^25 per chunk.  Counts of a closed scene are known; the image is that
of explicitly cut chunks (FP32 sums of at most 128 contributions: 1e-5 relative)."""
import numpy as np
import pytest

from tests.test_gpu_queue_edges import _render, closed  # noqa: F401  (module fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h,spp", [(1, 131071, 1), (1024, 128, 1), (512, 1025, 1), (1024, 512, 2), (1025, 512, 2),
                                     (1024, 768, 2)])
def test_default_chunks(closed, w, h, spp):  # noqa: F811
    sc, tree = closed
    a, st = _render(sc, tree, w, h, spp, 4, 3)
    assert st["rays"] == w * h * spp * 85 and st["primary_rays"] == w * h * spp
    b, sb = _render(sc, tree, w, h, spp, 4, 3, chunk=77777)
    assert (sb["rays"], sb["shadow_rays"]) == (st["rays"], st["shadow_rays"])
    assert np.allclose(a, b, rtol=1e-5, atol=1e-6)
