"""A wave of the shadow tests that takes more than 64 chunks of its queue adds the
rays that finish from then on directly.  One queue of more than 64 x 512 entries per
wave of the grid (eight blocks of four waves per compute unit) makes sure that some
wave does; the image is that of many small chunks (FP32 sums in another order: a
part in 2^24 per contribution).  In a process of its own: the queues take about
110 GB."""
import pytest

from tests import child

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("renderer", [0, 2])
def test_more_chunks_than_a_wave_notes(gpu, renderer):
    got = child.run("""
import json, sys
import numpy as np, torch
import turner_amd as T
from turner_amd import scenes
renderer = int(sys.argv[1])
_, cus = T.device_info()
sc = scenes.furnace(level=1)
light = [((0.0, 3.0, -3.0), (1.0, 0.5, 0.25, 1.0))]
tree = T.KDTree(sc["verts"], sc["normals"], sc["albedo"], sc["emission"])
line = 64 * 512 * 8 * 4 * cus  # entries
w, h = 1024, 512

def render(spp, chunk, flags):
    conf = T.TracerConfig(width=w, aspect=w / h, max_recursion_depth=0, num_pixel_samples=spp,
                          num_monte_carlo_samples=0, seed=5, chunk_paths=chunk, renderer=renderer, flags=flags)
    acc = torch.zeros((h, w, 4), device="cuda")
    st = T.render_accumulate(tree, sc["camera"], light, conf, acc)
    return acc.cpu().numpy(), st

spp = line // (w * h) + 2
a, st = render(spp, w * h * spp, 32)  # replayed chunks run in one pipeline: one queue
b, sb = render(spp, 1 << 22, 0)
print(json.dumps({"shadow": st["shadow_rays"], "line": line, "rays": [st["rays"], sb["rays"], w * h * spp],
                  "same": st["shadow_rays"] == sb["shadow_rays"],
                  "close": bool(np.allclose(a, b, rtol=spp * 2.0 ** -23, atol=0)), "lit": float(a[..., 0].max())}))
""", renderer)
    assert got["shadow"] > got["line"] and got["same"]
    assert len(set(got["rays"])) == 1
    assert got["close"] and got["lit"] > 0
