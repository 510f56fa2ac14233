"""Device memory of the ray queues: what a first render takes, what is left when
little is free, and that large queues go back with the last scene and batch of the
device.  Each in a process of its own, in bytes that the driver reports free."""
import pytest

from tests import child

pytestmark = pytest.mark.gpu

SETUP = """
import json, sys
import numpy as np, torch
import turner_amd as T
from turner_amd import scenes

def free():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]

def tree_of(sc):
    t = T.KDTree(sc["verts"], sc["normals"], sc["albedo"], sc["emission"])
    T.KDTreeIntersection(t).intersect([0, 0, 0], [0, 0, 1])
    return t

def render(t, sc, w, h, spp, m, depth, **kw):
    conf = T.TracerConfig(width=w, aspect=w / h, max_recursion_depth=depth, num_pixel_samples=spp,
                          num_monte_carlo_samples=m, seed=5, flags=3, **kw)
    acc = torch.zeros((h, w, 4), device="cuda")
    st = T.render_accumulate(t, sc["camera"], sc["lights"], conf, acc)
    return acc.cpu().numpy(), st["rays"]

def leave(n):  # a ballast that leaves n bytes free
    global ballast
    ballast = None
    torch.cuda.empty_cache()
    ballast = torch.empty(free() - n, dtype=torch.uint8, device="cuda")

sc = scenes.furnace(level=1)
sc["lights"] = [((0.0, 3.0, -3.0), (1.0, 1.0, 1.0, 1.0))]
t = tree_of(sc)
acc = torch.zeros((512, 1024, 4), device="cuda")
"""

MB = 1 << 20


def test_chunks_sized_by_the_caller(gpu):
    few, many = (child.run(SETUP + """
f = free()
render(t, sc, 1024, 1024, 1, 1, 2, chunk_paths=int(sys.argv[1]))
print(json.dumps(f - free()))
""", chunk) for chunk in (4096, 1 << 19))
    # two pipelines with 404 B per entry: what the larger chunks take more (what streams
    # take is in both); an allocation is a multiple of 2 MiB
    assert abs(many - few - 2 * 404 * ((1 << 19) - 4096)) <= 8 * MB


def test_small_render_with_little_memory_free(gpu):
    got = child.run(SETUP + """
leave(3 << 30)
f = free()
img, n = render(t, sc, 64, 64, 1, 2, 2)
print(json.dumps([f - free(), n, int(np.isfinite(img).all())]))
""")
    # at most a quarter of 3 GiB goes to queues that this render does not need
    assert got[0] <= 768 * MB and got[1] == 64 * 64 * 7 and got[2]


# 524,288 samples of 64 segments at the deepest level: 2 x 2^24 entries by default.
# With 40 GiB free they would be a third of it, with 60 a quarter of it at most.
@pytest.mark.parametrize("gib,most", [(40, 2 * 2**23 * 404), (60, 2 * 2**24 * 404)])
def test_queues_take_a_share_of_the_free_memory(gpu, gib, most):
    got = child.run(SETUP + """
want, rays = render(t, sc, 1024, 512, 1, 4, 3, chunk_paths=20000)
leave(int(sys.argv[1]) << 30)
f = free()
img, n = render(t, sc, 1024, 512, 1, 4, 3)
# sums of one sample: at most 85 contributions each, in another order
ok = bool(np.allclose(img, want, rtol=1e-5, atol=1e-6)) and n == rays == 1024 * 512 * 85
print(json.dumps([f - free(), ok]))
""", gib)
    assert got[0] <= most + 64 * MB and got[1]


def test_queues_go_back_with_the_last_scene_and_batch(gpu):
    got = child.run(SETUP + """
from turner_amd import batch
other = tree_of(scenes.cornell_box())
b = batch.Batch([t])
render(t, sc, 64, 64, 1, 1, 2, chunk_paths=1024)  # streams and events stay
jobs = [{"camera": sc["camera"], "lights": sc["lights"], "width": 64, "height": 64, "spp": 1}]
f = free()
img, n = render(t, sc, 1024, 512, 1, 4, 3)
taken = f - free()
t.close()
other.close()
kept = f - free()
b.render(jobs, max_depth=2, mc_samples=1, flags=3, seed=1)
b.close()
back = f - free()
t = tree_of(sc)
again, n2 = render(t, sc, 1024, 512, 1, 4, 3)
print(json.dumps([taken, kept, back, n == n2, bool(np.allclose(img, again, rtol=1e-5, atol=1e-6))]))
""")
    taken, kept, back, same, close = got
    # beyond what may stay (2 x 2^23 entries), kept while a batch lives, then all of it back
    assert taken > 2 * 2**23 * 404 and kept > 2 * 2**23 * 404 and back <= 64 * MB
    assert same and close


def test_scenes_of_several_threads(gpu):
    """Each thread makes a scene, renders it and destroys it, while the others do."""
    got = child.run(SETUP + """
import threading
want, rays = render(t, sc, 1024, 512, 1, 4, 3)
t.close()
failed = []

def turns():
    try:
        for _ in range(4):
            mine = T.KDTree(sc["verts"], sc["normals"], sc["albedo"], sc["emission"])
            img, n = render(mine, sc, 1024, 512, 1, 4, 3)
            assert n == rays and np.allclose(img, want, rtol=1e-5, atol=1e-6)
            mine.close()
    except Exception as e:
        failed.append(repr(e))

threads = [threading.Thread(target=turns) for _ in range(3)]
for x in threads:
    x.start()
for x in threads:
    x.join()
print(json.dumps(failed))
""")
    assert got == []
