"""Calls that use pinned host memory when they can get it, in a process where it is
refused: they work as they do with it.  And a batch whose host memory is refused is an
error, not an exception through the C interface."""
import os
import subprocess

import pytest

from tests import child

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def refuse(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("refuse") / "librefuse.so")
    src = os.path.join(child.ROOT, "tests", "cpp", "refuse_alloc.cpp")
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-o", so, src, "-ldl"], check=True)
    return so


SETUP = """
import ctypes, json, sys
shim = ctypes.CDLL(sys.argv[1], ctypes.RTLD_GLOBAL)
shim.refuse_host_blocks.argtypes = [ctypes.c_size_t]
import numpy as np, torch
import turner_amd as T
from turner_amd import scenes
"""


@pytest.mark.parametrize("refined", [0, 1])
def test_host_rays(gpu, refuse, refined):
    got = child.run(SETUP + """
tree = T.KDTree(scenes.intersect_scene(level=3)["verts"], refined=bool(int(sys.argv[2])))
q = T.KDTreeIntersection(tree)
res = {}
shim.refuse_pinned_memory(1)
o, d = scenes.random_rays(65536, seed=5)
for n in (1, 1000, 65536):
    res[n] = q.intersect_batch(o[:n], d[:n])
shim.refuse_pinned_memory(0)
print(json.dumps([all(np.array_equal(a.view(np.uint32), b.view(np.uint32))
                      for a, b in zip(res[n], q.intersect_batch(o[:n], d[:n]))) for n in res]))
""", refuse, refined)
    assert got == [True, True, True]


def test_renders(gpu, refuse):
    got = child.run(SETUP + """
from turner_amd import batch
sc = scenes.cornell_box()
tree = T.KDTree(sc["verts"], sc["normals"], sc["albedo"], sc["emission"])
b = batch.Batch([tree, tree])
jobs = [{"camera": sc["camera"], "lights": sc["lights"], "width": w, "height": 40, "spp": 2} for w in (30, 41)]
conf = T.TracerConfig(width=64, max_recursion_depth=2, num_pixel_samples=4, num_monte_carlo_samples=2, flags=4)

def all_of():
    img, st = T.render(tree, sc["camera"], sc["lights"], conf)
    images, bst, _ = b.render(jobs, max_depth=2, mc_samples=1, flags=3, seed=1)
    return [img, *(np.asarray(x.cpu() if hasattr(x, "cpu") else x) for x in images)], [st["rays"], st["shadow_rays"], bst["rays"]]

shim.refuse_pinned_memory(1)
a, sa = all_of()
shim.refuse_pinned_memory(0)
c, sc_ = all_of()
# FP32 sums of at most 4 x 7 contributions in another order
print(json.dumps([sa == sc_, all(bool(np.allclose(x, y, rtol=1e-5, atol=1e-6)) for x, y in zip(a, c)), sa[0] > 0]))
""", refuse)
    assert got == [True, True, True]


def test_batch_without_host_memory(gpu, refuse):
    got = child.run(SETUP + """
from turner_amd import _lib, batch
tree = T.KDTree(scenes.intersect_scene(level=5)["verts"])
before = torch.cuda.mem_get_info()[0]
codes = []
for size in (1 << 16, 1 << 18, 1 << 20):
    shim.refuse_host_blocks(size)
    try:
        batch.Batch([tree])
        codes.append(0)
    except T.TurnerError as e:
        codes.append(e.code)
    shim.refuse_host_blocks(0)
b = batch.Batch([tree])
b.close()
print(json.dumps([codes, before - torch.cuda.mem_get_info()[0], _lib.TN_ERR_OOM]))
""", refuse)
    codes, lost, oom = got
    assert codes[0] == oom and set(codes) <= {0, oom} and lost <= 4 << 20
