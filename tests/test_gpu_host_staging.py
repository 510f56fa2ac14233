"""Host-side calls exchange small inputs and results with the kernels through
pinned memory and larger ones by copies: both sides of each line, and again after
a smaller and a larger call, with concurrent callers."""
import threading

import numpy as np
import pytest

import oracle as O
import turner_amd as T
from turner_amd import scenes
from tests.test_gpu_render import _render
from turner_amd._lib import TN_RENDER_REF_JITTER

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("refined", [False, True])
def test_host_rays_equal_device_rays(gpu, refined):
    import torch
    sc = scenes.intersect_scene(level=3)
    q = T.KDTreeIntersection(T.KDTree(sc["verts"], refined=refined))
    rng = np.random.default_rng(7)

    def check(n, o, d):
        host = q.intersect_batch(o[:n], d[:n])
        dev = q.intersect_batch(torch.from_numpy(o[:n]).cuda(), torch.from_numpy(d[:n]).cuda())
        for a, b in zip(host, dev):
            assert np.array_equal(a.view(np.uint32), b.cpu().numpy().view(np.uint32)), n

    o = rng.uniform(-2, 2, (70000, 3)).astype(np.float32)
    d = rng.normal(size=o.shape).astype(np.float32)
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    for n in (1, 64, 65536, 3, 65537, 65535):
        check(n, o, d)
    failed = []

    def caller(k):
        try:
            for _ in range(20):
                a = slice(997 * k, 997 * k + 101 * (k + 1))
                want = ids[a]
                assert np.array_equal(q.intersect_batch(o[a], d[a])[0], want)
        except Exception as e:  # reported by the main thread
            failed.append(e)

    ids = q.intersect_batch(o, d)[0]
    threads = [threading.Thread(target=caller, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed


# 2 x width x spp floats of jitter: 1 MiB, then one sample more
@pytest.mark.parametrize("width,spp", [(64, 2048), (64, 2049), (3, 1)])
def test_jitter_tables(gpu, width, spp):
    sc = scenes.cornell_box()
    tree = T.KDTree(sc["verts"], sc.get("normals"), sc.get("albedo"), sc.get("emission"))
    conf = T.TracerConfig(width=width, aspect=float(width), max_recursion_depth=0, num_pixel_samples=spp,
                          num_monte_carlo_samples=1, flags=TN_RENDER_REF_JITTER)
    assert conf.height() == 1
    lin, st = _render(tree, sc, conf)
    ref, _, nr, _ = O.render(sc, O.Tree(sc["verts"]), width, 1, 0, 1, spp, flags=O.FLAG_REF_RNG, nthreads=4)
    assert st["rays"] == nr == width * spp
    # both sides sum spp FP32 contributions: spp * 2^-24 of the sum each at most
    np.testing.assert_allclose(lin, ref, rtol=1e-5 + spp * 2.0 ** -23, atol=1e-6)
    assert lin[..., :3].max() > 0
