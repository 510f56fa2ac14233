"""The cooperative traversal where its schedule has edges: ray counts around
the refill and wave sizes, trees from a single leaf up (a root that is a leaf,
one and two levels, odd and even depths), rays that start on a triangle's
plane (distance +-0), run along it, or have zero or negative-zero direction
components.  Every result is the oracle's, bit for bit."""
import numpy as np
import pytest

import oracle as O
import turner_amd as T
from turner_amd._lib import TN_ISECT_EXHAUSTIVE, TN_ISECT_REFINED
from tests import helpers as H

pytestmark = pytest.mark.gpu

SCENES = {
    "one": lambda: H.tri((0, 0, 1), (0, 1, 1), (1, 0, 1))[None],
    "two": lambda: np.stack([H.tri((0, 0, 1), (0, 1, 1), (1, 0, 1)), H.tri((2, 0, 2), (3, 0, 2), (3, 1, 2))]),
    "four": H.four_separated,
    "cube": H.cube12,
    "stack": lambda: H.coplanar_stack(1, np.random.default_rng(2)),
    "grid": lambda: H.grid_mesh(5),
    "soup": lambda: H.random_soup(300, np.random.default_rng(3), spread=2.0),
}
COUNTS = [1, 2, 15, 16, 17, 47, 48, 49, 63, 64, 65, 255, 257, 1000, 4099]


def _rays(verts, n, rng):
    o, d = H.hard_rays(verts, n, rng)
    v = verts.reshape(-1, 3, 3)
    k = rng.integers(0, len(v), n)
    w = rng.dirichlet((1, 1, 1), n)[:, :, None]
    kind = rng.integers(0, 5, n)
    on = (v[k] * w).sum(1).astype(np.float32)  # a point of a triangle (about)
    o[kind == 1] = on[kind == 1]
    o[kind == 2] = v[k, 0][kind == 2]  # a vertex itself: the plane distance is exactly +-0
    along = (v[k, 1] - v[k, 0]).astype(np.float32)
    d[kind == 3] = along[kind == 3]
    d[kind == 4] = rng.normal(size=(n, 3)).astype(np.float32)[kind == 4]
    d[(kind == 4) & (rng.random(n) < 0.3), 0] = -0.0
    return o.astype(np.float32), d.astype(np.float32)


@pytest.mark.parametrize("name", sorted(SCENES))
def test_edges_against_the_oracle(gpu, name):
    import torch
    verts = SCENES[name]()
    tree = T.KDTree(verts, refined=True)
    rng = np.random.default_rng(11)
    for n in COUNTS:
        o, d = _rays(verts, n, rng)
        want = O.intersect(tree.triangle_records(), tree.flat_nodes(), tree.box(), o, d)
        to, td = torch.from_numpy(o).cuda(), torch.from_numpy(d).cuda()
        for flags in (0, TN_ISECT_EXHAUSTIVE, TN_ISECT_REFINED, TN_ISECT_REFINED | TN_ISECT_EXHAUSTIVE):
            got = T.KDTreeIntersection(tree).intersect_batch(to, td, flags)
            for a, b, part in zip(got, want, "id r s t".split()):
                a, b = a.cpu().numpy().view(np.uint32), np.ascontiguousarray(b).view(np.uint32)
                assert np.array_equal(a, b), f"{name}, {n} rays, flags {flags}: {part} differs"
        ids, r = want[0], want[1]
        hit = ids != T.TN_INVALID_ID
        for scale in (0.5, 1.0, 2.0):
            tmax = np.where(hit, r, np.float32(1.0)) * np.float32(scale)
            tm = torch.from_numpy(tmax).cuda()
            expect = (hit & (r <= tmax)).astype(np.uint8)
            for flags in (0, TN_ISECT_REFINED):
                occ = torch.empty(n, dtype=torch.uint8, device="cuda")
                T.check(T.lib().tn_occluded(tree.handle, T.ptr(to), T.ptr(td), T.ptr(tm), n, T.ptr(occ), flags,
                                            torch.cuda.current_stream().cuda_stream))
                assert np.array_equal(occ.cpu().numpy(), expect), f"{name}, {n} rays, tmax x {scale}, flags {flags}"
