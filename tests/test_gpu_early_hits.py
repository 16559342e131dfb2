"""Grazing hits whose rounded t lies before the entry into their own leaf's box
(by more than the pruning's slack), with another triangle between the two
distances: pruning then decides whether the triangle is reached.  Queries of
every size give the walk in the reference's order with its pruning (the
oracle's), the same for each copy of a ray whatever rays share its wave, and so
do counted queries with one step an iteration."""
import dataclasses

import numpy as np
import pytest

from firefly_amd import abi, scenes

pytestmark = pytest.mark.gpu

QUAD_MAX = 131072


def sliver_scene(oracle, seed):
    """A stack of long triangles met at angles of 1e-6 to 1e-4 and a screen
    across the rays; rays whose hit on the top one is early: some with the screen
    between its t and its leaf's entry, some with the screen beyond it.
    (positions, rays, how many of the first kind)"""
    f = np.float32
    rng = np.random.default_rng(seed)
    size = 10 ** rng.uniform(1.0, 1.9)
    a, b = rng.normal(size=3), rng.normal(size=3)
    a /= np.linalg.norm(a)
    b -= a * (a @ b)
    b /= np.linalg.norm(b)
    nn = np.cross(a, b)
    v0 = rng.normal(size=3)
    tri = np.array([v0, v0 + a * size, v0 + a * size * 0.5 + b * size * 0.01])
    n = 60000
    w = rng.dirichlet((0.3, 0.3, 0.3), n)
    g = 10 ** rng.uniform(-6, -4, n)
    d = a + rng.uniform(-0.2, 0.2, n)[:, None] * b - g[:, None] * nn
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    rays = np.zeros((n, 8), f)
    rays[:, :3], rays[:, 4:7] = w @ tri - d * size * 2, d

    def alone(t3):
        p = t3[None].astype(f)
        nodes, ordered = oracle.bvh_build(p, 1)
        t, _, _, i = oracle.trace_closest(nodes, oracle.ordered_tris(p.reshape(-1, 9), ordered), rays)
        return np.where(i >= 0, t, f(np.inf))

    def lim(t):
        return ((t + (t * f(2.0 ** -12)).astype(f)).astype(f) + f(1e-6)).astype(f)

    t_long = alone(tri)
    lo, hi = tri.astype(f).min(0), tri.astype(f).max(0)
    inv = (f(1) / rays[:, 4:7]).astype(f)
    entry = (((np.where(inv < 0, hi, lo) - rays[:, :3]).astype(f)) * inv).astype(f).max(1)
    early = np.isfinite(t_long) & (lim(t_long) < entry)
    # a screen across the rays, where most of the early ones have it between
    best = (0, None, None)
    for q in (0.1, 0.3, 0.5, 0.7, 0.9):
        e = np.quantile(np.where(early, 0.5 * (t_long + entry), np.nan)[early], q)
        c = v0 - 2 * size * a + a * e
        screen = c + 0.1 * size * np.array([-b - nn, 2 * nn, 2 * b - nn])
        t_s = alone(screen)
        between = early & (t_long < t_s) & (lim(t_s) < entry)
        beyond = early & (entry <= lim(t_s))
        if between.sum() > best[0]:
            best = (int(between.sum()), screen, np.concatenate([np.nonzero(between)[0], np.nonzero(beyond)[0]]))
    k, screen, pick = best
    stack = tri - 0.003 * size * np.arange(7)[:, None, None] * nn
    return np.concatenate([stack, screen[None]]).astype(f), rays[pick], k


@pytest.mark.parametrize("seed", [0, 1, 2, 3])
def test_early_hits_do_not_depend_on_the_launch(gpu, oracle, seed):
    import torch
    pos, some, k = sliver_scene(oracle, seed)
    assert k >= 20 and len(some) > k
    base = scenes.spheres_scene(8, 8, 1, 1, segments=4, rings=3)
    nrm = np.tile(np.float32([0, 1, 0]), (len(pos), 3, 1))
    sd = dataclasses.replace(base, positions=pos, normals=nrm, uvs=np.zeros((len(pos), 3, 2), np.float32),
                             material_ids=np.zeros(len(pos), np.int32))
    sc = abi.Scene(gpu, pos, nrm, sd.uvs, sd.material_ids, sd.materials, max_prims=1)
    ps = oracle.PreparedScene(sd, *sc.bvh())
    tris = ps.tris_ordered()

    def walk(rays):
        return oracle.trace_walk(ps.nodes, tris, rays, prune=True, width=2)

    rng = np.random.default_rng(seed)
    lo, hi = float(pos.min()), float(pos.max())
    for n in (len(some), 20000, QUAD_MAX + 257):
        rays = scenes.random_rays(n, seed + n, lo=lo, hi=hi, y_lo=lo, y_hi=hi)
        at = rng.permutation(n)[:max(len(some), n // 2)]
        rays[at] = some[np.arange(len(at)) % len(some)]
        t, i = walk(rays)
        r = torch.from_numpy(rays).cuda()
        for counted in (False, True):
            print(seed, n, "counted" if counted else "", flush=True)
            h = torch.empty((n, 4), dtype=torch.float32, device="cuda")
            cnt = torch.zeros(2, dtype=torch.int64, device="cuda") if counted else None
            sc.trace_closest(r, h, False, cnt)
            torch.cuda.synchronize()
            g = h.cpu().numpy()
            assert np.array_equal(g[:, 3].view(np.int32), i)
            assert np.array_equal(g[i >= 0, 0].view(np.uint32), t[i >= 0].view(np.uint32))
    sc.close()
