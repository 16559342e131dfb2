"""The compressed wide walk of renders and ray queries against the oracle, bit
for bit, where it can go wrong: launch sizes at the limit between four lanes
and one lane to a ray and at wave edges, rays that meet two triangles at one
distance (the reference's visit order decides), leaves of many triangles, a
tree too deep for the four-lane walk's stack, coordinates far from the origin
and far apart, rays with zero direction components, and both triangle tests."""
import dataclasses

import numpy as np
import pytest

from firefly_amd import abi, scenes

pytestmark = pytest.mark.gpu

QUAD_MAX = 131072  # rays of the largest launch that gives each four lanes


def _soup(n, seed, edge):
    pos, nrm, uv = scenes.soup_in_cube(n, seed, edge)
    return pos, nrm, uv


def _chain(n):
    """Triangles along a line, each 1.5x farther: clustered from the near end
    one by one, a tree deeper than the four-lane walk's stack."""
    c = 1.5 ** np.arange(n)
    tri = np.zeros((n, 3, 3))
    tri[:, 0, 0] = c
    tri[:, 1, 0] = c * 1.2
    tri[:, 2, 0] = c
    tri[:, 2, 1] = c * 0.3
    tri[..., 2] = np.linspace(0.0, 1.0, n)[:, None]
    nrm = np.zeros_like(tri)
    nrm[..., 2] = 1.0
    return tri.astype(np.float32), nrm.astype(np.float32), np.zeros((n, 3, 2), np.float32)


def _scene(kind):
    """(positions, normals, uvs, largest leaf, box of the ray origins)"""
    if kind == "mesh":
        sd = scenes.icosphere_scene(8, 8, 1, 1, seed=3, subdiv=4, env_w=8, env_h=4)
        return sd.positions, sd.normals, sd.uvs, 8, (-1.5, 1.5)
    if kind == "doubled":  # every triangle twice: every hit is shared
        pos, nrm, uv = _soup(700, 5, 0.2)
        return np.repeat(pos, 2, 0), np.repeat(nrm, 2, 0), np.repeat(uv, 2, 0), 4, (-0.2, 1.2)
    if kind == "big_leaves":
        pos, nrm, uv = _soup(3000, 6, 0.05)
        return pos, nrm, uv, 200, (-0.2, 1.2)
    if kind == "one":
        pos, nrm, uv = _soup(1, 7, 0.5)
        return pos, nrm, uv, 8, (-0.2, 1.2)
    if kind == "five":
        pos, nrm, uv = _soup(5, 8, 0.5)
        return pos, nrm, uv, 1, (-0.2, 1.2)
    if kind == "far":  # far from the origin, scales mixed
        pos, nrm, uv = _soup(4000, 9, 0.05)
        pos = pos * np.float32(300.0) + np.float32(7000.0)
        pos[:1000] = pos[:1000] * np.float32(0.01) + np.float32(7000.0)
        return pos, nrm, uv, 8, (6900.0, 7400.0)
    assert kind == "chain"
    return (*_chain(140), 1, (0.0, 40.0))


def _rays(n, seed, box, axis_aligned):
    r = scenes.random_rays(n, seed, lo=box[0], hi=box[1], y_lo=box[0], y_hi=box[1])
    if axis_aligned:
        rng = np.random.default_rng(seed)
        d = np.zeros((n, 3), np.float32)
        a = rng.integers(0, 3, n)
        d[np.arange(n), a] = rng.choice([-1.0, 1.0], n)
        two = rng.random(n) < 0.5  # the others: one zero component only
        d[two, (a[two] + 1) % 3] = rng.choice([-0.5, 0.5], int(two.sum()))
        r[:, 4:7] = d
    return r


CASES = [("mesh", 1, False), ("mesh", 65, True), ("mesh", QUAD_MAX, False), ("mesh", QUAD_MAX + 1, False),
         ("mesh", QUAD_MAX + 1, True), ("doubled", 2049, False), ("doubled", QUAD_MAX + 257, False),
         ("big_leaves", 5000, True), ("big_leaves", QUAD_MAX + 1, False), ("one", 63, False), ("five", 1025, False),
         ("far", 16385, False), ("far", QUAD_MAX + 63, True), ("chain", 3000, False), ("chain", QUAD_MAX + 1, True)]


@pytest.mark.parametrize("kind,n,axis_aligned", CASES, ids=[f"{k}-{n}{'-axis' if a else ''}" for k, n, a in CASES])
def test_wide_walk_equals_the_reference_walk(gpu, oracle, kind, n, axis_aligned):
    import torch
    pos, nrm, uv, leaf, box = _scene(kind)
    base = scenes.spheres_scene(8, 8, 1, 1, segments=4, rings=3)
    sd = dataclasses.replace(base, positions=pos, normals=nrm, uvs=uv, material_ids=np.zeros(len(pos), np.int32))
    # (the SAH builder would split such leaves, and balance such a tree)
    builder = {"big_leaves": abi.FF_BVH_LBVH, "chain": abi.FF_BVH_PLOC}.get(kind, abi.FF_BVH_SAH)
    sc = abi.Scene(gpu, pos, nrm, uv, sd.material_ids, sd.materials, max_prims=leaf, builder=builder)
    nodes, ordered = sc.bvh()
    ps = oracle.PreparedScene(sd, nodes, ordered)
    if kind == "chain":
        assert sc.max_depth > 64
    if kind == "big_leaves":
        assert nodes["n_prims"].max() > 60
    rays = _rays(n, 100 + n, box, axis_aligned)
    print(kind, n, axis_aligned, flush=True)
    r = torch.from_numpy(rays).cuda()
    h = torch.empty((n, 4), dtype=torch.float32, device="cuda")
    for two_sided in (False, True):
        sc.trace_closest(r, h, two_sided)
        torch.cuda.synchronize()
        g = h.cpu().numpy()
        t, u, v, i = oracle.trace_closest(ps.nodes, ps.tris_ordered(), rays, two_sided=two_sided)
        assert np.array_equal(g[:, 3].view(np.int32), i)
        hit = i >= 0
        for a, b in ((g[:, 0], t), (g[:, 1], u), (g[:, 2], v)):
            assert np.array_equal(a[hit].view(np.uint32), b[hit].view(np.uint32))
    occ = torch.empty(n, dtype=torch.uint8, device="cuda")
    sc.trace_any(r, occ)
    torch.cuda.synchronize()
    assert np.array_equal(occ.cpu().numpy(), oracle.trace_any(ps.nodes, ps.tris_ordered(), rays))
    sc.close()
