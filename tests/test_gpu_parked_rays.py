"""Rays that the one-lane wide walk parks, to be traced again in the
reference's order: launches whose every ray meets two triangles at one distance
or has a box plane distance that is NaN, at the sizes where the number of lanes
a wave owns changes (a wave of a small launch owns fewer lanes than it may
park), queries and a render, on a tree too deep for the four-lane walk.  Bit for
bit the oracle's hits, occlusion and film."""
import dataclasses

import numpy as np
import pytest

from firefly_amd import abi, scenes

pytestmark = pytest.mark.gpu

QUAD_MAX = 131072


def _chain(n):
    """Triangles along z, each 1.5x farther: PLOC makes a tree of depth > 64."""
    c = 1.5 ** np.arange(n)
    tri = np.zeros((n, 3, 3))
    tri[:, 0, 2] = c
    tri[:, 1, 2] = c * 1.2
    tri[:, 2, 2] = c
    tri[:, 2, 1] = c * 0.3
    tri[..., 0] = np.linspace(0.0, 1.0, n)[:, None]
    nrm = np.zeros_like(tri)
    nrm[..., 0] = 1.0
    return tri.astype(np.float32), nrm.astype(np.float32), np.zeros((n, 3, 2), np.float32)


def _doubled(sd, pos, nrm, uv, mid):
    return dataclasses.replace(sd, positions=np.repeat(pos, 2, 0), normals=np.repeat(nrm, 2, 0),
                               uvs=np.repeat(uv, 2, 0), material_ids=np.repeat(mid, 2).astype(np.int32))


def _create(gpu, oracle, sd, builder):
    sc = abi.Scene(gpu, sd.positions, sd.normals, sd.uvs, sd.material_ids, sd.materials, max_prims=1, builder=builder)
    return sc, oracle.PreparedScene(sd, *sc.bvh())


def _check_queries(sc, ps, oracle, rays, min_hits):
    import torch
    n = len(rays)
    r = torch.from_numpy(rays).cuda()
    h = torch.empty((n, 4), dtype=torch.float32, device="cuda")
    occ = torch.empty(n, dtype=torch.uint8, device="cuda")
    for two_sided in (False, True):
        print(n, "rays, two-sided" if two_sided else "rays", flush=True)
        sc.trace_closest(r, h, two_sided)
        torch.cuda.synchronize()
        g = h.cpu().numpy()
        t, u, v, i = oracle.trace_closest(ps.nodes, ps.tris_ordered(), rays, two_sided=two_sided)
        assert np.array_equal(g[:, 3].view(np.int32), i)
        hit = i >= 0
        assert hit.sum() >= min_hits
        for a, b in ((g[:, 0], t), (g[:, 1], u), (g[:, 2], v)):
            assert np.array_equal(a[hit].view(np.uint32), b[hit].view(np.uint32))
    print(n, "rays, any hit", flush=True)
    sc.trace_any(r, occ)
    torch.cuda.synchronize()
    assert np.array_equal(occ.cpu().numpy(), oracle.trace_any(ps.nodes, ps.tris_ordered(), rays))


@pytest.mark.parametrize("n", [1, 63, 2047, 2048, 16384, 16831, 20000, 63487, 63488, 65537, QUAD_MAX + 1])
def test_every_ray_meets_two_triangles_at_once(gpu, oracle, n):
    pos, nrm, uv = _chain(140)
    base = scenes.spheres_scene(8, 8, 1, 1, segments=4, rings=3)
    sd = _doubled(base, pos, nrm, uv, np.zeros(len(pos), np.int32))
    sc, ps = _create(gpu, oracle, sd, abi.FF_BVH_PLOC)
    assert sc.max_depth > 64
    rng = np.random.default_rng(n)
    tri = pos[rng.integers(0, 50, n)]  # (farther ones overflow)
    w = rng.dirichlet((4.0, 4.0, 4.0), n)
    target = np.einsum("nk,nkc->nc", w, tri.astype(np.float64))
    front = np.cross(tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0])[:, 0] > 0
    d = np.zeros((n, 3))
    d[:, 0] = np.where(front, -1.0, 1.0)
    d[:, 1:] = rng.uniform(-1e-3, 1e-3, (n, 2))
    rays = np.zeros((n, 8), np.float32)
    rays[:, 0:3], rays[:, 4:7] = target - 0.002 * d, d
    _check_queries(sc, ps, oracle, rays, int(0.9 * n))
    sc.close()


@pytest.mark.parametrize("deep,n", [(True, 3000), (True, 20000), (True, 63487), (False, QUAD_MAX + 257)])
def test_box_plane_distances_that_are_nan(gpu, oracle, deep, n):
    base = scenes.spheres_scene(8, 8, 1, 1, segments=16, rings=8)
    sd = base
    if deep:
        pos, nrm, uv = _chain(140)
        pos = pos + np.float32(50.0)
        sd = dataclasses.replace(base, positions=np.concatenate([base.positions, pos]),
                                 normals=np.concatenate([base.normals, nrm]), uvs=np.concatenate([base.uvs, uv]),
                                 material_ids=np.concatenate([base.material_ids, np.zeros(len(pos), np.int32)]))
    sc, ps = _create(gpu, oracle, sd, abi.FF_BVH_PLOC if deep else abi.FF_BVH_SAH)
    nodes, _ = sc.bvh()
    assert not deep or sc.max_depth > 64
    near = np.nonzero((np.abs(nodes["bmin"]).max(1) < 20) & (np.abs(nodes["bmax"]).max(1) < 20))[0]
    rng = np.random.default_rng(n)
    box = nodes[near[rng.integers(0, len(near), n)]]
    lo, hi = box["bmin"], box["bmax"]
    rays = np.zeros((n, 8), np.float32)
    rays[:, :3] = (lo + rng.random((n, 3)) * (hi - lo)).astype(np.float32)
    d = rng.normal(size=(n, 3)).astype(np.float32)
    a = np.where(rng.random(n) < 0.8, 0, rng.integers(0, 3, n))  # (x decides: the others' NaNs are dropped)
    k = np.arange(n)
    rays[k, a] = np.where(rng.random(n) < 0.5, lo[k, a], hi[k, a])  # on the box's plane
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    d[k, a] = np.where(rng.random(n) < 0.5, 0.0, -0.0)  # parallel to it
    rays[:, 4:7] = d
    _check_queries(sc, ps, oracle, rays, n // 20)
    sc.close()


def test_render_of_a_doubled_surface_in_a_deep_tree(gpu, oracle):
    import torch
    base = scenes.spheres_scene(160, 128, 1, 3, segments=12, rings=6)
    pos, nrm, uv = _chain(140)
    pos = pos + np.float32(20.0)  # behind the camera
    sd = _doubled(base, np.concatenate([base.positions, pos]), np.concatenate([base.normals, nrm]),
                  np.concatenate([base.uvs, uv]), np.concatenate([base.material_ids, np.zeros(len(pos), np.int32)]))
    sc, ps = _create(gpu, oracle, sd, abi.FF_BVH_PLOC)
    assert sc.max_depth > 64
    env, cam = abi.EnvMap(gpu, sd.env), abi.make_camera(sd.inv_vp)
    for flags in (0, abi.FF_RENDER_TIMING):
        f = torch.zeros((sd.height, sd.width, 4), dtype=torch.float32, device="cuda")
        print("render, flags", flags, flush=True)
        abi.render(gpu, sc, env, cam, sd.width, sd.height, 1, 3, 5, f, flags=flags)
        st = abi.last_render_stats(gpu)
        with oracle.env_tables(*env.read()[:4]):
            ref, cst = ps.render(spp=1, max_depth=3, seed=5)
        assert np.array_equal(f.cpu().numpy(), ref)
        for k in ("rays_primary", "rays_extension", "rays_shadow", "rays_shadow_gated", "paths"):
            assert getattr(st, k) == getattr(cst, k), k
    sc.close()
    env.close()
