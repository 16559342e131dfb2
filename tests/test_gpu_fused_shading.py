"""Routing and shading in one launch against the same stages in launches of
their own (per-launch timing asks for those): every film value and ray count is
the same, at the limit between its two forms, at tile and chunk edges, with
paths left over from one tile to the next, with one and with all material
types, and with scenes that differ between requests.  Likewise the adjoint's
replay, whose vertices wait for their shadow rays until the next extension rays
are traced with them: its deterministic sums are the same either way."""
import numpy as np
import pytest

from firefly_amd import abi, scenes

pytestmark = pytest.mark.gpu

SMALL = 384 * 1024  # paths in flight of the largest call that takes 256-path tiles
COUNTS = ("rays_primary", "rays_extension", "rays_shadow", "paths")


def _scene(gpu, width, height, depth, seed, types):
    sd = scenes.spheres_scene(width=width, height=height, spp=1, max_depth=depth, seed=seed, segments=16, rings=8)
    mats = sd.materials.copy()
    mats[:, 0] = np.resize(types, len(mats))
    mats[mats[:, 0] == abi.FF_MAT_CONDUCTOR, 5] = 1.0
    sc = abi.Scene(gpu, sd.positions, sd.normals, sd.uvs, sd.material_ids, mats)
    return sc, abi.EnvMap(gpu, sd.env), abi.make_camera(sd.inv_vp)


def _render(gpu, items, k, flags):
    import torch
    films = [torch.zeros((h, w, 4), dtype=torch.float32, device="cuda") for _, _, _, w, h, *_ in items]
    abi.render_batch(gpu, [(*it, f) for it, f in zip(items, films)], flags=flags, spp_batch=k)
    torch.cuda.synchronize()
    st = abi.last_render_stats(gpu)
    return [f.cpu().numpy() for f in films], [getattr(st, c) for c in COUNTS]


ALL = [abi.FF_MAT_MIX, abi.FF_MAT_DIFFUSE, abi.FF_MAT_CONDUCTOR, abi.FF_MAT_DIELECTRIC]
CASES = [
    (1, 1, 1, 1, 3, ALL), (51, 5, 1, 1, 3, ALL), (257, 1, 1, 2, 4, [abi.FF_MAT_DIFFUSE]),
    (63, 31, 3, 5, 5, ALL), (512, 768, 1, 1, 4, ALL), (1024, 384, 1, 1, 3, [abi.FF_MAT_CONDUCTOR]),
    (SMALL + 1, 1, 1, 1, 4, ALL), (1031, 577, 2, 4, 5, ALL), (1031, 577, 2, 2, 2, [abi.FF_MAT_MIX]),
]


@pytest.mark.parametrize("width,height,k,spp,depth,types", CASES)
def test_one_launch_equals_stage_launches(gpu, width, height, k, spp, depth, types):
    sc, env, cam = _scene(gpu, width, height, depth, 11, types)
    items = [(sc, env, cam, width, height, spp, depth, 5)]
    films, counts = _render(gpu, items, k, 0)
    want, want_counts = _render(gpu, items, k, abi.FF_RENDER_TIMING)
    assert np.array_equal(films[0], want[0])
    assert counts == want_counts
    assert np.all(films[0][..., 3] == spp)


@pytest.mark.parametrize("sizes,k", [([(40, 31), (17, 9), (64, 64)], 2), ([(700, 500), (333, 777)], 1)])
def test_one_launch_equals_stage_launches_of_several_scenes(gpu, sizes, k):
    items = []
    for i, (w, h) in enumerate(sizes):
        types = [ALL, [abi.FF_MAT_DIFFUSE], ALL[::-1]][i]
        items.append((*_scene(gpu, w, h, 3 + i, i, types), w, h, 2, 3 + i, 7 + i))
    films, counts = _render(gpu, items, k, 0)
    want, want_counts = _render(gpu, items, k, abi.FF_RENDER_TIMING)
    for f, g in zip(films, want):
        assert np.array_equal(f, g)
    assert counts == want_counts


@pytest.mark.parametrize("types", [ALL, [abi.FF_MAT_DIFFUSE], [abi.FF_MAT_MIX, abi.FF_MAT_DIELECTRIC]])
@pytest.mark.parametrize("width,height,k,spp,depth", [(33, 17, 2, 3, 4), (512, 300, 1, 2, 3), (5, 1, 1, 1, 1)])
def test_replay_with_rays_traced_together(gpu, width, height, k, spp, depth, types):
    import torch
    sd = scenes.textured_spheres_scene(width=width, height=height, spp=spp, max_depth=depth, tex_size=16, env_w=32,
                                       env_h=16, segments=16, rings=8)
    mats = sd.materials.copy()
    mats[:, 0] = np.resize(types, len(mats))
    sc = abi.Scene(gpu, sd.positions, sd.normals, sd.uvs, sd.material_ids, mats, textures=sd.textures)
    env, cam = abi.EnvMap(gpu, sd.env), abi.make_camera(sd.inv_vp)
    paths = torch.zeros((spp, height, width, 4), dtype=torch.float32, device="cuda")
    film = torch.zeros((height, width, 4), dtype=torch.float32, device="cuda")
    abi.render_paths(gpu, sc, env, cam, width, height, spp, depth, 5, film, paths, spp_batch=k)
    d = torch.from_numpy(np.random.default_rng(1).normal(size=(height, width, 4)).astype(np.float32)).cuda()
    out = []
    for flags in (0, abi.FF_RENDER_TIMING):
        g_env = torch.zeros(sd.env.shape, dtype=torch.float32, device="cuda")
        g_tex = [torch.zeros(t.shape, dtype=torch.float32, device="cuda") for t in sd.textures]
        abi.adjoint(gpu, sc, env, cam, width, height, spp, depth, 5, paths, d, env_grad=g_env, tex_grads=g_tex,
                    flags=flags | abi.FF_ADJOINT_DETERMINISTIC, spp_batch=k)
        torch.cuda.synchronize()
        st = abi.last_render_stats(gpu)
        out.append([g_env.cpu().numpy(), *(t.cpu().numpy() for t in g_tex), [getattr(st, c) for c in COUNTS]])
    for a, b in zip(*out):
        assert np.array_equal(a, b)
    assert np.any(out[0][0] != 0)


@pytest.mark.parametrize("width,height,k", [(SMALL // 512, 512, 1), (SMALL // 512 + 1, 512, 1), (1031, 400, 2)])
def test_replay_forms_by_paths_in_flight(gpu, width, height, k):
    """The replay's one-launch forms on either side of their limit, with paths
    left over between tiles, of several scenes: deterministic sums as apart."""
    import torch
    depth, spp = 3, k
    d = torch.from_numpy(np.random.default_rng(2).normal(size=(height, width, 4)).astype(np.float32)).cuda()
    items, paths, grads = [], [], []
    for i, (w, h) in enumerate([(width, height), (40, 30)]):
        sc, env, cam = _scene(gpu, w, h, depth, i, ALL)
        film = torch.zeros((h, w, 4), dtype=torch.float32, device="cuda")
        items.append((sc, env, cam, w, h, spp, depth, 5 + i, film))
        paths.append(torch.zeros((spp, h, w, 4), dtype=torch.float32, device="cuda"))
    abi.render_batch(gpu, items, path_radiance=paths, spp_batch=k)
    out = []
    for flags in (0, abi.FF_RENDER_TIMING):
        grads = [torch.zeros((it[1].hgt, it[1].w, 3), dtype=torch.float32, device="cuda") for it in items]
        abi.adjoint_batch(gpu, items, paths, [d, d[:30, :40].contiguous()], env_grads=grads,
                          flags=flags | abi.FF_ADJOINT_DETERMINISTIC, spp_batch=k)
        torch.cuda.synchronize()
        st = abi.last_render_stats(gpu)
        out.append([*(g.cpu().numpy() for g in grads), [getattr(st, c) for c in COUNTS]])
    for a, b in zip(*out):
        assert np.array_equal(a, b)
    assert np.any(out[0][0] != 0) and np.any(out[0][1] != 0)
