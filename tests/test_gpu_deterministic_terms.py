"""The deterministic gradients keep every term apart: a vertex's light-sample
gradient and its continuation's go into the 64-bit sums one by one, although
they share a texel and an atomic.  Their bits are pinned: the file holds the
gradients of a renderer with an atomic for every term (parity unpinned by the
reference, which has no adjoint).  Adding the two terms in FP32 first moves the
last bits of the albedo and roughness gradients."""
import json
import os

import numpy as np
import pytest

from firefly_amd import abi, scenes

pytestmark = pytest.mark.gpu

GOLDEN = os.path.join(os.path.dirname(__file__), "golden", "adjoint_deterministic.json")
CASES = [(33, 17, 3, 4, 8), (160, 120, 2, 3, 5)]


def gradients(ctx, w, h, spp, depth, tex, flags=0):
    """Deterministic gradients of the albedo texture, the roughness texture and
    the environment: a mixed and a conductor material beside diffuse ones."""
    import torch
    sd = scenes.textured_spheres_scene(width=w, height=h, spp=spp, max_depth=depth, tex_size=tex, env_w=16, env_h=8,
                                       segments=16, rings=8)
    rng = np.random.default_rng(7)
    sd.textures = [*sd.textures, rng.uniform(0.2, 0.9, (tex, tex)).astype(np.float32)]
    mats = sd.materials.copy()
    mats[1:, 0] = np.resize([abi.FF_MAT_MIX, abi.FF_MAT_CONDUCTOR, abi.FF_MAT_DIFFUSE], len(mats) - 1)
    mats[1:, 11] = 1  # roughness texture
    sc = abi.Scene(ctx, sd.positions, sd.normals, sd.uvs, sd.material_ids, mats, textures=sd.textures)
    env, cam = abi.EnvMap(ctx, sd.env), abi.make_camera(sd.inv_vp)
    film = torch.zeros((h, w, 4), dtype=torch.float32, device="cuda")
    paths = torch.zeros((spp, h, w, 4), dtype=torch.float32, device="cuda")
    abi.render_paths(ctx, sc, env, cam, w, h, spp, depth, 3, film, paths)
    d = torch.from_numpy(rng.normal(size=(h, w, 4)).astype(np.float32)).cuda()
    g_env = torch.zeros(sd.env.shape, dtype=torch.float32, device="cuda")
    g_tex = [torch.zeros(t.shape, dtype=torch.float32, device="cuda") for t in sd.textures]
    abi.adjoint(ctx, sc, env, cam, w, h, spp, depth, 3, paths, d, env_grad=g_env, tex_grads=g_tex,
                flags=flags | abi.FF_ADJOINT_DETERMINISTIC)
    torch.cuda.synchronize()
    sc.close()
    env.close()
    return {"albedo": g_tex[0].cpu().numpy(), "roughness": g_tex[1].cpu().numpy(), "env": g_env.cpu().numpy()}


@pytest.mark.parametrize("flags", [0, abi.FF_RENDER_TIMING], ids=["one_launch", "stages"])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_terms_stay_apart(gpu, case, flags):
    with open(GOLDEN) as f:
        want = json.load(f)[case]
    got = gradients(gpu, *CASES[case], flags)
    for k, g in got.items():
        assert np.any(g != 0)
        assert g.ravel().view(np.uint32).tolist() == want[k], k
