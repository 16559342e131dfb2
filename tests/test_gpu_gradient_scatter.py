"""The adjoint's wave-cooperative gradient scatter against the oracle's FP64
adjoint at the sizes where footprints fold onto themselves or leave a wave
partly filled: textures of one to five texels a side (every footprint wraps),
images of fewer paths than a wave and of odd size, with FP32 atomics and with
the deterministic sums.  Tolerance as for the other adjoint tests: relative L2
error over all texels of a target at most 1e-3."""
import numpy as np
import pytest

from firefly_amd import abi, scenes
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _near(a, b):  # (a target that no path reaches has no gradient on either side)
    return np.linalg.norm((a - b).ravel()) <= 1e-3 * np.linalg.norm(b.ravel())


@pytest.mark.parametrize("flags", [0, abi.FF_ADJOINT_DETERMINISTIC], ids=["atomics", "deterministic"])
@pytest.mark.parametrize("w,h,spp,tex,env", [(7, 9, 1, 1, (4, 2)), (61, 33, 2, 5, (5, 3)), (64, 64, 3, 2, (16, 8))])
def test_scatter_matches_fp64_oracle(gpu, w, h, spp, tex, env, flags):
    import torch
    sd = scenes.textured_spheres_scene(width=w, height=h, spp=spp, max_depth=3, tex_size=tex, env_w=env[0],
                                       env_h=env[1], segments=16, rings=8)
    ps = O.PreparedScene(sd)
    rng = np.random.default_rng(w)
    d = rng.normal(size=(h, w, 3)).astype(np.float32) / (w * h)
    sc = abi.Scene(gpu, sd.positions, sd.normals, sd.uvs, sd.material_ids, sd.materials, textures=sd.textures)
    e = abi.EnvMap(gpu, sd.env)
    cam = abi.make_camera(sd.inv_vp)
    film = torch.zeros((h, w, 4), dtype=torch.float32, device="cuda")
    paths = torch.zeros((spp, h, w, 4), dtype=torch.float32, device="cuda")
    abi.render_paths(gpu, sc, e, cam, w, h, spp, 3, sd.seed, film, paths, spp_batch=spp)
    dd = torch.zeros((h, w, 4), dtype=torch.float32, device="cuda")
    dd[..., :3] = torch.from_numpy(d).cuda()
    g_env = torch.zeros(sd.env.shape, dtype=torch.float32, device="cuda")
    g_tex = torch.zeros(sd.textures[0].shape, dtype=torch.float32, device="cuda")
    abi.adjoint(gpu, sc, e, cam, w, h, spp, 3, sd.seed, paths, dd, env_grad=g_env, tex_grads=[g_tex], flags=flags,
                spp_batch=spp)
    torch.cuda.synchronize()
    _, r_env, r_tex = ps.adjoint(d)
    assert _near(g_env.cpu().numpy(), r_env)
    assert _near(g_tex.cpu().numpy(), r_tex[0])
    sc.close()
    e.close()
