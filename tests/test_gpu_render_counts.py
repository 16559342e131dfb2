"""Boxes and triangles in a render's statistics: four boxes a record of the wide
walk, and what a ray traced again in the reference's order tests.  Every camera
ray that hits a surface which lies twice in the scene is traced again: one
triangle pair in one leaf, whose root record holds both, with four lanes and
with one lane to a ray (FF_RENDER_TIMING: the kinds of rays apart)."""
import dataclasses

import numpy as np
import pytest

from firefly_amd import abi, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h", [(64, 48), (512, 400)], ids=["four_lanes", "one_lane"])
@pytest.mark.parametrize("flags", [0, abi.FF_RENDER_TIMING])
def test_rays_traced_again_are_counted(gpu, w, h, flags):
    import torch
    base = scenes.spheres_scene(w, h, 1, 1)
    tri = np.array([[[-2.0, 0, -2.0], [-2.0, 0, 2.0], [2.0, 0, -2.0]]], np.float32)
    nrm = np.tile(np.float32([0, 1, 0]), (2, 3, 1))
    sd = dataclasses.replace(base, positions=np.repeat(tri, 2, 0), normals=nrm, uvs=np.zeros((2, 3, 2), np.float32),
                             material_ids=np.zeros(2, np.int32))
    sc = abi.Scene(gpu, sd.positions, sd.normals, sd.uvs, sd.material_ids, sd.materials)
    assert sc.n_nodes == 1
    env, cam = abi.EnvMap(gpu, sd.env), abi.make_camera(sd.inv_vp)
    rays = torch.empty((w * h, 8), dtype=torch.float32, device="cuda")
    hits = torch.empty((w * h, 4), dtype=torch.float32, device="cuda")
    abi.generate_rays(gpu, cam, w, h, 5, 0, rays)
    sc.trace_closest(rays, hits)
    film = torch.zeros((h, w, 4), dtype=torch.float32, device="cuda")
    abi.render(gpu, sc, env, cam, w, h, 1, 1, 5, film, flags=flags)
    st = abi.last_render_stats(gpu)
    hit = int((hits[:, 3].view(torch.int32) >= 0).sum())
    assert w * h // 20 < hit < w * h
    # a record a ray; for a ray traced again the root's box and its two triangles
    again = st.ext_nodes - 4 * (st.rays_primary + st.rays_extension)
    assert hit <= again <= st.rays_primary + st.rays_extension
    assert st.ext_tris >= 4 * hit
    # shadow rays start on the surface: none is traced again
    assert st.shadow_nodes == 4 * st.rays_shadow
    sc.close()
    env.close()
