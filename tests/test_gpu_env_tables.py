"""Environment tables and their search guides where their one-pass build can
go wrong: fewer columns than threads, one column a thread and a column more,
runs that are no multiple of four, more rows than threads, rows that are black
but for one texel (all guide entries belong to one element), black at the
start or the end, or black altogether.  The oracle's render with the tables
read back searches them whole; the film is the same in every bit."""
import numpy as np
import pytest

from firefly_amd import abi, scenes

pytestmark = pytest.mark.gpu


def _env(w, h, kind):
    rgb = np.random.default_rng(w * 31 + h).uniform(0.1, 2.0, (h, w, 3)).astype(np.float32)
    if kind == "one_texel":  # (its neighbours take part: luminances are filtered)
        rgb[:] = 0.0
        rgb[h // 2, w // 3] = 50.0
    elif kind == "sun":
        rgb[h // 2, w // 3] = 1e6
    elif kind == "black_ends":
        rgb[:, : w // 3] = 0.0
        rgb[:, w - w // 4:] = 0.0
        rgb[h - 1] = 0.0
    return rgb


@pytest.mark.parametrize("kind", ["random", "one_texel", "sun", "black_ends"])
@pytest.mark.parametrize("w,h", [(2, 2), (3, 5), (255, 4), (256, 3), (257, 6), (1031, 9), (16, 1031), (2048, 8)])
def test_render_with_tables_read_back(gpu, oracle, w, h, kind):
    import torch
    sd = scenes.spheres_scene(width=24, height=16, spp=2, max_depth=3, segments=8, rings=4)
    sd.env = _env(w, h, kind)
    sc = abi.Scene(gpu, sd.positions, sd.normals, sd.uvs, sd.material_ids, sd.materials)
    env = abi.EnvMap(gpu, np.ones_like(sd.env))
    env.update(sd.env)
    film = torch.zeros((16, 24, 4), dtype=torch.float32, device="cuda")
    abi.render(gpu, sc, env, abi.make_camera(sd.inv_vp), 24, 16, 2, 3, sd.seed, film, spp_batch=2)
    ps = oracle.PreparedScene(sd, *sc.bvh())
    with oracle.env_tables(*env.read()[:4]):
        want, _ = ps.render(spp=2, max_depth=3, spp_batch=2)
    assert np.array_equal(film.cpu().numpy(), want, equal_nan=True)
    sc.close()
    env.close()
