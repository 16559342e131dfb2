"""The autotuner times what each setting decides: renders for the samples in
flight, counted traces for the traversal variant; a render's film does not
depend on what it found."""
import json

import pytest

from firefly_amd import abi, autotune, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("refine_spp", [0, 4])
def test_each_setting_is_timed_by_what_reads_it(gpu, monkeypatch, tmp_path, refine_spp):
    import torch
    sd = scenes.spheres_scene(width=64, height=48, spp=4, max_depth=3, segments=12, rings=6)
    sc = abi.Scene(gpu, sd.positions, sd.normals, sd.uvs, sd.material_ids, sd.materials)
    env, cam = abi.EnvMap(gpu, sd.env), abi.make_camera(sd.inv_vp)
    renders, traced, current = [], set(), [None]
    render, set_variant, trace = abi.render, abi.set_traversal_variant, abi.Scene.trace_closest
    monkeypatch.setattr(abi, "render", lambda *a, **k: (renders.append(k.get("spp_batch")), render(*a, **k)))
    monkeypatch.setattr(abi, "set_traversal_variant", lambda c, v: (current.__setitem__(0, v), set_variant(c, v)))

    def counted(self, rays, hits, two_sided=False, counts_dev=None, stream=None):
        assert counts_dev is not None and rays.shape[0] == 64 * 48
        traced.add(current[0])
        trace(self, rays, hits, two_sided, counts_dev, stream)

    monkeypatch.setattr(abi.Scene, "trace_closest", counted)
    path = str(tmp_path / "tuned.json")
    try:
        out = autotune.autotune(gpu, sc, env, cam, 64, 48, 3, probe_spp=2, batches=(1, 2), refine_batches=(4, 8),
                                refine_spp=refine_spp, reps=2, tail_candidates=(0, 1), out_json=path)
        best = out["best"]
        ks = [1, 2, 4] if refine_spp else [1, 2]
        assert renders[1:] == [k for k in ks for _ in range(2)]  # (the first: warm-up)
        assert [c["spp_batch"] for c in out["candidates"]] == ks
        assert best["seconds"] == min(c["seconds"] for c in out["candidates"])
        assert traced == {v[0] for v in abi.traversal_variants()}
        assert best["variant"] == current[0] == min(out["traces"], key=lambda t: t["seconds"])["variant"]
        assert best.get("tail_variant", -1) == -1
        assert json.load(open(path)) == out
    finally:
        set_variant(gpu, 0)
    film = torch.zeros((48, 64, 4), dtype=torch.float32, device="cuda")
    render(gpu, sc, env, cam, 64, 48, 4, 3, 0, film, spp_batch=best["spp_batch"])
    torch.cuda.synchronize()
    assert bool((film[..., 3] == 4).all())
    sc.close()
    env.close()
