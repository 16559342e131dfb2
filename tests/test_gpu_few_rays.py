"""Queries whose waves hold every ray at once and take theirs by number, at the
sizes where a wave's share changes, where the last wave has less than its share
or none, and at the limit beyond which the work counters hand rays out; each
after a query that left the counters used up.  Bit for bit the oracle's hits."""
import numpy as np
import pytest

from firefly_amd import abi, scenes

pytestmark = pytest.mark.gpu

# the chip's resident waves (256 CUs, 6 workgroups of 4) with 16 rays each
HELD = 256 * 6 * 4 * 16


@pytest.mark.parametrize("n", [1, 2, 1023, 1024, 1025, 2049, 16383, 16384, 16399, HELD - 1, HELD, HELD + 1, HELD + 17])
def test_rays_taken_by_number(gpu, oracle, n):
    import torch
    sd = scenes.spheres_scene(8, 8, 1, 1, segments=16, rings=8)
    sc = abi.Scene(gpu, sd.positions, sd.normals, sd.uvs, sd.material_ids, sd.materials)
    ps = oracle.PreparedScene(sd, *sc.bvh())
    many = torch.from_numpy(scenes.random_rays(140000, 3)).cuda()
    sc.trace_closest(many, torch.empty((len(many), 4), dtype=torch.float32, device="cuda"))
    rays = scenes.random_rays(n, n)
    r = torch.from_numpy(rays).cuda()
    h = torch.full((n, 4), 7.0, dtype=torch.float32, device="cuda")
    occ = torch.full((n,), 9, dtype=torch.uint8, device="cuda")
    sc.trace_closest(r, h)
    sc.trace_any(r, occ)
    torch.cuda.synchronize()
    g = h.cpu().numpy()
    t, u, v, i = oracle.trace_closest(ps.nodes, ps.tris_ordered(), rays)
    assert np.array_equal(g[:, 3].view(np.int32), i)
    hit = i >= 0
    for a, b in ((g[:, 0], t), (g[:, 1], u), (g[:, 2], v)):
        assert np.array_equal(a[hit].view(np.uint32), b[hit].view(np.uint32))
    assert np.array_equal(occ.cpu().numpy(), oracle.trace_any(ps.nodes, ps.tris_ordered(), rays))
    sc.close()
