"""Every traversal variant against the oracle, on traces that ask for counts
(only those run the variants' kernels): closest hits with and without culling
and any hits, bit for bit, on a flat scene, on a mesh whose stacks leave the
smaller LDS stacks and on a tree of depth > 64; and the no-allocation query,
counted and not, on both of its kernels."""
import numpy as np
import pytest

from firefly_amd import abi, scenes

pytestmark = pytest.mark.gpu

VARIANTS = 27


def _chain(n):
    """Triangles along a line, each 1.5x farther: PLOC makes a tree of depth > 64."""
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


@pytest.fixture(scope="module", params=["spheres", "mesh", "chain"])
def traced(request, gpu, oracle):
    """A scene, rays, and the oracle's answers to them."""
    import dataclasses
    if request.param == "mesh":
        sd = scenes.icosphere_scene(width=8, height=8, subdiv=6)
        rays = scenes.random_rays(30001, 21)
    else:
        sd = scenes.spheres_scene()
        rays = scenes.random_rays(30001, 4)
    kw = {}
    if request.param == "chain":
        pos, nrm, uv = _chain(140)
        sd = dataclasses.replace(sd, positions=pos, normals=nrm, uvs=uv, material_ids=np.zeros(140, np.int32))
        kw = {"max_prims": 1, "builder": abi.FF_BVH_PLOC}
        rng = np.random.default_rng(8)
        k = rng.integers(0, 50, 30001)  # (edge products of farther ones overflow)
        target = np.einsum("nk,nkc->nc", rng.dirichlet((1.0, 1.0, 1.0), 30001), pos[k].astype(np.float64))
        d = rng.normal(size=(30001, 3))
        rays[:, 0:3], rays[:, 4:7] = target - 0.5 * d, d
        rays[::5, 4:7] *= -1.0  # (away from the triangle)
    else:  # from the surfaces: the pruning behind the origin
        first = oracle.PreparedScene(sd)
        t, _, _, i = oracle.trace_closest(first.nodes, first.tris_ordered(), rays)
        on = np.nonzero(i >= 0)[0][::2]
        rays[on, 0:3] += rays[on, 4:7] * t[on, None]
    sc = abi.Scene(gpu, sd.positions, sd.normals, sd.uvs, sd.material_ids, sd.materials, **kw)
    ps = oracle.PreparedScene(sd, *sc.bvh())
    if request.param == "chain":
        assert sc.max_depth > 64
    tris = ps.tris_ordered()
    want = {two: oracle.trace_closest(ps.nodes, tris, rays, two_sided=two) for two in (False, True)}
    occ = oracle.trace_any(ps.nodes, tris, rays)
    assert (want[False][3] >= 0).sum() > 1000 and 0 < occ.sum() < len(rays)
    yield sc, rays, want, occ
    sc.close()


def _same_hits(g, want):
    t, u, v, i = want
    assert np.array_equal(g[:, 3].view(np.int32), i)
    hit = i >= 0
    for a, b in ((g[:, 0], t), (g[:, 1], u), (g[:, 2], v)):
        assert np.array_equal(a[hit].view(np.uint32), b[hit].view(np.uint32))


@pytest.mark.parametrize("variant", range(VARIANTS))
def test_counted_hits(gpu, traced, variant):
    import torch
    assert len(abi.traversal_variants()) == VARIANTS
    sc, rays, want, occ = traced
    r = torch.from_numpy(rays).cuda()
    h = torch.empty((len(rays), 4), dtype=torch.float32, device="cuda")
    o = torch.empty(len(rays), dtype=torch.uint8, device="cuda")
    abi.set_traversal_variant(gpu, variant)
    try:
        for two in (False, True):
            cnt = torch.zeros(2, dtype=torch.int64, device="cuda")
            h.fill_(7.0)
            sc.trace_closest(r, h, two, counts_dev=cnt)
            torch.cuda.synchronize()
            _same_hits(h.cpu().numpy(), want[two])
            assert bool((cnt > 0).all())
        cnt = torch.zeros(2, dtype=torch.int64, device="cuda")
        sc.trace_any(r, o, counts_dev=cnt)
        torch.cuda.synchronize()
        assert np.array_equal(o.cpu().numpy(), occ)
        assert bool((cnt > 0).all())
    finally:
        abi.set_traversal_variant(gpu, 0)


@pytest.mark.parametrize("counted", [False, True])
@pytest.mark.parametrize("variant", [0, 12, 23])
def test_noalloc_hits(gpu, traced, variant, counted):
    import torch
    sc, rays, want, _ = traced
    r = torch.from_numpy(rays).cuda()
    h = torch.full((len(rays), 4), 7.0, dtype=torch.float32, device="cuda")
    cnt = torch.zeros(2, dtype=torch.int64, device="cuda") if counted else None
    abi.set_traversal_variant(gpu, variant)
    try:
        if sc.max_depth > 39:  # deeper than the fixed scratch
            with pytest.raises(abi.FFError) as e:
                sc.trace_closest_noalloc(r, h, False, cnt)
            assert e.value.status == 5
            return
        sc.trace_closest_noalloc(r, h, False, cnt)
        torch.cuda.synchronize()
    finally:
        abi.set_traversal_variant(gpu, 0)
    _same_hits(h.cpu().numpy(), want[False])
