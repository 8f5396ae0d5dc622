"""BoundaryRouter.deal tests the segments of a wave against triangles together
(one lane per particle and triangle): lists longer than a wave, equal
parameters (every triangle twice, under two ids: the first one counts),
partial waves, waves with few segments and more particles than one round of
blocks give the oracle's hits, seeds and material actions.  TriangleMesh.detect
(a segment per lane) gives the same hits on the same scenes."""
import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _scene():
    from psum_amd import mesh as Mh
    noz = Mh.revolve_zr_curve([(-4, 1.0), (-2, 0.6), (-1, 0.6), (1, 1.4), (4, 2.0)], 12)
    cube = Mh.axis_aligned_cube(-5, -5, -5, 5, 5, 10)
    meshes = [(noz, 1), (cube, 0), (noz, 2), (cube, 3)]
    tri = np.concatenate([np.asarray(t).reshape(-1, 9) for t, _ in meshes])
    ids = np.concatenate([np.full(len(np.asarray(t).reshape(-1, 9)), i, np.int32) for t, i in meshes])
    return meshes, tri, ids


def _segments(n, few):
    rng = np.random.default_rng(n)
    p1 = rng.uniform([-4.9, -4.9, -4.9], [4.9, 4.9, 9.9], (n, 3))
    p2 = p1 + rng.normal(0, 2.0, (n, 3))
    if few:
        p1[np.arange(n) % 17 != 0, 2] = np.nan
    return p1, p2


def _cuda(arrays):
    return [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in arrays]


@pytest.mark.parametrize("shape", [(2, 2, 2), (9, 8, 11)])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 2500])
@pytest.mark.parametrize("few", [False, True])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_wave_boundary_matches_oracle(shape, n, few, dtype):
    from psum_amd import mesh as Mh
    meshes, tri, ids = _scene()
    router = Mh.BoundaryRouter(temperature=300.0, mass=6.67e-27).set(meshes, *shape)
    om = O.OracleMesh(tri, ids, *shape)
    if shape == (2, 2, 2):
        assert np.diff(om.cell_start.astype(np.int64)).max() > 64
    p1, p2 = (p.astype(dtype).T for p in _segments(n, few))
    rng = np.random.default_rng(n + 1)
    vel = rng.normal(0, 1.0, (3, n)).astype(dtype)
    seed = rng.integers(0, 2**32, n, dtype=np.uint64).astype(np.uint32)
    ref = om.boundary(list(p1), list(p2), list(vel), seed, temperature=300.0, mass=6.67e-27)
    gold, gp, gv = _cuda(p1), _cuda(p2), _cuda(vel)
    gs = torch.from_numpy(seed.view(np.int32).copy()).cuda()
    hits, hid = router.deal(gold, gp, gv, gs, hit_id=True)
    assert hits == ref["hits"] and np.array_equal(hid.cpu().numpy(), ref["hit_id"])
    assert n < 2500 or hits > (20 if few else 500)
    assert np.array_equal(gs.cpu().numpy().view(np.uint32), ref["seed"])
    # the actions' sqrt, log and trigonometric functions differ in the last
    # places of FP64: 1e-12, or one FP32 rounding
    speed = np.sqrt(sum(x.astype(np.float64) ** 2 for x in ref["vel"]))
    for c in range(3):
        a, b = gp[c].cpu().numpy(), ref["pos"][c]
        assert np.array_equal(np.isnan(a), np.isnan(b))
        m = ~np.isnan(b)
        tol = 1e-12 * (1 + np.abs(b[m])) if dtype == np.float64 else np.spacing(np.abs(b[m]))
        assert np.all(np.abs(a[m] - b[m]) <= tol), c
        va, vb = gv[c].cpu().numpy(), ref["vel"][c]
        tolv = 1e-12 * speed if dtype == np.float64 else np.spacing(np.abs(vb))
        assert np.all(np.abs(va - vb) <= tolv), c
    router.trigger.close()


def test_more_particles_than_one_round_of_blocks():
    """8192 blocks of 256 walk the particles: beyond 2^21 of them each block
    takes several batches.  The same particles in calls of one batch each give
    the same bits."""
    from psum_amd import mesh as Mh
    meshes, _, _ = _scene()
    router = Mh.BoundaryRouter(temperature=300.0, mass=6.67e-27).set(meshes, 9, 8, 11)
    n, part = (1 << 21) + 5001, 1 << 20
    p1, p2 = (p.T for p in _segments(n, False))
    vel = np.random.default_rng(2).normal(0, 1.0, (3, n))
    seed = np.arange(n, dtype=np.int32)

    def deal(s):
        a = [_cuda(x[:, s]) for x in (p1, p2, vel)]
        sd = torch.from_numpy(seed[s].copy()).cuda()
        hits, hid = router.deal(*a, sd, hit_id=True)
        return hits, [hid, sd] + [torch.nan_to_num(t, nan=-99.0) for t in a[1] + a[2]]
    hits, whole = deal(slice(0, n))
    pieces = [deal(slice(i, min(i + part, n))) for i in range(0, n, part)]
    assert hits == sum(p[0] for p in pieces) and hits > n // 5
    for k, t in enumerate(whole):
        assert torch.equal(t, torch.cat([p[1][k] for p in pieces]))
    router.trigger.close()


@pytest.mark.parametrize("shape", [(2, 2, 2), (9, 8, 11)])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 2500])
@pytest.mark.parametrize("few", [False, True])
def test_detect_matches_oracle(shape, n, few):
    from psum_amd import mesh as Mh
    meshes, tri, ids = _scene()
    tm = Mh.TriangleMesh(meshes, *shape)
    om = O.OracleMesh(tri, ids, *shape)
    p1, p2 = _segments(n, few)
    k, nrm, idt = (t.cpu().numpy() for t in tm.detect(_cuda(p1.T), _cuda(p2.T)))
    for i in range(n):
        if not np.isfinite(p1[i]).all():
            assert idt[i] == -1
            continue
        h, kk, nn, mid = om.detect(p1[i], p2[i], fast=False)
        assert (idt[i] >= 0) == h, i
        if h:
            assert k[i] == kk and idt[i] == mid and np.array_equal(nrm[i], nn), i
    tm.close()
