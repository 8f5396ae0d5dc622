"""The wave's segments are tested against triangles together: lists longer
than a wave, equal parameters (every triangle twice, under two ids: the first
one counts), partial waves and waves with few segments give the oracle's hit
per segment, bit for bit."""
import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("shape", [(2, 2, 2), (9, 8, 11)])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 2500])
@pytest.mark.parametrize("few", [False, True])
def test_wave_detect_matches_oracle(shape, n, few):
    from psum_amd import mesh as Mh
    noz = Mh.revolve_zr_curve([(-4, 1.0), (-2, 0.6), (-1, 0.6), (1, 1.4), (4, 2.0)], 12)
    cube = Mh.axis_aligned_cube(-5, -5, -5, 5, 5, 10)
    meshes = [(noz, 1), (cube, 0), (noz, 2), (cube, 3)]
    tri = np.concatenate([np.asarray(t).reshape(-1, 9) for t, _ in meshes])
    ids = np.concatenate([np.full(len(np.asarray(t).reshape(-1, 9)), i, np.int32) for t, i in meshes])
    tm = Mh.TriangleMesh(meshes, *shape)
    om = O.OracleMesh(tri, ids, *shape)
    rng = np.random.default_rng(n)
    p1 = rng.uniform([-4.9, -4.9, -4.9], [4.9, 4.9, 9.9], (n, 3))
    p2 = p1 + rng.normal(0, 2.0, (n, 3))
    if few:
        p1[np.arange(n) % 17 != 0, 2] = np.nan
    dev = [[torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in p.T] for p in (p1, p2)]
    k, nrm, idt = (t.cpu().numpy() for t in tm.detect(*dev))
    for i in range(n):
        if not np.isfinite(p1[i]).all():
            assert idt[i] == -1
            continue
        h, kk, nn, mid = om.detect(p1[i], p2[i], fast=False)
        assert (idt[i] >= 0) == h, i
        if h:
            assert k[i] == kk and idt[i] == mid and np.array_equal(nrm[i], nn), i
    tm.close()
