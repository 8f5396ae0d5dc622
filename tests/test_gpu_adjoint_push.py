"""The adjoint push sums a block's gradient-weight deposit in an LDS tile
where the block's box fits it and adds to the accumulator directly where it
does not.  The sums are integers, so particles in cell order (tiles),
shuffled (direct adds) and taken from an odd address give the same
accumulator and the same adjoint state, bit for bit."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _push(g, dtype, x, lx, lv, phi, scale, offset):
    """psum_hip_adjoint_push on arrays that start `offset` values into their
    allocation; returns acc, lx, lv"""
    from psum_amd import _lib
    from psum_amd import engine as E
    D = g.dim

    def put(a):
        t = torch.empty(a.size + offset, dtype=torch.from_numpy(a).dtype, device="cuda")
        t[offset:] = torch.from_numpy(a).cuda()
        return t[offset:]
    xs, lxs, lvs = [put(a) for a in x], [put(a) for a in lx], [put(a) for a in lv]
    acc = torch.zeros(E.num_nodes(g), dtype=torch.int64, device="cuda")
    sc = torch.tensor([scale, 1.0 / scale, 0.0, 0.0], dtype=torch.float64, device="cuda")
    ph = torch.from_numpy(phi).cuda()
    ptr = [(C.c_void_p * 3)(*([t.data_ptr() for t in v] + [None] * (3 - D))) for v in (xs, lxs, lvs)]
    _lib.check(_lib.lib().psum_hip_adjoint_push(C.byref(g), dtype, ptr[0], ptr[1], ptr[2], x[0].size, ph.data_ptr(),
                                                -1.0, 0.1, sc.data_ptr(), acc.data_ptr(), None), "adjoint_push")
    torch.cuda.synchronize()
    return acc.cpu().numpy(), [t.cpu().numpy() for t in lxs], [t.cpu().numpy() for t in lvs]


# one particle, a block short of and beyond 1024, rows of more nodes than a
# tile holds with one column of drift, a seam; dtype 2: FP32 positions with
# an FP64 adjoint
@pytest.mark.parametrize("nodes,periodic,n", [((2100, 6), True, 4097), ((24, 40), True, 1), ((24, 40), True, 1023),
                                              ((33, 17), False, 5003), ((9, 7, 11), False, 3001),
                                              ((12, 10, 8), True, 2048)])
@pytest.mark.parametrize("dtype", [0, 1, 2])
def test_tile_and_direct_adds_agree(nodes, periodic, n, dtype):
    from psum_amd import _lib
    from psum_amd import engine as E
    code = dtype                       # PSUM_F64, PSUM_F32, PSUM_F32_ADJ64
    xt, at = [(np.float64, np.float64), (np.float32, np.float32), (np.float32, np.float64)][dtype]
    rng = np.random.default_rng(sum(nodes) + n)
    g = E.periodic_grid(list(nodes)) if periodic else E.wall_grid([m - 1 for m in nodes])
    ext = [m if periodic else m - 1 for m in nodes]
    x = [(rng.random(n) * L).astype(xt) for L in ext]
    order = np.lexsort([np.floor(a) for a in x[::-1]])
    x = [a[order] for a in x]
    if n > 8:
        x[0][3] = np.nan                     # an absorbed particle
    lx = [rng.standard_normal(n).astype(at) for _ in nodes]
    lv = [rng.standard_normal(n).astype(at) for _ in nodes]
    phi = rng.standard_normal(int(np.prod(nodes))).astype(at)
    ref = _push(g, code, x, lx, lv, phi, 2.0 ** 36, 0)
    off = _push(g, code, x, lx, lv, phi, 2.0 ** 36, 1)
    p = rng.permutation(n)
    mix = _push(g, code, [a[p] for a in x], [a[p] for a in lx], [a[p] for a in lv], phi, 2.0 ** 36, 0)
    assert np.array_equal(ref[0], off[0]) and np.array_equal(ref[0], mix[0])
    for q in (1, 2):
        for a, b, c in zip(ref[q], off[q], mix[q]):
            assert np.array_equal(a, b) and np.array_equal(a[p], c)

    # the accumulator against the deposit -qm dt sum_e lvt_e d_e c_i in FP64:
    # each particle adds at most 2^D terms rounded to 2^-36; FP32 terms carry
    # their own rounding
    D = len(nodes)
    lb = 0.5 if periodic else 0.0
    ok = np.isfinite(x[0])
    t = [a[ok].astype(np.float64) - lb for a in x]
    base = [np.floor(a) for a in t]
    s = [a - b for a, b in zip(t, base)]
    lvt = [(v[ok] + at(0.1) * a[ok]).astype(np.float64) for v, a in zip(lv, lx)]
    want = np.zeros(int(np.prod(nodes)))
    for k in range(1 << D):
        bit = [(k >> (D - 1 - d)) & 1 for d in range(D)]
        lin = np.zeros(t[0].size, np.int64)
        for d in range(D):
            lin = lin * nodes[d] + np.mod(base[d] + bit[d], nodes[d]).astype(np.int64)
        term = 0.0
        for e in range(D):
            c = lvt[e] * (1.0 if bit[e] else -1.0)
            for d in range(D):
                if d != e:
                    c = c * (s[d] if bit[d] else 1.0 - s[d])
            term = term + c
        np.add.at(want, lin, 0.1 * term)
    got = ref[0] * 2.0 ** -36
    tol = (n * 2.0 ** -36 + 1e-14 * n) if at is np.float64 else n * 1e-6
    assert np.abs(got - want).max() <= tol
