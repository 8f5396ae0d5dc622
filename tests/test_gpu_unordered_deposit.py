"""Particles in no order: gather_push leaves the deposit of scattered blocks
to the per-domain kernel.  Sums are integers, so the accumulator, the
particles and the counters equal those of the call without workspace (block
tiles and direct adds), for any mix of ordered and unordered particles."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

N0 = 1 << 19           # the least particles the domains take


# one domain, several with a ragged last one, a plane near the tile's limit,
# walls (absorbed particles), and a row too long for a tile (no domains)
@pytest.mark.parametrize("nodes,periodic,dx", [((40, 30), True, 1.0), ((311, 257), True, 0.3), ((601, 400), False, 1.0),
                                               ((33, 40, 37), True, 0.5), ((9, 90, 88), False, 1.0),
                                               ((12, 14000), True, 1.0)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("n,ordered", [(N0, 0.0), (N0 - 1, 0.0), (N0 + 4097, 0.5), (N0 + 1, 1.0)])
def test_domains_equal_direct_adds(nodes, periodic, dx, dtype, n, ordered):
    from psum_amd import _lib
    from psum_amd import engine as E
    D = len(nodes)
    gen = torch.Generator(device="cuda").manual_seed(n + sum(nodes))
    g = E.periodic_grid(list(nodes), dx) if periodic else E.wall_grid([m - 1 for m in nodes], dx)
    ext = [m * dx if periodic else (m - 1) * dx for m in nodes]
    pos = [torch.rand(n, generator=gen, device="cuda", dtype=dtype) * L * 0.999999 for L in ext]
    k = int(n * ordered)
    if k:
        head = [a[:k].clone() for a in pos]
        keys, perm = E.stable_sort(E.cell_keys(g, head), E.num_nodes(g))
        for a, h in zip(pos, E.permute(head, perm)):
            a[:k] = h
    pos[0][::991] = float("nan")
    vel = [torch.randn(n, generator=gen, device="cuda", dtype=dtype) for _ in nodes]
    phi = torch.randn(E.num_nodes(g), generator=gen, device="cuda", dtype=dtype)
    wb = _lib.lib().psum_hip_gather_push_workspace(C.byref(g), n)
    assert (wb > 0) == (n >= N0 and nodes != (12, 14000))
    w, scale, code = -0.7, 2.0 ** 40, 1 if dtype == torch.float32 else 0
    p2, v2 = [a.clone() for a in pos], [a.clone() for a in vel]
    for cnt in (False, True):
        a, b = ([t.clone() for t in pos], [t.clone() for t in vel]), ([t.clone() for t in p2], [t.clone() for t in v2])
        ca, cb = (torch.zeros(4, dtype=torch.int64, device="cuda") for _ in range(2))
        acc, _ = E.gather_push(g, a[0], a[1], phi, -1.0, 0.05, 1.3, w_dep=w, scale=scale, counters=ca if cnt else None)
        ref = torch.zeros(E.num_nodes(g), dtype=torch.int64, device="cuda")
        ptr = [(C.c_void_p * 3)(*([t.data_ptr() for t in s] + [None] * (3 - D))) for s in b]
        _lib.check(_lib.lib().psum_hip_gather_push(C.byref(g), code, ptr[0], ptr[1], n, phi.data_ptr(), -1.0, 0.05, 1.3,
                                                   w, scale, ref.data_ptr(), None, cb.data_ptr() if cnt else None,
                                                   torch.cuda.current_stream().cuda_stream), "gather_push")
        assert torch.equal(acc, ref)
        assert torch.equal(ca, cb)
        for s, t in zip(a[0] + a[1], b[0] + b[1]):
            assert torch.equal(torch.nan_to_num(s, nan=-1.0), torch.nan_to_num(t, nan=-1.0))


@pytest.mark.parametrize("nodes,n,domains", [((1024, 800), N0, True), ((1024, 830), N0, False),
                                             ((1024, 830), 2 * N0 - 1, False), ((1024, 830), 2 * N0, True),
                                             ((80, 80, 80), N0, True)])
def test_many_domains_need_many_particles(nodes, n, domains):
    """In 2D more than 51 domains cost more than the atomics below 2^20
    particles: both sides of the line, the same sums"""
    from psum_amd import _lib
    from psum_amd import engine as E
    g = E.periodic_grid(list(nodes))
    assert (_lib.lib().psum_hip_gather_push_workspace(C.byref(g), n) > 0) == domains
    gen = torch.Generator(device="cuda").manual_seed(n)
    pos = [torch.rand(n, generator=gen, device="cuda") * m * 0.999999 for m in nodes]
    vel = [torch.zeros(n, device="cuda") for _ in nodes]
    ref, _ = E.deposit(g, pos, -0.7, scale=2.0 ** 40)
    acc, _ = E.gather_push(g, pos, vel, torch.zeros(E.num_nodes(g), device="cuda"), -1.0, 0.0, 1.0, w_dep=-0.7,
                           scale=2.0 ** 40)
    assert torch.equal(acc, ref)


def test_domain_sums_that_wrap_are_counted():
    """one cell takes 2^19 terms of 2^49..2^50: every node's sum leaves the
    int64 range in an LDS tile, and the counter says so"""
    from psum_amd import engine as E
    g = E.periodic_grid([300, 200])
    gen = torch.Generator(device="cuda").manual_seed(3)
    pos = [torch.rand(2 * N0, generator=gen, device="cuda", dtype=torch.float64) * m for m in (300, 200)]
    pos[0][::2], pos[1][::2] = 7.9, 9.1
    vel = [torch.zeros(2 * N0, device="cuda", dtype=torch.float64) for _ in range(2)]
    phi = torch.zeros(E.num_nodes(g), device="cuda", dtype=torch.float64)
    cnt = torch.zeros(4, dtype=torch.int64, device="cuda")
    E.gather_push(g, pos, vel, phi, -1.0, 0.1, 1.0, w_dep=1024.0, scale=2.0 ** 40, counters=cnt)
    assert int(cnt[3]) > 0
