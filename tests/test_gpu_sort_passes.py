"""The radix sort's digit widths (8 to 10 bits, 1 to 4 passes, key/index pairs
between them, both block sizes), and the stepper's sort of particles loaded
in random order, which takes them through records, against a stable sort."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


# 1 pass of 1 and 10 bits, 2 of 9 and 10, 3 of 7 (2^20 is a 21-bit count) and
# 8, 4 of 8; the large sizes lie on both sides of the 8-wave blocks' limit
@pytest.mark.parametrize("nkeys", [1, 1000, 1 << 17, (1 << 20) - 1, 1 << 20, 1 << 23, 0xFFFFFFFE])
@pytest.mark.parametrize("n", [1, 4097, 30_001, 512 * 8192 - 1, 512 * 8192 + 8195])
def test_every_pass_count_is_a_stable_sort(nkeys, n):
    from psum_amd import engine as E
    rng = np.random.default_rng(nkeys % 1000 + n)
    keys = rng.integers(0, nkeys, n, dtype=np.uint32)
    keys[rng.integers(0, n, n // 9)] = 0xFFFFFFFF
    keys[: n // 5] = keys[0]
    want = np.argsort(np.where(keys == 0xFFFFFFFF, np.uint64(nkeys), keys.astype(np.uint64)), kind="stable")
    sk, perm = E.stable_sort(torch.from_numpy(keys.view(np.int32)).cuda(), nkeys)
    assert np.array_equal(perm.cpu().numpy().view(np.uint32), want.astype(np.uint32))
    assert np.array_equal(sk.cpu().numpy().view(np.uint32), keys[want])


@pytest.mark.parametrize("n", [3, 5000, 70_001])
@pytest.mark.parametrize("nkeys", [1000, 1 << 17, 1 << 20])
def test_workspace_and_arrays_at_4_byte_alignment(n, nkeys):
    from psum_amd import _lib
    rng = np.random.default_rng(n)
    keys = rng.integers(0, nkeys, n, dtype=np.uint32)
    want = np.argsort(keys, kind="stable")
    lib = _lib.lib()
    wb = lib.psum_hip_sort_workspace(n)
    a = [torch.zeros(n + 1, dtype=torch.int32, device="cuda") for _ in range(3)]
    a[0][1:] = torch.from_numpy(keys.view(np.int32))
    work = torch.empty(wb + 4, dtype=torch.uint8, device="cuda")
    k, out, perm, w = (t.data_ptr() + 4 for t in a + [work])
    _lib.check(lib.psum_hip_sort(k, n, nkeys, out, perm, w, wb, torch.cuda.current_stream().cuda_stream), "sort")
    assert np.array_equal(a[2][1:].cpu().numpy().view(np.uint32), want.astype(np.uint32))
    assert np.array_equal(a[1][1:].cpu().numpy().view(np.uint32), keys[want])


# 1, 1, 2, 3 and 4 digits of up to 10 bits
@pytest.mark.parametrize("nkeys", [5, 1000, 60_000, 1 << 25, 0xFFFFFFFE])
@pytest.mark.parametrize("n", [4097, 500_001])
def test_sort_in_place(nkeys, n):
    from psum_amd import _lib
    rng = np.random.default_rng(n)
    keys = rng.integers(0, nkeys, n, dtype=np.uint32)
    want = np.argsort(keys, kind="stable")
    lib = _lib.lib()
    wb = lib.psum_hip_sort_workspace(n)
    k = torch.from_numpy(keys.view(np.int32)).cuda()
    perm, work = torch.empty_like(k), torch.empty(wb, dtype=torch.uint8, device="cuda")
    _lib.check(lib.psum_hip_sort(k.data_ptr(), n, nkeys, k.data_ptr(), perm.data_ptr(), work.data_ptr(), wb,
                                 torch.cuda.current_stream().cuda_stream), "sort")
    assert np.array_equal(perm.cpu().numpy().view(np.uint32), want.astype(np.uint32))
    assert np.array_equal(k.cpu().numpy().view(np.uint32), keys[want])


def _state(st, n):
    from psum_amd import _lib
    pos, vel, m = (C.c_void_p * 3)(), (C.c_void_p * 3)(), C.c_int64(0)
    _lib.check(_lib.lib().psum_stepper_state(st.h, 0, pos, vel, C.byref(m)), "state")

    class A:
        def __init__(self, p, t):
            self.__cuda_array_interface__ = {"shape": (m.value,), "typestr": t, "data": (p, False), "version": 3,
                                             "strides": None}
    torch.cuda.synchronize()
    return [torch.as_tensor(A(p, n), device="cuda").clone() for p in list(pos[:st.dim]) + list(vel[:st.dim])]


# n of components x n x size beyond 16 MB; n % components = 3, 0, 1, 5: the
# records of the last particles lie apart
@pytest.mark.parametrize("nodes,dtype,n", [((64, 48), "f32", 1_100_003), ((64, 48), "f64", 540_000),
                                           ((20, 18, 16), "f32", 720_001), ((20, 18, 16), "f64", 400_001)])
@pytest.mark.parametrize("batch", [False, True])
def test_random_load_is_sorted_through_records(nodes, dtype, n, batch):
    from psum_amd import _lib
    from psum_amd import engine as E
    t = torch.float32 if dtype == "f32" else torch.float64
    g = torch.Generator(device="cuda").manual_seed(n)
    pos = [torch.rand(n, generator=g, device="cuda", dtype=t) * (m - 1) for m in nodes]
    vel = [torch.randn(n, generator=g, device="cuda", dtype=t) for _ in nodes]
    pos[0][::1000] = float("nan")
    cfg = dict(g=E.periodic_grid(list(nodes)), species=[dict(q=-1.0, m=1.0, w=1.0, pos=pos, vel=vel)], dtype=dtype,
               depth=2, pre=1, post=1, max_cycles=2, tol=0.0, dt=0.1, rho_bg=1.0, sort_every=1)
    if batch:
        b = E.Batch([cfg])                # sorts in place: the arrays keep their addresses
        st = b.instances[0]
    else:
        st = E.Stepper(cfg.pop("g"), cfg.pop("species"), **cfg)
    # the stable order of cell, then velocity signs
    ok = torch.isfinite(pos[0])
    key = torch.zeros(n, dtype=torch.int64, device="cuda")
    for x, m in zip(pos, nodes):
        key = key * m + torch.remainder(torch.floor(torch.where(ok, x, 0).double() - 0.5).long(), m)
    for v in vel:
        key = key * 2 + (v >= 0)
    perm = torch.sort(torch.where(ok, key, 2 ** 40), stable=True)[1][:int(ok.sum())]
    want = [a[perm] for a in pos + vel]
    for again in range(2):                # in random order, then in order (the direct permutation)
        _lib.check(_lib.lib().psum_stepper_sort(st.h), "sort")
        for a, w in zip(_state(st, "<f4" if dtype == "f32" else "<f8"), want):
            assert torch.equal(a, w)
