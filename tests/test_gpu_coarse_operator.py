"""The coarse end of the V-cycle as one dense product (levels small enough
are merged into the matrix of the V-cycle from that level down): the iterates
are the oracle's per V-cycle, at level sizes on both sides of the limit, with
and without pre- or post-sweeps, after a change of the sweep counts, and in a
fixed-cycle solver.
"""
import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _walls(nodes, seed):
    og = O.wall_grid([n - 1 for n in nodes])
    fixed = np.zeros(nodes, np.uint8)
    for d in range(len(nodes)):
        s = [slice(None)] * len(nodes)
        for e in (0, -1):
            s[d] = e
            fixed[tuple(s)] = 1
    r, c, v = O.poisson_coo(og, 1.0, fixed.ravel())
    b = np.random.default_rng(seed).standard_normal(fixed.size)
    b[fixed.ravel() == 1] = 0.0
    return fixed.size, r, c, v, b


def _periodic(nodes, seed):
    og = O.periodic_grid(list(nodes))
    nn = O.num_nodes(og)
    fixed = np.zeros(nn, np.uint8)
    fixed[0] = 1
    r, c, v = O.poisson_coo(og, 1.0, fixed)
    b = np.random.default_rng(seed).standard_normal(nn)
    b -= b.mean()
    b[0] = 0.0
    return nn, r, c, v, b


# second level of 2025, 2070 (limit 2049), 4096 and 64, 49 nodes in 2D;
# 4913, 5832 (limit 5000) and 1100 in 3D
CASES = [("walls", (89, 89), 3), ("walls", (89, 90), 3), ("periodic", (128, 128), 3), ("periodic", (16, 16), 2),
         ("walls", (13, 14), 2), ("walls", (33, 33, 33), 3), ("walls", (35, 35, 35), 3), ("walls", (17, 20, 23), 2)]


@pytest.mark.parametrize("kind,nodes,depth", CASES)
@pytest.mark.parametrize("prepost", [(2, 1), (0, 2), (3, 0)])
def test_merged_levels_match_the_oracle_per_cycle(kind, nodes, depth, prepost):
    from psum_amd import engine as E
    nn, r, c, v, b = (_walls if kind == "walls" else _periodic)(nodes, 3)
    pre, post = prepost
    K = nodes[2] if len(nodes) == 3 else 1
    mg = O.MG(nn, r, c, v, nodes[0], nodes[1], K, depth=depth, pre=pre, post=post)
    s = E.SolverBackend("hip_multigrid_gpu")
    dims = f"I {nodes[0]} J {nodes[1]}" + (f" K {K}" if K > 1 else "")
    # set up with other sweep counts: set_options rebuilds the operator
    s.set_options(f"{dims} depth {depth} pre_relax 1 post_relax 1 max_cycles 1")
    s.set_matrix(nn, nn, r, c, v)
    s.set_options(f"{dims} depth {depth} pre_relax {pre} post_relax {post} max_cycles 1")
    x_ref, x = np.zeros(nn), torch.zeros(nn, dtype=torch.float64, device="cuda")
    for cyc in range(3):
        mg.vcycles(b, x_ref, 1)
        s.solve(torch.from_numpy(b).cuda(), x)
        err = np.max(np.abs(x.cpu().numpy() - x_ref)) / np.max(np.abs(x_ref))
        # FP64 sums of at most 5832 terms in another order
        assert err < 1e-11, (cyc, err)


@pytest.mark.parametrize("kind,nodes,depth", CASES)
def test_merged_levels_in_the_mixed_solver(kind, nodes, depth):
    """FP32 V-cycles in FP64 refinement: a single iteration is the oracle's to
    FP32 rounding, and the solve converges to the FP64 solver's answer."""
    from psum_amd import engine as E
    nn, r, c, v, b = (_walls if kind == "walls" else _periodic)(nodes, 5)
    K = nodes[2] if len(nodes) == 3 else 1
    dims = f"I {nodes[0]} J {nodes[1]}" + (f" K {K}" if K > 1 else "")

    def solve(backend, opt):
        s = E.SolverBackend(backend)
        s.set_options(f"{dims} depth {depth} pre_relax 2 post_relax 2 {opt}")
        s.set_matrix(nn, nn, r, c, v)
        x = torch.zeros(nn, dtype=torch.float64, device="cuda")
        s.solve(torch.from_numpy(b).cuda(), x)
        return x.cpu().numpy(), s.stats()
    one32, _ = solve("hip_multigrid32f_gpu", "max_cycles 1 correction_interval 1")
    one64, _ = solve("hip_multigrid_gpu", "max_cycles 1")
    # about 2^-24 times the condition of the sweeps; 1e-5 as for the whole
    # mixed solve against the oracle
    assert np.max(np.abs(one32 - one64)) <= 1e-5 * np.max(np.abs(one64))
    x32, (_, rel) = solve("hip_multigrid32f_gpu", "max_cycles 60 tol 1e-10")
    x64, _ = solve("hip_multigrid_gpu", "max_cycles 60 tol 1e-11")
    assert rel <= 1e-10
    assert np.max(np.abs(x32 - x64)) <= 1e-8 * np.max(np.abs(x64))


@pytest.mark.parametrize("n", [32, 64])
def test_merged_levels_lose_no_precision_in_the_mixed_solver(n):
    """A pair of far charges in a periodic box: the rows of the merged matrix
    cancel against each other, so the matrix itself has to be held in FP64
    (held in FP32: 3.7e-7).  What FP32 vectors round is the scaled and the
    restricted right-hand side, the coarse values and the sweep: 2^-24 each."""
    from psum_amd import engine as E
    nodes = (n, n, n)
    nn, r, c, v, _ = _periodic(nodes, 1)
    b = np.zeros(nodes)
    b[n // 4, n // 4, n // 4], b[3 * n // 4, 3 * n // 4, 3 * n // 4] = 1.0, -1.0
    x = []
    for backend in ("hip_multigrid_gpu", "hip_multigrid32f_gpu"):
        s = E.SolverBackend(backend)
        s.set_options(f"I {n} J {n} K {n} depth {n.bit_length() - 4} pre_relax 0 post_relax 1 max_cycles 1 "
                      "correction_interval 1")
        s.set_matrix(nn, nn, r, c, v)
        xd = torch.zeros(nn, dtype=torch.float64, device="cuda")
        s.solve(torch.from_numpy(b.ravel().copy()).cuda(), xd)
        x.append(xd.cpu().numpy())
    e = x[1] - x[0]
    e -= e[0]            # the gauge is the pinned node's
    assert np.linalg.norm(e) <= 4 * 2.0 ** -24 * np.linalg.norm(x[0])


@pytest.mark.parametrize("dtype", ["f64", "f32"])
def test_switching_to_fixed_cycles_keeps_the_solution(dtype):
    """A fixed cycle count takes a smaller limit (a matrix of its own): the
    step's potential stays that of the tolerance-controlled solve."""
    from psum_amd import engine as E
    from psum_amd.workloads import langmuir_2d
    wl = langmuir_2d(n=128, ppc=4, seed=3, dtype=np.float64 if dtype == "f64" else np.float32)
    phis = []
    for fixed in (0, 25):
        st = E.Stepper(wl["grid"], wl["species"], dtype=dtype, mixed_mg=dtype == "f32", depth=4, pre=2, post=2,
                       max_cycles=40, tol=1e-12, dt=wl["dt"], rho_bg=1.0)
        st.set_smoothing(3, 2)
        if fixed:
            st.set_schedule(fixed, 0, 0)
        st.run(1)
        phis.append(st.phi())
        st.close()
    assert np.max(np.abs(phis[0] - phis[1])) <= 1e-9 * np.max(np.abs(phis[0]))


def test_operator_follows_the_sweeps_of_a_refused_option_list():
    """An option list that is refused half-way has set the sweeps before the
    value it is refused for: the next solve runs with them on every level,
    merged ones included, like a solver set up with them."""
    from psum_amd import engine as E
    nn, r, c, v, b = _walls((65, 49), 4)
    out = []
    for late in (False, True):
        s = E.SolverBackend("hip_multigrid_gpu")
        s.set_options(f"I 65 J 49 depth 3 pre_relax {1 if late else 3} post_relax 1 max_cycles 2")
        s.set_matrix(nn, nn, r, c, v)
        if late:
            with pytest.raises(E.PsumError):
                s.set_options("I 65 J 49 pre_relax 3 correction_interval 0")
        x = torch.zeros(nn, dtype=torch.float64, device="cuda")
        s.solve(torch.from_numpy(b).cuda(), x)
        out.append(x.cpu().numpy())
    assert np.array_equal(out[0], out[1])


def test_switching_to_fixed_cycles_builds_nothing():
    """44 x 46 nodes are merged with a tolerance and 22 x 23 in a fixed-cycle
    solver: both matrices are there from the set-up on, so the switch neither
    allocates nor frees."""
    from psum_amd import engine as E
    from psum_amd.workloads import langmuir_2d
    wl = langmuir_2d(n=88, ppc=4, seed=3)
    g = E.periodic_grid([88, 92])
    st = E.Stepper(g, wl["species"], depth=3, pre=2, post=2, max_cycles=40, tol=1e-12, dt=wl["dt"], rho_bg=1.0)
    st.run(1)
    free = torch.cuda.mem_get_info()[0]
    st.set_schedule(25, 0, 0)
    assert torch.cuda.mem_get_info()[0] == free
    st.run(1)
    assert torch.cuda.mem_get_info()[0] == free
    st.close()


@pytest.mark.parametrize("backend", ["hip_multigrid_gpu", "hip_multigrid32f_gpu"])
@pytest.mark.parametrize("kind,nodes,depth", [
    ("walls", (1100, 300), 6),       # large tiles (210 blocks) with remainders on both axes
    ("walls", (823, 760), 6),        # large FP64 tiles (52 x 13 of 16 rows) with remainders on both axes
    ("periodic", (720, 704), 6),     # and across the seam
    ("walls", (301, 1153), 6),       # odd counts
    ("periodic", (512, 464), 5),     # large tiles across the seam
    ("walls", (199, 62), 3),         # small tiles, even last axis
    ("periodic", (72, 40), 4),       # 9 x 5 at the end: axes kept as they are
    ("periodic", (144, 6), 3),       # an axis shorter than a tile's halo
])
@pytest.mark.parametrize("prepost", [(1, 1), (2, 1), (4, 4), (7, 2), (0, 5)])
def test_tile_kernels_match_the_unfused_kernels(backend, kind, nodes, depth, prepost):
    """The tile kernels (sweeps, prolongation with staged coarse values, the
    downward half in one launch; both tile sizes) against one launch per
    sweep and transfer ("fuse 0"): equal bits."""
    from psum_amd import engine as E
    nn, r, c, v, b = (_walls if kind == "walls" else _periodic)(nodes, 7)
    pre, post = prepost
    out = []
    for fuse in (0, 1):
        s = E.SolverBackend(backend)
        s.set_options(f"I {nodes[0]} J {nodes[1]} depth {depth} pre_relax {pre} post_relax {post} max_cycles 3 "
                      f"correction_interval 1 fuse {fuse}")
        s.set_matrix(nn, nn, r, c, v)
        x = torch.zeros(nn, dtype=torch.float64, device="cuda")
        s.solve(torch.from_numpy(b).cuda(), x)
        out.append(x.cpu().numpy())
    assert np.array_equal(out[0], out[1])
