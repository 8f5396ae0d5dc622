"""Timed cases of the particle-in-cell engine, over the range its users run.

Each case is one pass through the public Python entry points (the Stepper
and Batch step loops, the multigrid solver backend, the particle / field
functions a program's own loop is made of, the differentiable step, Monte
Carlo collisions, the triangle-mesh boundary).  `exact` restates what a pass
returns in plain FP64 torch: CIC and B-spline coupling by index arithmetic,
the discrete Poisson problem by FFT (periodic) or sine transforms (walls).

Units are the workloads': dx = 1, omega_p = 1, v_th = 1, eps = 1 unless a
case says otherwise.
"""
import math

import numpy as np
import torch

from psum_amd import _lib
from psum_amd import engine as E
from psum_amd import mcc as M
from psum_amd import mesh as Mh
from psum_amd.pypsum import PicFieldEnergy

STEPS = 20          # steps of a step-loop pass: one sort period of the fast species


# ------------------------------------------------------------------ cases

def listed():
    return [
        # the plain FP64 2D Langmuir problem of the benchmark: a small
        # periodic run, bound by launches and the solver's latency
        dict(name="langmuir2d_128_f64", kind="step2d", n0=128, n1=128, ppc=64, load="langmuir",
             dtype="f64", order=1, pre=2, post=1, tol=1e-10),
        # the benchmark's 2D two-stream instability at its full size
        dict(name="twostream2d_1024_f32", kind="step2d", n0=1024, n1=1024, ppc=100, load="two_stream",
             dtype="f32", order=1, pre=3, post=3, tol=1e-8),
        # cubic B-spline coupling on a grid that is no power of two
        dict(name="spline2d_248x200_f32", kind="step2d", n0=248, n1=200, ppc=49, load="langmuir",
             dtype="f32", order=3, pre=2, post=2, tol=1e-8),
        # the bounded 3D box (grounded, absorbing walls; electrons and ions),
        # mixed precision, at the largest size that is quick to prepare
        dict(name="box3d_128_f32", kind="box3d", c0=128, c1=128, c2=128, ppc=32, dtype="f32",
             pre=5, post=5, tol=1e-8),
        # a small odd box in plain FP64
        dict(name="box3d_50x44x61_f64", kind="box3d", c0=50, c1=44, c2=61, ppc=10, dtype="f64",
             pre=3, post=3, tol=1e-8),
        # the field solver alone, as a frontend calls it through the backend
        dict(name="solve2d_641x385_f64", kind="solve", n0=641, n1=385, n2=1, mixed=False, pre=2, post=1,
             tol=1e-10),
        # a program's own loop over unsorted FP32 particles, some of them
        # invalid: push + deposit, field energy, compaction
        dict(name="loop2d_unsorted_f32", kind="loop", dim=2, n0=512, n1=384, n2=1, n=5_000_001, dx=0.5,
             dtype="f32", sort=False),
        # a program's own loop that bins and sorts FP64 particles each step
        dict(name="loop3d_sorted_f64", kind="loop", dim=3, n0=60, n1=52, n2=44, n=3_000_003, dx=1.0,
             dtype="f64", sort=True),
        # the differentiable two-stream step: recorded forward and reverse
        dict(name="adjoint2d_256_f32", kind="adjoint", n=256, ppc=64, steps=20, ckpt=10, dtype="f32"),
        # an ensemble of small independent problems stepped together
        dict(name="batch2d_12_f32", kind="batch", instances=12, small=64, large=256, ppc=48),
        # Monte Carlo collisions of electrons with a background gas
        dict(name="mcc_20m_f64", kind="mcc", n=20_000_000, dtype="f64", ionization=False),
        # the triangle-mesh particle boundary (router scene)
        dict(name="mesh_10m_f64", kind="mesh", n=10_000_000, dtype="f64", parts=100),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step2d", "step2d", "step2d", "box3d", "box3d", "solve", "loop", "loop", "adjoint", "batch",
                       "mcc", "mesh"])
    if kind == "step2d":
        # periodic node counts of 64..1024 per axis that halve to 31 or fewer
        # nodes, as a geometric multigrid needs
        n0, n1 = (_log_int(rng, 16, 32) * 2 ** rng.randint(2, 5) for _ in range(2))
        order = rng.choice([1, 1, 1, 2, 3, 4])
        load = rng.choice(["langmuir", "two_stream"])
        ppc = _log_int(rng, 4, 10) ** 2
        most = 100_000_000 if order == 1 else 8_000_000
        while n0 * n1 * ppc > most:
            ppc = (math.isqrt(ppc) - 1) ** 2
        dtype = rng.choice(["f32", "f64"])
        return dict(kind=kind, n0=n0, n1=n1, ppc=ppc, load=load, dtype=dtype, order=order, pre=rng.randint(2, 3),
                    post=rng.randint(1, 3), tol=1e-8 if dtype == "f32" else 1e-10)
    if kind == "box3d":
        c = [_log_int(rng, 24, 120) for _ in range(3)]
        return dict(kind=kind, c0=c[0], c1=c[1], c2=c[2], ppc=_log_int(rng, 8, 32),
                    dtype=rng.choice(["f32", "f64"]), pre=rng.randint(2, 5), post=rng.randint(2, 5), tol=1e-8)
    if kind == "solve":
        if rng.random() < 0.5:
            return dict(kind=kind, n0=_log_int(rng, 65, 1025), n1=_log_int(rng, 65, 1025), n2=1,
                        mixed=rng.random() < 0.5, pre=2, post=rng.randint(1, 2), tol=1e-8)
        n = [_log_int(rng, 25, 129) for _ in range(3)]
        return dict(kind=kind, n0=n[0], n1=n[1], n2=n[2], mixed=rng.random() < 0.5, pre=rng.randint(2, 3),
                    post=rng.randint(1, 3), tol=1e-8)
    if kind == "loop":
        dim = rng.choice([2, 3])
        n = [_log_int(rng, 40, 600 if dim == 2 else 100) for _ in range(dim)] + [1]
        return dict(kind=kind, dim=dim, n0=n[0], n1=n[1], n2=n[2] if dim == 3 else 1,
                    n=_log_int(rng, 50_000, 10_000_000), dx=rng.choice([1.0, 0.5, 0.3]),
                    dtype=rng.choice(["f32", "f64"]), sort=rng.random() < 0.5)
    if kind == "adjoint":
        return dict(kind=kind, n=8 * rng.randint(8, 32), ppc=_log_int(rng, 4, 8) ** 2, steps=rng.randint(8, 20),
                    ckpt=rng.randint(4, 10), dtype=rng.choice(["f32", "f64"]))
    if kind == "batch":
        return dict(kind=kind, instances=rng.randint(3, 12), small=64, large=rng.choice([128, 192, 256]),
                    ppc=_log_int(rng, 16, 64))
    if kind == "mcc":
        return dict(kind=kind, n=_log_int(rng, 20_000, 20_000_000), dtype=rng.choice(["f32", "f64"]),
                    ionization=rng.random() < 0.5)
    return dict(kind=kind, n=_log_int(rng, 20_000, 10_000_000), dtype=rng.choice(["f32", "f64"]),
                parts=rng.choice([40, 60, 100]))


# -------------------------------------------------------------- utilities

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _tdt(dtype):
    return torch.float32 if dtype == "f32" else torch.float64


def _periodic_depth(sizes):
    """coarsenings of a periodic grid, each halving the even axes, down to a
    coarsest grid of at most 512 nodes, or to where no axis of 16 nodes or
    more is even"""
    n, d = list(sizes), 0
    while math.prod(n) > 512 and any(m % 2 == 0 and m >= 16 for m in n):
        n = [m // 2 if m % 2 == 0 and m >= 4 else m for m in n]
        d += 1
    return max(1, d)


def _wall_depth(nodes):
    """coarsenings of a wall grid, each keeping every other node and the last
    one, down to a coarsest grid of at most 800 nodes"""
    n, d = list(nodes), 0
    while math.prod(n) > 800 and max(n) > 4:
        n = [max(2, m // 2 + 1) for m in n]
        d += 1
    return max(1, d)


class _DeviceArray:
    """A species array of a stepper as torch sees it, without a copy
    (psum_stepper_state); it keeps the stepper alive."""

    def __init__(self, owner, ptr, n, dtype):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": "<f4" if dtype == "f32" else "<f8",
                                         "data": (int(ptr), False), "version": 3, "strides": None}


def _state(st, species, dtype, owner=None):
    import ctypes as C
    pos, vel, n = (C.c_void_p * 3)(), (C.c_void_p * 3)(), C.c_int64(0)
    _lib.check(_lib.lib().psum_stepper_state(st.h, species, pos, vel, C.byref(n)), "psum_stepper_state")
    keep = (st, owner)
    return [torch.as_tensor(_DeviceArray(keep, p, n.value, dtype), device="cuda")
            for p in list(pos[:st.dim]) + list(vel[:st.dim])]


# ---------------------------------------------------------- initial loads

def _load_2d(case, seed, n0, n1, ppc, load, dtype):
    """positions and velocities of one electron species on [0, n0) x [0, n1)"""
    g = _gen(seed)
    t = _tdt(dtype)
    N = n0 * n1 * ppc

    def rand():
        return torch.rand(N, generator=g, device="cuda", dtype=t)

    def randn():
        return torch.randn(N, generator=g, device="cuda", dtype=t)
    if load == "two_stream":
        # a sqrt(ppc)^2 lattice in every cell with 1e-3 jitter; beams +-5
        m = int(round(math.sqrt(ppc)))
        i = torch.arange(N, device="cuda")
        x = (i // (n1 * ppc)).to(t)
        y = (i // ppc % n1).to(t)
        x += ((i // m % m).to(t) + 0.5) / m + 1e-3 * randn()
        y += ((i % m).to(t) + 0.5) / m + 1e-3 * randn()
        x, y = torch.remainder(x, n0), torch.remainder(y, n1)
        vx = torch.where(i % 2 == 0, 5.0, -5.0).to(t) + randn()
        del i
    else:
        # density 1 + 0.01 cos(2 pi x / L) to first order
        x = rand() * n0
        x = torch.remainder(x - 0.01 * n0 / (2 * math.pi) * torch.sin(2 * math.pi * x / n0), n0)
        y = rand() * n1
        vx = randn()
    x[x >= n0] = 0.0
    y[y >= n1] = 0.0
    return [x, y], [vx, randn()]


def _species_2d(case, seed, n0, n1, ppc, load, dtype):
    pos, vel = _load_2d(case, seed, n0, n1, ppc, load, dtype)
    return dict(q=-1.0, m=1.0, w=1.0 / ppc, pos=pos, vel=vel)


def _species_box(case, seed):
    t = _tdt(case["dtype"])
    c = [case["c0"], case["c1"], case["c2"]]
    N = c[0] * c[1] * c[2] * case["ppc"]
    out = []
    for s, (q, m, vth) in enumerate(((-1.0, 1.0, 1.0), (1.0, 1836.0, math.sqrt(0.1 / 1836.0)))):
        g = _gen(10 * seed + s)
        pos = [torch.rand(N, generator=g, device="cuda", dtype=t) * L for L in c]
        for x, L in zip(pos, c):
            x[x >= L] = 0.0
        vel = [torch.randn(N, generator=g, device="cuda", dtype=t) * vth for _ in range(3)]
        out.append(dict(q=q, m=m, w=1.0 / case["ppc"], pos=pos, vel=vel))
    return out


def _faces(nodes):
    f = np.zeros(nodes, np.uint8)
    for d in range(len(nodes)):
        s = [slice(None)] * len(nodes)
        for e in (0, -1):
            s[d] = e
            f[tuple(s)] = 1
    return f


def _batch_specs(case, seed):
    """instance i: a square periodic grid between `small` and `large` nodes"""
    sizes = [n for n in (64, 96, 128, 192, 256) if case["small"] <= n <= case["large"]]
    out = []
    for i in range(case["instances"]):
        n, ppc = sizes[i % len(sizes)], max(4, case["ppc"] - 3 * i)
        out.append((n, ppc, _species_2d(case, 100 * seed + i, n, n, ppc, "langmuir", "f32")))
    return out


def _mcc_inputs(case, seed):
    """electrons on [0, 0.067): a 2 eV core with a hot tail"""
    g, n, t = _gen(seed), case["n"], _tdt(case["dtype"])
    x = torch.rand(n, generator=g, device="cuda", dtype=t) * 0.067
    hot = (torch.rand(n, generator=g, device="cuda") < 0.1).to(t)
    v = [torch.randn(n, generator=g, device="cuda", dtype=t) * (6e5 + 2.4e6 * hot) for _ in range(3)]
    s = torch.randint(-2**31, 2**31 - 1, (n,), generator=g, device="cuda", dtype=torch.int32)
    return x, v, s


_X0 = 28.0
_ME, _MHE, _QE, _DENS, _MCC_DT = 9.10956e-31, 6.67e-27, 1.602e-19, 3e21, 1e-12


def _fit(a, b, c, x_on=None):
    row = [0.0, 0.0, c, b - 2 * c * _X0, a - b * _X0 + c * _X0 * _X0]
    if x_on is None:
        return dict(seg_hi=[], coef=[row])
    return dict(seg_hi=[x_on], coef=[[0, 0, 0, 0, -200.0], row])


def _channels():
    return [("elastic", _fit(-44.0, -0.4, -0.02), 0.0),
            ("excitation", _fit(-46.0, 0.8, -0.15, _X0 + 2.16), 19.82),
            ("excitation", _fit(-46.5, 0.7, -0.12, _X0 + 2.2), 20.61),
            ("ionization", _fit(-45.0, 0.9, -0.1, _X0 + 2.37), 24.587)]


def _scene():
    """an absorbing box, a specular 64-segment nozzle, a diffuse plane"""
    noz = Mh.revolve_zr_curve([(-4, 1.0), (-3.5, 1.0), (-3, 0.9), (-2.5, 0.8), (-2, 0.6), (-1.5, 0.5), (-1, 0.6),
                               (-0.5, 0.8), (0, 1.0), (0.5, 1.2), (1, 1.4), (1.5, 1.6), (2, 1.8), (2.5, 1.9),
                               (3, 2.0), (3.5, 2.0), (4, 2.0)], 64)
    return [(Mh.axis_aligned_cube(-5, -5, -5, 5, 5, 10), "absorb"), (noz, "specular"),
            (Mh.axis_aligned_plane(-5, -5, -4.0, 5, 5, -4.0), "diffuse")]


def _loop_inputs(case, seed):
    g, t, D = _gen(seed), _tdt(case["dtype"]), case["dim"]
    nodes = [case["n0"], case["n1"], case["n2"]][:D]
    pos = [torch.rand(case["n"], generator=g, device="cuda", dtype=t) * (n * case["dx"]) for n in nodes]
    for x, n in zip(pos, nodes):
        x[x >= n * case["dx"]] = 0.0
    # one particle in 33 was absorbed earlier
    gone = torch.randperm(case["n"], generator=g, device="cuda")[:case["n"] // 33]
    pos[0][gone] = float("nan")
    vel = [torch.randn(case["n"], generator=g, device="cuda", dtype=t) for _ in range(D)]
    phi = torch.zeros(nodes, device="cuda", dtype=torch.float64)
    for d, n in enumerate(nodes):
        shape = [1] * D
        shape[d] = n
        i = torch.arange(n, device="cuda", dtype=torch.float64).reshape(shape)
        phi = phi + torch.cos(2 * math.pi * (d + 1) * i / n)
    phi = phi + 0.01 * torch.randn(nodes, generator=g, device="cuda", dtype=torch.float64)
    return nodes, pos, vel, phi.reshape(-1)


_LOOP = dict(qm=-1.0, dt=0.05, mass=1.0, w=-0.03125)


# ---------------------------------------------------------------- prepare

def prepare(case, seed):
    kind = case["kind"]
    if kind == "step2d":
        sp = _species_2d(case, seed, case["n0"], case["n1"], case["ppc"], case["load"], case["dtype"])
        st = E.Stepper(E.periodic_grid([case["n0"], case["n1"]]), [sp], dtype=case["dtype"],
                       mixed_mg=case["dtype"] == "f32", depth=_periodic_depth([case["n0"], case["n1"]]),
                       pre=case["pre"], post=case["post"], max_cycles=60, tol=case["tol"], dt=0.05, rho_bg=1.0,
                       sort_every=STEPS, interp_order=case["order"])
        return dict(case=case, st=st, species=[sp])
    if kind == "box3d":
        sp = _species_box(case, seed)
        cells = [case["c0"], case["c1"], case["c2"]]
        nodes = [c + 1 for c in cells]
        st = E.Stepper(E.wall_grid(cells), sp, dtype=case["dtype"], mixed_mg=case["dtype"] == "f32",
                       depth=_wall_depth(nodes), pre=case["pre"], post=case["post"], max_cycles=60, tol=case["tol"],
                       dt=0.1, rho_bg=0.0, sort_every=STEPS, fixed=_faces(nodes).ravel())
        st.set_schedule(0, STEPS, 2)     # 4^3-cell bins
        return dict(case=case, st=st, species=sp)
    if kind == "solve":
        nodes = [n for n in (case["n0"], case["n1"], case["n2"]) if n > 1]
        grid = E.wall_grid([n - 1 for n in nodes])
        fixed = _faces(nodes)
        (r, c, v), _ = E.poisson_assemble(grid, eps=1.0, fixed=fixed.ravel())
        s = E.SolverBackend("hip_multigrid32f_gpu" if case["mixed"] else "hip_multigrid_gpu")
        opt = "I %d J %d" % (nodes[0], nodes[1]) + (" K %d" % nodes[2] if len(nodes) == 3 else "")
        s.set_options("%s depth %d pre_relax %d post_relax %d max_cycles 60 tol %g"
                      % (opt, _wall_depth(nodes), case["pre"], case["post"], case["tol"]))
        s.set_matrix(fixed.size, fixed.size, r, c, v)
        idx = np.flatnonzero(fixed.ravel())
        vals = np.zeros(idx.size)
        vals[:fixed[0].size] = 1.0       # the low face of the slowest axis at potential 1
        s.set_source_replace(idx, vals)
        b0 = torch.randn(fixed.size, generator=_gen(seed), device="cuda", dtype=torch.float64) * 0.1
        return dict(case=case, solver=s, b0=b0, b=torch.empty_like(b0), x=torch.empty_like(b0))
    if kind == "loop":
        nodes, pos, vel, phi = _loop_inputs(case, seed)
        return dict(case=case, grid=E.periodic_grid(nodes, case["dx"]), pos=pos, vel=vel, phi=phi,
                    phi_p=phi.to(_tdt(case["dtype"])))
    if kind == "adjoint":
        sp = _species_2d(case, seed, case["n"], case["n"], case["ppc"], "two_stream", case["dtype"])
        st = E.Stepper(E.periodic_grid([case["n"]] * 2), [sp], dtype=case["dtype"], mixed_mg=case["dtype"] == "f32",
                       depth=_periodic_depth([case["n"]] * 2), pre=3, post=3, max_cycles=60, tol=1e-9, dt=0.05,
                       rho_bg=1.0, sort_every=0)
        leaves = [a.requires_grad_(True) for a in sp["pos"] + sp["vel"]]
        return dict(case=case, st=st, leaves=leaves)
    if kind == "batch":
        specs = _batch_specs(case, seed)
        b = E.Batch([dict(g=E.periodic_grid([n, n]), species=[sp], dtype="f32", mixed_mg=True,
                          depth=_periodic_depth([n, n]), pre=2, post=2, max_cycles=60, tol=1e-8, dt=0.05, rho_bg=1.0,
                          sort_every=STEPS) for n, _, sp in specs])
        for i in range(len(b)):
            b.configure(i, 9, STEPS, 0)
        b.reset_history(1 << 14)
        return dict(case=case, batch=b, species=[sp for _, _, sp in specs])
    if kind == "mcc":
        x, v, s = _mcc_inputs(case, seed)
        n = case["n"]
        # the incident species and, with ionization, its products share arrays
        cap = n + (n // 10 + 64 if case["ionization"] else 0)
        el = M.Particles.empty(1, cap, dtype=_tdt(case["dtype"]))
        el.pos[0][:n], el.seed[:n] = x, s
        for c in range(3):
            el.vel[c][:n] = v[c]
        el.n = n
        ions = M.Particles.empty(1, n // 10 + 64, dtype=_tdt(case["dtype"])) if case["ionization"] else None
        ch = [M.channel(k, threshold_ev=thr, **f) for k, f, thr in _channels()[:4 if case["ionization"] else 3]]
        proc = [M.Process(ch, _DENS, incident_mass=_ME, target_mass=_MHE, target_temperature=300.0)]
        return dict(case=case, grid=E.wall_grid([1000], dx=0.067 / 1000), proc=proc, el=el, ions=ions)
    if kind == "mesh":
        g, n, t = _gen(seed), case["n"], _tdt(case["dtype"])
        router = Mh.BoundaryRouter().set(_scene(), case["parts"], case["parts"], case["parts"])
        r = torch.sqrt(torch.rand(n, generator=g, device="cuda", dtype=t)) * 0.45
        th = 2 * math.pi * torch.rand(n, generator=g, device="cuda", dtype=t)
        old = [r * torch.cos(th), r * torch.sin(th), -4 + 7.9 * torch.rand(n, generator=g, device="cuda", dtype=t)]
        vel = [torch.randn(n, generator=g, device="cuda", dtype=t) for _ in range(3)]
        seeds = torch.randint(-2**31, 2**31 - 1, (n,), generator=g, device="cuda", dtype=torch.int32)
        return dict(case=case, router=router, old=old, vel=vel, seeds=seeds, dt=0.1)
    raise ValueError(kind)


# -------------------------------------------------------------------- run

def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind in ("step2d", "box3d"):
        # a run from given particles: load, STEPS steps (a sort of every
        # species before the first), then phi and the particles
        st = state["st"]
        for q, sp in enumerate(state["species"]):
            st.load(q, sp["pos"], sp["vel"])
        hist = st.run(STEPS)
        return dict(hist=hist, phi=st.phi(),
                    particles=[_state(st, q, case["dtype"]) for q in range(len(state["species"]))])
    if kind == "solve":
        state["b"].copy_(state["b0"])
        state["x"].zero_()
        state["solver"].solve(state["b"], state["x"])
        return state["x"]
    if kind == "loop":
        g, pos, vel = state["grid"], state["pos"], state["vel"]
        keys = perm = None
        if case["sort"]:
            keys = E.cell_keys(g, pos)
            keys, perm = E.stable_sort(keys, E.num_nodes(g))
            pos = E.permute(pos, perm)
            vel = E.permute(vel, perm)
            state["pos"], state["vel"] = pos, vel
        acc, diag = E.gather_push(g, pos, vel, state["phi_p"], _LOOP["qm"], _LOOP["dt"], _LOOP["mass"],
                                  w_dep=_LOOP["w"])
        energy = E.field_energy(g, state["phi"])
        alive_pos, alive_vel = E.compact(pos, vel)
        out = dict(acc=acc, diag=diag, energy=energy, pos=alive_pos, vel=alive_vel)
        if perm is not None:
            out.update(keys=keys, perm=perm)
        return out
    if kind == "adjoint":
        loss = PicFieldEnergy.apply(state["st"], case["steps"], case["ckpt"], *state["leaves"])
        return dict(loss=loss.detach(), grads=list(torch.autograd.grad(loss, state["leaves"])))
    if kind == "batch":
        b = state["batch"]
        for st, sp in zip(b.instances, state["species"]):
            st.load(0, sp["pos"], sp["vel"])
        b.run(STEPS)
        return [dict(phi=st.phi(), particles=_state(st, 0, "f32", b)) for st in b.instances]
    if kind == "mcc":
        el, ions = state["el"], state["ions"]
        el.n = case["n"]
        if ions is not None:
            ions.n = 0
        made, _ = M.collide(state["grid"], state["proc"], el, _MCC_DT, electrons=el if ions is not None else None,
                            ions=ions, grow=False)
        out = dict(made=made, vel=el.vel, seed=el.seed)
        if ions is not None:
            out.update(pos=el.pos, ion_pos=ions.pos, ion_vel=ions.vel, ion_seed=ions.seed)
        return out
    if kind == "mesh":
        pos = [torch.add(o, v, alpha=state["dt"]) for o, v in zip(state["old"], state["vel"])]
        vel = [v.clone() for v in state["vel"]]
        seeds = state["seeds"].clone()
        hits, hit_id = state["router"].deal(state["old"], pos, vel, seeds, hit_id=True)
        return dict(hits=hits, hit_id=hit_id, pos=pos, vel=vel, seeds=seeds)
    raise ValueError(kind)


# ------------------------------------------------------------------- work

def _esz(dtype):
    return 4 if dtype == "f32" else 8


def work(case):
    """What a pass cannot do without: particle state read and written once a
    step, rho written, phi written and read; arithmetic of the weights."""
    kind = case["kind"]
    if kind == "step2d":
        nn = case["n0"] * case["n1"]
        N = nn * case["ppc"]
        s = (case["order"] + 1) ** 2
        return dict(bytes=STEPS * (N * 8 * _esz(case["dtype"]) + nn * 32), flops=STEPS * N * (30 + 10.0 * s))
    if kind == "box3d":
        N = 2 * case["c0"] * case["c1"] * case["c2"] * case["ppc"]
        nn = (case["c0"] + 1) * (case["c1"] + 1) * (case["c2"] + 1)
        return dict(bytes=STEPS * (N * 12 * _esz(case["dtype"]) + nn * 32), flops=STEPS * N * 120.0)
    if kind == "solve":
        nn = case["n0"] * case["n1"] * case["n2"]
        return dict(bytes=16.0 * nn, flops=100.0 * nn)
    if kind == "loop":
        N, D, e = case["n"], case["dim"], _esz(case["dtype"])
        nn = case["n0"] * case["n1"] * case["n2"]
        # push, then the survivors written once more; keys and permutation out
        return dict(bytes=N * (6 * D * e + (8 if case["sort"] else 0)) + nn * (16 + e), flops=N * 30.0 * 2 ** D)
    if kind == "adjoint":
        N = case["n"] ** 2 * case["ppc"]
        # the forward state, and per step x and the four adjoint components
        return dict(bytes=case["steps"] * N * (16.0 * _esz(case["dtype"]) + 64), flops=case["steps"] * N * 250.0)
    if kind == "batch":
        N = 0
        for i in range(case["instances"]):
            sizes = [n for n in (64, 96, 128, 192, 256) if case["small"] <= n <= case["large"]]
            N += sizes[i % len(sizes)] ** 2 * max(4, case["ppc"] - 3 * i)
        return dict(bytes=STEPS * N * 32.0, flops=STEPS * N * 70.0)
    if kind == "mcc":
        return dict(bytes=case["n"] * (4.0 * _esz(case["dtype"]) + 8), flops=case["n"] * 300.0)
    return dict(bytes=case["n"] * (15.0 * _esz(case["dtype"]) + 12), flops=case["n"] * 400.0)


# -------------------------------------------------------------- tolerance

def tolerance(case):
    """Sizes measured against `exact` or between two correct solves of the
    same inputs, times about four."""
    kind = case["kind"]
    f32 = case.get("dtype") == "f32"
    if kind in ("step2d", "batch", "box3d") and (f32 or kind == "batch"):
        # velocities 5e-5 .. 2.2e-4 (a particle whose FP32 position rounds into
        # the next cell feels another field), phi of the quiet start 1.4e-4
        return {"rel": 9e-4, "max": 0.99}
    if kind == "step2d":
        return {"rel": 3e-9, "max": 3e-8}       # phi 1e-12 .. 7e-10 at a residual of 1e-10
    if kind == "box3d":
        return {"rel": 8e-9, "max": 8e-8}       # phi 1.5e-9 at a residual of 1e-8
    if kind == "solve":
        # residual 1e-8 or 1e-10: 1.8e-12 at 1e-10
        return {"rel": 1e-8} if case["tol"] > 1e-9 else {"rel": 1e-10}
    if kind == "loop":
        return {"rel": 1e-7} if f32 else {"rel": 1e-15, "max": 4e-15}   # one rounding: 2.6e-8, 6.5e-17
    if kind == "adjoint":
        # FP32 trajectories cross cell edges at other steps: 5e-3
        return {"rel": 0.02, "max": 0.99} if f32 else {"rel": 1e-6, "max": 1e-4}
    # collisions and wall hits: the rounding of sin, cos and log
    return {"rel": 1e-7} if f32 else {"rel": 1e-14}


# ------------------------------------------------------- the exact results

def _bspline(u, p):
    """the centred cardinal B-spline of degree p"""
    if p == 0:
        return ((u >= -0.5) & (u < 0.5)).to(u.dtype)
    h = (p + 1) / 2
    return ((u + h) * _bspline(u + 0.5, p - 1) + (h - u) * _bspline(u - 0.5, p - 1)) / p


class _Pic:
    """Plain FP64 restatement of the step on unit spacing: periodic nodes at
    i + 1/2 with period n, or nodes 0..c between absorbing walls."""

    def __init__(self, nodes, periodic, fixed_zero, order=1, dx=1.0, lb=None):
        self.n, self.D, self.periodic, self.order, self.dx = list(nodes), len(nodes), periodic, order, dx
        self.lb = (0.5 * dx if periodic else 0.0) if lb is None else lb
        self.fixed_zero = fixed_zero

    def _axis(self, x, d, i, base, grad):
        """weight (or its derivative) of node base + i along axis d"""
        u = (x - self.lb) / self.dx - (base + i)
        if not grad:
            return _bspline(u, self.order) if self.order > 1 else (1 - u.abs())
        if self.order > 1:
            return (_bspline(u + 0.5, self.order - 1) - _bspline(u - 0.5, self.order - 1)) / self.dx
        return (torch.ones_like(u) if i else -torch.ones_like(u)) / self.dx

    def _bases(self, pos):
        out = []
        for x in pos:
            t = (x.detach() - self.lb) / self.dx
            if self.order % 2:
                out.append(torch.floor(t) - (self.order - 1) // 2)
            else:
                out.append(torch.floor(t + 0.5) - self.order // 2)
        return out

    def support(self, pos):
        """(node index, offsets) of every support node"""
        b = self._bases(pos)
        S = self.order + 1
        for k in range(S ** self.D):
            off = [k // S ** (self.D - 1 - d) % S for d in range(self.D)]
            lin = torch.zeros_like(pos[0], dtype=torch.int64)
            for d in range(self.D):
                i = (b[d] + off[d]).to(torch.int64)
                i = torch.remainder(i, self.n[d]) if self.periodic else i
                lin = lin * self.n[d] + i
            yield lin, off, b

    def deposit(self, pos, w):
        rho = torch.zeros(math.prod(self.n), dtype=torch.float64, device=pos[0].device)
        for lin, off, b in self.support(pos):
            c = w
            for d in range(self.D):
                c = c * self._axis(pos[d], d, off[d], b[d], False)
            rho = rho.index_add(0, lin, c)
        return rho

    def grad(self, phi, pos):
        out = [0.0] * self.D
        for lin, off, b in self.support(pos):
            ph = torch.index_select(phi, 0, lin)
            wv = [self._axis(pos[d], d, off[d], b[d], False) for d in range(self.D)]
            for e in range(self.D):
                c = ph * self._axis(pos[e], e, off[e], b[e], True)
                for d in range(self.D):
                    if d != e:
                        c = c * wv[d]
                out[e] = out[e] + c
        return out

    def solve(self, rho):
        """phi of the discrete problem: mean-free and phi[0] = 0 (periodic),
        or zero on the faces"""
        if self.periodic:
            f = torch.fft.fftn(rho.reshape(self.n))
            lam = torch.zeros(self.n, dtype=torch.float64, device=rho.device)
            for d, n in enumerate(self.n):
                shape = [1] * self.D
                shape[d] = n
                lam = lam + (2 - 2 * torch.cos(2 * math.pi * torch.arange(n, device=rho.device,
                                                                          dtype=torch.float64) / n)).reshape(shape)
            lam.reshape(-1)[0] = 1.0
            keep = torch.ones_like(lam)
            keep.reshape(-1)[0] = 0.0
            phi = torch.fft.ifftn(f * keep / lam).real.reshape(-1)
            return phi - phi[0]
        return dirichlet(rho.reshape(self.n)).reshape(-1)

    def energy(self, phi):
        p = phi.reshape(self.n)
        e = 0.0
        for d in range(self.D):
            g = (torch.roll(p, -1, d) - p) / self.dx if self.periodic else p.diff(dim=d) / self.dx
            e = e + (g * g).sum()
        return 0.5 * e * self.dx ** self.D

    def sorted(self, pos, vel, shift):
        """the stable order of bin, then velocity signs"""
        key = torch.zeros_like(pos[0], dtype=torch.int64)
        for d in range(self.D):
            c = torch.floor(pos[d] - self.lb).to(torch.int64)
            c = torch.remainder(c, self.n[d]) if self.periodic else c
            key = key * ((self.n[d] + (1 << shift) - 1) >> shift) + (c >> shift)
        for v in vel:
            key = key * 2 + (v >= 0).to(torch.int64)
        perm = torch.sort(key, stable=True)[1]
        return [x[perm] for x in pos], [v[perm] for v in vel]


def dirichlet(b, face=None):
    """(-Laplacian phi = b) with phi 0 on the faces (or `face` on the low
    face of axis 0), by sine transforms"""
    D, n = b.dim(), [m - 2 for m in b.shape]
    r = b[tuple(slice(1, -1) for _ in range(D))].clone()
    if face is not None:
        r[0] += face
    lam = torch.zeros_like(r)
    mats = []
    for d in range(D):
        k = torch.arange(1, n[d] + 1, device=b.device, dtype=torch.float64)
        mats.append(torch.sin(math.pi * torch.outer(k, k) / (n[d] + 1)))
        shape = [1] * D
        shape[d] = n[d]
        lam = lam + (2 - 2 * torch.cos(math.pi * k / (n[d] + 1))).reshape(shape)

    def sweep(a):
        for d in range(D):
            a = torch.tensordot(mats[d], a, dims=([1], [d])).movedim(0, d)
        return a
    r = sweep(sweep(r) / lam)
    for d in range(D):
        r = r * (2.0 / (n[d] + 1))
    out = torch.zeros_like(b)
    out[tuple(slice(1, -1) for _ in range(D))] = r
    if face is not None:
        out[0] = face
    return out


def _where_fp64(dtype, pos):
    """periodic positions: one that rounds across the period in FP32 wraps on
    one side only, so they are compared where they are FP64"""
    return pos if dtype == "f64" else [None] * len(pos)


def _exact_steps(pic, species, steps, dt, rho_bg, shift, sort=True):
    """`steps` steps of the loop; returns (hist, phi, species states)"""
    state = []
    for sp in species:
        pos, vel = [x.double() for x in sp["pos"]], [v.double() for v in sp["vel"]]
        state.append(list(pic.sorted(pos, vel, shift)) if sort else [pos, vel])
    hist = torch.zeros(steps, 5, dtype=torch.float64)
    phi = None
    for s in range(steps):
        rho = torch.full((math.prod(pic.n),), float(rho_bg), dtype=torch.float64, device="cuda")
        live = []
        for sp, (pos, vel) in zip(species, state):
            ok = torch.isfinite(pos[0])
            live.append(ok)
            w = sp["q"] * sp["w"] * ok.double()
            safe = [torch.where(ok, x, 0.5 * torch.ones_like(x)) for x in pos]
            rho += pic.deposit(safe, w)
        if pic.periodic:
            rho -= rho.mean()
        phi = pic.solve(rho)
        hist[s, 0] = pic.energy(phi).item()
        for sp, st, ok in zip(species, state, live):
            pos, vel = st
            mw = sp["m"] * sp["w"]
            hist[s, 1] += sum((0.5 * mw * v[ok] * v[ok]).sum().item() for v in vel)
            for d in range(pic.D):
                hist[s, 2 + d] += (mw * vel[d][ok]).sum().item()
            safe = [torch.where(ok, x, 0.5 * torch.ones_like(x)) for x in pos]
            g = pic.grad(phi, safe)
            out = torch.zeros_like(ok)
            for d in range(pic.D):
                v = vel[d] - g[d] * (sp["q"] / sp["m"]) * dt
                x = pos[d] + v * dt
                if pic.periodic:
                    x = torch.where(x < 0, x + pic.n[d], torch.where(x >= pic.n[d], x - pic.n[d], x))
                else:
                    out |= ok & ~((x >= 0) & (x < pic.n[d] - 1))
                st[1][d] = torch.where(ok, v, vel[d])
                st[0][d] = torch.where(ok, x, pos[d])
            st[0][0] = torch.where(out, torch.full_like(st[0][0], float("nan")), st[0][0])
    return hist.numpy(), phi, state


def exact(case, seed):
    kind = case["kind"]
    if kind == "step2d":
        sp = _species_2d(case, seed, case["n0"], case["n1"], case["ppc"], case["load"], case["dtype"])
        pic = _Pic([case["n0"], case["n1"]], True, False, case["order"])
        hist, phi, st = _exact_steps(pic, [sp], STEPS, 0.05, 1.0, 0)
        return dict(hist=hist, phi=phi, particles=[_where_fp64(case["dtype"], st[0][0]) + st[0][1]])
    if kind == "box3d":
        sp = _species_box(case, seed)
        pic = _Pic([case["c0"] + 1, case["c1"] + 1, case["c2"] + 1], False, True)
        hist, phi, st = _exact_steps(pic, sp, STEPS, 0.1, 0.0, 2)
        # the first coordinate of an FP32 particle within rounding of a wall
        # may be the NaN of an absorbed one on one side only
        return dict(hist=hist, phi=phi, particles=[([None] if case["dtype"] == "f32" else [p[0]]) + p[1:] + v
                                                   for p, v in st])
    if kind == "solve":
        nodes = [n for n in (case["n0"], case["n1"], case["n2"]) if n > 1]
        b = torch.randn(math.prod(nodes), generator=_gen(seed), device="cuda", dtype=torch.float64) * 0.1
        return dirichlet(b.reshape(nodes), 1.0).reshape(-1)
    if kind == "loop":
        nodes, pos, vel, phi = _loop_inputs(case, seed)
        dx = case["dx"]
        pic = _Pic(nodes, True, False, 1, dx)
        p = phi.to(_tdt(case["dtype"])).double()
        pos, vel = [x.double() for x in pos], [v.double() for v in vel]
        if case["sort"]:
            key = torch.zeros_like(pos[0], dtype=torch.int64)
            ok = torch.isfinite(pos[0])
            for d in range(pic.D):
                c = torch.floor((torch.where(ok, pos[d], 0.0) - pic.lb) / dx).to(torch.int64)
                key = key * nodes[d] + torch.remainder(c, nodes[d])
            key[~ok] = 2 ** 40
            perm = torch.sort(key, stable=True)[1]
            pos, vel = [x[perm] for x in pos], [v[perm] for v in vel]
        ok = torch.isfinite(pos[0])
        pos, vel = [x[ok] for x in pos], [v[ok] for v in vel]
        m = _LOOP["mass"]
        diag = torch.stack([sum((0.5 * m * v * v).sum() for v in vel)] + [(m * v).sum() for v in vel] +
                           [torch.zeros((), dtype=torch.float64, device="cuda")] * (3 - pic.D))
        g = pic.grad(p, pos)
        vel = [v - gd * _LOOP["qm"] * _LOOP["dt"] for v, gd in zip(vel, g)]
        pos = [x + v * _LOOP["dt"] for x, v in zip(pos, vel)]
        pos = [torch.where(x < 0, x + n * dx, torch.where(x >= n * dx, x - n * dx, x)) for x, n in zip(pos, nodes)]
        out = dict(acc=None, diag=diag, energy=pic.energy(phi), vel=vel,
                   pos=_where_fp64(case["dtype"], pos))
        if case["sort"]:
            out.update(keys=None, perm=None)
        return out
    if kind == "adjoint":
        n = case["n"]
        sp = _species_2d(case, seed, n, n, case["ppc"], "two_stream", case["dtype"])
        pic = _Pic([n, n], True, False)
        leaves = [a.double().requires_grad_(True) for a in sp["pos"] + sp["vel"]]
        pos, vel = leaves[:2], leaves[2:]

        def field(pos):
            rho = pic.deposit(pos, sp["q"] * sp["w"]) + 1.0
            return pic.solve(rho - rho.mean())
        for _ in range(case["steps"]):
            g = pic.grad(field(pos), pos)
            vel = [v + gd * 0.05 for v, gd in zip(vel, g)]
            pos = [x + v * 0.05 for x, v in zip(pos, vel)]
            pos = [x - n * torch.floor(x.detach() / n) for x in pos]
        loss = pic.energy(field(pos))
        return dict(loss=loss.detach(), grads=list(torch.autograd.grad(loss, leaves)))
    if kind == "batch":
        out = []
        for n, _, sp in _batch_specs(case, seed):
            _, phi, st = _exact_steps(_Pic([n, n], True, False), [sp], STEPS, 0.05, 1.0, 0)
            out.append(dict(phi=phi, particles=_where_fp64("f32", st[0][0]) + st[0][1]))
        return out
    if kind == "mcc" and not case["ionization"]:
        return _exact_mcc(case, seed)
    return None          # the mesh scene's exact hits and ionization products take too long in plain torch


def _exact_mcc(case, seed):
    x, v, s = _mcc_inputs(case, seed)
    v = [a.double() for a in v]
    lcg = s.to(torch.int64) & 0xFFFFFFFF

    def step(state):
        state = (state * 1664525 + 1013904223) & 0xFFFFFFFF
        return state, state.double() / 4294967295.0
    v2 = v[0] * v[0] + v[1] * v[1] + v[2] * v[2]
    lcg, r = step(lcg)
    areas = []
    for _, f, _ in _channels()[:3]:
        lx = torch.log(v2)
        y = [c[2] * lx * lx + c[3] * lx + c[4] for c in f["coef"]]
        y = y[0] if len(y) == 1 else torch.where(lx < f["seg_hi"][0], y[0], y[1])
        areas.append(torch.exp(y))
    total = areas[0] + areas[1] + areas[2]
    thr = r * total
    chosen = torch.where(thr <= areas[0], 0, torch.where(thr <= areas[0] + areas[1], 1, 2))
    chosen = torch.where(total > 0, chosen, -1)
    after, r2 = step(lcg)
    lcg = torch.where(chosen >= 0, after, lcg)
    hit = (chosen >= 0) & (r2 < total * _MCC_DT * _DENS * torch.sqrt(v2))
    a, ra = step(lcg)
    _, rb = step(a)
    c = 2 * ra - 1
    sn, ang = torch.sqrt(1 - c * c), 2 * math.pi * rb
    thr_ev = torch.tensor([t for _, _, t in _channels()[:3]], device="cuda", dtype=torch.float64)
    left = v2 - 2 * _QE * thr_ev[chosen.clamp(min=0)] / _ME
    speed = torch.sqrt(torch.where(chosen == 0, v2, left.clamp(min=0)))
    moved = hit & ((chosen == 0) | (left > 0))
    new = [c * speed, sn * torch.sin(ang) * speed, sn * torch.cos(ang) * speed]
    return dict(made=0, vel=[torch.where(moved, p, q) for p, q in zip(new, v)], seed=None)
