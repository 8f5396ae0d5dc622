"""A stepper's solves replay several V-cycles per graph (runs of 8, 4, 2 and 1
cycles, then checked cycles; one-cycle graphs in the first solve).  Histories,
potentials and cycle counts are those of the same steps without graphs."""
import os
import threading
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


# odd and even sweep counts (the iterate ends in either of its buffers);
# tolerances that take 1, a few and more cycles than one run holds, or the limit
@pytest.mark.parametrize("nodes,depth", [((64, 48), 2), ((17, 19, 21), 2)])
@pytest.mark.parametrize("pre,post", [(2, 1), (1, 1)])
@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("tol,cycles", [(0.9, 40), (1e-6, 40), (1e-11, 60), (1e-30, 21), (1e-30, 1)])
def test_runs_of_cycles_equal_direct_launches(nodes, depth, pre, post, dtype, tol, cycles):
    from psum_amd import engine as E
    rng = np.random.default_rng(3)
    t = np.float64 if dtype == "f64" else np.float32
    walls = len(nodes) == 3
    n = 20_000
    ext = [m - 1 if walls else m for m in nodes]
    pos = [(rng.random(n) * L * 0.999).astype(t) for L in ext]
    vel = [rng.standard_normal(n).astype(t) for _ in nodes]
    fixed = None
    if walls:
        f = np.zeros(nodes, np.uint8)
        for d in range(3):
            s = [slice(None)] * 3
            for e in (0, -1):
                s[d] = e
                f[tuple(s)] = 1
        fixed = f.ravel()
    out = []
    for graph in (1, 0):
        g = E.wall_grid(ext) if walls else E.periodic_grid(list(nodes))
        kw = dict(fixed=fixed) if walls else {}
        st = E.Stepper(g, [dict(q=-1.0, m=1.0, w=0.1, pos=[a.copy() for a in pos], vel=[a.copy() for a in vel])],
                       dtype=dtype, mixed_mg=dtype == "f32", depth=depth, pre=pre, post=post, max_cycles=cycles,
                       tol=tol, dt=0.05, rho_bg=0.0 if walls else 1.0, sort_every=0, mg_graph=graph, **kw)
        h = [st.run(4), st.run(3)]
        out.append((np.concatenate(h), np.array(st.phi())))
    assert np.array_equal(out[0][0], out[1][0])
    assert np.array_equal(out[0][1], out[1][1])


def test_steppers_whose_threads_share_a_core():
    """Waiting for a check's norms gives way to other threads: two steppers on
    threads of one core overlap (alone 30 ms each: 58 ms when the wait held
    the core, 32 ms now), and their histories are those of stepping alone."""
    from psum_amd import engine as E
    from psum_amd.workloads import langmuir_2d

    def stepper(i):
        wl = langmuir_2d(n=64, ppc=16, seed=i)
        return E.Stepper(wl["grid"], wl["species"], depth=3, pre=2, post=1, max_cycles=40, tol=1e-10, dt=wl["dt"],
                         rho_bg=1.0)
    rounds, steps = 5, 60
    alone, t_alone = [], []
    for i in range(2):
        st = stepper(i)
        h = [st.run(steps)]
        for _ in range(rounds):
            t = time.perf_counter()
            h.append(st.run(steps))
            t_alone.append(time.perf_counter() - t)
        alone.append(np.concatenate(h))
        st.close()
    sts = [stepper(i) for i in range(2)]
    h = [[st.run(steps)] for st in sts]
    t_shared, cores = [], os.sched_getaffinity(0)
    os.sched_setaffinity(0, {min(cores)})      # the threads started from here inherit it
    try:
        for _ in range(rounds):
            th = [threading.Thread(target=lambda i=i: h[i].append(sts[i].run(steps))) for i in range(2)]
            t = time.perf_counter()
            for x in th:
                x.start()
            for x in th:
                x.join()
            t_shared.append(time.perf_counter() - t)
    finally:
        os.sched_setaffinity(0, cores)
    for i in range(2):
        assert np.array_equal(np.concatenate(h[i]), alone[i])
        sts[i].close()
    assert min(t_shared) < 1.6 * min(t_alone), (t_shared, t_alone)
