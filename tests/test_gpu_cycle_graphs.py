"""A stepper's solves replay several V-cycles per graph (runs of 8, 4, 2 and 1
cycles, then checked cycles; one-cycle graphs in the first solve).  Histories,
potentials and cycle counts are those of the same steps without graphs."""
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
