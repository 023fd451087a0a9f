"""Multigrid CG at the sizes where its kernels change form, against the oracle bit for bit: the
levels that share one workgroup (a first level of exactly 4096 cells, levels that are too long for it,
a single coarse level), 1024- and 256-thread blocks (up to and past 2048 chunks of 4096 cells), and
restriction by child and by aggregate (up to and past 2^18 aggregates). The systems are random
weighted 7-point Laplacians on a random active set, so no scene has to be run."""
import numpy as np
import pytest

from tests.conftest import announce

pytestmark = pytest.mark.gpu


def system(n, nz, seed):
    """Symmetric diagonally dominant system on an active block with holes."""
    rng = np.random.default_rng(seed)
    act = np.zeros((n, n, nz), dtype=bool)
    m = max(1, min(n, 40))
    act[: m, : max(1, (3 * m) // 4), : min(nz, 60)] = True
    act &= rng.random(act.shape) < 0.9
    act[0, 0, 0] = True
    arr = {"active": act.astype(np.uint8)}
    diag = np.where(act, 0.05, 0.0)
    for axis, (lo, hi) in enumerate([("a_left", "a_right"), ("a_down", "a_up"), ("a_back", "a_front")]):
        w = np.where(act, rng.uniform(0.2, 1.0, act.shape), 0.0)
        prev = np.roll(act, 1, axis)
        edge = [slice(None)] * 3
        edge[axis] = 0
        prev[tuple(edge)] = False
        w = np.where(prev, w, 0.0)  # coupling to the neighbour before
        wn = np.roll(w, -1, axis)
        edge[axis] = -1
        wn[tuple(edge)] = 0.0
        arr[lo], arr[hi] = -w, -wn
        diag += w + wn
    arr["adiag"] = diag
    arr["rhs"] = np.where(act, rng.standard_normal(act.shape), 0.0)
    return arr


@pytest.mark.parametrize("n,nz,iters", [(1, 1, 300), (2, 1, 300), (8, 8, 300), (32, 32, 300), (33, 31, 300),
                                        (3, 6000, 300), (30, 300, 300), (130, 127, 4), (210, 192, 3)])
def test_mg_solve_shapes(hip, oracle, n, nz, iters):
    announce(f"multigrid shapes n={n} nz={nz}")
    kw = dict(nx=n, ny=n, nz=nz, size_z=nz / n, preconditioner=hip.PRECOND_MULTIGRID, cg_max_iterations=iters)
    g = hip.FluidSim(hip.default_config(**kw))
    o = oracle.OracleSim(oracle.default_config(**kw))
    for name, a in system(n, nz, 100 * n + nz).items():
        g.set(name, a)
        o.set(name, a)
    so, sg = o.solve_pressure(), g.solve_pressure()
    assert sg["cg_iterations"] == so["cg_iterations"] and sg["status"] == so["status"], (sg, so)
    assert sg["residual_inf"] == so["residual_inf"]
    assert np.array_equal(g.get("pg"), o.get("pg"))
    g.close()
    o.close()
