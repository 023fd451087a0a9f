"""P2G over every tile shape of its gather, against the oracle.

The gather's tile (y-nodes by x-planes) follows the particle count per z-extent, so each case here
has the count that selects one shape, on a small ragged grid: sides that no tile divides, two
z-tiles of unequal width (65 nodes), rows of bins with more records than one staged chunk, empty
tiles, and particles in random order (bins hold indices out of order before they are sorted).
FP64 must agree bit for bit; mixed precision within the worst-case rounding of an FP32 sum over the
particles that reach a node (weights and sums each contribute one rounding of 2^-24 per term).
"""
import numpy as np
import pytest

from tests.conftest import announce

pytestmark = pytest.mark.gpu

# a shape of yh x x nodes is taken from 350 * 64 * 8 / 3 * yh * x particles on (three face grids
# together), from 350 * 64 * 8 * yh * x above 2^22 particles (one face grid at a time); 8 x 16, from
# 23 M on, is the 256^3 workload's
CASES = [(0, 33), (3, 33), (20_000, 33), (250_000, 65), (500_000, 33), (1_000_000, 65), (2_000_000, 33),
         (4_000_000, 33), (4_300_000, 33)]
ARRAYS = ["u", "v", "w", "uw", "vw", "ww", "u_last", "v_last", "w_last"]


def scene(count, n, nz):
    rng = np.random.default_rng(count + nz)
    size = np.array([1.0, 1.0, nz / n])
    lo, hi = 0.1 * size, np.array([0.62, 0.95, 1.0]) * size  # empty planes at high x, walls touched in z
    pos = lo + (hi - lo) * rng.random((count, 3))
    if count > 100:  # a crowded bin and particles on the walls
        pos[: count // 50] = 0.5 * size + 0.2 / n * rng.random((count // 50, 3))
        pos[count // 50: count // 50 + 3] = 0.0
        pos[-3:] = size
    return pos, rng.uniform(-1.0, 1.0, (count, 3))


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "mixed"])
@pytest.mark.parametrize("count,nz", CASES)
def test_p2g_tile_shapes(hip, oracle, count, nz, precision):
    n = 21
    announce(f"p2g shapes count={count} nz={nz} precision={precision}")
    kw = dict(nx=n, ny=n, nz=nz, size_z=nz / n)
    pos, vel = scene(count, n, nz)
    if precision:
        pos, vel = pos.astype(np.float32).astype(np.float64), vel.astype(np.float32).astype(np.float64)
        pos = np.minimum(pos, np.array([1.0, 1.0, nz / n]))
    g = hip.FluidSim(hip.default_config(precision=precision, **kw))
    o = oracle.OracleSim(oracle.default_config(**kw))
    for s in (g, o):
        s.set_particles(pos, vel)
        s.p2g(0.0)
    for nm in ("u_valid", "v_valid", "w_valid"):
        if not precision:
            assert np.array_equal(g.get(nm), o.get(nm)), nm
    for nm in ARRAYS:
        a, b = g.get(nm), o.get(nm)
        if not precision:
            assert np.array_equal(a, b), nm
            continue
        # terms per node: at most 64 bins of the fullest bin's particles
        terms = 64 * max(1, int(count / 50 + 16 * count / (n * n * nz)))
        tol = 2.0 * terms * 2.0 ** -24 + 1e-5
        scale = max(float(np.abs(b).max()), 1e-30)
        w = o.get(nm[0] + "w")
        mask = w > 1e-2 * max(float(w.max()), 1e-30)  # a node only grazed by a stencil has no accurate quotient
        if mask.any():
            assert float(np.abs(a - b)[mask].max()) <= tol * scale, nm


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "mixed"])
@pytest.mark.parametrize("count,nz", [(0, 33), (3, 33), (20_000, 33), (250_000, 65), (500_000, 33), (2_000_000, 33)])
def test_p2g_apic_tile_shapes(hip, oracle, count, nz, precision):
    """APIC's P2G over the same tiles, with the affine rows that G2P takes from random face grids. (Mixed
    precision: nodes four or more from every wall; a stencil cut by a wall has an ill-conditioned D.)"""
    n = 21
    announce(f"apic p2g shapes count={count} nz={nz} precision={precision}")
    kw = dict(nx=n, ny=n, nz=nz, size_z=nz / n, advection=hip.ADVECT_APIC)
    pos, vel = scene(count, n, nz)
    if precision:
        pos, vel = pos.astype(np.float32).astype(np.float64), vel.astype(np.float32).astype(np.float64)
        pos = np.minimum(pos, np.array([1.0, 1.0, nz / n]))
    g = hip.FluidSim(hip.default_config(precision=precision, **kw))
    o = oracle.OracleSim(oracle.default_config(**kw))
    for s in (g, o):
        s.set_particles(pos, vel)
        for nm in ("u", "v", "w"):
            shape, _ = g.array_info(nm)
            s.set(nm, np.random.default_rng(len(nm) + shape[0]).uniform(-1.0, 1.0, shape).astype(np.float32))
        s.g2p(0.0)
        s.clear()  # the oracle adds to the grids it finds
        s.p2g(0.0)
    inner = (slice(4, -4),) * 3
    for nm in ("u", "v", "w", "uw", "vw", "ww", "u_valid", "v_valid", "w_valid"):
        a, b = g.get(nm), o.get(nm)
        if not precision:
            assert np.array_equal(a, b), nm
        elif not nm.endswith("valid"):
            # terms as above; an affine row comes from 64 nodes and reaches two cells
            terms = 64 * max(1, int(count / 50 + 16 * count / (n * n * nz)))
            tol = 4.0 * (terms + 64) * 2.0 ** -24 + 1e-5
            w = o.get(nm[0] + "w")[inner]
            mask = w > 1e-2 * max(float(w.max()), 1e-30)
            if mask.any():
                assert float(np.abs(a - b)[inner][mask].max()) <= tol * max(float(np.abs(b).max()), 1e-30), nm
