"""Host copies through the pinned lanes: what is put in comes back, in both precisions, at sizes
around a piece's edge (2^20 device bytes), with one lane and with several, and the domain check
names the first particle that lies outside whichever thread finds it."""
import numpy as np
import pytest

from tests.conftest import announce

pytestmark = pytest.mark.gpu

# particles: 3 values each, 4 or 8 bytes a value; 87382 * 12 and 43691 * 24 are just past a piece
COUNTS = [0, 1, 43690, 43691, 87381, 87382, 262_144, 1_500_001]


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "mixed"])
@pytest.mark.parametrize("count", COUNTS)
def test_particles_round_trip(hip, count, precision):
    announce(f"particles round trip count={count} precision={precision}")
    rng = np.random.default_rng(count)
    pos, vel = rng.random((count, 3)), rng.standard_normal((count, 3))
    if count:
        vel[0] = [1e-310, -0.0, 3e-42]  # subnormals of FP64 and FP32, signed zero
    sim = hip.FluidSim(hip.default_config(nx=8, ny=8, nz=8, precision=precision))
    for v in (vel, None, vel):
        sim.set_particles(pos, v)
        p, u = sim.particles()
        cast = np.float32 if precision else np.float64
        want = np.zeros_like(vel) if v is None else vel
        assert np.array_equal(p, pos.astype(cast).astype(np.float64))
        assert np.array_equal(u, want.astype(cast).astype(np.float64))
        assert np.array_equal(np.signbit(u), np.signbit(want.astype(cast)))
    if count:
        c = rng.standard_normal((count, 3, 3))
        sim.set_particle_affine(c)
        assert np.array_equal(sim.particle_affine(), c.astype(cast).astype(np.float64))


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "mixed"])
@pytest.mark.parametrize("n,nz", [(1, 1), (7, 5), (64, 63), (100, 101)])
def test_arrays_round_trip(hip, n, nz, precision):
    announce(f"arrays round trip n={n} nz={nz} precision={precision}")
    rng = np.random.default_rng(n)
    sim = hip.FluidSim(hip.default_config(nx=n, ny=n, nz=nz, precision=precision))
    cast = np.float32 if precision else np.float64
    for name in ("u", "w", "fluid_sdf", "w_valid"):
        shape, dtype = sim.array_info(name)
        a = rng.integers(0, 2, shape).astype(dtype) if dtype == np.uint8 else rng.standard_normal(shape)
        sim.set(name, a)
        want = a if dtype == np.uint8 else a.astype(cast).astype(np.float64)
        assert np.array_equal(sim.get(name), want), name


@pytest.mark.parametrize("bad", [[0], [1_400_000, 900_000], [1_499_999]])
def test_first_particle_outside_is_named(hip, bad):
    pos = np.random.default_rng(3).random((1_500_000, 3))
    for k, i in enumerate(bad):
        pos[i, (i + k) % 3] = [1.5, np.nan][k]
    sim = hip.FluidSim(hip.default_config(nx=8, ny=8, nz=8))
    with pytest.raises(hip.FluidSimError, match=f"particle {min(bad)} lies outside"):
        sim.set_particles(pos)
    assert sim.num_particles() == 0
