"""The branches of the WENO stencils, the streaming solver's walk over row density classes and the
host transfers at the sizes and values where they can go wrong."""
import numpy as np
import pytest

from tests._cases import inner

pytestmark = pytest.mark.gpu


def _tank(nx, ny, nz, jdir, dx=0.02, stretch=0.0):
    from oracle.oracle import Domain as ODomain
    from reef3d_amd import Domain as DDomain
    from reef3d_amd.cases import wave_tank
    f = wave_tank(nx, ny, nz, dx, depth=0.6 * nz * dx, amp=0.05 * 0.6 * nz * dx, wavelength=1.0)
    ZN = f["ZN"] + stretch * dx * np.sin(0.37 * np.arange(f["ZN"].size))
    kw = dict(nx=nx, ny=ny, nz=nz, XN=f["XN"], YN=f["YN"], ZN=ZN, DYM=dx, DZM=dx, jdir=jdir, top_group=3,
              g=(0.0, 0.0, -9.81), dt=0.005, N44=-1e-10, N46=20000)
    return f, ODomain(**kw), DDomain(**kw)


@pytest.mark.parametrize("shape", [(37, 9, 21, 1), (130, 5, 18, 1), (130, 1, 33, 0)])
@pytest.mark.parametrize("sides", ["above", "below", "per lane"])
@pytest.mark.parametrize("scale", [1.0, 1e40, 1e-40])
def test_weno_sides_and_guard(shape, sides, scale):
    """One upwind side per wavefront or one per lane, and values whose smoothness indicators
    leave the range of the unscaled divisions in part of the domain (scale 1e40): the bits of
    the oracle, as everywhere else."""
    nx, ny, nz, jdir = shape
    print(shape, sides, scale, flush=True)
    f, O, D = _tank(nx, ny, nz, jdir, stretch=0.1)
    rng = np.random.default_rng(nx + nz)
    vel = [{"above": -1.0, "below": 1.0, "per lane": 0.0}[sides] + 0.3 * rng.standard_normal(O.shape) for _ in range(3)]
    if sides != "per lane":
        vel = [np.sign(a.mean()) * np.abs(a) for a in vel]
    if not jdir:
        vel[1][...] = 0.0
    phi = f["phi"] + 0.1 * 0.02 * rng.standard_normal(O.shape)
    phi[: nz // 2] *= scale
    for kind, gcv, a in ((4, 52, phi), (1, 10, vel[0]), (2, 11, vel[1]), (3, 12, vel[2])):
        O.ghost(a, kind, gcv)
    for n, a in zip(("phi", "u", "v", "w"), (phi, *vel)):
        D.put(n, a)
    L = np.zeros(O.shape)
    O.hj(phi, *vel, L)
    D.zero("L")
    D.convection("phi", 4)
    assert np.array_equal(inner(D.get("L")), inner(L))
    # the transported component in the same range
    for ipol, acc in ((1, "F"), (2, "G"), (3, "H")):
        if ipol == 2 and not jdir:
            continue
        q = vel[ipol - 1].copy()
        q[: nz // 2] *= scale
        ref = np.zeros(O.shape)
        O.flux(ipol, q, *vel, ref)
        D.put("work0", q)
        D.zero(acc)
        D.convection("work0", ipol)
        assert np.array_equal(inner(D.get(acc)), inner(ref)), acc
    O.reini(phi, 2)
    D.reini("phi", 2)
    assert np.array_equal(inner(D.get("phi")), inner(phi))


@pytest.mark.parametrize("shape", [(37, 9, 21, 1), (130, 1, 33, 0)])
def test_quotients_that_overflow(shape):
    """Cells of +-1e307, whose differences overflow when divided by the width (0.02): infinities
    decide the upwind side of the reinitialisation and end in NaN, cell for cell as the oracle's."""
    nx, ny, nz, jdir = shape
    print(shape, flush=True)
    f, O, D = _tank(nx, ny, nz, jdir, stretch=0.1)
    rng = np.random.default_rng(nx)
    phi = f["phi"].copy()
    at = rng.integers(0, [nz, ny, nx], (12, 3))
    for q, (k, j, i) in enumerate(at):
        inner(phi)[k, j, i] = (-1e307, 1e307, 1e305)[q % 3]
    O.ghost(phi, 4, 52)
    vel = [rng.standard_normal(O.shape) for _ in range(3)]
    if not jdir:
        vel[1][...] = 0.0
    for kind, gcv, a in ((1, 10, vel[0]), (2, 11, vel[1]), (3, 12, vel[2])):
        O.ghost(a, kind, gcv)
    for n, a in zip(("phi", "u", "v", "w"), (phi, *vel)):
        D.put(n, a)
    L = np.zeros(O.shape)
    O.hj(phi, *vel, L)
    D.zero("L")
    D.convection("phi", 4)
    assert np.array_equal(inner(D.get("L")), inner(L), equal_nan=True)
    O.reini(phi, 1)
    D.reini("phi", 1)
    assert np.isnan(phi).any() and np.isfinite(inner(phi)).any()
    assert np.array_equal(inner(D.get("phi")), inner(phi), equal_nan=True)


@pytest.mark.parametrize("shape", [(300, 33, 75, 1), (129, 65, 70, 1), (64, 70, 131, 1)])
@pytest.mark.parametrize("stretch", [0.0, 0.2])
def test_class_walk(shape, stretch):
    """3-D tanks of more than 2048 tiles, ragged in every direction, uniform and stretched in z,
    with rows of water, of air and of both.  Tolerances: the first iterations follow the oracle's
    within what other summation orders allow (sqrt(N) eps = 2e-13, amplified by 12 iterations;
    1e-10 as for the other solver tests); the solutions meet the stop criterion in the oracle's
    residual (1.5 times it in FP64, whose iterated residual drifts from the true one)."""
    nx, ny, nz, jdir = shape
    print(shape, stretch, flush=True)
    f, O, D = _tank(nx, ny, nz, jdir, stretch=stretch)
    phi = f["phi"].copy()
    O.ghost(phi, 4, 52)
    b = np.random.default_rng(nx).standard_normal(nx * ny * nz)
    b -= b.mean()
    M = O.poisson(phi, np.zeros(O.shape), b.copy())
    D.put("phi", phi)
    rhs = np.zeros(O.shape)
    inner(rhs)[...] = b.reshape(nx, ny, nz).transpose(2, 1, 0)
    D.put("work1", rhs)
    for it in (1, 12):
        D.zero("work0")
        assert D.solver("work0", "work1", 1e-300, it)[0] == it
        x = np.zeros(O.shape)
        O.bicgstab(x, M, b.copy(), 1e-300, it)
        got, ref = inner(D.get("work0")), inner(x)
        np.testing.assert_allclose(got, ref, rtol=0, atol=1e-10 * np.abs(ref).max(), err_msg=f"it={it}")
    for solve, slack in ((D.solver, 1.5), (D.solver_mixed, 1.0)):
        D.zero("work0")
        solve("work0", "work1", -1e-10, 20000)
        assert O.residual(D.get("work0"), M, b.copy()) <= slack * 1e-10 * np.linalg.norm(b)


@pytest.mark.parametrize("shape", [(4, 1, 4), (150, 40, 60), (200, 60, 62), (401, 64, 64), (70000, 1, 4)])
def test_transfers_round_trip(shape):
    """Fields of one chunk, of several, of every copying thread and with slots used again, also
    after a field of another size; the reference layout takes another path to the same values."""
    from reef3d_amd import Domain as DDomain
    nx, ny, nz = shape
    print(shape, flush=True)
    nodes = [0.1 * np.arange(-5, n + 6, dtype=np.float64) for n in shape]
    D = DDomain(nx=nx, ny=ny, nz=nz, XN=nodes[0], YN=nodes[1], ZN=nodes[2], DYM=0.1, DZM=0.1, jdir=1 if ny > 1 else 0,
                top_group=3, g=(0.0, 0.0, -9.81), dt=0.005, N44=1e-10, N46=100)
    rng = np.random.default_rng(nx)
    a, b = rng.standard_normal(D.shape), rng.standard_normal(D.shape)
    D.put("work0", a)
    D.put("work1", b)
    assert np.array_equal(D.get("work0"), a)
    assert np.array_equal(D.get("work1"), b)
    assert np.array_equal(D.get("work1", layout="ref"), b.transpose(2, 1, 0))
    D.put("work2", np.ascontiguousarray(a.transpose(2, 1, 0)), layout="ref")
    assert np.array_equal(D.get("work2"), a)
