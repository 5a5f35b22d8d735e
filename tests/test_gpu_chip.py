"""The on-chip BiCGStab (tanks of up to 2048 tiles) at the edges of its blocks: one tile, ragged
tiles in every direction, one block and many, one and two tiles per work item, the largest
tank, and the first size above it, which the streaming phases solve.

On chip and streamed, and by row classes and from the faces, a solve has the same bits.  The
first iterations follow the oracle's, as those of the streaming solver do.  Tolerance:
the device adds its dot products in another order than the oracle's serial loop, about
sqrt(N) eps = 1.6e-13 relative for the largest tank, and 12 iterations amplify that by less
than the 1e-10 that the first 40 iterations on the reference's fixture are held to."""
import numpy as np
import pytest

from tests._cases import inner
from tests.test_gpu_mixed import TOL, _system

pytestmark = pytest.mark.gpu

SHAPES = [(64, 1, 4, 0), (65, 1, 9, 0), (37, 1, 130, 0), (1150, 1, 157, 0), (2048, 1, 256, 0), (2049, 1, 256, 0),
          (16, 6, 12, 1), (65, 5, 33, 1), (130, 33, 37, 1), (192, 39, 64, 1)]


@pytest.mark.parametrize("shape", SHAPES)
def test_first_iterations_follow_the_oracle(shape):
    nx, ny, nz, jdir = shape
    O, D, M, b = _system(nx, ny, nz, jdir, seed=77 + nx)
    print(shape, flush=True)
    for it in (1, 3, 12):
        D.zero("work0")
        n, _ = D.solver("work0", "work1", 1e-300, it)
        x = np.zeros(O.shape)
        O.bicgstab(x, M, b.copy(), 1e-300, it)
        assert n == it
        got, ref = inner(D.get("work0")), inner(x)
        np.testing.assert_allclose(got, ref, rtol=0, atol=1e-10 * np.abs(ref).max(), err_msg=f"it={it}")


def _forms(D, forms, solve):
    """The results of solve() with the controls of each form, and the on-chip launches."""
    out = []
    D.timing(True)
    for controls in forms:
        for key, value in controls.items():
            D.set_control(key, value)
        for limit in (1, 3, 12, 20000):
            D.timing_reset()
            out.append((controls, limit, solve(limit), min(D.timing_get("chip")[1], 1)))
    n = len(out) // len(forms)
    for q, (controls, limit, (r, x), _) in enumerate(out):
        want = out[q % n][2]
        assert r == want[0], f"{controls} maxiter {limit}: {r} for {want[0]}"
        assert np.array_equal(x, want[1]), f"{controls} maxiter {limit}"
    return [launches for _, _, _, launches in out[::n]]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_on_chip_and_streamed_are_the_same_bits(shape, precision):
    nx, ny, nz, jdir = shape
    _, D, _, _ = _system(nx, ny, nz, jdir, seed=41 + nz)
    print(shape, precision, flush=True)

    def solve(limit):
        D.zero("work0")
        r = (D.solver if precision == "fp64" else D.solver_mixed)("work0", "work1", -TOL, limit)
        return r, D.get("work0")

    assert _forms(D, [dict(onchip=1024), dict(onchip=0)], solve) == [0 if nx > 2048 else 1, 0]


@pytest.mark.parametrize("shape,var", [(s, var) for s in [(64, 1, 4, 0), (65, 1, 9, 0), (700, 1, 130, 0), (16, 6, 12, 1),
                                                          (65, 5, 33, 1), (130, 33, 37, 1)]
                                       for var in (1, 2, 3, 4) if s[3] or var != 2])
def test_explicit_operator_on_chip_and_streamed_are_the_same_bits(shape, var):
    """The caller's matrix (diagonally dominant, of random coefficients) over the cells of each
    grid; the cells outside keep their values and take part in a restart."""
    nx, ny, nz, jdir = shape
    _, D, _, _ = _system(nx, ny, nz, jdir, seed=51)
    ie, je, ke = nx - (var == 1), ny - (var == 2), nz - (var == 3)
    rng = np.random.default_rng(nx + var)
    n = ie * je * ke
    M7 = -rng.uniform(0.5, 1.5, (7, n))
    at = np.indices((ie, je, ke)).reshape(3, -1)
    for q, (axis, end) in {1: (0, ie - 1), 2: (0, 0), 3: (1, je - 1), 4: (1, 0), 5: (2, ke - 1), 6: (2, 0)}.items():
        M7[q][at[axis] == end] = 0.0
    if not jdir:
        M7[3:5] = 0.0
    M7[0] = 1.05 * np.abs(M7[1:]).sum(axis=0)
    b, x0 = rng.standard_normal(n), rng.standard_normal((nz + 6, ny + 6, nx + 6))
    print(shape, var, flush=True)

    def solve(limit):
        D.put("work0", x0)
        r = D.solver_start(var, M7, b, "work0", -TOL, limit)
        return r, D.get("work0")

    assert _forms(D, [dict(onchip=1024), dict(onchip=0)], solve) == [1, 0]


@pytest.mark.parametrize("shape", [(16, 6, 12, 1), (65, 5, 33, 1), (130, 33, 37, 1), (193, 37, 101, 1), (64, 4, 65, 1),
                                   (70, 9, 129, 1)])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_row_classes_and_faces_are_the_same_bits(shape, precision):
    """Streamed, with the operator from the row classes and from the faces of every row."""
    nx, ny, nz, jdir = shape
    _, D, _, _ = _system(nx, ny, nz, jdir, seed=61)
    D.set_control("onchip", 0)
    print(shape, precision, flush=True)

    def solve(limit):
        D.zero("work0")
        r = (D.solver if precision == "fp64" else D.solver_mixed)("work0", "work1", -TOL, limit)
        return r, D.get("work0")

    _forms(D, [dict(rowclass=1), dict(rowclass=0)], solve)


@pytest.mark.parametrize("shape", [(64, 1, 4, 0), (1150, 1, 157, 0), (65, 5, 33, 1), (192, 39, 64, 1)])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_solution_and_its_scaling(shape, precision):
    """The oracle's residual of the solution meets the stop criterion (1.5 times it in FP64,
    whose iterated residual drifts from the true one), and the right-hand side 2b gives
    exactly 2x: a power of two changes no rounding, so a lost or stale value breaks it."""
    nx, ny, nz, jdir = shape
    O, D, M, b = _system(nx, ny, nz, jdir, seed=5 + nz)
    solve = D.solver if precision == "fp64" else D.solver_mixed
    print(shape, precision, flush=True)
    out = []
    for scale in (1.0, 2.0):
        rhs = np.zeros(O.shape)
        inner(rhs)[...] = scale * b.reshape(nx, ny, nz).transpose(2, 1, 0)
        D.put("work1", rhs)
        D.zero("work0")
        solve("work0", "work1", -TOL, 20000)
        out.append(D.get("work0"))
    assert O.residual(out[0], M, b.copy()) <= (1.5 if precision == "fp64" else 1.0) * TOL * np.linalg.norm(b)
    assert np.array_equal(inner(out[1]), 2.0 * inner(out[0]))


def test_iterations_beyond_one_launch():
    """More iterations than one launch runs (1024): the solve goes on where it stopped, in the
    same way each time, and stops at the asked count."""
    _, D, _, _ = _system(65, 5, 33, 1, seed=9)
    xs = []
    for _ in range(2):
        D.zero("work0")
        n, _ = D.solver("work0", "work1", 0.0, 1500)
        assert n == 1500
        xs.append(D.get("work0"))
    assert np.isfinite(xs[0]).all() and np.array_equal(xs[0], xs[1])


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_a_solve_streams_where_there_is_no_workspace(precision):
    """A limit below the workspace (25 MiB at the least): the solve runs by the streaming phases,
    with the same bits, and on chip again once the limit allows it."""
    _, D, _, _ = _system(65, 5, 33, 1, seed=21)
    solve = D.solver if precision == "fp64" else D.solver_mixed
    D.timing(True)
    out = []
    for mib, launches in ((1024, 1), (1, 0), (0, 0), (1024, 1)):
        D.set_control("onchip", mib)
        D.timing_reset()
        D.zero("work0")
        print(precision, mib, flush=True)
        r = solve("work0", "work1", -TOL, 20000)
        assert min(D.timing_get("chip")[1], 1) == launches
        out.append((r, D.get("work0")))
    for r, x in out[1:]:
        assert r == out[0][0] and np.array_equal(x, out[0][1])


@pytest.mark.parametrize("shape", [(64, 1, 4, 0), (1150, 1, 157, 0), (65, 5, 33, 1)])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_a_launch_that_is_given_up_streams_on(shape, precision):
    """The abort bit set before a launch: the blocks of a tank leave at the latest at the commit with
    nothing stored, and the solve streams, with the same bits.  The next 63 solves stream without a launch, the 64th
    tries again, and without it the solves run on chip.  A tank of one block waits for nothing
    and is not given up."""
    nx, ny, nz, jdir = shape
    _, D, _, _ = _system(nx, ny, nz, jdir, seed=31)
    solve = D.solver if precision == "fp64" else D.solver_mixed
    phase = "bicg_v" if precision == "fp64" else "mix_v"
    D.timing(True)
    one_block = nx * nz <= 256

    def run(limit):
        D.timing_reset()
        D.zero("work0")
        r = solve("work0", "work1", -TOL, limit)
        return r, D.get("work0"), min(D.timing_get("chip")[1], 1), min(D.timing_get(phase)[1], 1)

    print(shape, precision, flush=True)
    r, x, chip, stream = run(20000)
    assert (chip, stream) == (1, 0)
    D.set_control("onchip_giveup", 1)
    r2, x2, chip, stream = run(20000)
    assert (chip, stream) == ((1, 0) if one_block else (1, 1))
    assert r2 == r and np.array_equal(x2, x)
    first = run(3)
    for _ in range(62):
        again = run(3)
        assert again[0] == first[0] and np.array_equal(again[1], first[1]) and again[2] == (1 if one_block else 0)
    assert run(3)[2] == 1
    D.set_control("onchip_giveup", 0)
    r2, x2, chip, stream = run(20000)
    assert (chip, stream) == (1, 0) and r2 == r and np.array_equal(x2, x)
