"""The on-chip BiCGStab (tanks of up to 2048 tiles) at the edges of its blocks: one tile, ragged
tiles in every direction, one block and many, one and two tiles per work item, the largest
tank, and the first size above it, which the streaming phases solve.

The first iterations follow the oracle's, as those of the streaming solver do.  Tolerance:
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
    """A wait limit of 0: the blocks of a tank leave at the commit with nothing stored, and the
    solve streams, with the same bits.  The next 63 solves stream without a launch, the 64th
    tries again, and a limit that allows it runs on chip.  A tank of one block waits for nothing
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
    D.set_control("onchip_wait", 0)
    r2, x2, chip, stream = run(20000)
    assert (chip, stream) == ((1, 0) if one_block else (1, 1))
    assert r2 == r and np.array_equal(x2, x)
    first = run(3)
    for _ in range(62):
        again = run(3)
        assert again[0] == first[0] and np.array_equal(again[1], first[1]) and again[2] == (1 if one_block else 0)
    assert run(3)[2] == 1
    D.set_control("onchip_wait", 0.5)
    r2, x2, chip, stream = run(20000)
    assert (chip, stream) == (1, 0) and r2 == r and np.array_equal(x2, x)
