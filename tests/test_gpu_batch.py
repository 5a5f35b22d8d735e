"""Batched tanks on the GPU: many tanks advanced by the same launches.

A tank's arithmetic depends on the tank alone (its chunks and reduction order are fixed
by its own size), so every field of every tank after a batched momentum_FC3 step must be
bit-identical to the same tank run alone, in FP64 and in the mixed-precision projection;
and a tank run alone matches the CPU oracle within the solver tolerance.
"""
import numpy as np
import pytest

from tests._cases import inner

pytestmark = pytest.mark.gpu

FIELDS = ("phi", "u", "v", "w", "press", "ro", "visc")
SOLVED_RTOL = 1e-8


def _tank(nx, ny, nz, dx, depth, amp, wavelength, dt, jdir):
    from reef3d_amd.cases import wave_tank
    f = wave_tank(nx, ny, nz, dx, depth, amp, wavelength)
    kw = dict(nx=nx, ny=ny, nz=nz, XN=f["XN"], YN=f["YN"], ZN=f["ZN"], DYM=dx, DZM=dx, jdir=jdir, top_group=3,
              g=(0.0, 0.0, -9.81), dt=dt, N44=-1e-10, N46=20000)
    return kw, f


TANKS = [
    _tank(96, 9, 40, 0.02, 0.5, 0.02, 1.0, 0.004, 1),
    _tank(300, 1, 64, 0.025, 0.96, 0.05, 1.5, 0.005, 0),
    _tank(70, 5, 24, 0.03, 0.45, 0.03, 0.8, 0.003, 1),
    _tank(130, 1, 40, 0.04, 0.96, 0.08, 2.0, 0.006, 0),
]


def _initial(B, tid, kw, f):
    B.put(tid, "phi", f["phi"])
    for n in ("u", "v", "w", "press"):
        B.put(tid, n, f[n])


def _prepare(B):
    B.ghost_fill("phi", 4, 52)
    B.ghost_fill("u", 1, 10)
    B.ghost_fill("v", 2, 11)
    B.ghost_fill("w", 3, 12)
    B.ghost_fill("press", 4, 40)
    B.fluid_update()


def _run(tanks, steps, precision, graphs=False, every_step=False, d20=0):
    from reef3d_amd import Batch
    B = Batch()
    ids = [B.add(**kw) for kw, _ in tanks]
    for tid, (kw, f) in zip(ids, tanks):
        _initial(B, tid, kw, f)
    B.solver_config(precision)
    B.set_control("graphs", 1 if graphs else 0)
    B.set_control("D20", d20)
    _prepare(B)
    iters, history = [], []
    for _ in range(steps):
        it, _ = B.fc3_step()
        iters.append(it)
        if every_step:
            history.append([{n: B.get(tid, n) for n in FIELDS} for tid in ids])
    out = [{n: B.get(tid, n) for n in FIELDS} for tid in ids]
    B.close()
    return (history if every_step else out), iters


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_batch_results_identical_to_alone(precision):
    mixed, it_mixed = _run(TANKS, 2, precision)
    for q, t in enumerate(TANKS):
        alone, it_alone = _run([t], 2, precision)
        for n in FIELDS:
            assert np.array_equal(mixed[q][n], alone[0][n]), f"tank {q} {n} differs between batch and alone"
        assert [s[q] for s in it_mixed] == [s[0] for s in it_alone]


def test_batch_with_explicit_diffusion_identical_to_alone():
    """D20 = 1 (ediff2) on a batch: each tank's steps are the bits of the tank run alone,
    and the control reaches the batched launches (the results differ from D20 = 0)."""
    mixed, _ = _run(TANKS, 2, "fp64", graphs=True, d20=1)
    plain, _ = _run(TANKS, 2, "fp64", graphs=True)
    for q, t in enumerate(TANKS):
        alone, _ = _run([t], 2, "fp64", d20=1)
        for n in FIELDS:
            assert np.array_equal(mixed[q][n], alone[0][n]), f"tank {q} {n} differs between batch and alone"
        assert not np.array_equal(mixed[q]["u"], plain[q]["u"]), f"tank {q}: D20 = 1 changed nothing"


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_graph_replay_identical(precision):
    """Steps replayed from captured hipGraphs (segments and iteration batches) give the
    same bits as launch-by-launch steps, on every replay; the host reads all fields back
    between the replays."""
    eager, it_eager = _run(TANKS[:3], 3, precision, graphs=False, every_step=True)
    graph, it_graph = _run(TANKS[:3], 3, precision, graphs=True, every_step=True)
    assert it_eager == it_graph
    for step in range(3):
        for q in range(3):
            for n in FIELDS:
                assert np.array_equal(eager[step][q][n], graph[step][q][n]), \
                    f"step {step} tank {q} {n}: graph replay differs"


def test_batched_tank_matches_oracle():
    from oracle.oracle import Domain as ODomain
    res, _ = _run(TANKS, 1, "fp64")
    for q, (kw, f) in enumerate(TANKS):
        O = ODomain(**kw)
        st = {n: f[n].copy() for n in ("phi", "u", "v", "w", "press")}
        for n, kind, gcv in (("phi", 4, 52), ("u", 1, 10), ("v", 2, 11), ("w", 3, 12), ("press", 4, 40)):
            O.ghost(st[n], kind, gcv)
        st["ro"], st["visc"] = np.zeros_like(st["phi"]), np.zeros_like(st["phi"])
        O.fluid_update(st["phi"], st["ro"], st["visc"])
        O.fc3_step(*(st[n] for n in FIELDS))
        for n in ("phi", "u", "w", "press"):
            ref = inner(st[n])
            err = np.abs(inner(res[q][n]) - ref).max() / (np.abs(ref).max() or 1.0)
            assert err < SOLVED_RTOL, f"tank {q} {n}: rel err {err:.2e}"


def test_batch_slots_and_budget():
    from reef3d_amd import Batch, ReefError
    kw0, f0 = TANKS[0]
    # the grid with its boundary groups (the ghost programs of a free-surface top differ
    # from a wall's)
    need = Batch.tank_bytes(**{k: kw0[k] for k in ("nx", "ny", "nz", "XN", "YN", "ZN", "DYM", "DZM", "jdir",
                                                   "top_group")})
    assert need > 0
    B = Batch(hbm_budget_bytes=2.5 * need)
    a = B.add(**kw0)
    b = B.add(**kw0)
    with pytest.raises(ReefError):
        B.add(**kw0)
    B.remove(a)
    c = B.add(**kw0)
    assert c == a                      # the freed slot is reused
    slots, active, used = B.info()
    assert slots == 2 and active == 2 and used <= 2.5 * need
    # tank_bytes is exactly what a tank takes from the device pool, ghost programs included
    assert used == 2 * need
    # a tank added after others were stepped is advanced only once made active with them
    for t in (b, c):
        _initial(B, t, kw0, f0)
    _prepare(B)
    B.set_active([c])
    it, _ = B.fc3_step()
    assert it[c] > 0 and it[b] == 0
    B.close()


def test_autotune_plans_and_identity():
    """The autotuner leaves every tank's state unchanged, records a valid plan for each
    size bucket, and with that plan table a tank's step is the same alone and in the batch."""
    from reef3d_amd import Batch
    B = Batch()
    ids = [B.add(**kw) for kw, _ in TANKS]
    for tid, (kw, f) in zip(ids, TANKS):
        _initial(B, tid, kw, f)
    B.solver_config("mixed")
    _prepare(B)
    before = [{n: B.get(tid, n) for n in FIELDS} for tid in ids]
    nb = B.autotune(reps=1)
    plans = B.plans()
    assert nb == len(plans) >= 2
    for jdir, lg, ty, tz, cpt in plans:
        assert (ty, tz) in ((4, 1), (2, 2), (1, 4)) and (jdir == 1 or ty == 1) and 1 <= cpt <= 64
    for q, tid in enumerate(ids):
        for n in FIELDS:
            assert np.array_equal(before[q][n], B.get(tid, n)), f"autotune changed tank {q} {n}"
    B.fc3_step()
    batch = [{n: B.get(tid, n) for n in FIELDS} for tid in ids]
    B.close()
    for q, (kw, f) in enumerate(TANKS):
        A = Batch()
        for p in plans:
            A.set_plan(*p)
        t = A.add(**kw)
        _initial(A, t, kw, f)
        A.solver_config("mixed")
        _prepare(A)
        A.fc3_step()
        for n in FIELDS:
            assert np.array_equal(batch[q][n], A.get(t, n)), f"tank {q} {n}: tuned plan, alone != batch"
        A.close()


@pytest.mark.parametrize("precision,graphs", [("fp64", False), ("mixed", False), ("mixed", True)])
def test_scheduled_run_identical_to_lockstep(precision, graphs):
    """Iteration-level scheduling (each tank moves through its own steps, no lockstep at the
    pressure solves) gives the same bits and iteration counts as lockstep steps, also when
    the batches of recurring solving sets replay from captured graphs."""
    from reef3d_amd import Batch
    lock, it_lock = _run(TANKS, 2, precision)
    B = Batch()
    ids = [B.add(**kw) for kw, _ in TANKS]
    for tid, (kw, f) in zip(ids, TANKS):
        _initial(B, tid, kw, f)
    B.solver_config(precision)
    B.set_control("graphs", 1 if graphs else 0)
    _prepare(B)
    it = B.run(2)
    sched = [{n: B.get(tid, n) for n in FIELDS} for tid in ids]
    B.close()
    assert [it[t] for t in ids] == [it_lock[-1][q] for q in range(len(TANKS))]
    for q in range(len(TANKS)):
        for n in FIELDS:
            assert np.array_equal(sched[q][n], lock[q][n]), f"tank {q} {n}: scheduled != lockstep"


# more than 2048 tiles, which the streaming phases solve: 3-D (class walk) and 2-D
LARGE = [_tank(224, 40, 96, 0.03, 1.7, 0.05, 2.0, 0.004, 1), _tank(2049, 1, 256, 0.02, 3.0, 0.1, 3.0, 0.004, 0)]


@pytest.mark.parametrize("tanks", [TANKS[1:2], LARGE[:1], TANKS[1:3] + LARGE[1:]], ids=["small", "large", "several"])
@pytest.mark.parametrize("added", [0, 1, 8])
def test_run_after_a_change_of_precision(tanks, added):
    """A scheduled run in another precision than the run before, and back, with tanks added in
    between (8 more outgrow the device's tank table): the bits and the iteration counts of the
    same steps of each tank alone, in lockstep.  The same tanks solve in each run, so a launch
    plan kept for them from the other precision would be used again."""
    from reef3d_amd import Batch
    runs = ["fp64", "mixed", "fp64", "mixed"]
    more = [TANKS[2 + q % 2] for q in range(added)]
    B = Batch()
    print(len(tanks), added, flush=True)
    ids = [B.add(**kw) for kw, _ in tanks]
    for tid, (kw, f) in zip(ids, tanks):
        _initial(B, tid, kw, f)
    _prepare(B)
    its = []
    for step, precision in enumerate(runs):
        if step == 2 and more:
            new = [B.add(**kw) for kw, _ in more]
            for tid, (kw, f) in zip(new, more):
                _initial(B, tid, kw, f)
            B.set_active(new)
            _prepare(B)
            B.set_active()
            ids += new
        B.solver_config(precision)
        it = B.run(1)
        its.append([it[t] for t in ids])
    got = [{n: B.get(t, n) for n in FIELDS} for t in ids]
    B.close()
    for q, (kw, f) in enumerate((tanks + more)[:len(tanks) + 2]):
        first = 0 if q < len(tanks) else 2
        A = Batch()
        t = A.add(**kw)
        _initial(A, t, kw, f)
        _prepare(A)
        for step in range(first, len(runs)):
            A.solver_config(runs[step])
            it, _ = A.fc3_step()
            assert its[step][q] == it[t] > 0, f"tank {q} run {step}"
        for n in FIELDS:
            assert np.array_equal(got[q][n], A.get(t, n)), f"tank {q} {n}: scheduled != lockstep"
        A.close()


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_scheduled_run_whose_launches_are_given_up(precision):
    """Every on-chip launch given up (onchip_giveup), in lockstep and scheduled: the same bits."""
    from reef3d_amd import Batch
    lock, it_lock = _run(TANKS, 2, precision)
    for scheduled in (False, True):
        B = Batch()
        ids = [B.add(**kw) for kw, _ in TANKS]
        for tid, (kw, f) in zip(ids, TANKS):
            _initial(B, tid, kw, f)
        B.solver_config(precision)
        B.set_control("onchip_giveup", 1)
        _prepare(B)
        print(precision, scheduled, flush=True)
        it = B.run(2) if scheduled else [B.fc3_step()[0] for _ in range(2)][-1]
        assert [it[t] for t in ids] == [it_lock[-1][q] for q in range(len(TANKS))]
        for q, t in enumerate(ids):
            for n in FIELDS:
                assert np.array_equal(B.get(t, n), lock[q][n]), f"tank {q} {n}"
        B.close()


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("graphs", [False, True])
def test_class_walked_and_other_tanks_in_one_launch(precision, graphs):
    """3-D tanks with row classes and 2-D tanks in one set, all streamed, or the small ones on chip
    once the large ones have ended, in lockstep and scheduled: the bits and iterations of each
    tank alone, whose phases are launched for its own kind."""
    from reef3d_amd import Batch
    tanks = [TANKS[0], LARGE[0], TANKS[1], LARGE[1], TANKS[3]]
    alone = [_run([t], 2, precision) for t in tanks]
    for onchip in (0, 1024):
        for scheduled in (False, True):
            B = Batch()
            ids = [B.add(**kw) for kw, _ in tanks]
            for tid, (kw, f) in zip(ids, tanks):
                _initial(B, tid, kw, f)
            B.solver_config(precision)
            B.set_control("graphs", 1 if graphs else 0)
            B.set_control("onchip", onchip)
            _prepare(B)
            print(precision, graphs, onchip, scheduled, flush=True)
            it = B.run(2) if scheduled else [B.fc3_step()[0] for _ in range(2)][-1]
            assert [it[t] for t in ids] == [a[1][-1][0] for a in alone]
            for q, t in enumerate(ids):
                for n in FIELDS:
                    assert np.array_equal(B.get(t, n), alone[q][0][0][n]), f"tank {q} {n}"
            B.close()


def test_a_set_too_large_for_the_chip_streams_until_it_is_smaller():
    """Twelve mixed tanks of 1344 tiles: streamed together first, on chip when few are left (the
    iterations of a solve done partly in each form), the bits of the tanks alone."""
    from reef3d_amd import Batch
    tanks = [_tank(1300 - 24 * q, 1, 256, 0.02, 3.0, 0.1, 3.0 - 0.1 * q, 0.004, 0) for q in range(12)]
    B = Batch()
    ids = [B.add(**kw) for kw, _ in tanks]
    for tid, (kw, f) in zip(ids, tanks):
        _initial(B, tid, kw, f)
    B.solver_config("mixed")
    _prepare(B)
    B.timing(True)
    it = B.run(1)
    assert B.timing_get("mix_v")[1] > 0 and B.timing_get("chip")[1] > 0
    for q, t in enumerate(ids):
        alone, it1 = _run([tanks[q]], 1, "mixed")
        assert it[t] == it1[0][0]
        for n in FIELDS:
            assert np.array_equal(B.get(t, n), alone[0][n]), f"tank {q} {n}"
    B.close()


def test_ghost_fills_of_uneven_tanks():
    """One fill of 1 and of many tanks from 4 to 2049 columns, 2-D and 3-D: each has the ghost
    layers it gets alone, for every program of a step."""
    from reef3d_amd import Batch
    sizes = [(4, 1, 4, 0), (2049, 1, 256, 0), (65, 5, 33, 1), (12, 10, 8, 1), (130, 33, 37, 1), (64, 1, 9, 0)]

    def fill(shapes, fields):
        B = Batch()
        ids = []
        for nx, ny, nz, jdir in shapes:
            f = [0.02 * np.arange(-5, n + 6, dtype=np.float64) for n in (nx, ny, nz)]
            ids.append(B.add(nx, ny, nz, *f, 0.02, 0.02, jdir=jdir, top_group=3, g=(0.0, 0.0, -9.81)))
        out = []
        for name, kind, gcv in (("phi", 4, 52), ("u", 1, 10), ("v", 2, 11), ("w", 3, 12), ("press", 4, 40), ("ro", 4, 1)):
            for t, a in zip(ids, fields):
                B.put(t, name, a)
            B.ghost_fill(name, kind, gcv)
            out.append([B.get(t, name) for t in ids])
        B.close()
        return out

    fields = [np.random.default_rng(q).standard_normal((nz + 6, ny + 6, nx + 6)) for q, (nx, ny, nz, _) in enumerate(sizes)]
    together = fill(sizes, fields)
    for q, s in enumerate(sizes):
        alone = fill([s], [fields[q]])
        assert all(np.array_equal(t[q], a[0]) for t, a in zip(together, alone)), s


def test_batch_refuses_differing_shared_parameters():
    """Only dt and F45 may differ between the tanks of a batch; the shared values stay
    those of the first tank added to the empty batch, also after that tank is removed."""
    from reef3d_amd import Batch, ReefError
    kw0, _ = TANKS[0]
    kw2, _ = TANKS[2]
    B = Batch()
    a = B.add(**kw0)
    b = B.add(**dict(kw2, dt=0.001, F45=1.5))
    for bad in (dict(rho=(998.0, 1.205)), dict(g=(0.0, 0.0, -9.8)), dict(N44=-1e-9), dict(F43=0.5),
                dict(N46=100), dict(visc=(2.0e-6, 1.4938e-5))):
        with pytest.raises(ReefError):
            B.add(**dict(kw2, **bad))
    B.remove(a)
    with pytest.raises(ReefError):
        B.add(**dict(kw2, rho=(998.0, 1.205)))
    B.remove(b)
    B.add(**dict(kw2, rho=(998.0, 1.205)))   # an empty batch takes new shared values
    B.close()
