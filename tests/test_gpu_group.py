"""BiCGStab iterated inside one launch (csrc/group.hip): sizes at the edges of
its work-groups (512 faces; 256 for three species or hexahedra), remainders,
the smallest systems, both precisions, both face orders, batches, and the
launched iteration that takes over when a wait in the kernel gives up.  Solved
to 1e-13, so the oracle's solution is met to 1e-10 (the parity bar)."""
import dataclasses

import numpy as np
import pytest

from mhfem_amd import capi, problems
import _group
import pyoracle

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300)


CASES = {
    # 5, 456, 533, 1008 and 2080 faces
    "tri1": lambda: problems.heat_2d(s=1, dt=1e-3),
    "tri12": lambda: problems.heat_2d(s=12, dt=1e-3),
    "tri13": lambda: problems.heat_2d(s=13, dt=1e-3),
    "tri18_n2": lambda: problems.adr_2d(s=18, n=2),
    "tri26_n3": lambda: problems.adr_2d(s=26, n=3),
    # 480, 1012 and 41 faces
    "quad15": lambda: problems.heat_quads(s=15),
    "quad22_n2": lambda: problems.adr_quads(s=22, n=2),
    "edge40": lambda: problems.adr_1d(s=40, n=2),
    # 18, 378, 864, 1650 and 6528 faces
    "tet1": lambda: problems.darcy_3d(s=1, preconditioner="diagonal"),
    "tet3": lambda: problems.darcy_3d(s=3, preconditioner="diagonal"),
    "tet4_n2": lambda: problems.adr_3d(s=4, n=2, preconditioner="diagonal"),
    "tet5_n3": lambda: problems.adr_3d(s=5, n=3, preconditioner="diagonal"),
    "tet8": lambda: problems.darcy_3d(s=8, preconditioner="diagonal", shuffle_cells=3),
    # 756, 756 and 450 faces
    "hex6": lambda: problems.adr_hexes(s=6, n=1),
    "hex6_n2": lambda: problems.adr_hexes(s=6, n=2),
    "hex5_n3": lambda: problems.adr_hexes(s=5, n=3),
}


def _steps(pr, s, o, steps=2):
    t = 0.0
    for k in range(steps):
        st = s.step(t, pr.dt)
        o.step(t, pr.dt, tol=1e-13)
        t += pr.dt
        assert st.converged and st.iterations > 0
        assert rel(s.get_array("Z_iF"), o.array("Z_iF")) < 1e-10, k
        assert rel(s.get_array("Z_iK"), o.array("Z_iK")) < 1e-10, k


@pytest.mark.parametrize("groups", [0, 1])
@pytest.mark.parametrize("precision", ["fp64", "fp32-reliable", "fp32-refined"])
@pytest.mark.parametrize("case", sorted(CASES))
def test_one_launch_matches_oracle(case, precision, groups):
    print(f"\n[group] {case} {precision} groups {groups}", flush=True)
    pr = CASES[case]()
    s = capi.Solver(pr, preconditioner="diagonal", tol=1e-13, precision=precision, inner_tol=0.03, face_groups=groups)
    _steps(pr, s, pyoracle.Oracle(pr))
    assert _group.iterated_in_one_launch(s), _group.info(s)
    s.close()


@pytest.mark.parametrize("precision", ["fp64", "fp32-reliable", "fp32-refined"])
@pytest.mark.parametrize("mesh", ["tet", "tri", "hex"])
def test_neighbours_share_work_groups(mesh, precision):
    """Whatever the order of the matrix copy, the work-groups hold the same
    faces, and most of a face's neighbours are in its own."""
    pr = {"tet": lambda: problems.darcy_3d(s=12, preconditioner="diagonal"), "tri": lambda: problems.heat_2d(s=60),
          "hex": lambda: problems.adr_hexes(s=12, n=1)}[mesh]()
    share = []
    for groups in (0, 1):
        s = capi.Solver(pr, preconditioner="diagonal", tol=1e-8, precision=precision, inner_tol=1e-2,
                        face_groups=groups)
        assert s.step(0.0, pr.dt).converged
        i = _group.info(s)
        share.append(i["remote"] / i["neighbours"])
        if groups and precision == "fp64":  # the captured step iterates on the natural order
            s.step_graph(pr.dt, pr.dt)
            i = _group.info(s)
            share.append(i["remote"] / i["neighbours"])
        s.close()
    assert set(share) == {share[0]} and share[0] < 0.3, share


@pytest.mark.parametrize("restart", [3, 30, 32])
@pytest.mark.parametrize("case", sorted(CASES))
def test_gmres_cycles_match_oracle(case, restart):
    """GMRES(m) with each cycle in one launch; restarts of 3 (a part of a
    group of four dot products), 30 (the default) and 32 (the largest)."""
    print(f"\n[group] gmres {case} m {restart}", flush=True)
    pr = CASES[case]()
    s = capi.Solver(pr, solver="gmres", preconditioner="diagonal", tol=1e-13, gmres_restart=restart)
    _steps(pr, s, pyoracle.Oracle(pr))
    assert _group.iterated_in_one_launch(s), _group.info(s)
    s.close()


@pytest.mark.parametrize("solver,precision", [("bicgstab", "fp64"), ("bicgstab", "fp32-reliable"), ("gmres", "fp64")])
def test_a_wait_that_gives_up_hands_over(solver, precision):
    """With a bound of zero the first wait between two work-groups gives up:
    the solve is finished by the launched iteration, the next one tries one
    launch again, and after two in a row that gave up one does not.  With the
    bound back, solves run in one launch again."""
    pr = problems.adr_3d(s=6, n=2, preconditioner="diagonal")
    print(f"\n[group] handed over, {solver} {precision}", flush=True)
    s = capi.Solver(pr, solver=solver, preconditioner="diagonal", tol=1e-13, precision=precision, inner_tol=0.03)
    _group.wait_bound(s, 0)
    _steps(pr, s, pyoracle.Oracle(pr), steps=3)
    i = _group.info(s)
    # the second solve tries one launch again, the third does not
    assert (i["gave_up"], i["cooldown"]) == (2, 1) and i["launches"] >= 2, i
    _group.wait_bound(s, 500000)
    t = 3 * pr.dt
    for k in range(2):
        assert s.step(t, pr.dt).converged
        t += pr.dt
    j = _group.info(s)
    assert j["gave_up"] == 2 and j["cooldown"] == 0 and j["launches"] > i["launches"], j
    s.close()


@pytest.mark.parametrize("precision", ["fp32-reliable", "fp32-refined"])
def test_scaled_right_hand_side(precision):
    """A right-hand side times 2^117 gives the solution times 2^117, bit for
    bit, in as many iterations.  On edges every lane has two unused neighbour
    slots.  In the 15 iterations of this solve (one round, simulated in FP32,
    with perturbed inputs too) the vectors stay below 81 (1.4e37 scaled), while
    p carried along in an unused slot, if its neighbour's values are added
    there, passes 7.4e4 (1.2e40: past FP32)."""
    pr = problems.adr_1d(s=30, n=1)
    b = np.random.default_rng(9).standard_normal(pr.num_faces)
    b[0] *= 100.0
    s = capi.Solver(pr, preconditioner="diagonal", tol=1e-5, precision=precision, inner_tol=1e-5)
    s.preIterate(0.0, pr.dt)
    s.assembleLinearSystem(0.0, pr.dt)
    x, st = s.solve_rhs(b, np.zeros_like(b))
    xs, sts = s.solve_rhs(b * 2.0 ** 117, np.zeros_like(b))
    assert _group.iterated_in_one_launch(s), _group.info(s)
    assert st.converged and st.fallback_iterations == 0 and sts.fallback_iterations == 0
    assert st.iterations == sts.iterations and st.outer_iterations == sts.outer_iterations
    assert np.array_equal(xs, x * 2.0 ** 117)
    s.close()


@pytest.mark.parametrize("case", ["tet", "edge", "tri"])
def test_breakdown_inside_a_round(case):
    """Values on Dirichlet faces only, from zero: (r, r*) vanishes after the
    first iteration.  The restart belongs to its round, in one launch as by
    launches: a solve whose only round aims at the tolerance takes one FP64
    update, and the breakdown is no stall."""
    pr = {"tet": lambda: problems.adr_3d(s=6, n=2, preconditioner="diagonal"), "edge": lambda: problems.adr_1d(s=60),
          "tri": lambda: problems.adr_2d(s=18)}[case]()
    for off in (False, True):
        s = capi.Solver(pr, preconditioner="diagonal", tol=1e-2, precision="fp32-reliable", inner_tol=1e-2)
        _group.launched(s, off)
        s.preIterate(0.0, pr.dt)
        s.assembleLinearSystem(0.0, pr.dt)
        _, _, _, rhs = s.export_system()
        x, st = s.solve_rhs(rhs, np.zeros_like(rhs))
        i = _group.info(s)
        assert st.converged and st.fallback_iterations == 0 and st.iterations > 1
        # the round, and its second launch after the breakdown
        assert i["gave_up"] == 0 and i["launches"] == (0 if off else 2), i
        assert st.outer_iterations == 1, off
        s.close()


def test_no_round_behind_the_end_of_a_solve():
    """Rounds that end at nine tenths of the residual they start from do not
    halve it: two of them hand the solve to FP64.  The round queued behind the
    second does nothing; behind one that aims at the tolerance none is queued."""
    pr = dataclasses.replace(problems.heat_2d(s=40), dt=10.0)
    b = np.random.default_rng(0).standard_normal(pr.num_faces)
    s = capi.Solver(pr, preconditioner="diagonal", tol=1e-10, precision="fp32-reliable", inner_tol=0.9)
    s.preIterate(0.0, pr.dt)
    s.assembleLinearSystem(0.0, pr.dt)
    x, st = s.solve_rhs(b, np.zeros_like(b))
    i = _group.info(s)
    assert st.converged and st.fallback_iterations > 0
    assert i["launches"] == st.outer_iterations + 1 and i["iterations"] == 0, (st.outer_iterations, i)
    s.close()
    pr = problems.heat_2d(s=40)
    s = capi.Solver(pr, preconditioner="diagonal", tol=1e-3, precision="fp32-reliable", inner_tol=1e-3)
    st = s.step(0.0, pr.dt)
    i = _group.info(s)
    assert st.outer_iterations == i["launches"] == 1 and i["iterations"] > 0, (st.outer_iterations, i)
    s.close()


@pytest.mark.parametrize("graph", [False, True])
def test_a_batch_that_gives_up_hands_over(graph):
    """The same in a batch, where the launched iteration then narrows to the
    instances still running, and in captured steps, which are captured again
    with and without iterations."""
    members = [problems.ensemble_member(sd, 500 + k) for k, sd in enumerate([14, 30, 22, 3, 40, 26, 9])]
    batch = problems.concatenate(members)
    s = capi.Solver(batch, tol=1e-13)
    co, fo = s.batch_info()
    oracles = [pyoracle.Oracle(m) for m in members]
    t = 0.0
    for k, ticks in enumerate([500000, 0, 0, 0, 500000, 500000]):
        print(f"\n[group] batch, graph {graph}, step {k}, bound {ticks}", flush=True)
        _group.wait_bound(s, ticks)
        before = _group.info(s)
        (s.step_graph if graph else s.step)(t, batch.dt)
        i = _group.info(s)
        # in one launch; two tries that give up; by launches; in one launch
        assert i["gave_up"] - before["gave_up"] == (k in (1, 2)), (k, i)
        assert (i["launches"] > before["launches"]) == (k != 3), (k, i)
        z, zk = s.get_array("Z_iF"), s.get_array("Z_iK")
        for j, (m, o) in enumerate(zip(members, oracles)):
            o.step(t, m.dt, tol=1e-13)
            assert rel(z[fo[j]:fo[j + 1]], o.array("Z_iF")) < 1e-10, (k, j)
            assert rel(zk[co[j]:co[j + 1]], o.array("Z_iK")) < 1e-10, (k, j)
        t += batch.dt
    s.close()


@pytest.mark.parametrize("precision", ["fp64", "fp32-refined", "fp32-reliable"])
@pytest.mark.parametrize("limit", [1, 2, 7])
def test_iteration_limit_inside_the_launch(limit, precision):
    """A solve that stops at max_iterations stops there in both forms, with
    the same iterate up to the rounding of a few iterations (FP32: of its
    6e-8 numbers)."""
    pr = problems.adr_3d(s=6, n=2, preconditioner="diagonal")
    b = np.random.default_rng(1).standard_normal(pr.n * pr.num_faces)
    out = []
    for off in (False, True):
        s = capi.Solver(pr, preconditioner="diagonal", tol=1e-12, precision=precision, inner_tol=1e-4,
                        max_iterations=limit)
        _group.launched(s, off)
        s.preIterate(0.0, pr.dt)
        s.assembleLinearSystem(0.0, pr.dt)
        out.append(s.solve_rhs(b, np.zeros_like(b)))
        s.close()
    (x, st), (y, su) = out
    assert not st.converged and not su.converged
    assert st.iterations == su.iterations == limit
    assert np.linalg.norm(x - y) <= (1e-10 if precision == "fp64" else 1e-4) * np.linalg.norm(y)


def test_breakdown_inside_the_launch():
    """Values on Dirichlet faces only, from zero, in FP64: (r, r*) is zero
    after the first iteration, the launch ends, the host restarts it."""
    pr = problems.adr_2d(s=18)
    x = []
    for off in (False, True):
        s = capi.Solver(pr, preconditioner="diagonal", tol=1e-13)
        _group.launched(s, off)
        s.preIterate(0.0, pr.dt)
        s.assembleLinearSystem(0.0, pr.dt)
        _, _, _, rhs = s.export_system()
        z, st = s.solve_rhs(rhs, np.zeros_like(rhs))
        i = _group.info(s)
        assert st.converged and i["gave_up"] == 0 and (i["launches"] == 0 if off else i["launches"] >= 2), i
        x.append(z)
        s.close()
    assert rel(x[0], x[1]) < 1e-10


def test_batch_larger_than_the_chip():
    """More work-groups than fit at once: segments start in turn."""
    members = [problems.ensemble_member(sd, 40 + k) for k, sd in enumerate([150, 20, 90, 150, 150, 7, 150])]
    batch = problems.concatenate(members)
    s = capi.Solver(batch, tol=1e-12)
    co, fo = s.batch_info()
    assert fo[-1] > 2 * 131072
    s.step(0.0, batch.dt)
    rp, col, val, rhs = s.export_system()
    x = s.get_array("Z_iF")
    r = rhs - np.add.reduceat(val * x[col], rp[:-1])
    for k in range(len(members)):
        a, b = fo[k], fo[k + 1]
        assert np.linalg.norm(r[a:b]) < 2e-12 * np.linalg.norm(rhs[a:b]), k
    assert _group.iterated_in_one_launch(s) and _group.info(s)["total"] > 256, _group.info(s)
    s.close()


def test_batch_of_large_instances():
    """Instances of 130 to 163 shares, ten of them: while one iterates the
    work-groups left hold a part of the next, whose other shares must be taken
    once they are free, on every XCD.  No wait gives up."""
    sides = [3, 230, 230, 230, 230, 220, 215, 230, 210, 230, 235]
    members = [problems.ensemble_member(sd, 40 + k) for k, sd in enumerate(sides)]
    batch = problems.concatenate(members)
    s = capi.Solver(batch, tol=1e-12)
    co, fo = s.batch_info()
    for k in range(2):
        print(f"\n[group] large instances, step {k}", flush=True)
        s.step(k * batch.dt, batch.dt)
        assert _group.iterated_in_one_launch(s), _group.info(s)
    rp, col, val, rhs = s.export_system()
    r = rhs - np.add.reduceat(val * s.get_array("Z_iF")[col], rp[:-1])
    for k in range(len(members)):
        a, b = fo[k], fo[k + 1]
        assert np.linalg.norm(r[a:b]) < 2e-12 * np.linalg.norm(rhs[a:b]), k
    s.close()


@pytest.mark.parametrize("case,precision", [("tri", "fp64"), ("tri", "fp32-reliable"), ("tet", "fp32-reliable"),
                                            ("tet", "fp32-refined")])
def test_two_parts_per_work_group(case, precision):
    """Past 131,072 faces a work-group of 1024 threads takes two parts, the
    last one here a single part: 275 and 331 parts of 512 faces."""
    pr = {"tri": lambda: problems.heat_2d(s=216), "tet": lambda: problems.darcy_3d(s=24, preconditioner="diagonal")}[case]()
    assert -(-pr.num_faces // 512) == {"tri": 275, "tet": 331}[case]
    s = capi.Solver(pr, preconditioner="diagonal", tol=1e-12, precision=precision, inner_tol=0.03)
    assert s.step(0.0, pr.dt).converged
    assert _group.iterated_in_one_launch(s) and _group.info(s)["threads"] == 1024, _group.info(s)
    rp, col, val, rhs = s.export_system()
    r = rhs - np.add.reduceat(val * s.get_array("Z_iF")[col], rp[:-1])
    assert np.linalg.norm(r) < 2e-12 * np.linalg.norm(rhs)
    s.close()


def test_rows_read_from_memory():
    """Three species on hexahedra, past the faces whose rows fit in LDS (128
    per CU) and below those that fit on the chip at all."""
    pr = problems.adr_hexes(s=22, n=3)
    assert 128 * 256 < pr.num_faces < 256 * 256
    s = capi.Solver(pr, tol=1e-12)
    s.step(0.0, pr.dt)
    rp, col, val, rhs = s.export_system()
    r = rhs - np.add.reduceat(val * s.get_array("Z_iF")[col], rp[:-1])
    assert np.linalg.norm(r) < 2e-12 * np.linalg.norm(rhs)
    assert _group.iterated_in_one_launch(s) and _group.info(s)["hold"] == "memory", _group.info(s)
    s.close()


def test_overlapping_contexts():
    """Two contexts solve at the same time on their own streams."""
    import threading

    prs = [problems.heat_2d(s=60, dt=1e-3), problems.darcy_3d(s=9, preconditioner="diagonal")]
    oracles = [pyoracle.Oracle(p) for p in prs]
    for p, o in zip(prs, oracles):
        o.step(0.0, p.dt, tol=1e-13)
    solvers = [capi.Solver(p, preconditioner="diagonal", tol=1e-13) for p in prs]
    errors = []

    def work(p, s, o):
        for _ in range(5):
            s.set_array("Z_iK", p.Z_iK0)
            capi.lib().mhfem_init(s.ctx)
            s.step(0.0, p.dt)
            e = rel(s.get_array("Z_iF"), o.array("Z_iF"))
            if not e < 1e-10:
                errors.append(e)

    threads = [threading.Thread(target=work, args=a) for a in zip(prs, solvers, oracles)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors
    for s in solvers:
        assert _group.iterated_in_one_launch(s), _group.info(s)
        s.close()
