"""The solve as one resident launch (small meshes) against the same solve by
launches: the fields and the solver records are the same bits, whatever the
number of workgroups, the preconditioner form and the precision, also when a
workgroup gives up its wait (residentPolls 1) and the solve is run again by
launches from the saved theta.  residentPolls 0 never uses the resident launch."""
import threading

import numpy as np
import pytest

from rheotool_amd import abi, cases

pytestmark = pytest.mark.gpu

FORMS = [("PBiCGStab", "DILU"), ("PBiCGStab", "diagonal"), ("PBiCGStab", "none"), ("PBiCG", "DILU")]


def step(m, f, controls, steps=2):
    """The steps in a context of their own: results, records, fields, solve counts."""
    with abi.Context(0) as ctx:
        eq = ctx.constitutiveEq("", ctx.mesh(m), abi.model_dict("GiesekusLog", lam=2.0, alpha=0.2))
        eq.set_solver(controls)
        eq.set_state(f.theta, f.eigVals, f.eigVecs)
        eq.set_flow(f.U, f.Ub, f.phi)
        rcs = [eq.correct(0.2 / max(m.nCells ** 0.5, 1.0)) for _ in range(steps)]
        perf = [(q.initialResidual, q.finalResidual, q.nIterations, q.nRefinements, q.converged, q.solved)
                for q in eq.solver_perf()]
        return rcs, perf, eq.theta(), eq.tau(), ctx.solve_counts


def workgroups(n, solver, precond):
    """Workgroups of the solve of an n-cell two-colourable mesh whose rows have at
    most six entries; 0: by launches."""
    rb = solver == "PBiCGStab" and precond == "DILU"
    P = -(-(n - n // 2 if rb else n) // 256)
    kept = rb or solver == "PBiCG"
    return P if P <= 128 and n <= (65536 if kept else 32768) else 0


# a workgroup takes 256 rows (red-black: 256 of each colour).  One row; one, two and
# more workgroups, full and not; just more than one XCD's 32 CUs hold in FP64 (8192
# rows; red-black 16384); the largest mesh the forms other than red-black take
# resident (32768 rows) and one row less than a workgroup below; red-black's (65536)
# and the first that is not
@pytest.mark.parametrize("shape", [(1, 1, 1), (16, 16, 1), (32, 16, 1), (27, 19, 1), (33, 32, 1), (13, 11, 9),
                                   (91, 91, 1), (129, 128, 1), (181, 181, 1), (256, 128, 1), (256, 256, 1),
                                   (257, 255, 1), (257, 256, 1)])
@pytest.mark.parametrize("precision", ["double", "mixed"])
def test_resident_solve_equals_launches(shape, precision):
    nx, ny, nz = shape
    m = cases.cartesian(nx, ny, nz, twoD=nz == 1 and nx > 1, channel=True)
    f = cases.make_fields(m, cases.FIELDS_CHANNEL, seed=nx + ny)
    for solver, precond in FORMS:
        base = abi.solver_dict(1e-10, solver=solver, precond=precond, precision=precision)
        print(f"[case] resident {shape} {solver} {precond} {precision}", flush=True)
        want = step(m, f, base + " residentPolls 0;")
        assert want[4] == (0, 0, 2)
        P = workgroups(m.nCells, solver, precond)
        for controls, gives_up in ((base, False), (base + " residentPolls 1;", True)):
            got = step(m, f, controls)
            assert got[0] == want[0] and got[1] == want[1]
            assert np.array_equal(got[2], want[2]) and np.array_equal(got[3], want[3])
            if P == 0:
                assert got[4] == (0, 0, 2)
            elif not gives_up or P == 1:
                assert got[4] == (2, 0, 0)
            else:
                assert got[4][0] + got[4][2] == 2
                assert got[4][1] >= 1 or P < 8  # a few workgroups may all arrive within a poll


@pytest.mark.parametrize("n", [500, 5000, 20000])
@pytest.mark.parametrize("noalloc", [False, True])
def test_resident_symm_solve_equals_launches(n, noalloc):
    """A general LDU system on a random face graph (rows wider than the kept
    width, no two-colouring) and on a box (Schur pivots)."""
    rng = np.random.default_rng(n)
    for m in (cases.random_graph(n, kNear=5, sigma=0.5, seed=3), cases.cartesian(n // 100, 10, 10)):
        lo, up = -rng.uniform(0.1, 1.0, m.nInternal), -rng.uniform(0.1, 1.0, m.nInternal)
        d = np.full(m.nCells, 0.5)
        np.add.at(d, m.owner[:m.nInternal], -lo)
        np.add.at(d, m.neighbour, -up)
        src, psi = rng.normal(size=(m.nCells, 6)), rng.normal(size=(m.nCells, 6))
        for solver, precond in FORMS:
            base = abi.solver_dict(1e-10, solver=solver, precond=precond)
            print(f"[case] resident system {m.nCells} {solver} {precond} noalloc={noalloc}", flush=True)
            out = []
            for controls in (base + " residentPolls 0;", base, base + " residentPolls 1;"):
                with abi.Context(0) as ctx:
                    got = ctx.symm_solve(ctx.mesh(m), d, lo, up, src, psi, controls, noalloc=noalloc)
                    out.append((got[0], [q.nIterations for q in got[1]], ctx.solve_counts))
            assert [o[2][:2] for o in out[:2]] == [(0, 0), (1, 0)]
            assert out[2][2][1] == 1 or n < 2048
            for o in out[1:]:
                assert np.array_equal(o[0], out[0][0]) and o[1] == out[0][1]


# members on one XCD; on more than one (above 64 workgroups in FP32, 32 in FP64), beside small ones
@pytest.mark.parametrize("precision,sides", [("mixed", (40, 60, 80)), ("mixed", (220, 30, 190, 16)),
                                             ("double", (150, 30, 180, 140, 16))])
def test_resident_server_batch_gives_up_and_finishes(precision, sides):
    """A batch of resident solves whose waits give up finishes by launches,
    with the same bits."""
    with abi.Context(0) as ctx:
        reqs = []
        for i, n in enumerate(sides):
            m = cases.cartesian(n, n, 1, twoD=True, channel=True)
            reqs.append((ctx.mesh(m), cases.make_fields(m, cases.FIELDS_CHANNEL, seed=i), 0.1 / n))
        out, counts = {}, {}
        for polls in ("0", "1", "200000"):
            print(f"[case] server {sides} {precision} residentPolls {polls}", flush=True)
            srv = abi.Server(ctx, max_inflight=8)
            base = abi.solver_dict(1e-10, precision=precision) + f" residentPolls {polls};"
            ts = [srv.submit(dm, f, abi.model_dict("Oldroyd-BLog"), dt, base) for dm, f, dt in reqs]
            while srv.progress():
                pass
            out[polls] = [srv.poll(t) for t in ts]
            counts[polls] = srv.solve_counts
            srv.close()
        assert counts["0"] == (0, 0, len(sides)) and counts["200000"] == (len(sides), 0, 0)
        assert counts["1"][1] >= 1 and counts["1"][0] + counts["1"][2] == len(sides)
        for polls in ("1", "200000"):
            for a, b in zip(out[polls], out["0"]):
                assert np.array_equal(a["theta"], b["theta"]) and np.array_equal(a["tau"], b["tau"])


@pytest.mark.parametrize("precision,precond,side", [("mixed", "DILU", 220), ("double", "DILU", 150),
                                                    ("double", "diagonal", 120)])
def test_resident_modes_equal_launches(precision, precond, side):
    """The modes of a multiMode step as one group of resident solves, each more
    than an XCD holds."""
    m = cases.cartesian(side, side, 1, twoD=True, channel=True)
    f = cases.make_fields(m, cases.FIELDS_CHANNEL, seed=5)
    modes = [abi.model_dict("GiesekusLog", lam=lam, alpha=0.2, etaP=0.2) for lam in (0.5, 1.0, 2.0)]
    body = "\n".join("M%d {%s}" % (i, t.split("{", 1)[1].rsplit("}", 1)[0]) for i, t in enumerate(modes))
    text = "parameters\n{\n    type multiMode;\n    models\n    (\n" + body + "\n    );\n}\n"
    out = []
    for polls, counts in (("0", (0, 0, 6)), ("200000", (6, 0, 0)), ("1", None)):
        print(f"[case] modes {side} {precision} {precond} residentPolls {polls}", flush=True)
        with abi.Context(0) as ctx:
            eq = ctx.constitutiveEq("", ctx.mesh(m), text)
            eq.set_solver(abi.solver_dict(1e-10, precision=precision, precond=precond) + f" residentPolls {polls};")
            for u in eq.modes():
                u.set_state(f.theta, f.eigVals, f.eigVecs)
            eq.set_flow(f.U, f.Ub, f.phi)
            for _ in range(2):
                eq.correct(0.1 / side)
            got = [eq.tau()] + [u.theta() for u in eq.modes()]
            n = ctx.solve_counts
        out.append(got)
        assert n == counts if counts else n[1] >= 1 and n[0] + n[2] == 6
        assert all(np.array_equal(a, b) for a, b in zip(got, out[0]))


def test_resident_solves_of_several_threads_do_not_wait_for_each_other():
    """Threads whose resident solves take up to half the chip each, and a server's
    batch beside them: those there is no room for run by launches, none gives up."""
    sides, steps = (240, 225, 250, 240, 200, 240), 60
    ms = [cases.cartesian(n, n, 1, twoD=True, channel=True) for n in sides]
    fs = [cases.make_fields(m, cases.FIELDS_CHANNEL, seed=i) for i, m in enumerate(ms)]
    controls = [abi.solver_dict(1e-10, precision="mixed" if i == 4 else "double") for i in range(len(sides))]
    want = [step(m, f, c, steps) for m, f, c in zip(ms, fs, controls)]
    got, served = {}, {}

    def serve():
        with abi.Context(0) as ctx:
            reqs = [cases.cartesian(n, n, 1, twoD=True, channel=True) for n in (150, 100, 210, 60)]
            flds = [cases.make_fields(m, cases.FIELDS_CHANNEL, seed=9) for m in reqs]
            dms = [ctx.mesh(m) for m in reqs]
            srv = abi.Server(ctx, max_inflight=8)
            for _ in range(steps // 2):
                for dm, f in zip(dms, flds):
                    srv.submit(dm, f, abi.model_dict("Oldroyd-BLog"), 1e-3, abi.solver_dict(1e-10, precision="mixed"))
                while srv.progress():
                    pass
            served["counts"] = srv.solve_counts
            srv.close()

    def run(i):
        got[i] = step(ms[i], fs[i], controls[i], steps)

    ts = [threading.Thread(target=run, args=(i,)) for i in range(len(sides))] + [threading.Thread(target=serve)]
    print("[case] resident solves of seven threads", flush=True)
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    counts = [got[i][4] for i in range(len(sides))] + [served["counts"]]
    print(counts)
    assert all(c[1] == 0 for c in counts) and sum(counts[-1]) == 4 * (steps // 2)
    for i in range(len(sides)):
        assert want[i][4] == (steps, 0, 0)
        assert got[i][:2] == want[i][:2] and all(np.array_equal(a, b) for a, b in zip(got[i][2:4], want[i][2:4]))


def test_after_a_wait_gave_up_the_next_solves_run_by_launches():
    m = cases.cartesian(128, 128, 1, twoD=True, channel=True)
    f = cases.make_fields(m, cases.FIELDS_CHANNEL, seed=1)
    with abi.Context(0) as ctx:
        eq = ctx.constitutiveEq("", ctx.mesh(m), abi.model_dict("GiesekusLog", lam=2.0, alpha=0.2))
        eq.set_state(f.theta, f.eigVals, f.eigVecs)
        eq.set_flow(f.U, f.Ub, f.phi)
        solves = []
        for polls, steps in (("1", 1), ("200000", 64), ("1", 1), ("200000", 128), ("200000", 128), ("1", 1), ("200000", 65)):
            eq.set_solver(abi.solver_dict(1e-10) + f" residentPolls {polls};")
            for _ in range(steps):
                eq.correct(1e-4)
            solves.append(ctx.solve_counts)
        print(solves)
        # (resident, gave up, by launches): 64 solves by launches after the first,
        # 128 after the second; 64 again once 128 resident solves have finished
        assert solves == [(0, 1, 1), (0, 1, 65), (0, 2, 66), (0, 2, 194), (128, 2, 194), (128, 3, 195), (129, 3, 259)]


@pytest.mark.parametrize("precision", ["double", "mixed"])
def test_a_budget_that_holds_the_launches_holds_the_step(precision):
    """The memory a resident solve saves its start in is taken if there is room:
    a context whose budget is just what the same steps take by launches runs them
    by launches, also with two modes, and one with more runs them resident."""
    m = cases.cartesian(120, 110, 1, twoD=True, channel=True)
    f = cases.make_fields(m, cases.FIELDS_CHANNEL, seed=2)
    one = abi.model_dict("GiesekusLog", lam=2.0, alpha=0.2)
    body = "\n".join("M%d {%s}" % (i, one.split("{", 1)[1].rsplit("}", 1)[0]) for i in range(2))
    for text, solves in ((one, 2), ("parameters\n{\n    type multiMode;\n    models\n    (\n" + body + "\n    );\n}\n", 4)):
        def run(budget, polls):
            with abi.Context(0, hbm_budget=budget) as ctx:
                eq = ctx.constitutiveEq("", ctx.mesh(m), text)
                eq.set_solver(abi.solver_dict(1e-10, precision=precision) + polls)
                for u in eq.modes() or [eq]:
                    u.set_state(f.theta, f.eigVals, f.eigVecs)
                eq.set_flow(f.U, f.Ub, f.phi)
                for _ in range(2):
                    eq.correct(1e-3)
                used = ctx.bytes_in_use
                return eq.tau(), ctx.solve_counts, used
        want, counts, used = run(0, " residentPolls 0;")
        assert counts == (0, 0, solves)
        used_at_most = used + (16 << 10)  # a group's argument tables, held during a step
        for budget, polls, counts in ((used_at_most, " residentPolls 0;", (0, 0, solves)),
                                      (used_at_most, "", (0, 0, solves)), (2 * used, "", (solves, 0, 0))):
            print(f"[case] budget {budget} {precision} {solves}{polls}", flush=True)
            got = run(budget, polls)
            assert got[1] == counts and got[2] == used and np.array_equal(got[0], want)


def test_a_servers_budget_admits_what_it_admitted_without_resident_solves():
    m = cases.cartesian(120, 110, 1, twoD=True, channel=True)
    f = cases.make_fields(m, cases.FIELDS_CHANNEL, seed=2)
    with abi.Context(0) as ctx:
        dm = ctx.mesh(m)
        est = abi.lib().rt_request_bytes_estimate(dm.h, 1, 0)
        out = []
        for budget, counts in ((est, (0, 0, 3)), (2 * est, (3, 0, 0))):
            print(f"[case] server budget {budget}", flush=True)
            srv = abi.Server(ctx, hbm_budget=budget, max_inflight=1)
            ts = [srv.submit(dm, f, abi.model_dict("Oldroyd-BLog"), 1e-3) for _ in range(3)]
            while srv.progress():
                pass
            out += [srv.poll(t)["theta"] for t in ts]
            assert srv.solve_counts == counts
            srv.close()
        assert all(np.array_equal(a, out[0]) for a in out)


def test_a_servers_groups_share_their_streams_cus():
    """The forms of a burst run in groups of their own, one after another on the
    server's stream: none is kept from running resident by another."""
    with abi.Context(0) as ctx:
        ms = [cases.cartesian(n, n, 1, twoD=True, channel=True) for n in (170, 120, 150, 60)]
        dms = [ctx.mesh(m) for m in ms]
        fs = [cases.make_fields(m, cases.FIELDS_CHANNEL, seed=4) for m in ms]
        text = abi.model_dict("Oldroyd-BLog")
        controls = [abi.solver_dict(1e-10, precision=p, precond=c) for p in ("mixed", "double") for c in ("DILU", "diagonal")]
        print("[case] server, four forms", flush=True)
        out = {}
        for polls in ("", " residentPolls 0;"):
            srv = abi.Server(ctx, max_inflight=16)
            ts = [srv.submit(dm, f, text, 1e-3, c + polls) for c in controls for dm, f in zip(dms, fs)]
            while srv.progress():
                pass
            out[polls] = [srv.poll(t)["theta"] for t in ts]
            assert srv.solve_counts == ((16, 0, 0) if not polls else (0, 0, 16))
            srv.close()
        assert all(np.array_equal(a, b) for a, b in zip(*out.values()))
