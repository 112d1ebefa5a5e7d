"""The solve as one resident launch (small meshes) against the same solve by
launches: the fields and the solver records are the same bits, whatever the
number of workgroups, the preconditioner form and the precision, also when a
workgroup gives up its wait (residentPolls 1) and the solve is run again by
launches from the saved theta.  residentPolls 0 never uses the resident launch."""
import numpy as np
import pytest

from rheotool_amd import abi, cases

pytestmark = pytest.mark.gpu

FORMS = [("PBiCGStab", "DILU"), ("PBiCGStab", "diagonal"), ("PBiCGStab", "none"), ("PBiCG", "DILU")]


@pytest.fixture(scope="module")
def ctx():
    c = abi.Context(0)
    yield c
    c.close()


def step(ctx, dm, m, f, controls, steps=2):
    eq = ctx.constitutiveEq("", dm, abi.model_dict("GiesekusLog", lam=2.0, alpha=0.2))
    eq.set_solver(controls)
    eq.set_state(f.theta, f.eigVals, f.eigVecs)
    eq.set_flow(f.U, f.Ub, f.phi)
    rcs = [eq.correct(0.2 / max(m.nCells ** 0.5, 1.0)) for _ in range(steps)]
    perf = [(q.initialResidual, q.finalResidual, q.nIterations, q.nRefinements, q.converged, q.solved)
            for q in eq.solver_perf()]
    return rcs, perf, eq.theta(), eq.tau()


# a workgroup takes 256 rows (red-black: 256 of each colour).  One row; one, two and
# more workgroups, full and not; just more than one XCD's 32 CUs hold in FP64 (8192
# rows; red-black 16384); the largest mesh the forms other than red-black take
# resident (32768 rows) and one row less than a workgroup below; red-black's (65536)
# and the first that is not
@pytest.mark.parametrize("shape", [(1, 1, 1), (16, 16, 1), (32, 16, 1), (27, 19, 1), (33, 32, 1), (13, 11, 9),
                                   (91, 91, 1), (129, 128, 1), (181, 181, 1), (256, 128, 1), (256, 256, 1),
                                   (257, 255, 1), (257, 256, 1)])
@pytest.mark.parametrize("precision", ["double", "mixed"])
def test_resident_solve_equals_launches(ctx, shape, precision):
    nx, ny, nz = shape
    m = cases.cartesian(nx, ny, nz, twoD=nz == 1 and nx > 1, channel=True)
    f = cases.make_fields(m, cases.FIELDS_CHANNEL, seed=nx + ny)
    dm = ctx.mesh(m)
    for solver, precond in FORMS:
        base = abi.solver_dict(1e-10, solver=solver, precond=precond, precision=precision)
        print(f"[case] resident {shape} {solver} {precond} {precision}", flush=True)
        want = step(ctx, dm, m, f, base + " residentPolls 0;")
        for controls in (base, base + " residentPolls 1;", base):
            got = step(ctx, dm, m, f, controls)
            assert got[0] == want[0] and got[1] == want[1]
            assert np.array_equal(got[2], want[2]) and np.array_equal(got[3], want[3])


@pytest.mark.parametrize("n", [500, 5000, 20000])
@pytest.mark.parametrize("noalloc", [False, True])
def test_resident_symm_solve_equals_launches(ctx, n, noalloc):
    """A general LDU system on a random face graph (rows wider than the staged
    width, no two-colouring) and on a box (Schur pivots)."""
    rng = np.random.default_rng(n)
    for m in (cases.random_graph(n, kNear=5, sigma=0.5, seed=3), cases.cartesian(n // 100, 10, 10)):
        dm = ctx.mesh(m)
        lo, up = -rng.uniform(0.1, 1.0, m.nInternal), -rng.uniform(0.1, 1.0, m.nInternal)
        d = np.full(m.nCells, 0.5)
        np.add.at(d, m.owner[:m.nInternal], -lo)
        np.add.at(d, m.neighbour, -up)
        src, psi = rng.normal(size=(m.nCells, 6)), rng.normal(size=(m.nCells, 6))
        for solver, precond in FORMS:
            base = abi.solver_dict(1e-10, solver=solver, precond=precond)
            want = ctx.symm_solve(dm, d, lo, up, src, psi, base + " residentPolls 0;", noalloc=noalloc)
            for controls in (base, base + " residentPolls 1;"):
                got = ctx.symm_solve(dm, d, lo, up, src, psi, controls, noalloc=noalloc)
                assert np.array_equal(got[0], want[0])
                assert [q.nIterations for q in got[1]] == [q.nIterations for q in want[1]]


def test_resident_server_batch_gives_up_and_finishes(ctx):
    """A batch of resident solves whose waits give up finishes by launches,
    with the same bits."""
    reqs = []
    for i, n in enumerate((40, 60, 80)):
        m = cases.cartesian(n, n, 1, twoD=True, channel=True)
        reqs.append((ctx.mesh(m), cases.make_fields(m, cases.FIELDS_CHANNEL, seed=i), 0.1 / n))
    out = {}
    for polls in ("0", "1", "200000"):
        srv = abi.Server(ctx, max_inflight=4)
        base = abi.solver_dict(1e-10, precision="mixed") + f" residentPolls {polls};"
        ts = [srv.submit(dm, f, abi.model_dict("Oldroyd-BLog"), dt, base) for dm, f, dt in reqs]
        while srv.progress():
            pass
        out[polls] = [srv.poll(t) for t in ts]
        srv.close()
    for polls in ("1", "200000"):
        for a, b in zip(out[polls], out["0"]):
            assert np.array_equal(a["theta"], b["theta"]) and np.array_equal(a["tau"], b["tau"])
