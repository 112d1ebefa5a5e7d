"""A server's requests run on their slots' streams, which nothing orders
against the meshes' own: bursts of requests of mixed sizes all converge to
what each gives alone."""
import numpy as np
import pytest

from rheotool_amd import abi, cases

pytestmark = pytest.mark.gpu


def test_every_request_of_every_burst_is_solved():
    controls = abi.solver_dict(1e-10, precision="mixed")
    text = abi.model_dict("Oldroyd-BLog", lam=1.0)
    sides = [24, 40, 56, 72]
    ms = [cases.cartesian(n, n, n, channel=True) for n in sides]
    fs = [cases.make_fields(m, cases.FIELDS_CHANNEL, seed=7 + i) for i, m in enumerate(ms)]
    with abi.Context(0) as ctx:
        dms = [ctx.mesh(m) for m in ms]
        want = []
        for dm, f, n in zip(dms, fs, sides):
            eq = ctx.constitutiveEq("", dm, text)
            eq.set_solver(controls)
            eq.set_state(f.theta, f.eigVals, f.eigVecs)
            eq.set_flow(f.U, f.Ub, f.phi)
            eq.correct(0.1 / n)
            want.append(eq.theta())
        srv = abi.Server(ctx, hbm_budget=0, max_inflight=16)
        for burst in range(30):
            tickets = [(i, srv.submit(dms[i], fs[i], text, 0.1 / sides[i], controls))
                       for i in (3, 0, 2, 1, 2, 0, 3, 1, 2, 3, 0, 3)]
            while srv.progress():
                pass
            srv.finished()
            for i, t in tickets:
                d = srv.poll(t)
                assert np.array_equal(d["theta"], want[i]), (burst, sides[i])
        srv.close()
