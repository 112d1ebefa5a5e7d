"""The fields' way between the caller's cell order and the device's rows, at
the edges of a workgroup's cells: theta and tau come back the bits that were
set, U arrives and div(tau) leaves in the caller's order (tauTotal and div(tau)
against the oracle: per-row arithmetic in its operation order, 1e-13)."""
import numpy as np
import pytest

from oracle import oracle as O
from rheotool_amd import abi, cases

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = abi.Context(0)
    yield c
    c.close()


def close(a, b):
    return np.linalg.norm(a - b) <= 1e-13 * np.linalg.norm(b)


@pytest.mark.parametrize("renumber", [0, 1])
@pytest.mark.parametrize("shape", [(1, 1, 1), (5, 17, 1), (2, 43, 1), (5, 51, 1), (8, 8, 4), (257, 1, 1),
                                   (19, 27, 1), (10, 10, 10)])
def test_fields_in_and_out(ctx, shape, renumber):
    print(f"[case] rows {shape} renumber={renumber}", flush=True)
    m = cases.cartesian(*shape, twoD=shape[2] == 1)
    f = cases.make_fields(m, cases.FIELDS_TG, seed=3, lnLo=-2.0, lnHi=2.0)
    tau = np.random.default_rng(6).normal(size=f.theta.shape)
    eq = ctx.constitutiveEq("", ctx.mesh(m, renumber),
                            abi.model_dict("Oldroyd-BLog", lam=1.0, rho=1.0, etaS=0.3, stabilization="none"))
    eq.set_state(f.theta, f.eigVals, f.eigVecs, tau)
    eq.set_flow(f.U, f.Ub, f.phi)
    assert np.array_equal(eq.theta(), f.theta)
    assert np.array_equal(eq.tau(), tau)
    assert close(eq.tau_total(), O.tau_total(m, f.U, f.Ub, tau, 0.3))
    assert close(eq.div_tau(), O.div_tau(m, tau, None, 1.0))


@pytest.mark.parametrize("shape,precision,was", [((40, 36, 30), "double", 47418112), ((40, 36, 30), "mixed", 42081280),
                                                 ((96, 96, 96), "double", 1015474432), ((120, 110, 1), "mixed", 14131200)])
def test_a_step_fits_the_device_memory_it_fitted(shape, precision, was):
    """A mesh, a model and its step take what they took before the meshes kept
    the face loops' column words and the cells' rows (`was`, bytes measured then;
    half a per cent for the size classes), so that a context's budget holds them
    as before."""
    print(f"[case] memory {shape} {precision}", flush=True)
    m = cases.cartesian(*shape, twoD=shape[2] == 1, channel=True)
    f = cases.make_fields(m, cases.FIELDS_CHANNEL, seed=2)
    with abi.Context(0) as c:
        eq = c.constitutiveEq("", c.mesh(m), abi.model_dict("GiesekusLog", lam=2.0, alpha=0.2))
        eq.set_solver(abi.solver_dict(1e-10, precision=precision))
        eq.set_state(f.theta, f.eigVals, f.eigVecs)
        eq.set_flow(f.U, f.Ub, f.phi)
        eq.correct(1e-3)
        assert c.bytes_in_use <= 1.005 * was
