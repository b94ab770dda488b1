"""Face fluxes formed inside the element update, at every order on meshes with
all eight face orientations: the RHS, and RK steps in calls of one and two (an
odd number of stages leaves the trace arrays exchanged), against the oracle.

Tolerance 1e-12 relative L2 per field for the RHS, the bound of the other RHS
parity tests, and on the change of the state over three steps (5e-12 with
per-element metrics, whose reference is the per-point geometry)."""
import numpy as np
import pytest

import oracle as O
from dsem_amd import cases
from dsem_amd import mesh as M
from dsem_amd.solver import DSEM
from helpers import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p", range(1, 9))
@pytest.mark.parametrize("metrics,tol", [("per_point", 1e-12), ("per_element", 5e-12)])
def test_rotated_faces_rhs_and_steps(p, metrics, tol):
    print(f"\n[case] face fluxes p={p} {metrics}", flush=True)
    mesh = M.rotated_box(3, p, seed=p)
    g = O.Geometry(mesh)
    JQ = cases.tgv_state(g.xg, g.jacob, "isothermal", perturb=1e-2, seed=p)
    ph = O.phys(re=400.0)
    dt = 0.5 * O.dtcalc(g, JQ, ph)
    ref = JQ.copy()
    for _ in range(3):
        O.rk_step(g, ref, dt, ph)
    with DSEM(mesh, re=400.0, metrics=metrics) as s:
        s.set_state(JQ)
        rhs = s.rhs()
        s.steps(1, dt)
        s.steps(2, dt)
        got = s.get_state()
    e1, e2 = rel_l2(rhs, O.rhs(g, JQ, ph)), rel_l2(got - JQ, ref - JQ)
    print("rhs", e1, "steps", e2, flush=True)
    assert np.all(e1 <= tol) and np.all(e2 <= tol)


@pytest.mark.parametrize("p", range(1, 9))
def test_recorded_steps_are_the_plain_steps(p):
    """A recorded step leaves each stage's state and traces in the tape and the
    last ones in the context: the state after recorded and plain steps in turn,
    and after a write to the state in between, equals plain steps bit for bit."""
    print(f"\n[case] recorded steps p={p}", flush=True)
    mesh = M.rotated_box(3, p, seed=p)
    with DSEM(mesh, re=400.0) as s:
        xg, jac = s.gauss_points()
        JQ = cases.tgv_state(xg, jac, "isothermal", perturb=1e-2, seed=p)
        s.set_state(JQ)
        dt = 0.3 * s.dtcalc()
        s.steps(4, dt)
        want = s.get_state()
        s.tape_reserve(2)
        for recorded in ((True, True, False, True), (False, True, False, False)):
            s.set_state(JQ)
            for i, rec in enumerate(recorded):
                if rec:
                    s.rk_step_record(dt, i % 2)
                else:
                    s.steps(1, dt)
            assert np.array_equal(s.get_state(), want)
        s.set_state(JQ)
        s.rk_step_record(dt, 0)
        s.set_state(JQ)
        s.rk_step_record(dt, 1)
        s.steps(3, dt)
        assert np.array_equal(s.get_state(), want)
