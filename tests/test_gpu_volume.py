"""FP64 volume kernels over every instance they come in: each order (matrix
cores from p = 5 on, vector form below), without and with the model
viscosities, with the staggered states saved, and on more elements than
workgroups are resident (p >= 5 loops over elements).

Tolerance 1e-12 relative L2 per field, the parity bound of the RHS: the sums
are those of the oracle up to order and rounding, about 20 roundings of
2^-53 on values whose cancellation the other parity tests bound."""
import ctypes as C

import numpy as np
import pytest

import oracle as O
from dsem_amd import cases
from dsem_amd.solver import DSEM
from helpers import distorted_box, graded_box, rel_l2

pytestmark = pytest.mark.gpu

TOL = 1e-12


def _oracle_rhs(g, JQ, ph, muh, nut):
    Qt, m = np.zeros_like(JQ), g.cmesh()
    rc = O.lib().or_rhs_les(C.byref(m), C.byref(ph), O.ptr(np.ascontiguousarray(JQ)), O.ptr(muh), O.ptr(nut),
                            O.ptr(Qt), None, 0)
    assert rc == 0
    return Qt


@pytest.mark.parametrize("p", range(1, 9))
def test_rhs_of_every_viscosity_instance(p):
    print(f"\n[case] volume instances p={p}", flush=True)
    mesh = distorted_box(3 if p < 6 else 2, p, amp=0.06, seed=p)
    g = O.Geometry(mesh)
    JQ = cases.tgv_state(g.xg, g.jacob, "isothermal", perturb=1e-2, seed=p)
    ph = O.phys(re=300.0)
    rng = np.random.default_rng(p)
    muh, nut = (np.abs(rng.standard_normal((mesh.K, 3, g.ns))) * 0.1 for _ in range(2))
    for ev in (False, True):
        with DSEM(mesh, re=300.0, shock=ev) as s:
            s.set_state(JQ)
            if ev:
                s.set_viscosity(muh)
            for les in (False, True):
                if les:
                    s.set_les(True, 0.17, 1.0)
                    s.set_les_viscosity(nut)
                want = _oracle_rhs(g, JQ, ph, muh if ev else None, nut if les else None)
                err = rel_l2(s.rhs(), want)
                print(f"ev {ev} les {les}: rel L2 {err}", flush=True)
                assert np.all(err <= TOL)


@pytest.mark.parametrize("p", range(1, 9))
def test_saved_staggered_states(p):
    print(f"\n[case] saved staggered states p={p}", flush=True)
    mesh = distorted_box(2, p, amp=0.05, seed=p)
    g = O.Geometry(mesh)
    JQ = cases.tgv_state(g.xg, g.jacob, "isothermal", perturb=1e-3, seed=p)
    ph = O.phys(re=500.0)
    dt = 0.3 * O.dtcalc(g, JQ, ph)
    ref, stag = JQ.copy(), np.zeros((mesh.K, 3, 5, g.ns))
    O.rk_step(g, ref, dt, ph, stag_out=stag)
    with DSEM(mesh, re=500.0) as s:
        s.set_state(JQ)
        s.keep_lagged_states(True)
        s.tstep(0.0, dt)
        got, lag = s.get_state(), s.get_lagged_states()
    assert np.all(rel_l2(got, ref) <= TOL)
    assert np.linalg.norm(lag - stag) <= TOL * np.linalg.norm(stag)


@pytest.mark.parametrize("shape,p", [((9, 7, 11), 5), ((7, 6, 7), 6), ((5, 8, 7), 7), ((6, 9, 5), 8)])
def test_more_elements_than_workgroups(shape, p):
    """270 to 693 elements against 256 or 512 resident workgroups: first,
    middle and last trips of the element loop, on one context twice."""
    print(f"\n[case] element loop {shape} p={p}", flush=True)
    mesh = graded_box(*shape, p)
    g = O.Geometry(mesh)
    JQ = cases.tgv_state(g.xg, g.jacob, "isothermal", perturb=1e-2, seed=p)
    want = O.rhs(g, JQ, O.phys(re=400.0))
    with DSEM(mesh, re=400.0) as s:
        s.set_state(JQ)
        one, two = s.rhs(), s.rhs()
    print("rel L2", rel_l2(one, want), flush=True)
    assert np.all(rel_l2(one, want) <= TOL)
    assert np.array_equal(one, two)
