"""Reverse volume kernel over the instances it comes in at p >= 5: each order
without and with the model viscosities, and on more elements than workgroups
are resident (a workgroup loops over elements); the reverse of the face fluxes
at every order on faces of all orientations.

Central differences bound the error as in the other adjoint tests, 1e-6
relative: with steps of 1e-6 (1e-7 where a viscosity's switches lie near) the
truncation is below 1e-9 and rounding, 2^-53 / h on sums of 1e4 to 1e6 terms
of random sign, below 1e-7."""
import numpy as np
import pytest

from dsem_amd import cases
from dsem_amd import mesh as M
from dsem_amd.solver import DSEM
from helpers import distorted_box, graded_box, periodic_state

pytestmark = pytest.mark.gpu


def _close(ad, fd):
    print(f"adjoint {ad:.12e} fd {fd:.12e}", flush=True)
    return abs(ad - fd) <= 1e-6 * abs(fd)


@pytest.mark.parametrize("shape,p", [((9, 7, 11), 5), ((7, 6, 7), 6), ((5, 8, 7), 7), ((6, 9, 5), 8)])
def test_more_elements_than_workgroups(shape, p):
    print(f"\n[case] reverse element loop {shape} p={p}", flush=True)
    mesh = graded_box(*shape, p)
    rng = np.random.default_rng(p)
    with DSEM(mesh, re=400.0) as s:
        xg, jac = s.gauss_points()
        JQ = periodic_state(xg, jac, (2 * np.pi, 3.0, 5.0), seed=p)
        lam = rng.standard_normal(JQ.shape)
        s.set_state(JQ)
        jb, nub = s.rhs_vjp(lam)
        jb2, nub2 = s.rhs_vjp(lam)
        assert np.array_equal(jb, jb2) and nub == nub2
        K = mesh.K
        h = 1e-6
        # directions on the first, middle and last trips of the loop
        for sel in (slice(0, K // 3), slice(K // 3, 2 * K // 3), slice(2 * K // 3, K)):
            v = np.zeros_like(JQ)
            v[sel] = rng.standard_normal(JQ[sel].shape) * np.abs(JQ).mean(axis=(0, 2), keepdims=True)
            s.set_state(JQ + h * v)
            rp = s.rhs()
            s.set_state(JQ - h * v)
            rm = s.rhs()
            assert _close(float(np.sum(jb * v)), float(np.sum(lam * (rp - rm)) / (2 * h)))


@pytest.mark.parametrize("les", [False, True])
@pytest.mark.parametrize("ev", [False, True])
@pytest.mark.parametrize("p", [5, 6, 7, 8])
def test_gradient_of_every_viscosity_instance(p, ev, les):
    import torch
    from dsem_amd import autograd as A
    print(f"\n[case] reverse volume p={p} ev {ev} les {les}", flush=True)
    mesh = distorted_box(2, p, amp=0.04, seed=p)
    kw = dict(shock=True, cmu=2.0, mumax=0.05) if ev else {}
    with DSEM(mesh, re=200.0, **kw) as s:
        if les:
            s.set_les(True, 0.12, 1e9)
        xg, jac = s.gauss_points()
        JQ = cases.tgv_state(xg, jac, "isothermal", perturb=3e-2, seed=p)
        s.set_state(JQ)
        dt, nsteps = 0.3 * s.dtcalc(), 3
        x = torch.tensor(JQ, device="cuda", requires_grad=True)
        J = A.kinetic_energy_integral(A.solve(s, x, nsteps, dt), A.bmat_tensor(s, "cuda"))
        J.backward()
        g = x.grad.cpu().numpy()
        bm = s.quadrature_weights()

        def Jf(q0):
            s.set_state(q0)
            s.steps(nsteps, dt, check=False)
            q = s.get_state()
            return 0.5 * float(np.sum(bm * (q[:, 1] ** 2 + q[:, 2] ** 2 + q[:, 3] ** 2) / q[:, 0]))

        h = 1e-7 if ev else 1e-6
        d = np.random.default_rng(p).standard_normal(JQ.shape) * np.abs(JQ).mean(axis=(0, 2), keepdims=True)
        assert _close(float(np.sum(g * d)), (Jf(JQ + h * d) - Jf(JQ - h * d)) / (2 * h))


@pytest.mark.parametrize("p", range(1, 9))
def test_face_flux_adjoint_on_rotated_faces(p):
    print(f"\n[case] reverse face fluxes p={p}", flush=True)
    mesh = M.rotated_box(3, p, seed=p)
    rng = np.random.default_rng(p)
    nu, h = 1.0 / 200.0, 1e-6
    with DSEM(mesh, re=1.0 / nu) as s:
        xg, jac = s.gauss_points()
        JQ = cases.tgv_state(xg, jac, "isothermal", perturb=2e-2, seed=p)
        lam = rng.standard_normal(JQ.shape)
        v = rng.standard_normal(JQ.shape) * np.abs(JQ).mean(axis=(0, 2), keepdims=True)
        s.set_state(JQ)
        jb, nub = s.rhs_vjp(lam)
        s.set_state(JQ + h * v)
        rp = s.rhs()
        s.set_state(JQ - h * v)
        rm = s.rhs()
        assert _close(float(np.sum(jb * v)), float(np.sum(lam * (rp - rm)) / (2 * h)))
    r = []
    for f in (1.5, 0.5):   # R is linear in nu: any step will do
        with DSEM(mesh, re=1.0 / (f * nu)) as s:
            s.set_state(JQ)
            r.append(s.rhs())
    assert _close(nub, float(np.sum(lam * (r[0] - r[1])) / nu))
