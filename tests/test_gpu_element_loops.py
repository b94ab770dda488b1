"""The persistent volume kernels (p >= 5) on more elements than workgroups are
resident, in the modes whose tables or buffers the element loop carries along:
model viscosities, saved staggered states and their adjoint, per-element
metrics, rotated faces.

A box of copies of eight distorted elements, holding copies of their state,
must give every copy the result of the eight alone, which fit one trip.  The
copies differ by the rounding of corners up to 20 edges from the origin, 4e-15
relative in the metrics; the pressure background, a few hundred times the
changes of the momentum flux, brings that to 1e-12 in a right-hand side, and
steps and their adjoints to some times that: bound 1e-10, gradients 1e-9."""
import numpy as np
import pytest

import oracle as O
from dsem_amd import cases
from dsem_amd import mesh as M
from dsem_amd.solver import DSEM
from helpers import graded_box, periodic_state, rel_l2

pytestmark = pytest.mark.gpu

# copies along each axis: 800 elements at p = 5 (two or three workgroups per
# CU), above 256 beyond
COPIES = {5: (4, 5, 5), 6: (3, 3, 5), 7: (3, 3, 4), 8: (3, 3, 4)}


def _copies(nx, ny, nz, p):
    """Box of nx x ny x nz copies of a 2^3 box of unit cubes with its middle
    node moved, and for each element the one of the eight it copies."""
    mid = np.array([3.0, -2.0, 5.0]) / 64.0
    def node(i, j, k):
        return np.array([i, j, k], dtype=float) + (mid if i % 2 and j % 2 and k % 2 else 0.0)
    corners, of = [], []
    for k in range(2 * nz):
        for i in range(2 * nx):
            for j in range(2 * ny):
                corners.append([node(*c) for c in ((i, j, k), (i + 1, j, k), (i + 1, j + 1, k), (i, j + 1, k),
                                                   (i, j, k + 1), (i + 1, j, k + 1), (i + 1, j + 1, k + 1),
                                                   (i, j + 1, k + 1))])
                of.append(j % 2 + 2 * (i % 2) + 4 * (k % 2))
    return M.build_topology(p, np.array(corners)), np.array(of)


def _gradient(mesh, JQ, models, nsteps, dt):
    """State, gradients with respect to state and viscosity after nsteps."""
    import torch
    from dsem_amd import autograd as A
    kw = dict(shock=True, cmu=2.0, mumax=0.05) if models else {}
    with DSEM(mesh, re=200.0, **kw) as s:
        if models:
            s.set_les(True, 0.12, 1e9)
        x = torch.tensor(JQ, device="cuda", requires_grad=True)
        nu = torch.tensor(1.0 / 200.0, dtype=torch.float64, device="cuda", requires_grad=True)
        y = A.solve(s, x, nsteps, dt, nu=nu)
        A.kinetic_energy_integral(y, A.bmat_tensor(s, "cuda")).backward()
        return y.detach().cpu().numpy(), x.grad.cpu().numpy(), float(nu.grad)


@pytest.mark.parametrize("models", [False, True])
@pytest.mark.parametrize("p", [5, 6, 7, 8])
def test_copies_step_and_differentiate_alike(p, models):
    print(f"\n[case] copies p={p} models {models}", flush=True)
    one, _ = _copies(1, 1, 1, p)
    many, of = _copies(*COPIES[p], p)
    with DSEM(one, re=200.0) as s, DSEM(many, re=200.0) as t:
        xg, jac = s.gauss_points()
        JQ = periodic_state(xg, jac, (2.0, 2.0, 2.0), seed=p)
        s.set_state(JQ)
        dt = 0.3 * s.dtcalc()
        t.set_state(JQ[of])
        for c in (s, t):
            c.keep_lagged_states(True)
            c.steps(2, dt)
        lag, lags = s.get_lagged_states()[of], t.get_lagged_states()
        assert np.linalg.norm(lags - lag) <= 1e-10 * np.linalg.norm(lag)
    y, g, gn = _gradient(one, JQ, models, 3, dt)
    ys, gs, gns = _gradient(many, JQ[of], models, 3, dt)
    print("state", rel_l2(ys, y[of]), "gradient", rel_l2(gs, g[of]), "nu", gns / gn / (many.K // 8) - 1.0, flush=True)
    assert np.all(rel_l2(ys, y[of]) <= 1e-10)
    assert np.all(rel_l2(gs, g[of]) <= 1e-9)
    assert abs(gns - gn * (many.K // 8)) <= 1e-9 * abs(gns)


@pytest.mark.parametrize("shape,p", [((9, 7, 11), 5), ((7, 6, 7), 6), ((5, 8, 7), 7), ((6, 9, 5), 8)])
def test_adjoint_with_per_element_metrics(shape, p):
    """The two ways to store affine metrics differ by rounding alone."""
    print(f"\n[case] adjoint per-element metrics {shape} p={p}", flush=True)
    mesh = graded_box(*shape, p)
    out = []
    for metrics in ("per_point", "per_element"):
        with DSEM(mesh, re=400.0, metrics=metrics) as s:
            xg, jac = s.gauss_points()
            JQ = periodic_state(xg, jac, (2 * np.pi, 3.0, 5.0), seed=p)
            s.set_state(JQ)
            out.append(s.rhs_vjp(np.random.default_rng(p).standard_normal(JQ.shape)))
    (jb, nb), (je, ne) = out
    print("rel L2", rel_l2(je, jb), "nu", ne / nb - 1.0, flush=True)
    assert np.all(rel_l2(je, jb) <= 1e-10) and abs(ne - nb) <= 1e-9 * abs(nb)


@pytest.mark.parametrize("n,p", [(9, 5), (7, 8)])
def test_rotated_faces_rhs_and_adjoint(n, p):
    """The state and the bounds of the other tests on rotated faces: RHS
    against the oracle 1e-12, adjoint against a central difference 1e-6."""
    print(f"\n[case] rotated element loop n={n} p={p}", flush=True)
    mesh = M.rotated_box(n, p, seed=p)
    g = O.Geometry(mesh)
    JQ = cases.tgv_state(g.xg, g.jacob, "isothermal", perturb=1e-2, seed=p)
    rng = np.random.default_rng(p)
    lam = rng.standard_normal(JQ.shape)
    v = rng.standard_normal(JQ.shape) * np.abs(JQ).mean(axis=(0, 2), keepdims=True)
    h = 1e-6
    with DSEM(mesh, re=400.0) as s:
        s.set_state(JQ)
        err = rel_l2(s.rhs(), O.rhs(g, JQ, O.phys(re=400.0)))
        jb, _ = s.rhs_vjp(lam)
        s.set_state(JQ + h * v)
        rp = s.rhs()
        s.set_state(JQ - h * v)
        rm = s.rhs()
    ad, fd = float(np.sum(jb * v)), float(np.sum(lam * (rp - rm)) / (2 * h))
    print("rhs", err, "adjoint", ad, "fd", fd, flush=True)
    assert np.all(err <= 1e-12) and abs(ad - fd) <= 1e-6 * abs(fd)
