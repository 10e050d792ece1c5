"""Whole-run kernel of small 1-D Euler meshes against the per-stage kernels (eager launches take
them): element counts around a wavefront and at the limit of the kernel and just above it, P1-P5, with
and without artificial viscosity, bounded and periodic, one call against several, and the NaN stop. Both
evaluate the same scheme in FP64: a few rounding errors of values of order one, times the step count."""
import numpy as np
import pytest

import problems as P
from subrosadg_amd import _lib as L

pytestmark = pytest.mark.gpu


def _pair(order, n, av, periodic, rk=L.RK_SSPRK3, flux=L.FLUX_HLLC):
    bc = None if periodic else ((L.BC_RIEMANN_FARFIELD, L.BC_ADIABATIC_SLIP_WALL),)
    mesh = L.Mesh(L.ELEM_LINE, order, (n,), (0.0,), (1.0,), **({} if periodic else {"boundary": bc}))
    kw = dict(cp=3.5, cv=2.5, equation=L.EQ_EULER, convective_flux=flux, time_integration=rk)
    if av:
        kw.update(shock_capturing=L.SHOCK_ARTIFICIAL_VISCOSITY, artificial_viscosity_factor=1.0, empirical_tolerance=0.5)
    prob = L.problem_desc(**kw)
    eager = L.ProblemDesc.from_buffer_copy(prob)
    eager.launch = L.LAUNCH_EAGER
    x = mesh.field("quad_coord").reshape(mesh.E, mesh.nq, 1)
    if av:  # Sod's tube, its jump smoothed over an element (the scheme undershoots to p < 0 on a jump inside one)
        w = 0.5 * (1.0 - np.tanh((x[..., 0] - 0.47) * n))
        rho = 0.125 + 0.875 * w
        prim = np.stack([rho, 0.1 + 0.0 * rho, (0.1 + 0.9 * w) / rho], -1)
    else:
        prim = np.stack([1.0 + 0.2 * np.sin(2 * np.pi * x[..., 0]), 0.3 + 0.1 * np.cos(2 * np.pi * x[..., 0]),
                         1.0 + 0.1 * np.cos(4 * np.pi * x[..., 0])], -1)
    out = []
    for p in (prob, eager):
        s = L.Solver(p, mesh)
        s.set_initial_primitive(prim)
        if mesh.Fb:
            b = P.sod_primitive(P.boundary_points(mesh))
            b[..., 1] = 0.1
            s.set_boundary_primitive(b)
        out.append(s)
    return out


CASES = [(1, 2, False, True), (1, 65, True, False), (2, 63, True, False), (2, 64, False, False), (3, 512, True, True),
         (3, 513, True, False), (4, 100, True, False), (4, 511, False, True), (5, 33, True, False)]


@pytest.mark.parametrize("order,n,av,periodic", CASES)
def test_whole_run_matches_stage_kernels(order, n, av, periodic):
    print(f"line run P{order} n={n} av={av} periodic={periodic}", flush=True)
    a, b = _pair(order, n, av, periodic)
    dt = a.compute_dt(0.1)
    for k in (1, 4, 7):  # odd and even trace parities, state kept between calls
        ra, na, ta = a.step(dt, k)
        rb, nb, tb = b.step(dt, k)
        assert (na, ta) == (nb, tb) == (0, k)
        np.testing.assert_allclose(ra, rb, rtol=1e-10, atol=1e-11)
        ua, ub = a.get_state(), b.get_state()
        assert np.abs(ua - ub).max() <= 1e-12 * np.abs(ub).max()
        ar, br = a.residual(), b.residual()  # the traces the run leaves
        assert np.abs(ar - br).max() <= 1e-10 * max(np.abs(br).max(), 1.0)
    if av:
        va, vb = a.artificial_viscosity(), b.artificial_viscosity()
        assert np.abs(va - vb).max() <= 1e-9 * max(np.abs(vb).max(), 1e-3)


@pytest.mark.parametrize("rk", [L.RK_FORWARD_EULER, L.RK_HEUN2])
def test_other_runge_kutta_schemes(rk):
    a, b = _pair(2, 40, False, True, rk=rk, flux=L.FLUX_ROE)
    dt = a.compute_dt(0.05)
    a.step(dt, 5), b.step(dt, 5)
    ua, ub = a.get_state(), b.get_state()
    assert np.abs(ua - ub).max() <= 1e-13 * np.abs(ub).max()


def test_nan_stop():
    a, b = _pair(3, 80, True, False)
    dt = 200.0 * a.compute_dt(1.0)
    _, na, ta = a.step(dt, 50)
    _, nb, tb = b.step(dt, 50)
    assert na == nb == 1 and ta == tb < 50
    assert a.step(dt, 0)[2] == 0


def test_calls_of_several_launches():
    """A launch takes at most 4096 steps: a longer call is bit-identical to the same steps in two calls of
    other lengths (trace parity, step count and state cross from one launch to the next)."""
    (a, _), (b, _) = _pair(1, 8, False, True), _pair(1, 8, False, True)
    dt = a.compute_dt(0.1)
    ra, na, ta = a.step(dt, 4099)
    _, n1, t1 = b.step(dt, 2050)
    rb, n2, t2 = b.step(dt, 2049)
    assert (na, n1, n2) == (0, 0, 0) and (ta, t1, t2) == (4099, 2050, 2049)
    assert np.array_equal(ra, rb)
    assert np.array_equal(a.get_state(), b.get_state())
    assert np.array_equal(a.residual(), b.residual())


def test_nan_stop_in_the_first_of_two_launches():
    """The launch behind the one that stopped leaves state and step count alone."""
    a, b = _pair(3, 80, True, False)
    dt = 200.0 * a.compute_dt(1.0)
    ra, na, ta = a.step(dt, 4100)
    rb, nb, tb = b.step(dt, 50)
    assert na == nb == 1 and ta == tb < 50
    assert np.isnan(ra).all() and np.isnan(rb).all()
    ua = a.get_state()
    assert np.isnan(ua).any()
    c, _ = _pair(3, 80, True, False)
    c.step(dt, ta)
    assert np.array_equal(c.get_state(), ua, equal_nan=True)


@pytest.mark.parametrize("order", [1, 2, 3])
@pytest.mark.parametrize("right", [True, False])
def test_nan_stop_of_an_infinite_boundary_flux(order, right):
    """An infinite flux at one end point alone: the end point's basis values are 1 and exact zeros, so it
    makes the residual's modes NaN, and both launch modes stop after the same step."""
    ends = (L.BC_RIEMANN_FARFIELD, L.BC_VELOCITY_INFLOW)
    mesh = L.Mesh(L.ELEM_LINE, order, (5,), (0.0,), (1.0,), boundary=(ends if right else ends[::-1],))
    prob = L.problem_desc(cp=3.5, cv=2.5, equation=L.EQ_EULER, convective_flux=L.FLUX_HLLC)
    prim = np.zeros((mesh.E, mesh.nq, 3))
    prim[..., 0], prim[..., 1], prim[..., 2] = 1.0, 0.1, 1.0
    b = np.zeros((mesh.Fb, mesh.nfq, 3))
    b[..., 0], b[..., 1], b[..., 2] = 1.0, 0.1, 1.0
    end = (P.boundary_points(mesh)[..., 0] > 0.5) == right
    b[end] = [1e200, -1e200, 1.0]
    out = []
    for launch in (L.LAUNCH_GRAPH, L.LAUNCH_EAGER):
        p = L.ProblemDesc.from_buffer_copy(prob)
        p.launch = launch
        s = L.Solver(p, mesh)
        s.set_initial_primitive(prim)
        s.set_boundary_primitive(b)
        out.append(s.step(1e-3, 6)[1:])
    assert out[0] == out[1] == (1, 1)
