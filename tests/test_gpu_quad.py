"""Sum-factorised quadrangle kernels at the sizes where their layout can go wrong: element counts that
fill no wavefront evenly (8, 5, 4, 2 and 1 elements each at P1..P5), sheared cells,
walls on two sides. Residual, lifted gradient and 3 SSP-RK3 steps against the oracle at the FP64 bar of
the parity tests, and against the vector kernels (a few rounding errors of values of order one)."""
import numpy as np
import pytest

import oracle as O
import problems as P
from subrosadg_amd import _lib as L

pytestmark = pytest.mark.gpu

KINDS = ["euler", "av", "br1", "br2"]
SHEAR = np.array([[1.0, 0.0], [0.3, 1.0]])


def _mesh(order, n):
    """n[0] x n[1] sheared cells of [0,1]^2: isothermal walls below and above, far field left and right."""
    nx, ny = n
    ii, jj = np.meshgrid(np.arange(nx + 1), np.arange(ny + 1), indexing="xy")
    xy = np.stack([ii / nx, jj / ny], -1).reshape(-1, 2) @ SHEAR
    a = (jj[:-1, :-1] * (nx + 1) + ii[:-1, :-1]).reshape(-1)
    quad = np.stack([a, a + 1, a + nx + 2, a + nx + 1], -1)
    j, i = np.arange(ny), np.arange(nx)
    sides = [np.stack([j * (nx + 1), (j + 1) * (nx + 1)], -1), np.stack([j * (nx + 1) + nx, (j + 1) * (nx + 1) + nx], -1),
             np.stack([i, i + 1], -1), np.stack([ny * (nx + 1) + i, ny * (nx + 1) + i + 1], -1)]
    return xy, quad, np.concatenate(sides), nx, ny, order


def _case(kind, order, n):
    xy, quad, faces, nx, ny, _ = _mesh(order, n)
    wall = L.BC_ISOTHERMAL_NONSLIP_WALL if kind.startswith("br") else L.BC_ADIABATIC_SLIP_WALL
    types = np.concatenate([np.full(2 * ny, L.BC_RIEMANN_FARFIELD), np.full(2 * nx, wall)])
    mesh = L.Mesh.from_arrays(L.ELEM_QUADRANGLE, order, xy, quad, boundary_faces=faces, boundary_type=types)
    kw = dict(cp=3.5, cv=2.5, convective_flux=L.FLUX_HLLC)
    if kind == "av":
        kw.update(shock_capturing=L.SHOCK_ARTIFICIAL_VISCOSITY, artificial_viscosity_factor=1.0, empirical_tolerance=4.0)
    if kind.startswith("br"):
        kw.update(equation=L.EQ_NS, viscous_flux=L.VISC_BR1 if kind == "br1" else L.VISC_BR2,
                  transport=L.TRANSPORT_CONSTANT, dynamic_viscosity=0.01)
    else:
        kw.update(equation=L.EQ_EULER)
    x = mesh.field("quad_coord").reshape(mesh.E, mesh.nq, 2)
    prim = np.zeros(x.shape[:2] + (4,))
    prim[..., 0] = 1.0 + 0.2 * np.sin(3.0 * x[..., 0] + 1.0) * np.cos(2.0 * x[..., 1])
    prim[..., 1] = 0.3 + 0.1 * np.cos(2.0 * x[..., 0] + x[..., 1])
    prim[..., 2] = -0.2 + 0.1 * np.sin(4.0 * x[..., 1])
    prim[..., 3] = 1.0 + 0.1 * np.cos(3.0 * x[..., 1] - x[..., 0])
    b = np.zeros((mesh.Fb, mesh.nfq, 4))
    b[..., 0], b[..., 1], b[..., 3] = 1.0, 0.3, 1.0
    return mesh, L.problem_desc(**kw), prim, b


@pytest.mark.parametrize("order,n", [(1, (1, 2)), (1, (3, 3)), (2, (2, 3)), (2, (2, 1)), (3, (5, 1)), (3, (3, 3)), (4, (3, 1)),
                                     (5, (1, 2))])
@pytest.mark.parametrize("kind", KINDS)
def test_quad_kernels(kind, order, n):
    print(f"quad {kind} P{order} {n}", flush=True)
    mesh, prob, prim, b = _case(kind, order, n)
    s = L.Solver(prob, mesh)
    s.set_initial_primitive(prim)
    s.set_boundary_primitive(b)
    u0 = s.get_state()
    o, x = O.Oracle(prob, mesh), O.Oracle(prob, mesh, extended=True)
    for c in (o, x):
        c.set_state(u0)
        c.set_boundary_primitive(b)
    v = L.Solver(P.with_kernels(prob, L.KERNELS_VECTOR), mesh)
    v.set_state(u0)
    v.set_boundary_primitive(b)
    P.fp64_parity(s.residual(), o.residual(), x.residual(), u0, mesh.dim, tol=1e-12)
    assert P.parity_error(s.residual(), v.residual(), u0, mesh.dim) <= 1e-11
    if kind.startswith("br"):
        h = float(mesh.field("min_edge").min())
        P.fp64_parity(s.gradient(), o.gradient(), x.gradient(), u0, mesh.dim, tol=5e-11, h=h)
    dt = o.compute_dt(0.1)
    for c in (o, x):
        c.step(dt, 3)
    rel, nan, taken = s.step(dt, 3)
    assert nan == 0 and taken == 3
    vrel, _, _ = v.step(dt, 3)
    # means of non-negative values that round differently; an unchanged variable's mean is rounding itself
    assert np.abs(rel - vrel).max() <= 1e-10 * np.abs(vrel).max()
    uo = o.get_state()
    P.fp64_parity(s.get_state(), uo, x.get_state(), uo, mesh.dim, tol=1e-12)
    for c in (s, v):
        c.close()
