"""The FP64 line kernel with the viscous terms and on curvilinear grids (Chandrashekar and Ranocha
split forms) against the oracle where its blocking can go wrong: two cells a side (a cell is its own
neighbour's neighbour on both sides), cell counts that leave a part of the last block empty, every
degree, both viscous numerical fluxes; and boundary faces, whose exterior states are the traces of
its face items.  Bar: 1e-12 of the sum of the absolute values of a DoF's terms, as in the other
residual parity tests."""
import numpy as np
import pytest

import oracle as O
import philip_amd as P

pytestmark = pytest.mark.gpu


def check(kw, seed):
    print(kw, flush=True)
    o, d = O.Oracle(**kw), P.DG(**kw)
    rng = np.random.default_rng(seed)
    u = o.vec().reshape(o.ncells, o.ns, o.Np)
    rho = rng.uniform(0.8, 1.2, (o.ncells, o.Np))
    v = rng.uniform(-0.5, 0.5, (o.ncells, o.dim, o.Np))
    p = rng.uniform(0.8, 1.2, (o.ncells, o.Np)) / (1.4 * 0.09)
    u[:, 0] = rho
    u[:, 1:1 + o.dim] = rho[:, None] * v
    u[:, -1] = p / 0.4 + 0.5 * rho * (v * v).sum(axis=1)
    u = u.ravel()
    ref = o.residual(u)
    m = o.residual_magnitude(u).reshape(o.ncells, o.ns, o.Np)
    d.set_solution(u)
    r = d.assemble_residual()
    den = np.maximum(m, 1e-8 * m.max(axis=(0, 2), keepdims=True))
    err = float((np.abs(r - ref).reshape(m.shape) / den).max())
    print(f"  per-DoF err {err:.2e}", flush=True)
    assert err <= 1e-12
    d.close()


SPLIT = dict(use_split_form=1, mach_inf=0.3)
NS = dict(pde=P.NAVIER_STOKES, use_constant_viscosity=0, reynolds_inf=200.0, prandtl=0.71)


@pytest.mark.parametrize("p,n", [(1, 2), (1, 5), (2, 3), (3, 2), (3, 3), (4, 3), (5, 2), (6, 2)])
@pytest.mark.parametrize("tp,cf,diss", [(P.CH, P.TWO_POINT_ROE, P.SIPG), (P.RA, P.TWO_POINT_LXF, P.BR2),
                                        (P.RA, P.CENTRAL, P.SIPG), (P.IR, P.TWO_POINT_ROE, P.BR2)])
@pytest.mark.parametrize("warp", [0, 1])
def test_navier_stokes(p, n, tp, cf, diss, warp):
    check(dict(SPLIT, **NS, dim=3, poly_degree=p, n_cells_1d=n, two_point_flux=tp, conv_flux=cf, diss_flux=diss,
               grid_warp=warp), 7 * p + n)


@pytest.mark.parametrize("dim,p,n", [(2, 1, 7), (2, 2, 3), (2, 4, 5), (2, 6, 3), (3, 1, 5), (3, 2, 4), (3, 3, 3),
                                     (3, 4, 3), (3, 5, 2), (3, 6, 2)])
@pytest.mark.parametrize("tp,cf", [(P.CH, P.TWO_POINT_ROE), (P.RA, P.ROE), (P.KG, P.TWO_POINT_LXF)])
def test_curved_euler(dim, p, n, tp, cf):
    lo, hi = (-1.0, 1.0) if dim == 2 else (0.0, 2 * np.pi)
    check(dict(SPLIT, dim=dim, poly_degree=p, n_cells_1d=n, two_point_flux=tp, conv_flux=cf, grid_warp=1,
               domain_left=lo, domain_right=hi), 11 * p + n)


@pytest.mark.parametrize("dim,p,n", [(2, 1, 9), (2, 3, 5), (2, 6, 3), (3, 1, 5), (3, 3, 3), (3, 4, 3), (3, 6, 2)])
@pytest.mark.parametrize("tp,cf", [(P.CH, P.TWO_POINT_ROE), (P.RA, P.LXF), (P.IR, P.TWO_POINT)])
@pytest.mark.parametrize("bc", [1002, 1003, 1004, 1006, 1007])
def test_boundary_traces(dim, p, n, tp, cf, bc):
    check(dict(SPLIT, dim=dim, poly_degree=p, n_cells_1d=n, two_point_flux=tp, conv_flux=cf,
               boundary_type=[bc, 1005, 0, 0, bc, bc]), 13 * p + n)
