"""The FP64 line kernel against the oracle where its blocking can go wrong, in every form it takes
(split and conservative, the viscous terms, curvilinear grids), on small meshes and above: two cells a side (a cell is its own
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
# more blocks than compute units: the meshes that take the default block, not the small meshes'
LARGE = [(2, 1, 130), (2, 2, 86), (2, 3, 66), (2, 4, 52), (2, 6, 37), (3, 1, 21), (3, 2, 14), (3, 3, 11), (3, 4, 9),
         (3, 5, 7), (3, 6, 7)]


@pytest.mark.parametrize("dim,p,n", LARGE)
@pytest.mark.parametrize("form", ["ch", "ir", "conservative"])
def test_default_block(dim, p, n, form):
    kw = dict(use_split_form=0, conv_flux=P.ROE) if form == "conservative" else \
        dict(use_split_form=1, two_point_flux=P.CH if form == "ch" else P.IR, conv_flux=P.TWO_POINT_ROE)
    check(dict(kw, dim=dim, poly_degree=p, n_cells_1d=n, mach_inf=0.3), 17 * p + n)


@pytest.mark.parametrize("dim,p,n", [(2, 1, 5), (2, 2, 4), (2, 3, 7), (2, 4, 9), (2, 5, 8), (2, 6, 5), (3, 1, 3), (3, 2, 4),
                                     (3, 3, 5), (3, 4, 4), (3, 5, 3), (3, 6, 3)])
@pytest.mark.parametrize("form", ["ra", "conservative"])
def test_small_mesh_block(dim, p, n, form):
    kw = dict(use_split_form=0, conv_flux=P.LXF) if form == "conservative" else \
        dict(use_split_form=1, two_point_flux=P.RA, conv_flux=P.TWO_POINT_LXF)
    check(dict(kw, dim=dim, poly_degree=p, n_cells_1d=n, mach_inf=0.3), 19 * p + n)


@pytest.mark.parametrize("precision", [P.FP64, P.MIXED])
@pytest.mark.parametrize("dim,p,n", [(2, 1, 9), (2, 4, 33), (2, 6, 12), (3, 1, 5), (3, 2, 4), (3, 3, 5), (3, 4, 3), (3, 5, 3),
                                     (3, 6, 3)])
def test_small_mesh_block_has_the_bits_of_every_batch_tile(precision, dim, p, n):
    """A solve of a small mesh (a wave per direction and kind of item) and the same solve in a batch in
    every tile: block layouts must not change a bit."""
    kw = dict(dim=dim, poly_degree=p, n_cells_1d=n, use_split_form=1, two_point_flux=P.CH, conv_flux=P.TWO_POINT_ROE,
              mach_inf=0.3, precision=precision)
    if dim == 2:
        kw.update(domain_left=-5.0, domain_right=5.0, mach_inf=1.195)
    d = P.DG(**kw)
    start = (lambda x: x.set_initial_condition_tgv()) if dim == 3 else (lambda x: x.set_initial_condition_vortex())
    start(d)
    dt = d.constant_time_step(0.01)
    d.allocate_ode_system("rk4")
    d.step_in_time(dt, 3)
    ref = d.solution()
    for tile in range(13 if dim == 2 else 3):
        print(kw, tile, flush=True)
        b = P.Batch([kw, kw])
        for x in b.instances:
            start(x)
        b.set_tile(tile)
        b.allocate("rk4", [dt, dt])
        b.step_in_time(3)
        b.synchronize()
        for x in b.instances:
            assert np.array_equal(x.solution(), ref)
        b.close()


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
