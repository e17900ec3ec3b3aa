"""Small jumps between cells on the FP64 path: the penalty and dissipation terms subtract the states
of the two sides, and a side whose momentum is rebuilt as rho v brings that product's rounding, which
is 1e-4 of a jump of 2^-40.

States are constant in each cell and p = 1, so that derivatives are exactly zero and the differences
exact, and the term in question is made to dominate what else rounds (a convective flux of 10 rounds
to 2e-15): a Reynolds number of 1e-6, where the jump's flux is above 1e-6; cells 2^20 times longer
along y and z than along x, where the faces that see the jump weigh 2^20 times the others.  The bar,
1e-7 of the largest value, is ten times what the other terms can round to and a thousandth of the
error that the test is for."""
import numpy as np
import pytest

import oracle as O
import philip_amd as P

pytestmark = pytest.mark.gpu
BAR = 1e-7
STEP = 2.0 ** -40


def base(dim, n):
    return dict(dim=dim, poly_degree=1, n_cells_1d=n, domain_left=0.0, domain_right=float(n), mach_inf=0.3,
                use_split_form=1, two_point_flux=P.CH)


def compare(o, d, u, components):
    ref = o.residual(u).reshape(o.ncells, o.ns, o.Np)
    d.set_solution(u)
    r = d.assemble_residual().reshape(ref.shape)
    for s in components:
        big = np.abs(ref[:, s]).max()
        err = np.abs(r[:, s] - ref[:, s]).max() / big
        print(f"  component {s}: largest {big:.2e}, err {err:.2e}", flush=True)
        assert big > 0 and err <= BAR
    d.close()


@pytest.mark.parametrize("n", [3, 5])
@pytest.mark.parametrize("cf", [P.TWO_POINT, P.TWO_POINT_ROE, P.TWO_POINT_LXF])
@pytest.mark.parametrize("warp", [0, 1])
def test_penalty_of_a_small_momentum_jump(n, cf, warp):
    kw = dict(base(3, n), conv_flux=cf, pde=P.NAVIER_STOKES, diss_flux=P.SIPG, use_constant_viscosity=1,
              constant_viscosity=1.0, reynolds_inf=1e-6, prandtl=0.71)
    print(kw, warp, flush=True)
    o, d = O.Oracle(**kw), P.DG(**kw)
    if warp:  # the same box as a curvilinear grid
        x = o.node_coords()
        o.set_grid_nodes(x)
        d.set_grid_nodes(x)
    rng = np.random.default_rng(n + cf)
    u = o.vec().reshape(o.ncells, o.ns, o.Np)
    u[:, 0] = 0.7
    u[:, 1:4] = 0.5 + STEP * rng.integers(-8, 9, (o.ncells, 3, 1))
    u[:, 4] = 20.0
    compare(o, d, u.ravel(), (1, 2, 3))


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("n", [3, 7])
@pytest.mark.parametrize("pde", [P.EULER, P.NAVIER_STOKES])
@pytest.mark.parametrize("cf", [P.LXF, P.TWO_POINT_LXF])
def test_dissipation_of_a_small_momentum_jump(dim, n, pde, cf):
    """Against the dissipation itself: with v_x = 0 nothing else reaches the transverse momenta at the
    faces along x (the oracle's split form passes face states through the entropy variables, which
    rounds them)."""
    kw = dict(base(dim, n), conv_flux=cf)
    if pde == P.NAVIER_STOKES:
        if dim == 2:
            pytest.skip("Navier-Stokes is 3D")
        kw.update(pde=pde, diss_flux=P.BR2, use_constant_viscosity=1, constant_viscosity=1.0, reynolds_inf=1e9,
                  prandtl=0.71)
    print(kw, flush=True)
    o, d = O.Oracle(**kw), P.DG(**kw)
    x = o.node_coords()
    x[..., 1:dim] *= 2.0 ** 20
    d.set_grid_nodes(x)
    rng = np.random.default_rng(n + cf)
    u = o.vec().reshape(o.ncells, o.ns, o.Np)
    at = np.rint(x[:, 0, 0]).astype(int)  # a cell's place along x
    m = 0.5 + STEP * rng.integers(-8, 9, (n, dim - 1))
    u[:, 0] = 0.7
    u[:, 1] = 0.0
    u[:, 2:-1] = m[at][..., None]
    u[:, -1] = 20.0
    d.set_solution(u.ravel())
    r = d.assemble_residual().reshape(u.shape)
    d.close()
    c = np.sqrt(1.4 * 0.4 * (20.0 - 0.5 * (m * m).sum(1) / 0.7) / 0.7)
    scale = 2.0 * 0.5 ** dim * 2.0 ** (20 * (dim - 1))  # lift, weight of the node, det J
    for side in (0, 1):  # a node of p = 1 is on one of the two faces along x
        nb = np.roll(np.arange(n), 1 - 2 * side)
        want = scale * (0.5 * np.maximum(c, c[nb]))[:, None] * (m[nb] - m)
        got = r[:, 2:-1, side::2]
        err = np.abs(got - want[at][..., None]).max() / np.abs(want).max()
        print(f"  side {side}: largest {np.abs(want).max():.2e}, err {err:.2e}", flush=True)
        assert err <= BAR
