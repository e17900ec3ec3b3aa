"""Integrated quantities, numerical entropy and the maximum wave speed against the oracle where the
quadrature kernels' shapes can go wrong: one point per direction more than nodes and the widest rule
(32 points), more columns than threads (17^2), more cells than the summing block has threads.
Bar: 1e-12 relative, the bar of the other integrated-quantity tests."""
import numpy as np
import pytest

import oracle as O
import philip_amd as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,p,n,over", [(2, 1, 2, 0), (2, 6, 33, 10), (2, 3, 5, 28), (3, 1, 11, 10), (3, 2, 2, 0),
                                          (3, 3, 3, 28), (3, 4, 3, 9), (3, 6, 2, 10)])
def test_quadrature_kernels(dim, p, n, over):
    lo, hi = (-5.0, 5.0) if dim == 2 else (0.0, 2 * np.pi)
    kw = dict(dim=dim, poly_degree=p, n_cells_1d=n, domain_left=lo, domain_right=hi, use_split_form=1,
              two_point_flux=P.CH, conv_flux=P.TWO_POINT_ROE, mach_inf=0.3)
    o, d = O.Oracle(**kw), P.DG(**kw)
    u = (o.ic_tgv() if dim == 3 else o.ic_vortex()).reshape(o.ncells, o.ns, o.Np)
    u *= 1.0 + 0.05 * np.random.default_rng(p).uniform(-1, 1, u.shape)
    u = u.ravel()
    d.set_solution(u)
    print(dim, p, n, over, flush=True)
    a, b = d.integrated(over), o.integrated(u, over)
    for k in ("kinetic_energy", "enstrophy", "incompressible_kinetic_energy"):
        assert abs(a[k] - b[k]) <= 1e-12 * abs(b[k]), k
    assert abs(d.max_wave_speed(over) - o.max_wave_speed(u, over)) <= 1e-12 * o.max_wave_speed(u, over)
    assert abs(d.numerical_entropy() - o.numerical_entropy(u)) <= 1e-12 * abs(o.numerical_entropy(u))
