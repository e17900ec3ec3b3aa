"""CPU check of the FP64 line kernels' surface and viscous fluxes along a general unit normal
(dg_fast.hpp, host build) against the oracle's point physics.

Bars: the numerical flux within 1e-13 of its largest component (the bar of the axis-aligned check);
the flux from the other side along the opposite normal is its exact negative, which is what makes a
face evaluated in two blocks conservative to the last bit; viscous fluxes within 1e-13 of the sum of
the magnitudes of their terms, bounded by the flux of the gradient with every sign made the same."""
import os
import subprocess

import numpy as np
import pytest

import oracle as O

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def host_exe(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("line64") / "line_fluxes64_host")
    subprocess.run(["g++", "-O2", "-std=c++17", "-o", exe, os.path.join(HERE, "host", "line_fluxes64_host.cpp")],
                   check=True)
    return exe


def states(rng, n, mach):
    rho = 1.0 + 0.3 * rng.uniform(-1, 1, n)
    vel = 0.5 * rng.standard_normal((n, 3))
    p = (1.0 / (1.4 * mach * mach)) * (1.0 + 0.3 * rng.uniform(-1, 1, n))
    return np.column_stack([rho, rho[:, None] * vel, p / 0.4 + 0.5 * rho * (vel ** 2).sum(1)])


@pytest.mark.parametrize("mach", [0.1, 1.2])
@pytest.mark.parametrize("tp,cf", [(O.CH, O.TWO_POINT_ROE), (O.RA, O.TWO_POINT_LXF), (O.CH, O.TWO_POINT),
                                   (O.RA, O.ROE), (O.CH, O.LXF), (O.RA, O.CENTRAL), (O.KG, O.TWO_POINT_ROE),
                                   (O.IR, O.TWO_POINT_LXF)])
def test_normal_fluxes_match_oracle_and_are_antisymmetric(host_exe, tp, cf, mach):
    rng = np.random.default_rng(3 + 10 * tp + cf)
    n = 48
    ui, ue = states(rng, n, mach), states(rng, n, mach)
    ue[: n // 2] = ui[: n // 2] * (1 + 1e-3 * rng.standard_normal((n // 2, 5)))
    nm = rng.standard_normal((n, 3))
    nm /= np.linalg.norm(nm, axis=1, keepdims=True)
    g = rng.standard_normal((n, 5, 3))
    const = tp % 2
    inp = f"{n} {tp} {cf} {mach} {const}\n" + "\n".join(
        " ".join(f"{x:.17g}" for x in np.r_[a, b, c, d.ravel()]) for a, b, c, d in zip(ui, ue, nm, g))
    out = subprocess.run([host_exe], input=inp, capture_output=True, text=True, check=True).stdout
    got = np.array([[float(x) for x in line.split()] for line in out.strip().splitlines()])
    o = O.Oracle(dim=3, poly_degree=1, n_cells_1d=2, two_point_flux=tp, conv_flux=cf, mach_inf=mach,
                 use_split_form=1 if cf >= O.TWO_POINT else 0, pde=O.NAVIER_STOKES, reynolds_inf=100.0, prandtl=0.71,
                 use_constant_viscosity=const, constant_viscosity=1.3, temperature_inf=273.15)
    # a face looks the same from either side, to the last bit
    assert (got[:, 5:10] == -got[:, :5]).all()
    for i in range(n):
        ref = o.numerical_flux(cf, ui[i], ue[i], nm[i])
        assert np.abs(got[i, :5] - ref).max() < 1e-13 * np.abs(ref).max()
        fv = o.dissipative_flux(ui[i], g[i])
        jump = (ui[i] - ue[i])[:, None] * nm[i][None, :]
        fj = o.dissipative_flux(ui[i], jump) @ nm[i]
        for a, b, grad in ((got[i, 10:22].reshape(3, 4), fv[1:].T, g[i]), (got[i, 22:], fj[1:], jump)):
            # terms of the energy flux reach E |grad| / rho times the conductivity
            big = np.abs(grad).max() * (1.0 + ui[i, 4] / ui[i, 0]) * 1.4 / 0.71 / 100.0 * 10.0
            assert np.abs(a - b).max() < 1e-13 * max(big, np.abs(b).max())
