"""CPU check that an FP64 line kernel's node cache loses nothing that a flux reads (dg_fast.hpp, host
build): the Kennedy-Gruber flux averages E / rho, so it has to get the node's own E.  Equal to the
last bit: the same evaluation on the same values."""
import os
import subprocess

import numpy as np
import pytest

import oracle as O

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def host_exe(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("form") / "form_cache_host")
    subprocess.run(["g++", "-O2", "-std=c++17", "-o", exe, os.path.join(HERE, "host", "form_cache_host.cpp")],
                   check=True)
    return exe


@pytest.mark.parametrize("tp", [O.KG, O.IR])
@pytest.mark.parametrize("mach", [0.1, 1.2])
def test_two_point_flux_reads_the_nodes_energy(host_exe, tp, mach):
    rng = np.random.default_rng(int(10 * mach) + tp)
    n = 200
    rho = rng.uniform(0.7, 1.3, (n, 2))
    v = rng.uniform(-0.5, 0.5, (n, 2, 3))
    p = rng.uniform(0.7, 1.3, (n, 2)) / (1.4 * mach * mach)
    u = np.concatenate([rho[..., None], rho[..., None] * v, (p / 0.4 + 0.5 * rho * (v * v).sum(-1))[..., None]], -1)
    text = f"{n} {tp}\n" + "\n".join(" ".join(f"{x:.17g}" for x in r.ravel()) for r in u)
    out = subprocess.run([host_exe], input=text, capture_output=True, text=True, check=True).stdout
    f = np.array([[float(x) for x in line.split()] for line in out.splitlines()]).reshape(n, 3, 5)
    assert (f[:, 0] == f[:, 2]).all()
    assert (f[:, 1] == f[:, 2]).all()
