"""When the ordered plane sums are scanned and when they are walked: the rule
of ordered_sum.hpp compiled for the host, and the kernel's bits on signed
planes, whose sums cancel."""
import dataclasses
import os
import shutil
import subprocess

import numpy as np
import pytest

from overlappingbls_amd import config

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_pace(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("no g++")
    exe = str(tmp_path / "pace")
    subprocess.run([gxx, "-O2", "-std=c++17", "-ffp-contract=off", "-o", exe,
                    os.path.join(ROOT, "tests", "cpp", "ordered_sum_pace.cpp")], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("nx,ny", [(48, 48), (64, 64), (64, 72), (128, 144), (256, 256), (512, 288)])
@pytest.mark.parametrize("kind", ["signed", "drifting", "waves", "back to zero", "ties"])
def test_signed_plane_sum_on_the_gpu(nx, ny, kind, gpu_lib):
    """obukhov's neutral friction velocity with a psi_m plane of either sign,
    large beside the logarithm: it follows the plane sum to its last bits."""
    nl = dataclasses.replace(config.workload("wide"), nxt=nx, nyt=ny, theta_flag=False, restart_theta=True)
    p = nl.params()
    g = gpu_lib.create(p)
    r = np.random.default_rng(nx + ny)
    n = nx * ny
    i = np.arange(n)
    psi = {"signed": r.standard_normal(n), "drifting": 0.3 + r.standard_normal(n),
           "waves": np.sin(0.05 * i) + 0.2 * r.standard_normal(n),
           "back to zero": np.where(i % 2, -1.3, 1.3) + np.where(i == n - 1, 7.0, 0.0),
           "ties": np.ldexp(r.integers(-3, 4, n).astype(float), -2)}[kind] * 2.0 ** 40
    u = np.zeros((g.nlev, ny, nx))
    u[1] = 3.0
    g.set("U", u)
    g.set("PSI_M_SFC", psi.reshape(ny, nx))
    g.obukhov(1)
    s = 0.0
    for x in psi.tolist():
        s += x
    assert s != 0.0
    dz = p.lz_tot / (p.nzt - 1)
    want = 3.0 * 0.4 / (np.log(0.5 * dz / p.zo) - s / n)
    got = g.get("USTAR_SFC")
    assert np.all(got == got[0, 0])
    # a division, a difference from a logarithm below 2^-30 of it, a division
    # and products of 3 n, which is exact: four roundings
    assert abs(got[0, 0] - want) <= 5e-16 * abs(want), (got[0, 0], want)
