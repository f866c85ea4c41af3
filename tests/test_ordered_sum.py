"""The scanned plane sums have the bits of the sequential loop: the maps of
ordered_sum.hpp, which the kernels scan, compiled for the host and compared
with the loop over sums that grow, stay zero, cancel, tie and overflow."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_scanned_sum_equals_the_loop(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("no g++")
    exe = str(tmp_path / "check")
    subprocess.run([gxx, "-O2", "-std=c++17", "-ffp-contract=off", "-o", exe,
                    os.path.join(ROOT, "tests", "cpp", "ordered_sum_check.cpp")], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("nx,ny", [(32, 64), (48, 48), (64, 64), (96, 72), (128, 144), (256, 256), (512, 288)])
@pytest.mark.parametrize("kind", ["noise", "uniform", "zero head", "wide", "rising"])
def test_plane_sum_on_the_gpu(nx, ny, kind, gpu_lib):
    """obukhov's neutral friction velocity is the plane sum of the speed times
    constants: equal to the sequential sum's to the last bits of the
    constants (a tree sum is off by 1e-14 and more)."""
    import dataclasses

    import numpy as np
    from overlappingbls_amd import config

    nl = dataclasses.replace(config.workload("wide"), nxt=nx, nyt=ny, theta_flag=False)
    p = nl.params()
    g = gpu_lib.create(p)
    r = np.random.default_rng(nx * ny)
    n = nx * ny
    u = {"noise": 20.0 + r.standard_normal(n), "uniform": np.full(n, 7.3),
         "zero head": np.where(np.arange(n) < n // 3, 0.0, 1.0 + r.random(n)),
         "wide": np.ldexp(1.0 + r.random(n), r.integers(-40, 40, n)),
         "rising": np.ldexp(1.0 + r.random(n), np.arange(n) * 90 // n)}[kind]
    v = np.where(np.arange(n) % 2, 0.25, 0.5) * u
    for name, a in (("U", u), ("V", v)):
        f = np.zeros((g.nlev, ny, nx))
        f[1] = a.reshape(ny, nx)
        g.set(name, f)
    g.obukhov(1)
    s = 0.0
    for x in np.sqrt(u * u + v * v).tolist():
        s += x
    dz = p.lz_tot / (p.nzt - 1)
    want = s / n * 0.4 / np.log(0.5 * dz / p.zo)
    got = g.get("USTAR_SFC")
    assert np.all(got == got[0, 0])
    assert abs(got[0, 0] - want) <= 1e-15 * want, (got[0, 0], want)
