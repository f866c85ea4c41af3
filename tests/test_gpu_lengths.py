"""Every compile-time line length against the oracle: derivatives, Nyquist
filter, the one-plane transforms, the test filter, and steps through a
dynamic SGS update (the fused 3/2-grid passes and the Lagrangian contraction
of each length).  Bars as in the parity tests: 1e-12 for FP64 lines and the
velocity and temperature after a step; 1e-6 for FP32 lines."""
import dataclasses

import numpy as np
import pytest

from overlappingbls_amd import config
from overlappingbls_amd.abi import LES_MIXED

pytestmark = pytest.mark.gpu

TOL = 1e-12
# each length once along x and once along y
PAIRS = [(16, 24), (24, 32), (32, 36), (36, 48), (48, 64), (64, 72), (72, 96), (96, 108), (108, 128), (128, 144),
         (144, 192), (192, 216), (216, 256), (256, 288), (288, 384), (384, 512), (512, 16)]


def rel(a, b):
    return float(np.linalg.norm((a - b).ravel()) / np.linalg.norm(b.ravel()))


def grid(nx, ny, nzt):
    return dataclasses.replace(config.workload("tiny_ragged"), nxt=nx, nyt=ny, nzt=nzt)


@pytest.mark.parametrize("nx,ny", PAIRS)
def test_lines(nx, ny, oracle_mod, gpu_lib):
    p = grid(nx, ny, 4).params()
    o, g = oracle_mod.create(p), gpu_lib.create(p)
    a = config.uniform(31, 2, (o.nlev, ny, nx))
    for c in (o, g):
        c.set("WORK0", a)
        c.ddx("WORK1", "WORK0")
        c.ddy("WORK2", "WORK0")
    bad = {n: rel(g.get(n), o.get(n)) for n in ("WORK1", "WORK2")}
    for c in (o, g):
        c.filter_data("WORK0")
        c.test_filter("WORK1", 2, 2)
    bad["filter"] = rel(g.get("WORK0"), o.get("WORK0"))
    bad["test_filter"] = rel(g.get("WORK1", 2, 1), o.get("WORK1", 2, 1))
    plane, big = a[1], config.uniform(32, 2, (1, 3 * ny // 2, 3 * nx // 2))[0]
    spec = o.fftn(plane)
    bad["fftn"] = rel(g.fftn(plane), spec)
    bad["ifftn"] = rel(g.ifftn(spec), o.ifftn(spec))
    bad["pad"] = rel(g.zero_padding(plane), o.zero_padding(plane))
    bad["unpad"] = rel(g.zero_unpadding(big), o.zero_unpadding(big))
    bad = {k: v for k, v in bad.items() if not v < TOL}
    # single precision, from FP64 state (U) and from a work field
    g.set_precision(LES_MIXED)
    for c in (o, g):
        c.set("U", a)
        c.ddx("DUDX", "U")
        c.ddy("DUDY", "U")
        c.set("TXX", a.astype(np.float32).astype(np.float64))
        c.ddx("TXY", "TXX")
        c.ddy("TYY", "TXX")
    for n in ("DUDX", "DUDY", "TXY", "TYY"):
        r = rel(g.get(n), o.get(n))
        if not r < 1e-6:
            bad["fp32 " + n] = r
    assert not bad, bad


@pytest.mark.parametrize("nx,ny", PAIRS)
def test_steps(nx, ny, oracle_mod, gpu_lib):
    """Three steps with the dynamic update at step 2 (cs_count 2)."""
    nl = grid(nx, ny, 6)
    nl = dataclasses.replace(nl, dt=nl.dt * min(1.0, 64.0 / max(nx, ny)))
    p = nl.params()
    o, g = oracle_mod.create(p), gpu_lib.create(p)
    f = config.initial_fields(nl, seed=41, vw_noise=True)
    bad = {}
    for c in (o, g):
        config.load_state(c, f)
    for jt in (1, 2, 3):
        for c in (o, g):
            c.step(jt)
        for n in ("U", "V", "W", "THETA"):
            sl = config.physical_levels(n, o.nz)
            r = rel(g.get(n)[sl], o.get(n)[sl])
            if not r < TOL:
                bad[jt, n] = r
    assert not bad, bad
