"""The cross product's kernel takes three, two or one levels a workgroup,
whichever fits the row length: its last workgroup of a column has one to three
levels left.  Each value is formed and rounded as by the separate kernels, and
the row transforms are the same, so one step from a start must equal the step
of a context with LES_FUSE=0 bit for bit, at every remainder."""
import dataclasses

import numpy as np
import pytest

from overlappingbls_amd import config
from overlappingbls_amd.abi import LES_MIXED

pytestmark = pytest.mark.gpu


def step(gpu_lib, monkeypatch, nl, fuse, mixed):
    monkeypatch.setenv("LES_FUSE", fuse)
    g = gpu_lib.create(nl.params())
    if mixed:
        g.set_precision(LES_MIXED)
    config.load_state(g, config.initial_fields(nl, seed=53, vw_noise=True))
    g.run(1, 1)
    return {n: g.get(n) for n in ("CX", "CY", "CZ", "U", "V", "W", "THETA")}


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("nx,ny,nzt", [(16, 24, 4), (16, 24, 5), (48, 16, 6), (48, 16, 7), (96, 36, 8), (96, 36, 9),
                                       (384, 16, 5), (384, 16, 6), (512, 16, 4), (512, 16, 5)])
def test_level_remainders(nx, ny, nzt, mixed, gpu_lib, monkeypatch):
    nl = dataclasses.replace(config.workload("tiny_ragged"), nxt=nx, nyt=ny, nzt=nzt)
    nl = dataclasses.replace(nl, dt=nl.dt * min(1.0, 64.0 / max(nx, ny)))
    a, b = (step(gpu_lib, monkeypatch, nl, f, mixed) for f in ("1", "0"))
    assert all(np.isfinite(v).all() for v in a.values())
    assert not [n for n in a if not np.array_equal(a[n], b[n])]
