"""Host transfers with and without row padding: set_field and get_field move
values unchanged and leave the caller's padding columns alone, for blocks
smaller and larger than a transfer chunk, whole and partial level ranges."""
import ctypes as C

import numpy as np
import pytest

from overlappingbls_amd import config
from overlappingbls_amd.abi import FIELD, LES_MIXED, LesError

pytestmark = pytest.mark.gpu


def _pd(a):
    return a.ctypes.data_as(C.POINTER(C.c_double))


# 24 x 12: rows of 192 bytes; 256 x 256: 512 rows a chunk, so five levels are
# two chunks and a half
@pytest.mark.parametrize("case", ["tiny_ragged", "wide"])
@pytest.mark.parametrize("pad", [0, 2, 7])
@pytest.mark.parametrize("name", ["U", "TXX"])
@pytest.mark.parametrize("mixed", [False, True])
def test_round_trip(case, pad, name, mixed, gpu_lib):
    g = gpu_lib.create(config.workload(case).params())
    if mixed:
        g.set_precision(LES_MIXED)
    for lev0, nlev in ((0, g.nlev), (1, g.nlev - 2), (g.nlev - 1, 1), (2, 0)):
        ld = g.nx + pad
        a = np.full((nlev, g.ny, ld), 3.0e30)
        val = config.uniform(5 + lev0, 1, (max(nlev, 1), g.ny, g.nx))[:nlev]
        if mixed and name == "TXX":           # a work field: single precision on the device
            val = val.astype(np.float32).astype(np.float64)
        a[:, :, :g.nx] = val
        if mixed and name == "TXX" and nlev == 0:     # an empty range of a single-precision field is refused
            with pytest.raises(LesError):
                g._call("set_field", g._h, FIELD[name], _pd(a), ld, lev0, nlev)
            continue
        g._call("set_field", g._h, FIELD[name], _pd(a), ld, lev0, nlev)
        b = np.full((nlev, g.ny, ld), -7.0)
        g._call("get_field", g._h, FIELD[name], _pd(b), ld, lev0, nlev)
        assert np.array_equal(b[:, :, :g.nx], val)
        assert np.all(b[:, :, g.nx:] == -7.0)


@pytest.mark.parametrize("pad", [0, 2])
def test_linear_state_round_trip(pad, gpu_lib):
    g = gpu_lib.create(config.workload("wide").params())
    ld = g.nx + pad
    a = np.full((g.nz - 1, g.ny, ld), 3.0e30)
    a[:, :, :g.nx] = config.uniform(9, 1, (g.nz - 1, g.ny, g.nx))
    g._call("lin_set", g._h, FIELD["V"], _pd(a), ld, 1, g.nz - 1)
    b = np.full(a.shape, -7.0)
    g._call("lin_get", g._h, FIELD["V"], _pd(b), ld, 1, g.nz - 1)
    assert np.array_equal(b[:, :, :g.nx], a[:, :, :g.nx])
    assert np.all(b[:, :, g.nx:] == -7.0)
