"""The library's host code without a GPU: tests/cpp/fake_hip.cpp stands in for
the HIP runtime in a child process (kernels are not run), so that memory that
runs out, a launch that fails and the stream each kernel goes to can be
checked on the CPU."""
import os
import shutil
import subprocess
import sys

import pytest

from overlappingbls_amd import build, lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PREAMBLE = """
import ctypes as C, dataclasses, sys
import numpy as np
fake = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
for f in ("fake_nmalloc", "fake_held", "fake_nlaunch", "fake_stream"):
    getattr(fake, f).restype = C.c_long
fake.fake_kernel.restype = C.c_char_p
fake.fake_kernel.argtypes = fake.fake_stream.argtypes = fake.fake_budget.argtypes = [C.c_long]
from overlappingbls_amd import config, lib
from overlappingbls_amd.abi import LES_E_HIP, LES_E_NOMEM, LES_MIXED, LES_OK, LesError

def grid(nx, ny, nzt=6, **kw):
    return dataclasses.replace(config.workload("tiny_ragged"), nxt=nx, nyt=ny, nzt=nzt, **kw).params()

def launches():
    return [(fake.fake_kernel(i).decode(), fake.fake_stream(i)) for i in range(fake.fake_nlaunch())]
"""


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    gxx, rocm = shutil.which("g++"), os.path.dirname(os.path.dirname(os.path.realpath(build.HIPCC)))
    if gxx is None:
        pytest.skip("no g++")
    if not os.path.exists(lib.LIB):
        build.build()
    so = str(tmp_path_factory.mktemp("fake") / "fake_hip.so")
    subprocess.run([gxx, "-O1", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I",
                    os.path.join(rocm, "include"), "-o", so, os.path.join(ROOT, "tests", "cpp", "fake_hip.cpp")],
                   check=True)

    def child(code, **env):
        r = subprocess.run([sys.executable, "-c", PREAMBLE + code, so], cwd=ROOT, env={**os.environ, **env},
                           capture_output=True, text=True)
        assert r.returncode == 0, r.stdout + r.stderr
    return child


# rows of 24 and 324 values have no contraction kernel, rows of 32 have one
@pytest.mark.parametrize("nx,fuse", [(24, "1"), (324, "1"), (32, "0"), (32, "1")])
def test_memory_is_taken_by_create(nx, fuse, fake):
    """All device memory of a step, dynamic SGS updates among them, belongs to
    les_create: none is allocated later, a shortage is refused there with
    LES_E_NOMEM and everything is given back."""
    fake(f"""
g = lib.create(grid({nx}, 12))
n, held = fake.fake_nmalloc(), fake.fake_held()
g.run(1, 4)
assert fake.fake_nmalloc() == n, "allocated in a step"
assert any("lagrange" in k or "lag_" in k for k, s in launches())
g.close()
assert fake.fake_held() == 0
fake.fake_budget(held - 1)
try:
    lib.create(grid({nx}, 12))
except LesError as e:
    assert e.status == LES_E_NOMEM, e.status
else:
    raise AssertionError("created without its memory")
assert fake.fake_held() == 0
""", LES_FUSE=fuse)


@pytest.mark.parametrize("why", ["query", "host_malloc"])
def test_a_failed_launch_is_reported(why, fake):
    """A launch that fails before a strided read-back is reported, also when
    the read-back's own query of the host pointer, or its page-locked chunks,
    fail and are done without."""
    fake(f"""
g = lib.create(grid(24, 12))
ld = g.nx + 2
out, spec, big = np.zeros((g.ny, ld)), np.zeros((g.ny, g.nx // 2 + 1, 2)), np.zeros((18, 36))
p = lambda a: a.ctypes.data_as(C.POINTER(C.c_double))
calls = dict(ifftn=("x_c2r", p(spec), p(out), ld), zero_unpadding=("yline", p(big), p(out), ld))
fake.fake_fail_{why}(1)
for name, (kernel, *args) in calls.items():
    fake.fake_fail_kernel(kernel.encode())
    assert g._f[name](g._h, *args) == LES_E_HIP, name
    fake.fake_fail_kernel(b"")
    assert g._f[name](g._h, *args) == LES_OK, name
""")


def test_a_refused_creation_leaves_nothing_behind(fake):
    """After memory ran out (les_create, les_set_precision) the next calls
    that have what they need succeed."""
    fake("""
g = lib.create(grid(24, 12))
held = fake.fake_held()
fake.fake_budget(held)
try:
    g.set_precision(LES_MIXED)
except LesError as e:
    assert e.status == LES_E_NOMEM, e.status
else:
    raise AssertionError("mixed mode without its memory")
g.ddx("WORK1", "WORK0")
try:
    lib.create(grid(24, 12))
except LesError as e:
    assert e.status == LES_E_NOMEM, e.status
fake.fake_budget(-1)
lib.create(grid(24, 12)).close()
""")


@pytest.mark.parametrize("overlap", ["0", "1"])
def test_serial_order_uses_one_stream(overlap, fake):
    """With LES_OVERLAP=0 every kernel of a step but the ordered plane sums (and
    the fills of their inputs) is launched on the context's stream; the filter's
    y pass, which otherwise runs beside the pressure solve, among them."""
    fake(f"""
for precision in (0, LES_MIXED):
    g = lib.create(grid(24, 12))
    g.set_precision(precision)
    fake.fake_clear()
    g.run(1, 3)
    of = launches()
    main = [s for k, s in of if "tdma" in k][0]
    sums = ("k_obukhov_sums", "k_level_means", "k_fill")
    away = {{k for k, s in of if s != main and not any(n in k for n in sums)}}
    assert bool(away) == {overlap == "1"}, away
    g.close()
""", LES_OVERLAP=overlap)


@pytest.mark.parametrize("fuse", ["0", "1"])
def test_pressure_routes(fuse, fake):
    """Plain steps form the pressure's right-hand side inside its row transform,
    with LES_FUSE=0 too (there the filter's row pass is a kernel of its own);
    statistics steps and rows without a table prepare it."""
    fake(f"""
for nx, stats in ((32, 0), (32, 1), (12, 0)):
    g = lib.create(grid(nx, 12))
    if stats:
        g.set_avgslice(True, 1, 100)
    fake.fake_clear()
    g.run(1, 1)
    names = [k for k, s in launches()]
    fused = [k for k in names if "kr_x_press" in k]
    assert bool(fused) == (nx == 32 and not stats), (nx, stats)
    assert any("k_press_prep" in k for k in names) != bool(fused), (nx, stats)
    if fused:
        assert fused[0].count("Lb1") == {fuse}, fused   # the FILTER argument
    g.close()
""", LES_FUSE=fuse)
