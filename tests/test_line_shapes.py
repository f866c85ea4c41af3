"""The launch shapes of the line kernels are those their comments were measured
with (compiled for the host: static_asserts in tests/cpp/line_shapes.hip)."""
import os
import subprocess

import pytest

from overlappingbls_amd import build

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_line_shapes():
    if not os.path.exists(build.HIPCC):
        pytest.skip("no hipcc")
    r = subprocess.run([build.HIPCC, "-std=c++17", f"--offload-arch={build.ARCH}", "--offload-host-only",
                        "-fsyntax-only", os.path.join(ROOT, "tests", "cpp", "line_shapes.hip")],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
