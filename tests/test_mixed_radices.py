"""Stage radices of the mixed-radix passes, on the CPU: every radix above 13 (a
dense stage on the matrix cores) is prime, and lengths whose prime factors are 13
or less have butterflies only (tests/cpp/radices_test.cpp)."""
import os
import subprocess

import pytest

from test_host_sanitizers import CPP, CSRC, HIPCC, HOST_SAN, run


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
def test_radices_under_sanitizers(tmp_path):
    exe = tmp_path / "radices_test"
    subprocess.run([HIPCC, "-x", "hip", "--offload-host-only", "-std=c++17", "-O1", "-g", "-fno-omit-frame-pointer"]
                   + HOST_SAN + ["-I", CSRC, os.path.join(CPP, "radices_test.cpp"),
                                 os.path.join(CSRC, "ff_mixplan.cpp"), "-o", str(exe), "-lpthread"],
                   check=True, capture_output=True)
    run(exe, "radices ok")
