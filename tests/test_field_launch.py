"""Launches of the driver kernels (fishfry_amd/csrc/ff_field.hip) on the CPU:
the host code runs under AddressSanitizer and UndefinedBehaviorSanitizer with the
HIP launch calls replaced by stand-ins (tests/cpp/field_launch.cpp) that refuse
dynamic LDS above 64 KB unless the kernel has been given it, and grids without
workgroups, for grids of every planes-per-tile and extents up to 2^31 - 1."""
import os
import subprocess

import pytest

from test_host_sanitizers import CPP, CSRC, HIPCC, HOST_SAN, run


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
def test_field_launches(tmp_path):
    exe = tmp_path / "field_launch"
    # (the device code is not built: its fat binary stays an unresolved symbol)
    subprocess.run([HIPCC, "-x", "hip", "--offload-host-only", "-std=c++17", "-O1", "-g", "-fno-omit-frame-pointer"]
                   + HOST_SAN + ["-Wl,--unresolved-symbols=ignore-all", "-I", CSRC,
                                 os.path.join(CPP, "field_launch.cpp"), os.path.join(CSRC, "ff_field.hip"),
                                 "-o", str(exe), "-lpthread"], check=True, capture_output=True)
    run(exe, "field launches ok")
