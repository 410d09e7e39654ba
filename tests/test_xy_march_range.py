"""The x and y sweeps of the hybrid scheme in one march address the listed
faces' fluxes with 32 bits: blocks whose 5 x (faces per axis) does not fit --
from 858 993 460 faces on, below ocfd_create's limit of 2^30 -- must take the
two sweeps, smaller large blocks the march."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIBDIR = os.path.join(ROOT, "opencfd-sc_amd")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def test_blocks_of_the_march(tmp_path):
    if not os.path.exists(HIPCC) or shutil.which("g++") is None:
        pytest.skip("hipcc not available")
    exe = str(tmp_path / "xy_march_range")
    r = subprocess.run([HIPCC, "-x", "hip", "--offload-host-only", "-std=c++17", "-I", os.path.join(LIBDIR, "csrc"),
                        os.path.join(ROOT, "tests", "c_abi", "xy_march_range.cpp"), "-o", exe, "-L" + LIBDIR,
                        "-locfd_hip", "-Wl,-rpath," + LIBDIR], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    # (nx, ny, nz), faces per axis below and above (2^32 - 1) / 5
    shapes = [((512, 512, 512), 1), ((896, 896, 896), 1), ((948, 950, 950), 1), ((960, 960, 960), 0),
              ((1024, 1000, 1000), 0)]
    r = subprocess.run([exe], input="".join("%d %d %d\n" % s for s, _ in shapes), capture_output=True, text=True,
                       timeout=60)
    assert r.returncode == 0, r.stderr
    for line, (s, takes) in zip(r.stdout.splitlines(), shapes):
        faces = max((s[0] + 1) * s[1] * s[2], s[0] * (s[1] + 1) * s[2])
        assert (5 * faces <= 2 ** 32 - 1) == bool(takes)
        assert line.split() == [str(takes)] * 2, s
