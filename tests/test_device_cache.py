"""The launchers' per-device values are shared by the handles of all threads:
no data race (ThreadSanitizer), and the launchers keep them nowhere else."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "opencfd-sc_amd", "csrc")


def test_threads_share_the_cache(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path / "device_cache")
    r = subprocess.run(["g++", "-std=c++17", "-g", "-O1", "-fsanitize=thread", "-pthread", "-I", CSRC,
                        os.path.join(ROOT, "tests", "c_abi", "device_cache.cpp"), "-o", exe],
                       capture_output=True, text=True)
    if r.returncode != 0 and "tsan" in r.stderr:
        pytest.skip("ThreadSanitizer not available")
    assert r.returncode == 0, r.stderr
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    if "unexpected memory mapping" in r.stderr:
        pytest.skip("ThreadSanitizer cannot run here")
    assert r.returncode == 0 and r.stdout == "wrong 0\n", r.stdout + r.stderr[-2000:]


def test_launchers_keep_no_plain_statics():
    """Function-local statics of the library are the caches and constant tables."""
    for name in sorted(os.listdir(CSRC)):
        if not name.endswith((".h", ".hip")):
            continue
        text = open(os.path.join(CSRC, name)).read()
        for line in re.findall(r"^[ \t]+static\s+(?!const\b|constexpr\b|_assert|inline\b|__device__\b)[^\n(]*[;=\[][^\n]*", text,
                               re.M):
            assert "DeviceCache" in line, "%s: %s" % (name, line.strip())
