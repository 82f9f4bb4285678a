"""The facet lists' FP32 certificates, built for the host with g++ and checked
against the FP64 test they stand for: tests/host/cert_check.cpp."""
import os
import shutil
import subprocess

import pytest

from test_headers_host import CSRC, ROOT, host_copy


def test_certificates_never_contradict_fp64(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    for h in ("twg_math.hpp", "twg_geom.hpp", "twg_bvh.hpp"):
        host_copy(os.path.join(CSRC, h), str(tmp_path / h))
    exe = str(tmp_path / "cert_check")
    r = subprocess.run(["g++", "-O1", "-std=c++17", "-ffp-contract=off", "-fsanitize=address,undefined",
                        "-fno-sanitize=float-cast-overflow", "-I", str(tmp_path),
                        os.path.join(ROOT, "tests", "host", "cert_check.cpp"), "-o", exe],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=600)
    print(r.stdout)
    assert r.returncode == 0, r.stdout[-3000:] + r.stderr[-3000:]
    assert "\n0 failures" in r.stdout
