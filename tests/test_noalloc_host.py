"""kspace_field_noalloc allocates nothing on the host either (it runs inside
serving loops and captures): tests/link/count_new.cpp counts operator new
while it calls the entry point without sites, which stops before the device."""
import os
import shutil
import subprocess

import pytest

from molmodel_amd import engine as E

HERE = os.path.dirname(os.path.abspath(__file__))


def test_no_host_allocation(tmp_path):
    if not shutil.which("g++"):
        pytest.skip("g++ not present")
    if not os.path.exists(E.LIB_PATH):
        pytest.skip("libmolmodel_amd.so not built")
    exe = str(tmp_path / "count_new")
    build = ["g++", "-std=c++17", "-O1", os.path.join(HERE, "link", "count_new.cpp"), "-o", exe,
             E.LIB_PATH, "-Wl,-rpath," + os.path.dirname(E.LIB_PATH), "-Wl,-rpath-link=/opt/rocm/lib"]
    p = subprocess.run(build, capture_output=True, text=True, timeout=300)
    assert p.returncode == 0, p.stderr
    p = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    print(p.stdout)
    assert p.returncode == 0, p.stdout + p.stderr
