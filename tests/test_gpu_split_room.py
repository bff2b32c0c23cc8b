"""A launch that would split its tiles over the source pencils, on a GPU without
room for the planes that takes: it runs with whole tiles, bitwise the same."""
import os
import shutil
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "sanitize")


def test_planes_without_room(tmp_path):
    if not shutil.which("g++"):
        pytest.skip("g++ not found")
    shim = str(tmp_path / "malloc_limit.so")
    subprocess.run(["g++", "-O1", "-fPIC", "-shared", os.path.join(HERE, "malloc_limit.cpp"), "-ldl", "-o", shim],
                   check=True)
    r = subprocess.run([sys.executable, "-u", os.path.join(HERE, "malloc_limit_child.py"), shim], capture_output=True,
                       text=True, timeout=100)
    assert r.returncode == 0 and "same without room" in r.stdout, r.stdout[-2000:] + r.stderr[-2000:]
