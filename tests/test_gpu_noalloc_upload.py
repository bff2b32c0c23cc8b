"""nf_execute_sic_noalloc uploads the work list it made, not the list's bound."""
import os
import shutil
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "sanitize")


def test_upload_ends_with_the_list(tmp_path):
    if not shutil.which("g++"):
        pytest.skip("g++ not found")
    shim = str(tmp_path / "upload_count.so")
    subprocess.run(["g++", "-O1", "-fPIC", "-shared", os.path.join(HERE, "upload_count.cpp"), "-ldl", "-o", shim],
                   check=True)
    r = subprocess.run([sys.executable, "-u", os.path.join(HERE, "upload_count_child.py"), shim], capture_output=True,
                       text=True, timeout=100)
    assert r.returncode == 0 and "uploaded" in r.stdout, r.stdout[-2000:] + r.stderr[-2000:]
    whole, may_split, split = (int(v) for v in r.stdout.split("uploaded")[1].split())
    # The same list where no tile costs enough to be split; longer, by 16 bytes an item, where all are.
    assert may_split == whole
    assert split > whole and (split - whole) % 16 == 0
