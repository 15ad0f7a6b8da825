"""The list of pinned blocks that sizes are read back through (csrc/qpip_mailbox.hpp),
checked on the host (tests/cpp/mailbox_check.cc): a call that fails gives its block back,
or, with a kernel in flight, leaves it to the next trim."""

import os
import shutil
import subprocess

import pytest
from conftest import ROOT


def test_blocks_of_failed_calls_are_freed(tmp_path):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no C++ compiler")
    exe = str(tmp_path / "mailbox_check")
    subprocess.run([cxx, "-O1", "-std=c++17", "-pthread", "-Wall", "-Werror",
                    "-I", os.path.join(ROOT, "cuspatial_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "mailbox_check.cc"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
