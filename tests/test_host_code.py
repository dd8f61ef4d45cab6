"""Host code of the library that a CPU can check: built with hipcc for the host
alone and run, against stand-ins where it calls the GPU runtime."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
HOST = os.path.join(ROOT, "tests", "host")

pytestmark = pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs hipcc")


def _run(tmp_path, *sources):
    exe = str(tmp_path / "host")
    subprocess.run([HIPCC, "-x", "hip", "--offload-host-only", "--offload-arch=gfx950", "-O1", "-std=c++17", "-pthread",
                    "-o", exe, *sources], check=True, timeout=300)
    return subprocess.run([exe], capture_output=True, text=True, timeout=120)


def test_work_items_are_numbered_past_32_bits(tmp_path):
    r = _run(tmp_path, os.path.join(HOST, "items_host.hip"))
    assert r.returncode == 0, r.stdout + r.stderr


def test_field_copies_leave_nothing_in_flight(tmp_path):
    r = _run(tmp_path, os.path.join(HOST, "copy_host.hip"), os.path.join(ROOT, "streams-2_amd", "csrc", "st_copy.hip"))
    assert r.returncode == 0, r.stdout + r.stderr
