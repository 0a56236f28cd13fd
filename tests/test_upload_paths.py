"""Host test of the factor upload's failure paths (stars-h_amd/csrc/hip/
copyin.hip compiled for the host, the runtime's calls replaced by
copyin_host.cpp): where the pinned ring or its threads cannot be had, the
arrays go through ordinary memory; after a failed copy nothing is left queued
and no slot is refilled under a queued copy."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "stars-h_amd", "csrc")


@pytest.fixture(scope="module")
def upload_bin(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("copyin") / "copyin")
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    obj = []
    for src in (os.path.join(CSRC, "hip", "copyin.hip"),
                os.path.join(ROOT, "tests", "copyin_host.cpp")):
        obj.append(f"{out}{len(obj)}.o")
        subprocess.check_call(
            [hipcc, "-x", "hip", "--offload-host-only", "-O1", "-fPIC",
             "-std=c++17",
             "-I", os.path.join(ROOT, "include"),
             "-I", os.path.join(CSRC, "include"), "-c", src, "-o", obj[-1]])
    subprocess.check_call(["g++", "-o", out] + obj + ["-pthread", "-ldl"])
    return out


def _run(binary, mode):
    res = subprocess.run([binary, mode], capture_output=True, text=True,
                         timeout=100, check=True)
    return [int(x) for x in res.stdout.split()]


@pytest.mark.parametrize("mode", ["ok", "pin", "thread"])
def test_arrays_arrive(upload_bin, mode):
    assert _run(upload_bin, mode) == [0, 1, 0, 0]


def test_a_failed_copy_leaves_nothing_queued(upload_bin):
    info, arrived, left, changed = _run(upload_bin, "copy")
    assert info != 0 and not arrived
    assert (left, changed) == (0, 0)
