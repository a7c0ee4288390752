"""CPU test of the staged transfers (m3lb_amd/csrc/transfer.hip) with the runtime's
entry points stood in for (tests/cpp/transfer_test.cpp): what the host reads after a
wait is visible to it, slots of a failed call are not handed on while the device
may write them, calls of several threads share at most kSlots slots, and running
out of pinned memory is an error, not a hang."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    tmp = tmp_path_factory.mktemp("transfer")
    objs = []
    for name, src in (("transfer", "m3lb_amd/csrc/transfer.hip"),
                      ("test", "tests/cpp/transfer_test.cpp")):
        o = str(tmp / (name + ".o"))
        subprocess.run([HIPCC, "-x", "hip", "--offload-host-only", "--offload-arch=gfx950", "-O1", "-fPIC",
                        "-std=c++17", "-I", os.path.join(ROOT, "include"), "-c",
                        os.path.join(ROOT, src), "-o", o], check=True)
        objs.append(o)
    exe = str(tmp / "transfer_test")
    subprocess.run(["g++", *objs, "-o", exe, "-lpthread"], check=True)
    return exe


@pytest.mark.parametrize("case", ["visible", "failed_wait", "threads", "no_memory"])
def test_staged_transfers(program, case):
    r = subprocess.run([program, case], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.strip() == "ok"
