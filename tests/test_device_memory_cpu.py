"""CPU test of the device allocations (m3lb_amd/csrc/device_memory.hip) with the
runtime's entry points stood in for (tests/cpp/device_memory_test.cpp): an
allocation that finds no memory takes the handles' spare arrays of that device, and
only then; the current device stays as it was."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def test_device_memory(tmp_path):
    objs = []
    for name, src in (("unit", "m3lb_amd/csrc/device_memory.hip"),
                      ("test", "tests/cpp/device_memory_test.cpp")):
        o = str(tmp_path / (name + ".o"))
        subprocess.run([HIPCC, "-x", "hip", "--offload-host-only", "--offload-arch=gfx950", "-O1",
                        "-fPIC", "-std=c++17", "-c", os.path.join(ROOT, src), "-o", o], check=True)
        objs.append(o)
    exe = str(tmp_path / "device_memory_test")
    subprocess.run(["g++", *objs, "-o", exe, "-lpthread"], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.strip() == "ok"
