"""CPU check of the passes' periodic coordinates (m3lb_amd/csrc/wrap.hpp): beside
axes of up to 2^31 nodes, where a product of the extent and the margin would not
fit an int (tests/cpp/wrap_test.cpp), and that the kernels use it."""
import os
import re
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_wrapped_coordinates(tmp_path):
    exe = tmp_path / "wrap_test"
    src = os.path.join(ROOT, "tests", "cpp", "wrap_test.cpp")
    subprocess.run(["g++", "-std=c++17", "-O1", "-ftrapv", "-Wall", "-Werror", src, "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.strip() == "ok"


def test_the_passes_wrap_without_products():
    for name in ("plane.hpp", "march.hpp"):
        with open(os.path.join(ROOT, "m3lb_amd", "csrc", name)) as fh:
            text = fh.read()
        assert "wrapped(X, d.sx)" in text
        assert not re.search(r"d\.s[xyz] \* H|2 \* d\.s[xyz]", text)
