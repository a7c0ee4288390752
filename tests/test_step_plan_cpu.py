"""CPU check of the rules that choose a box's pass and its blocks
(m3lb_amd/csrc/step_plan.hpp) through a g++-built program
(tests/cpp/step_plan_test.cpp)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("step_plan") / "step_plan_test")
    src = os.path.join(ROOT, "tests", "cpp", "step_plan_test.cpp")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", src, "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("case", ["squares", "covers", "thin", "walls", "two_steps", "march", "runs",
                                  "long_boxes"])
def test_step_plan(program, case):
    r = subprocess.run([program, case], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.strip() == "ok"
