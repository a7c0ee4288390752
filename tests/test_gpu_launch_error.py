"""A pass whose launch reports an error leaves the box as it was: the populations of
the time it still shows, which later calls step on from.  The error is one that the
runtime already holds, of an allocation of 2^60 bytes that it refused: the launch
itself is sound."""
import ctypes

import numpy as np
import pytest

from m3lb_amd import abi, cases, solver
from m3lb_amd.solver import FluidSolver

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def announce(request):
    print(f"\n[gpu-case] {request.node.name}", flush=True)
    yield


def refused_allocation():
    """Leaves an out-of-memory error as the runtime's last error of this thread."""
    hip = solver.load()  # its dependency libamdhip64 resolves hipMalloc
    p = ctypes.c_void_p()
    assert hip.hipMalloc(ctypes.byref(p), ctypes.c_size_t(1 << 60)) != 0


@pytest.mark.parametrize("kind", ["plane", "walls", "march"])
def test_a_reported_launch_error_leaves_the_state(kind):
    if kind == "march":
        cfg = abi.make_config(abi.D3Q27, abi.OP_CM, abi.SHIFTED, abi.F32, (70, 20, 12), omega=1.4)
    else:
        cfg = abi.make_config(abi.D2Q9, abi.OP_CM, abi.SHIFTED, abi.F64, (50, 50, 1), omega=1.4,
                              periodic=(kind == "plane",) * 2 + (True,))
    r = np.random.default_rng(5)
    n = abi.domain_of(cfg)[9]
    field = [1.0 + 0.01 * r.uniform(-1, 1, n)] + [0.03 * r.uniform(-1, 1, n) for _ in range(3)]

    def start(s):
        if kind == "walls":
            s.set_regularized_walls(*cases.cavity_walls(50, 0.05))
        s.test_march_always(True)
        s.initialize_field(*field)
        s.step(2)
        return s
    with FluidSolver(cfg) as s:
        start(s).step(4)
        want = s.storage()
    with FluidSolver(cfg) as s:
        start(s)
        before = s.storage()
        refused_allocation()
        with pytest.raises(RuntimeError, match="kernel launch"):
            s.step(4)
        assert s.timestep() == 2
        assert np.array_equal(s.storage(), before)
        s.step(4)
        assert s.timestep() == 6
        assert np.array_equal(s.storage(), want)
