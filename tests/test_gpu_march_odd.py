"""Even numbers of steps from an odd one: the passes in place take them (either
parity), short of the counts where two single steps around the passes through LDS
cost less."""
import numpy as np
import pytest

from m3lb_amd import abi
from m3lb_amd.solver import FluidSolver

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def announce(request):
    print(f"\n[gpu-case] {request.node.name}", flush=True)
    yield


@pytest.mark.parametrize("dtype,shape,last", [(abi.F32, (192, 182, 190), 8),
                                              (abi.F64, (160, 132, 140), 8)])
@pytest.mark.parametrize("store", [False, True])
def test_even_counts_from_an_odd_step(dtype, shape, last, store):
    cfg = abi.make_config(abi.D3Q27, abi.OP_CM, abi.SHIFTED, dtype, shape, omega=1.7)
    out = []
    for fusion in (abi.FUSION_OFF, abi.FUSION_AUTO):
        with FluidSolver(cfg) as s:
            s.set_step_fusion(fusion)
            s.initialize_taylor_green(0.04)
            base = s.device_bytes()
            s.step(1)
            passes = []
            for n in (2, last, last + 2):
                before = s.fused_passes()
                s.step(n + (1 if store else 0), store_macroscopic=store)
                if store:
                    s.step(1)  # to an odd step again
                passes.append(s.fused_passes() - before)
                if n < last + 2:
                    assert s.device_bytes() < 1.5 * base  # no second array
            assert s.timestep() == 1 + 2 + last + last + 2 + (6 if store else 0)
            if fusion == abi.FUSION_AUTO:
                # the last count: one step, the passes, one step
                assert passes == [1, last // 2, last // 2]
            else:
                assert passes == [0, 0, 0]
            out.append(np.stack(s.compute_macroscopic()))
    assert np.array_equal(*out)
