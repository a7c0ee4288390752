"""Readouts of several threads at once: the pinned staging slots are shared by every
handle, so calls wait for each other and small slots give way to large ones.  The
fields are those of the same calls one after the other."""
import threading

import numpy as np
import pytest

from m3lb_amd import abi
from m3lb_amd.solver import FluidSolver

pytestmark = pytest.mark.gpu


def test_readouts_of_several_threads():
    boxes = [(abi.F64, (70, 64, 50)), (abi.F32, (128, 128, 96)), (abi.F32, (16, 12, 8)),
             (abi.F64, (96, 80, 60)), (abi.F16, (64, 64, 64)), (abi.F32, (33, 21, 17))]
    print("\n[gpu-case] readouts of several threads", flush=True)
    solvers = []
    for k, (dtype, shape) in enumerate(boxes):
        cfg = abi.make_config(abi.D3Q27, abi.OP_CM, abi.SHIFTED, dtype, shape, omega=1.5)
        r = np.random.default_rng(k)
        n = abi.domain_of(cfg)[9]
        s = FluidSolver(cfg)
        s.initialize_field(1.0 + 0.01 * r.uniform(-1, 1, n),
                           *[0.03 * r.uniform(-1, 1, n) for _ in range(3)])
        s.step(3)
        solvers.append(s)

    def read(s):
        return [np.stack(s.compute_macroscopic()), s.gather_populations(), s.storage(),
                np.array([s.total_mass(), *s.energy_enstrophy()[:2]])]
    want = [read(s) for s in solvers]
    got = [[] for _ in solvers]
    errors = []

    def work(k):
        try:
            for _ in range(4):
                got[k].append(read(solvers[k]))
        except Exception as e:  # shown by the assertion below
            errors.append(e)
    threads = [threading.Thread(target=work, args=(k,)) for k in range(len(solvers))]
    for t in threads:
        t.start()
    for t in threads:
        t.join(100)
    assert not errors
    for k in range(len(solvers)):
        assert len(got[k]) == 4
        for r in got[k]:
            for a, b in zip(r, want[k]):
                assert np.array_equal(a, b)
    for s in solvers:
        s.close()
