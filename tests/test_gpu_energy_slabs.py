"""m3lb_energy_enstrophy of boxes whose velocities do not fit its scratch (64 MB):
slabs of planes with the planes beside them, the wrap and a shorter last slab
included, against NumPy sums over compute_macroscopic().  The sums run over 3 to 6
million terms of like size in FP64 in another order: 1e-12 relative is about
ten times their rounding (2^-53 sqrt(n) to 2^-53 log2(n) blocks)."""
import numpy as np
import pytest

from m3lb_amd import abi
from m3lb_amd.solver import FluidSolver

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def announce(request):
    print(f"\n[gpu-case] {request.node.name}", flush=True)
    yield


def interior(cfg, a):
    nx, ny, nz, hx, hy, hz, sx, sy, sz, _ = abi.domain_of(cfg)
    return a.reshape(sz, sy, sx)[hz:hz + nz, hy:hy + ny, hx:hx + nx]


def reference(u, v, w):
    def d(a, axis):  # wraps at every face, as the reference's central differences do
        return 0.5 * (np.roll(a, -1, axis) - np.roll(a, 1, axis))
    e = 0.5 * (u * u + v * v + w * w)
    om = 0.5 * ((d(w, 1) - d(v, 0)) ** 2 + (d(u, 0) - d(w, 2)) ** 2 + (d(v, 2) - d(u, 1)) ** 2)
    return e, om


@pytest.mark.parametrize("dtype,shape", [(abi.F32, (200, 180, 163)), (abi.F64, (150, 140, 141)),
                                         (abi.F64, (1200, 800, 5))])
@pytest.mark.parametrize("periodic", [(1, 1, 1), (1, 1, 0), (0, 1, 0)])
def test_slabs_match_the_fields(dtype, shape, periodic):
    cfg = abi.make_config(abi.D3Q27, abi.OP_CM, abi.SHIFTED, dtype, shape, periodic=periodic,
                          omega=1.4)
    r = np.random.default_rng(3)
    n = abi.domain_of(cfg)[9]
    with FluidSolver(cfg) as s:
        s.initialize_field(1.0 + 0.01 * r.uniform(-1, 1, n),
                           *[0.03 * r.uniform(-1, 1, n) for _ in range(3)])
        s.step(2)
        e, om, finite = s.energy_enstrophy()
        _, u, v, w = [interior(cfg, a) for a in s.compute_macroscopic()]
    we, wom = [float(a.sum()) for a in reference(u, v, w)]
    assert finite
    assert abs(e - we) <= 1e-12 * we
    assert abs(om - wom) <= 1e-12 * wom


@pytest.mark.parametrize("plane", [0, 70, 140])
def test_slabs_report_a_node_that_is_not_finite(plane):
    shape = (150, 140, 141)
    cfg = abi.make_config(abi.D3Q27, abi.OP_CM, abi.SHIFTED, abi.F64, shape, omega=1.4)
    n = abi.domain_of(cfg)[9]
    f = [np.ones(n)] + [np.full(n, 0.01) for _ in range(3)]
    f[1][plane * 150 * 140 + 1234] = np.nan
    with FluidSolver(cfg) as s:
        s.initialize_field(*f)
        e, _, finite = s.energy_enstrophy()
        _, u, v, w = s.compute_macroscopic()
        assert not finite
        ok = np.isfinite(u) & np.isfinite(v) & np.isfinite(w)
        assert (~ok).sum() == 1
        want = float(0.5 * (u[ok] ** 2 + v[ok] ** 2 + w[ok] ** 2).sum())
        assert abs(e - want) <= 1e-12 * want
