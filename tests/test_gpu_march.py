"""Two D3Q27 steps per pass through LDS (m3lb_amd/csrc/march.hpp) against one
launch per step (M3LB_FUSION_OFF), through the C-ABI.

Every node runs the same update on the same inputs, so the whole slot image,
halo and Solid slots included, is bit-identical.  Sizes lie around the edges of
a block's core (64 x 13 nodes FP32, 32 x 12 FP64) and its runs of planes; the
test hook takes small boxes to the passes, the last case takes the rule's way.
"""
import numpy as np
import pytest

from m3lb_amd import abi
from m3lb_amd.solver import FluidSolver

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def announce(request):
    print(f"\n[gpu-case] {request.node.name}", flush=True)
    yield


def noise(cfg, seed=1):
    r = np.random.default_rng(seed)
    n = abi.domain_of(cfg)[9]
    return [1.0 + 0.01 * r.uniform(-1, 1, n)] + [0.03 * r.uniform(-1, 1, n) for _ in range(3)]


def blocks(shape):
    """A Solid ball and an Excluded corner patch."""
    nx, ny, nz = shape
    z, y, x = np.meshgrid(np.arange(nz), np.arange(ny), np.arange(nx), indexing="ij")
    fl = np.zeros((nz, ny, nx), dtype=np.uint8)
    fl[(x - nx // 3) ** 2 + (y - ny // 2) ** 2 + (z - nz // 2) ** 2
       <= max(1, min(shape) // 4) ** 2] = abi.SOLID
    fl[-2:, -2:, -2:] = abi.EXCLUDED
    return fl


def compare(cfg, setup, chunks=(1, 5, 2), passes=3, always=True):
    out = []
    for fusion in (abi.FUSION_OFF, abi.FUSION_AUTO):
        with FluidSolver(cfg) as s:
            s.set_step_fusion(fusion)
            s.test_march_always(always)
            setup(s)
            img = []
            for n in chunks:
                s.step(n)
                img.append(s.storage())
            assert s.fused_passes() == (passes if fusion == abi.FUSION_AUTO else 0)
            s.step(3, store_macroscopic=True)
            img.append(np.stack(s.macroscopic_stored()))
            out.append(img)
    for a, b in zip(*out):
        assert np.isfinite(a).all()
        assert np.array_equal(a, b)


@pytest.mark.parametrize("shape", [(1, 1, 1), (2, 3, 1), (5, 4, 3), (32, 12, 7), (64, 13, 20),
                                   (65, 14, 9), (33, 25, 30), (130, 27, 5)])
@pytest.mark.parametrize("periodic,geometry", [((1, 1, 1), False), ((1, 0, 1), True),
                                               ((0, 1, 1), False), ((1, 1, 0), True),
                                               ((0, 0, 0), False)])
@pytest.mark.parametrize("dtype", [abi.F32, abi.F64])
def test_march_sizes_halos_and_solids(shape, periodic, geometry, dtype):
    if any(n == 1 and not p for n, p in zip(shape, periodic)):
        pytest.skip("an axis of one node without wrap or halo")
    cfg = abi.make_config(abi.D3Q27, abi.OP_CM, abi.SHIFTED, dtype, shape, periodic=periodic,
                          omega=1.6, force=(1e-5, -2e-6, 3e-6) if geometry else None)

    def setup(s):
        if geometry:
            s.set_geometry(blocks(shape))
        s.initialize_field(*noise(cfg))
    compare(cfg, setup)


@pytest.mark.parametrize("op", [abi.OP_BGK, abi.OP_BGK_PRODUCT, abi.OP_TRT, abi.OP_TRT_PRODUCT,
                                abi.OP_MRT, abi.OP_CM])
@pytest.mark.parametrize("dtype,storage", [(abi.F64, abi.SHIFTED), (abi.F32, abi.SHIFTED),
                                           (abi.F64, abi.RAW), (abi.F32, abi.RAW)])
@pytest.mark.parametrize("force", [None, (2e-5, -1e-5, 1e-5)])
@pytest.mark.parametrize("pz", [0, 1])
def test_march_every_operator(op, dtype, storage, force, pz):
    """Operators without a march kernel take one launch per step."""
    shape = (67, 15, 11)
    cfg = abi.make_config(abi.D3Q27, op, storage, dtype, shape, periodic=(1, 1, pz), omega=1.3,
                          omega_minus=1.1, force=force)
    marches = op in (abi.OP_BGK_PRODUCT, abi.OP_MRT, abi.OP_CM)
    compare(cfg, lambda s: s.initialize_field(*noise(cfg)), passes=3 if marches else 0)


def test_march_after_a_change_of_state():
    """New flags, a new seeding and a loaded checkpoint between passes: the slots
    no node moves are those of one launch per step."""
    shape = (70, 20, 12)
    cfg = abi.make_config(abi.D3Q27, abi.OP_MRT, abi.SHIFTED, abi.F32, shape,
                          periodic=(1, 0, 1), omega=1.4)

    def run(s):
        s.initialize_field(*noise(cfg, 2))
        s.step(4)
        s.set_geometry(blocks(shape))
        s.step(5)
        img = [s.storage()]
        s.seed_populations(s.gather_populations())
        s.step(4)
        img.append(s.storage())
        s.initialize(1.0, 0.02, 0.01)
        s.step(4)
        img.append(s.storage())
        return img
    out = []
    for fusion in (abi.FUSION_OFF, abi.FUSION_AUTO):
        with FluidSolver(cfg) as s:
            s.set_step_fusion(fusion)
            s.test_march_always(True)
            out.append(run(s))
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("dtype,shape", [(abi.F32, (192, 182, 190)), (abi.F64, (160, 132, 140))])
def test_march_runs_by_default_beyond_the_cache(dtype, shape):
    cfg = abi.make_config(abi.D3Q27, abi.OP_CM, abi.SHIFTED, dtype, shape, omega=1.9)
    out = []
    for fusion in (abi.FUSION_OFF, abi.FUSION_AUTO):
        with FluidSolver(cfg) as s:
            s.set_step_fusion(fusion)
            s.initialize_taylor_green(0.04)
            base = s.device_bytes()
            s.step(5)
            assert s.fused_passes() == (2 if fusion == abi.FUSION_AUTO else 0)
            assert (s.device_bytes() > 1.5 * base) == (fusion == abi.FUSION_AUTO)
            out.append(np.stack(s.compute_macroscopic()))
    assert np.array_equal(*out)
