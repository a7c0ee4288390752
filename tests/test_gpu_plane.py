"""Several D2Q9 steps per launch (m3lb_amd/csrc/plane.hpp) against one launch
per step (M3LB_FUSION_OFF), through the C-ABI.

A pass runs every node's update on the same inputs with the same arithmetic,
so the whole slot image, halo and Solid slots included, is bit-identical after
any number of steps of either parity.  Sizes lie around the regions' edges:
boxes smaller than a margin, of one region, of several, and large enough for
each region and step count the library chooses.
"""
import sys

import numpy as np
import pytest

from m3lb_amd import abi, cases
from m3lb_amd.solver import FluidSolver

pytestmark = pytest.mark.gpu

OPS = [abi.OP_BGK, abi.OP_BGK_PRODUCT, abi.OP_TRT, abi.OP_TRT_PRODUCT, abi.OP_MRT, abi.OP_CM]
CHUNKS = [1, 9, 2, 30, 3, 8]


@pytest.fixture(autouse=True)
def announce(request):
    print(f"\n[gpu-case] {request.node.name}", flush=True)
    sys.stdout.flush()
    yield


def images(cfg, setup, chunks=CHUNKS, passes=True):
    out = []
    for fusion in (abi.FUSION_OFF, abi.FUSION_AUTO):
        with FluidSolver(cfg) as s:
            s.set_step_fusion(fusion)
            base = s.device_bytes()
            setup(s)
            img = []
            for n in chunks:
                s.step(n)
                img.append(s.storage())
            # a second population array is held once passes have run
            assert (s.device_bytes() > 1.5 * base) == (passes and fusion == abi.FUSION_AUTO)
            s.step(3, store_macroscopic=True)
            img.append(np.stack(s.macroscopic_stored()))
            img.append(np.stack(s.compute_macroscopic()))
            out.append(img)
    for a, b in zip(*out):
        assert np.isfinite(a).all()
        assert np.array_equal(a, b)


def noise(cfg, seed=1):
    r = np.random.default_rng(seed)
    n = abi.domain_of(cfg)[9]
    return [1.0 + 0.01 * r.uniform(-1, 1, n)] + [0.03 * r.uniform(-1, 1, n) for _ in range(2)] + [
        np.zeros(n)]


def blocks(shape):
    """Interior flags: a Solid disc and an Excluded corner patch."""
    nx, ny, _ = shape
    y, x = np.meshgrid(np.arange(ny), np.arange(nx), indexing="ij")
    fl = np.zeros((1, ny, nx), dtype=np.uint8)
    fl[0][(x - nx // 3) ** 2 + (y - ny // 2) ** 2 <= max(1, ny // 6) ** 2] = abi.SOLID
    fl[0][-2:, -2:] = abi.EXCLUDED
    return fl


@pytest.mark.parametrize("op", OPS)
@pytest.mark.parametrize("dtype,storage", [(abi.F64, abi.SHIFTED), (abi.F32, abi.SHIFTED),
                                           (abi.F32, abi.RAW)])
@pytest.mark.parametrize("geometry", [False, True])
def test_plane_is_bit_identical_every_operator(op, dtype, storage, geometry):
    shape = (43, 37, 1)
    cfg = abi.make_config(abi.D2Q9, op, storage, dtype, shape,
                          periodic=(True, not geometry, True), omega=1.3, omega_minus=1.1,
                          omega_bulk=1.1 if op in (abi.OP_MRT, abi.OP_CM) else -1.0,
                          force=(2e-5, -1e-5, 0.0))

    def setup(s):
        if geometry:
            s.set_geometry(blocks(shape))
        s.initialize_field(*noise(cfg))
    images(cfg, setup)


@pytest.mark.parametrize("dtype", [abi.F16, abi.BF16, abi.I16, abi.E2M13])
def test_plane_is_bit_identical_16bit(dtype):
    for shape in ((50, 21, 1), (420, 300, 1)):
        cfg = abi.make_config(abi.D2Q9, abi.OP_CM, abi.SHIFTED, dtype, shape, omega=1.6)
        images(cfg, lambda s: s.initialize_field(*noise(cfg)), chunks=[1, 13, 4])


@pytest.mark.parametrize("shape", [(1, 1), (1, 7), (5, 3), (16, 16), (17, 33), (8, 18), (130, 77),
                                   (33, 300), (261, 250), (401, 323)])
@pytest.mark.parametrize("periodic", [(1, 1), (1, 0), (0, 1), (0, 0)])
@pytest.mark.parametrize("dtype", [abi.F64, abi.F32])
def test_plane_sizes_and_halos(shape, periodic, dtype):
    shape = (*shape, 1)
    cfg = abi.make_config(abi.D2Q9, abi.OP_CM, abi.SHIFTED, dtype, shape,
                          periodic=(*periodic, True), omega=1.2)
    # an axis of one node that does not wrap has no halo: one launch per step
    plain = any(n == 1 and not p for n, p in zip(shape, periodic))
    if plain:
        pytest.skip("an axis of one node without wrap or halo")
    images(cfg, lambda s: s.initialize_field(*noise(cfg)), chunks=[1, 9, 22])


def test_plane_after_a_change_of_state():
    """New flags, a new seeding, new scales and a loaded checkpoint between
    passes: the slots no node moves are those of one launch per step."""
    shape = (60, 45, 1)
    cfg = abi.make_config(abi.D2Q9, abi.OP_MRT, abi.SHIFTED, abi.I16, shape,
                          periodic=(True, False, True), omega=1.4)
    out = []
    for fusion in (abi.FUSION_OFF, abi.FUSION_AUTO):
        with FluidSolver(cfg) as s:
            s.set_step_fusion(fusion)
            s.initialize_field(*noise(cfg, 2))
            s.step(12)
            s.set_geometry(blocks(shape))
            s.step(10)
            img = [s.storage()]
            s.calibrate_scales()
            s.step(7)
            pops = s.gather_populations()
            s.seed_populations(pops)
            s.step(8)
            img.append(s.storage())
            s.initialize(1.0, 0.02, 0.01)
            s.step(8)
            img.append(s.storage())
            s.set_geometry(np.zeros(60 * 45, dtype=np.uint8))
            s.step(9)
            img.append(s.storage())
            out.append(img)
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("op", OPS)
@pytest.mark.parametrize("dtype", [abi.F64, abi.F32])
@pytest.mark.parametrize("n", [7, 33])
def test_plane_cavity_walls(op, dtype, n):
    cfg = abi.make_config(abi.D2Q9, op, abi.SHIFTED, dtype, (n, n, 1), periodic=(0, 0, 1),
                          omega=1.7, omega_minus=1.2)

    def setup(s):
        s.set_regularized_walls(*cases.cavity_walls(n, 0.05))
        s.initialize(1.0)
    images(cfg, setup)


@pytest.mark.parametrize("n", [131, 210])
def test_plane_cavity_walls_many_blocks(n):
    cfg = abi.make_config(abi.D2Q9, abi.OP_CM, abi.SHIFTED, abi.F64, (n, n, 1), periodic=(0, 0, 1),
                          omega=1.8)

    def setup(s):
        s.set_regularized_walls(*cases.cavity_walls(n, 0.05))
        s.initialize_field(*noise(cfg))
    images(cfg, setup, chunks=[1, 8, 40])


@pytest.mark.parametrize("variant", ["fd_off", "field", "force", "solid", "scale", "outlet"])
def test_plane_wall_variants(variant):
    """Corners without the finite-difference stress, per-node wall velocities,
    a forced channel with the Guo correction off, a Solid block beside the
    walls, a scaled table; an outlet keeps one launch per step."""
    shape = (40, 26, 1)
    nx, ny, _ = shape
    force = (1e-5, 2e-6, 0.0) if variant == "force" else None
    periodic = (variant == "force", False, True)
    cfg = abi.make_config(abi.D2Q9, abi.OP_CM, abi.SHIFTED, abi.F64, shape, periodic=periodic,
                          omega=1.6, force=force)

    def setup(s):
        if variant == "solid":
            fl = np.zeros((1, ny, nx), dtype=np.uint8)
            fl[0, 10:14, 0:9] = abi.SOLID
            s.set_geometry(fl)
        if variant == "force":
            walls = cases.channel_walls(shape, 0.02)
            s.set_regularized_walls(*walls)
            s.set_force_correction(False)
        else:
            nrm = np.zeros((ny, nx), dtype=np.uint8)
            tag = np.zeros((ny, nx), dtype=np.uint16)
            nrm[:, 0], nrm[:, -1], nrm[0, :], nrm[-1, :] = (cases.NRM_XM, cases.NRM_XP,
                                                           cases.NRM_YM, cases.NRM_YP)
            tag[-1, :] = 1
            for j in (0, -1):
                for i in (0, -1):
                    nrm[j, i], tag[j, i] = cases.NRM_CORNER, 0
            if variant == "outlet":
                nrm[1:-1, -1] = cases.NRM_OUT_XP
            if variant == "solid":
                nrm[10:14, 0] = 0
            s.set_regularized_walls(nrm, tag, np.array([[0, 0, 0, 1.0], [0.04, 0.01, 0.02, 1.0]]))
            if variant == "fd_off":
                s.set_fd_corners(False)
            if variant == "scale":
                s.set_wall_velocity_scale(0.7)
            if variant == "field":
                r = np.random.default_rng(3)
                s.set_wall_velocity_field(*[0.01 * r.uniform(-1, 1, nx * ny) for _ in range(3)])
                s.set_wall_velocity_field_scale(1.3)
        s.initialize_field(*noise(cfg))
    images(cfg, setup, passes=variant != "outlet")


@pytest.mark.parametrize("n,walls", [(128, False), (129, False), (192, False), (193, False),
                                     (300, False), (385, False), (128, True), (129, True),
                                     (192, True), (193, True), (257, True)])
@pytest.mark.parametrize("dtype", [abi.F64, abi.F32])
def test_plane_at_the_steps_of_the_rule(n, walls, dtype):
    """Both sides of the sizes where the region or the steps per launch change."""
    shape = (n, n - 1, 1)
    cfg = abi.make_config(abi.D2Q9, abi.OP_CM, abi.SHIFTED, dtype, (n, n, 1) if walls else shape,
                          periodic=(not walls, not walls, True), omega=1.6)

    def setup(s):
        if walls:
            s.set_regularized_walls(*cases.cavity_walls(n, 0.05))
        s.initialize_field(*noise(cfg))
    images(cfg, setup, chunks=[1, 9, 22])


@pytest.mark.parametrize("chain", [False, True])
def test_plane_many_corners(chain):
    """More corners per region than one wave takes at once, and corners whose
    stencils follow one another along an axis (one launch per step)."""
    shape = (70, 36, 1)
    nx, ny, _ = shape
    cfg = abi.make_config(abi.D2Q9, abi.OP_CM, abi.SHIFTED, abi.F64, shape, periodic=(1, 0, 1),
                          omega=1.2)
    nrm = np.zeros((ny, nx), dtype=np.uint8)
    nrm[0], nrm[-1] = cases.NRM_YM, cases.NRM_YP
    if chain:
        nrm[8, 20:30] = cases.NRM_YM
        nrm[8, 20:30:3] = cases.NRM_CORNER
    else:
        nrm[4:-4:2, 3:-3:2] = cases.NRM_CORNER

    def setup(s):
        s.set_regularized_walls(nrm, np.zeros((ny, nx), dtype=np.uint16), np.zeros((1, 4)))
        s.set_fd_corners(False)
        s.initialize_field(*noise(cfg))
    images(cfg, setup, chunks=[1, 9, 2], passes=not chain)
