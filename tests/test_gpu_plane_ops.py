"""The D2Q9 passes of several steps (m3lb_amd/csrc/plane.hpp) against one launch
per step for every operator, storage type and region, forced and not: each is an
instantiation of its own, whose multiply-adds the compiler contracts by itself, so
bit identity is checked for each.  Walls in raw and in 16-bit storage too."""
import numpy as np
import pytest

from m3lb_amd import abi, cases
from test_gpu_plane import OPS, announce, blocks, images, noise  # noqa: F401

pytestmark = pytest.mark.gpu

# one box per region and step count of the rule: 24 x 24, 32 x 32, and beyond one
# round 64 x 32 (4-byte and 2-byte storage) or 32 x 32 with 4 steps (8-byte)
SHAPES = [(60, 57, 1), (256, 250, 1), (420, 400, 1)]
FORMS = [(abi.F64, abi.SHIFTED), (abi.F64, abi.RAW), (abi.F32, abi.SHIFTED), (abi.F32, abi.RAW),
         (abi.F16, abi.SHIFTED), (abi.BF16, abi.SHIFTED), (abi.I16, abi.SHIFTED),
         (abi.E2M13, abi.SHIFTED)]


def config(op, dtype, storage, shape, force, periodic=(True, True, True)):
    return abi.make_config(abi.D2Q9, op, storage, dtype, shape, periodic=periodic, omega=1.3,
                           omega_minus=1.1,
                           omega_bulk=1.1 if op in (abi.OP_MRT, abi.OP_CM) else -1.0, force=force)


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("op", OPS)
@pytest.mark.parametrize("dtype,storage", FORMS)
@pytest.mark.parametrize("force", [None, (2e-5, -1e-5, 0.0)])
def test_plane_every_operator_in_every_region(op, dtype, storage, shape, force):
    cfg = config(op, dtype, storage, shape, force)
    images(cfg, lambda s: s.initialize_field(*noise(cfg)), chunks=[1, 8, 2])


@pytest.mark.parametrize("op", OPS)
@pytest.mark.parametrize("dtype,storage", FORMS)
def test_plane_every_operator_with_solids(op, dtype, storage):
    shape = (90, 77, 1)
    cfg = config(op, dtype, storage, shape, None, periodic=(False, True, True))

    def setup(s):
        s.set_geometry(blocks(shape))
        s.initialize_field(*noise(cfg))
    images(cfg, setup, chunks=[1, 8, 2])


@pytest.mark.parametrize("dtype", [abi.F64, abi.F32])
@pytest.mark.parametrize("shape", SHAPES)
def test_plane_identity_collision(dtype, shape):
    cfg = abi.make_config(abi.D2Q9, abi.OP_NULL, abi.RAW, dtype, shape, omega=1.0)
    images(cfg, lambda s: s.initialize_field(*noise(cfg)), chunks=[1, 8, 2])


@pytest.mark.parametrize("op", OPS)
@pytest.mark.parametrize("dtype,storage", FORMS)
@pytest.mark.parametrize("n", [33, 140])
def test_plane_walls_every_storage(op, dtype, storage, n):
    cfg = config(op, dtype, storage, (n, n, 1), None, periodic=(False, False, True))

    def setup(s):
        s.set_regularized_walls(*cases.cavity_walls(n, 0.05))
        s.initialize_field(*noise(cfg))
    images(cfg, setup, chunks=[1, 8, 3])


@pytest.mark.parametrize("dtype,storage", FORMS)
def test_plane_forced_channel_walls(dtype, storage):
    """Straight walls without corners, a Guo force, several regions a side."""
    shape = (70, 41, 1)
    cfg = config(abi.OP_CM, dtype, storage, shape, (1e-5, 0.0, 0.0), periodic=(True, False, True))

    def setup(s):
        s.set_regularized_walls(*cases.channel_walls(shape, 0.02))
        s.initialize_field(*noise(cfg))
    images(cfg, setup, chunks=[1, 8, 3])
