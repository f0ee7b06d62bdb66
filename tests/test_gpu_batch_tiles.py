"""Batch tiles at the ends of their range: every order whose halo a tile's width
admits runs on it, and tuning times all of them.  Members equal the surfaces made
alone to the last bit."""
import numpy as np
import pytest
import torch

import arma_amd
from arma_amd import _abi

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def made(ctx, shape, pshape, prec):
    phi = np.random.default_rng(11).standard_normal(pshape) * (0.3 / np.prod(pshape) ** 0.5)
    phi[0, 0, 0] = 0.0
    return ctx.ar_desc(shape, phi, 1.0, _abi.dcmt_p521_params(1), seeds=np.array([5], np.uint32),
                       noise_mode=arma_amd.NOISE_PARTITIONED, partition=shape,
                       algorithm=arma_amd.AR_WAVEFRONT, precision=prec)


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
@pytest.mark.parametrize("tile_x,pshape", [
    (8, (3, 9, 10)), (8, (2, 9, 9)), (16, (3, 10, 10)), (32, (3, 10, 9)), (32, (1, 10, 1)),
])
def test_widest_orders(hip_ctx, tile_x, pshape, prec):
    p = arma_amd.FP32 if prec == "fp32" else arma_amd.FP64
    dt = torch.float32 if prec == "fp32" else torch.float64
    shapes = [(21, 37, 70), (30, 40, 33)]
    descs = [made(hip_ctx, s, pshape, p) for s in shapes]
    batch = hip_ctx.batch(descs, None, p)
    arena = torch.empty(batch.arena_elements, dtype=dt, device=DEV)
    batch.set_config((tile_x, arma_amd.BATCH_SURFACE_MAJOR, 0))
    batch.generate(arena)
    hip_ctx.synchronize()
    for i, s in enumerate(shapes):
        z = torch.empty(s, dtype=dt, device=DEV)
        hip_ctx.ar_generate(descs[i], z)
        assert torch.equal(batch.surface(arena, i), z)
    if tile_x == 8:
        widths = {t[0][0] for t in batch.tune(arena, reps=1)}
        # 10 columns of a row are wider than 8 + 1
        assert widths == ({8, 16} if pshape[2] == 10 else {8, 16, 32})
    batch.close()


def test_device_bytes_of_many_tiles(hip_ctx):
    """A batch holds its mailboxes and little else: no slots for stores that its
    kernels do not make."""
    shape, es = (1, 2048, 4096), 8
    tiles = shape[1] // 16 * (shape[2] // 16)
    # rows of 16 + 15 boundary values at 1 + 30 + 2 steps
    mailboxes = tiles * (shape[0] + 32) * 31 * es
    d = made(hip_ctx, shape, (2, 2, 2), arma_amd.FP64)
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    batch = hip_ctx.batch([d], None, arma_amd.FP64)
    used = before - torch.cuda.mem_get_info()[0]
    batch.close()
    # (what the runtime had kept of earlier buffers does not count as used)
    assert used <= mailboxes + (64 << 20)
