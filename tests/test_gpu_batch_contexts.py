"""A batch made on one context and generated on another of the same device: its
tables are on the device when it has been made, whatever its maker's stream was
doing."""
import ctypes as C

import numpy as np
import pytest
import torch

import arma_amd
from arma_amd import _abi

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def made(ctx, shape, seed):
    phi = np.random.default_rng(seed).standard_normal((3, 3, 2)) * 0.05
    phi[0, 0, 0] = 0.0
    n = -(-shape[0] // 16)
    return ctx.ar_desc(shape, phi, 0.5, _abi.dcmt_p521_params(n),
                       seeds=np.arange(n, dtype=np.uint32) + seed,
                       noise_mode=arma_amd.NOISE_PARTITIONED, partition=(16,) + shape[1:],
                       algorithm=arma_amd.AR_WAVEFRONT, precision=arma_amd.FP32)


def test_batch_of_a_busy_context():
    maker = arma_amd.Context(0, torch_stream=False)
    user = arma_amd.Context(0, torch_stream=False)
    shapes = [(40, 33, 50), (17, 64, 20)]
    descs = [made(maker, s, 3 + i) for i, s in enumerate(shapes)]
    alone = []
    for d, s in zip(descs, shapes):
        z = torch.empty(s, dtype=torch.float32, device=DEV)
        maker.ar_generate(d, z)
        maker.rescale(z, s, arma_amd.FP32, 1.0)
        alone.append(z)
    big = torch.empty((512, 256, 256), dtype=torch.float32, device=DEV)
    work = made(maker, tuple(big.shape), 9)
    arena = torch.full((1 << 18,), float("nan"), dtype=torch.float32, device=DEV)
    torch.cuda.synchronize()
    for _ in range(20):
        maker.ar_generate(work, big)
    batch = maker.batch(descs, [1.0] * len(shapes), arma_amd.FP32)
    assert batch.arena_elements <= arena.numel()
    stream = torch.cuda.ExternalStream(_abi.lib().arma_hip_get_stream(maker.h), device=DEV)
    assert stream.query()
    _abi.check(_abi.lib().arma_hip_batch_generate(user.h, batch.h, C.c_void_p(arena.data_ptr())))
    user.synchronize()
    for i, z in enumerate(alone):
        assert torch.equal(batch.surface(arena, i), z)
    batch.close()
    user.close()
    maker.close()
