"""The no-allocation entry point at the end of its range: one tile, order 10, whose
mailboxes leave a few kilobytes of 32 MiB for the tables."""
import numpy as np
import pytest
import torch

import arma_amd
from arma_amd import _abi

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def made(ctx, nt):
    shape = (nt, 16, 16)
    phi = np.random.default_rng(5).standard_normal((10, 10, 10)) * 0.005
    phi[0, 0, 0] = 0.0
    return shape, ctx.ar_desc(shape, phi, 1.0, _abi.dcmt_p521_params(1),
                              seeds=np.array([4], np.uint32),
                              noise_mode=arma_amd.NOISE_PARTITIONED, partition=shape,
                              precision=arma_amd.FP64, algorithm=arma_amd.AR_WAVEFRONT)


def test_the_longest_tile(hip_ctx):
    # 207 boundary values of 8 bytes at each of nt + 48 steps
    nt = ((32 << 20) - 13000) // (207 * 8) - 48
    shape, d = made(hip_ctx, nt)
    want = torch.empty(shape, dtype=torch.float64, device=DEV)
    hip_ctx.ar_generate(d, want)
    got = torch.zeros(shape, dtype=torch.float64, device=DEV)
    hip_ctx.ar_generate_noalloc(d, got)
    torch.cuda.synchronize()
    assert torch.equal(got, want)
    shape, d = made(hip_ctx, nt + 30)
    with pytest.raises(ValueError, match="no-allocation entry point has"):
        hip_ctx.ar_generate_noalloc(d, torch.empty(shape, dtype=torch.float64, device=DEV))
