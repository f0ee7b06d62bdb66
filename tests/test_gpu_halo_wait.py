"""Checked launches report a halo value that does not arrive in time.

Consumers of a neighbouring tile's values wait for them.  A checked launch
(ARMA_HIP_CHECK_HALO=1) waits for a bounded time only, gives up and says so; the
limit is set below the time that the far end of a chain of tiles waits in earnest,
so that launches whose values all arrive give up too, run to their end and fail the
call.  The next call is as if nothing had been."""
import numpy as np
import pytest
import torch

import arma_amd

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
# tiles of 16 columns in one chain: the last waits for several milliseconds
CHAIN = (40, 8192, 16)


def run(ctx, shape, prec, seed=1):
    phi = np.random.default_rng(4).standard_normal((3, 3, 2)) * 0.05
    phi[0, 0, 0] = 0.0
    dt = torch.float32 if prec == arma_amd.FP32 else torch.float64
    z = torch.from_numpy(np.random.default_rng(seed).standard_normal(shape)).to(DEV).to(dt)
    ctx.ar_recurrence(ctx.ar_desc(shape, phi, 1.0, [arma_amd.mt19937_params()],
                                  algorithm=arma_amd.AR_WAVEFRONT, precision=prec), z)
    torch.cuda.synchronize()
    return z


@pytest.mark.parametrize("prec", [arma_amd.FP32, arma_amd.FP64])
def test_a_late_value_fails_the_call(hip_ctx, monkeypatch, prec):
    plain = run(hip_ctx, CHAIN, prec)
    monkeypatch.setenv("ARMA_HIP_CHECK_HALO", "1")
    assert torch.equal(run(hip_ctx, CHAIN, prec), plain)
    monkeypatch.setenv("ARMA_HIP_CHECK_HALO_POLLS", "16")
    with pytest.raises(arma_amd._abi.ArmaHipError):
        run(hip_ctx, CHAIN, prec)
    monkeypatch.delenv("ARMA_HIP_CHECK_HALO_POLLS")
    assert torch.equal(run(hip_ctx, CHAIN, prec), plain)
    monkeypatch.delenv("ARMA_HIP_CHECK_HALO")
    assert torch.equal(run(hip_ctx, CHAIN, prec), plain)


def test_checked_quad_tile(hip_ctx, monkeypatch):
    monkeypatch.setenv("ARMA_HIP_QUAD_TILE", "1")
    plain = run(hip_ctx, (40, 70, 90), arma_amd.FP32)
    monkeypatch.setenv("ARMA_HIP_CHECK_HALO", "1")
    assert torch.equal(run(hip_ctx, (40, 70, 90), arma_amd.FP32), plain)
