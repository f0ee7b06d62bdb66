"""The wavefront tile's forms: one or two groups of lanes, resident coefficients
of P0 x P0 x 2 and P0 x P0 x P0 orders, streamed ones of any other, one or two
workgroups per CU, and the order in which tiles start.

Bars, from the existing tests of the recurrence: 1e-12 of the largest value in
FP64 (sums of at most 1000 terms), 1e-6 rms and 2e-5 in FP32 (compensated sums
of at most 100-term FP32 partials).  Batch members equal their single surfaces
bit for bit.
"""
import numpy as np
import pytest
import torch

import arma_amd
import pyoracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

# orders in time 1 .. 10, of the known shapes and of others
ORDERS = ([(p, p, 2) for p in range(1, 11)] + [(p, p, p) for p in range(1, 11)] +
          [(1, 3, 4), (2, 10, 10), (4, 1, 6), (6, 3, 1), (9, 2, 7), (10, 4, 3)])
# one ragged tile; no step on which all lanes are in the grid; several tiles
# along both axes, more along y, with steady steps
SHAPES = [(5, 3, 9), (33, 20, 40), (70, 33, 81)]


def phi_of(pshape, seed):
    rng = np.random.default_rng(seed)
    phi = rng.standard_normal(pshape) * (0.3 / np.prod(pshape) ** 0.5)
    phi[0, 0, 0] = 0.0
    return phi


def desc(ctx, shape, phi, prec):
    return ctx.ar_desc(shape, phi, 1.0, [arma_amd.mt19937_params()],
                       algorithm=arma_amd.AR_WAVEFRONT, precision=prec)


@pytest.mark.parametrize("pshape", ORDERS)
def test_forms_match_oracle(hip_ctx, pshape):
    phi = phi_of(pshape, 3)
    for shape in SHAPES:
        eps = np.random.default_rng(4).standard_normal(shape)
        ref = O.ar_generate(eps, phi)
        z = torch.from_numpy(eps.copy()).to(DEV)
        hip_ctx.ar_recurrence(desc(hip_ctx, shape, phi, arma_amd.FP64), z)
        err = np.max(np.abs(z.cpu().numpy() - ref)) / max(1.0, np.max(np.abs(ref)))
        assert err <= 1e-12, (shape, err)
        e32 = eps.astype(np.float32)
        ref = O.ar_generate(e32.astype(np.float64), phi)
        z = torch.from_numpy(e32).to(DEV)
        hip_ctx.ar_recurrence(desc(hip_ctx, shape, phi, arma_amd.FP32), z)
        d = z.cpu().numpy().astype(np.float64) - ref
        rms = np.sqrt(np.mean(d ** 2)) / np.sqrt(np.mean(ref ** 2))
        mx = np.max(np.abs(d)) / np.max(np.abs(ref))
        assert rms <= 1e-6 and mx <= 2e-5, (shape, rms, mx)


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
@pytest.mark.parametrize("pshapes", [
    [(5, 5, 2), (3, 3, 3), (4, 2, 3), (2, 2, 2), (1, 3, 3)],          # two workgroups per CU
    [(9, 9, 9), (7, 7, 2), (10, 10, 2), (8, 8, 8), (6, 4, 9), (3, 3, 2)],  # one
])
def test_batched_forms_equal_singles(hip_ctx, pshapes, prec):
    p = arma_amd.FP32 if prec == "fp32" else arma_amd.FP64
    dt = torch.float32 if prec == "fp32" else torch.float64
    params = arma_amd._abi.dcmt_p521_params(1)
    descs, singles = [], []
    for i, ps in enumerate(pshapes):
        shape = (40 + 9 * i, 20 + 13 * i, 70 - 7 * i)
        d = hip_ctx.ar_desc(shape, phi_of(ps, 10 + i), 1.0, params, seeds=np.array([7 + i], np.uint32),
                            noise_mode=arma_amd.NOISE_PARTITIONED, partition=shape,
                            algorithm=arma_amd.AR_WAVEFRONT, precision=p)
        descs.append(d)
        z = torch.empty(shape, dtype=dt, device=DEV)
        hip_ctx.ar_generate(d, z)
        hip_ctx.rescale(z, shape, p, 1.0)
        singles.append(z)
    batch = hip_ctx.batch(descs, [1.0] * len(descs), p)
    arena = torch.empty(batch.arena_elements, dtype=dt, device=DEV)
    for cfg in [(16, arma_amd.BATCH_SURFACE_MAJOR, 0), (16, arma_amd.BATCH_INTERLEAVED, 0)]:
        batch.set_config(cfg)
        arena.fill_(float("nan"))
        torch.cuda.synchronize()
        batch.generate(arena)
        hip_ctx.synchronize()
        for i, z in enumerate(singles):
            assert torch.equal(batch.surface(arena, i), z), (cfg, pshapes[i])
    batch.close()


@pytest.mark.parametrize("pshape", [(1, 1, 1), (1, 3, 3), (3, 1, 3), (3, 3, 1), (5, 5, 2), (4, 4, 4)])
def test_infinite_noise_spreads_as_in_the_sum(hip_ctx, pshape):
    """One infinite value makes non-finite what depends on it and nothing else."""
    shape = (40, 21, 37)
    eps = np.random.default_rng(8).standard_normal(shape)
    eps[9, 5, 18] = np.inf
    phi = phi_of(pshape, 6)
    with np.errstate(invalid="ignore"):
        ref = O.ar_generate(eps, phi)
    z = torch.from_numpy(eps.copy()).to(DEV)
    hip_ctx.ar_recurrence(desc(hip_ctx, shape, phi, arma_amd.FP64), z)
    assert np.array_equal(np.isfinite(z.cpu().numpy()), np.isfinite(ref))
