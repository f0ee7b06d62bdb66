"""White noise of long streams, generated by parts: every normal equals the
sequential generator's (the oracle's) within the bar of the other noise
tests, 4 ulp, at the sizes where a stream is cut into few and many pieces,
where pieces differ between ragged blocks, and where it is not cut at all."""
import math

import numpy as np
import pytest
import torch

import arma_amd
from arma_amd import _abi
import pyoracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def ulps(a, b):
    return float(np.max(np.abs(a - b) / np.spacing(np.maximum(np.abs(a), np.abs(b)))))


def blocks(shape, part):
    np_ = [-(-s // p) for s, p in zip(shape, part)]
    for a in range(np_[0]):
        for b in range(np_[1]):
            for c in range(np_[2]):
                lo = (a * part[0], b * part[1], c * part[2])
                yield tuple(slice(lo[d], min(lo[d] + part[d], shape[d])) for d in range(3))


def check(got, shape, part, params, seeds, varwn, sem):
    fp32 = sem == arma_amd.NOISE_FLOAT
    sd = np.float32(np.sqrt(np.float32(varwn))) if fp32 else math.sqrt(varwn)
    dt = np.float32 if fp32 else np.float64
    for p, where in enumerate(blocks(shape, part)):
        block = got[where]
        ref = O.noise_sequential(O.MtParams(*params[p].as_tuple()), int(seeds[p]), sd, block.size,
                                 dtype=dt).reshape(block.shape)
        assert ulps(block, ref) <= 4, (p, where)


@pytest.mark.parametrize("sem", [arma_amd.NOISE_DOUBLE, arma_amd.NOISE_FLOAT])
@pytest.mark.parametrize("shape,part", [
    ((1, 1, 2000), (1, 1, 2000)),        # one short stream, whole
    ((1, 1, 3001), (1, 1, 3001)),
    ((31, 33, 35), (31, 33, 35)),        # one stream in many pieces, odd rows
    ((64, 128, 128), (64, 128, 128)),    # the most pieces
    ((40, 50, 70), (32, 48, 48)),        # ragged blocks, some too short to cut
    ((64, 96, 97), (16, 32, 32)),
])
def test_long_streams(hip_ctx, shape, part, sem):
    n = sum(1 for _ in blocks(shape, part))
    params = _abi.dcmt_p521_params(n)
    seeds = np.arange(n, dtype=np.uint32) * 11 + 3
    prec = arma_amd.FP32 if sem == arma_amd.NOISE_FLOAT else arma_amd.FP64
    d = hip_ctx.ar_desc(shape, np.zeros((1, 1, 1)), 1.3, params, seeds=seeds,
                        noise_mode=arma_amd.NOISE_PARTITIONED, partition=part, precision=prec,
                        noise_semantics=sem)
    eps = torch.empty(shape, dtype=torch.float32 if prec == arma_amd.FP32 else torch.float64,
                      device=DEV)
    for _ in range(2):
        eps.fill_(float("nan"))
        hip_ctx.white_noise(d, eps)
    check(eps.cpu().numpy(), shape, part, params, seeds, 1.3, sem)


def test_long_streams_in_a_batch():
    """A batch's streams (two members of different block sizes) by parts, and
    again from a captured graph with other work between the replays."""
    ctx = arma_amd.Context(0, torch_stream=False)
    shapes, part = [(40, 50, 70), (33, 31, 90)], (32, 48, 48)
    descs, seeds, params = [], [], []
    for i, s in enumerate(shapes):
        n = sum(1 for _ in blocks(s, part))
        params.append(_abi.dcmt_p521_params(n))
        seeds.append(np.arange(n, dtype=np.uint32) + 100 * i)
        descs.append(ctx.ar_desc(s, np.zeros((1, 1, 1)), 0.7, params[i], seeds=seeds[i],
                                 noise_mode=arma_amd.NOISE_PARTITIONED, partition=part,
                                 precision=arma_amd.FP64, algorithm=arma_amd.AR_WAVEFRONT))
    batch = ctx.batch(descs, None, arma_amd.FP64)
    arena = torch.empty(batch.arena_elements, dtype=torch.float64, device=DEV)
    torch.cuda.synchronize()
    for run in ("generate", "capture", "replay", "replay"):
        if run == "capture":
            batch.capture(arena)
            continue
        arena.fill_(float("nan"))
        torch.cuda.synchronize()
        batch.generate(arena) if run == "generate" else batch.replay()
        ctx.synchronize()
        for i, s in enumerate(shapes):
            check(batch.surface(arena, i).cpu().numpy(), s, part, params[i], seeds[i], 0.7,
                  arma_amd.NOISE_DOUBLE)
    batch.close()
    ctx.close()


@pytest.mark.parametrize("sem", [arma_amd.NOISE_DOUBLE, arma_amd.NOISE_FLOAT])
@pytest.mark.parametrize("p", [0, 1279, 44497])
@pytest.mark.parametrize("shape,part", [
    ((1, 1, 8191), (1, 1, 8191)),
    ((1, 1, 8192), (1, 1, 8192)),
    ((33, 35, 31), (33, 35, 31)),
    ((20, 40, 61), (20, 24, 61)),
])
def test_large_states(hip_ctx, shape, part, p, sem):
    """MT19937 (p = 0 here) and the largest dynamic-creator states; several
    seeds, so that some streams need more words than were drawn ahead."""
    n = sum(1 for _ in blocks(shape, part))
    one = arma_amd.mt19937_params()
    if p:
        one.nn, one.mm = p // 32 + 1, (p // 32 + 1) // 2
        one.rr = one.nn * 32 - p
        one.umask = (0xFFFFFFFF << one.rr) & 0xFFFFFFFF
        one.lmask = ~one.umask & 0xFFFFFFFF
    params = [one] * n
    prec = arma_amd.FP32 if sem == arma_amd.NOISE_FLOAT else arma_amd.FP64
    eps = torch.empty(shape, dtype=torch.float32 if prec == arma_amd.FP32 else torch.float64,
                      device=DEV)
    for seed in range(3):
        seeds = np.arange(n, dtype=np.uint32) * 5 + 17 * seed
        d = hip_ctx.ar_desc(shape, np.zeros((1, 1, 1)), 0.8, params, seeds=seeds,
                            noise_mode=arma_amd.NOISE_PARTITIONED, partition=part,
                            precision=prec, noise_semantics=sem)
        eps.fill_(float("nan"))
        hip_ctx.white_noise(d, eps)
        check(eps.cpu().numpy(), shape, part, params, seeds, 0.8, sem)
