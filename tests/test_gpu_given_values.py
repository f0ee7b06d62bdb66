"""Given leading slices may hold any bits, those of the pattern among them that stands
for a value that a neighbouring tile has not stored yet: the launch takes them as the
NaNs that they are, leaves them as they were, and ends."""
import numpy as np
import pytest
import torch

import arma_amd
from arma_amd import _abi

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
SHAPE, GIVEN = (30, 40, 37), 4


@pytest.mark.parametrize("prec,word,pattern", [
    (arma_amd.FP64, np.uint64, 0x7ff4a5a5a5a5a5a5),
    (arma_amd.FP64, np.uint64, 0x7ff4a5a500000001),
    (arma_amd.FP32, np.uint32, 0x7fa5a5a5),
])
@pytest.mark.parametrize("tile_x", [8, 16, 32])
def test_given_bits(hip_ctx, prec, word, pattern, tile_x):
    dt = np.float64 if prec == arma_amd.FP64 else np.float32
    phi = np.random.default_rng(6).standard_normal((3, 3, 3)) * 0.05
    phi[0, 0, 0] = 0.0
    d = hip_ctx.ar_desc(SHAPE, phi, 1.0, _abi.dcmt_p521_params(1), seeds=np.array([2], np.uint32),
                        noise_mode=arma_amd.NOISE_PARTITIONED, partition=(26, 40, 37),
                        algorithm=arma_amd.AR_WAVEFRONT, precision=prec)
    batch = hip_ctx.batch([d], None, prec, history=[GIVEN],
                          config=(tile_x, arma_amd.BATCH_SURFACE_MAJOR, 0))
    given = np.random.default_rng(7).standard_normal((GIVEN,) + SHAPE[1:]).astype(dt)
    # the last rows and columns of tiles, which their neighbours read
    places = [(3, 15, 15), (2, 31, 20), (3, 7, 31), (1, 20, 7), (3, 39, 36)]
    out = []
    for bits in (pattern, np.array(np.nan, dt).view(word)):
        mine = given.copy()
        for p in places:
            mine.view(word)[p] = bits
        arena = torch.zeros(batch.arena_elements, dtype=torch.from_numpy(mine).dtype, device=DEV)
        z = batch.surface(arena, 0)
        z[:GIVEN] = torch.from_numpy(mine).to(DEV)
        torch.cuda.synchronize()
        batch.generate(arena)
        batch.factors()  # raises where the launch gave up
        got = z.cpu().numpy()
        np.testing.assert_array_equal(got[:GIVEN].view(word), mine.view(word))
        assert np.isnan(got[GIVEN:]).any() and not np.isnan(got[GIVEN:]).all()
        out.append(got[GIVEN:])
    np.testing.assert_array_equal(out[0], out[1])
    batch.close()
