"""Buffers that only make a call faster are done without when the device has no memory
left for them: what ran before they were there still runs, with the same bits."""
import numpy as np
import pytest
import torch

import arma_amd

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
N = 20_000_000  # normals of one MT19937 stream: 204 MB of words


def taken():
    """All device memory but pieces of less than 128 MB, the last of them left free."""
    free = torch.cuda.mem_get_info()[0]
    held = []
    for size in (free - (1 << 30), 512 << 20, 128 << 20):
        for _ in range(20):
            try:
                held.append(torch.empty(size, dtype=torch.uint8, device=DEV))
            except torch.cuda.OutOfMemoryError:
                break
    return held


def test_words_ahead_without_memory():
    desc = arma_amd.Context.ar_desc((1, 1, N), np.zeros((1, 1, 1)), 1.0,
                                    [arma_amd.mt19937_params()], seeds=np.array([3], np.uint32),
                                    noise_mode=arma_amd.NOISE_SEQUENTIAL,
                                    precision=arma_amd.FP32)
    want = torch.empty(N, dtype=torch.float32, device=DEV)
    with_room = arma_amd.Context(0)
    with_room.white_noise(desc, want)
    torch.cuda.synchronize()
    with_room.close()
    got = torch.zeros_like(want)
    ctx = arma_amd.Context(0)
    small = torch.empty(64, dtype=torch.float32, device=DEV)
    ctx.white_noise(arma_amd.Context.ar_desc((1, 1, 64), np.zeros((1, 1, 1)), 1.0,
                                             [arma_amd.mt19937_params()],
                                             seeds=np.array([1], np.uint32),
                                             noise_mode=arma_amd.NOISE_SEQUENTIAL,
                                             precision=arma_amd.FP32), small)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    held = taken()
    try:
        ctx.white_noise(desc, got)
        torch.cuda.synchronize()
    finally:
        del held
        torch.cuda.empty_cache()
    assert torch.equal(got, want)
    ctx.close()
