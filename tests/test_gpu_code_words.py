"""GPU: the KV writers' codes and scales, bit for bit against the oracle, on
values at and next to half-integer quotients (where the fast rounding hands
over to the true division), over maxima of every fp16 magnitude."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import kv_quant as kq

pytestmark = pytest.mark.gpu


def _rows(n, qmax, seed):
    """[n, 128] fp16: column 0 the row's maximum, the rest near half-integer
    multiples of the row's scale (exact ties, one step either side) or random."""
    rng = np.random.default_rng(seed)
    amax = rng.integers(1, 0x7C00, (n, 1)).astype(np.uint16).view(np.float16)
    s = np.maximum(amax.astype(np.float32) / np.float32(qmax), np.float32(1e-8)).astype(np.float64)
    half = ((rng.integers(-qmax, qmax, (n, 127)) + 0.5) * s).astype(np.float16)
    step = rng.integers(-1, 2, (n, 127))
    x = np.where(step == 0, half, np.nextafter(half, np.where(step > 0, np.inf, -np.inf).astype(np.float16)))
    pick = rng.random((n, 127))
    x = np.where(pick < 0.2, amax / np.float16(2), x)
    x = np.where(pick > 0.7, (rng.uniform(-1, 1, (n, 127)) * amax.astype(np.float64)).astype(np.float16), x)
    x = np.where(np.abs(x) <= amax, x, amax).astype(np.float16)
    return np.concatenate([amax, x], axis=1)


def _same(t, a):
    return np.array_equal(t.cpu().numpy().view(np.uint8), np.ascontiguousarray(a).view(np.uint8))


@pytest.mark.parametrize("n", [1, 31, 32, 33, 5000])
def test_per_token(llmik, cuda, n):
    for qmax, fn in ((127, llmik.quantize_per_token), (7, llmik.quantize_v_per_token_int4)):
        x = _rows(n, qmax, n)[None, None]
        q, s = fn(torch.from_numpy(x).to(cuda))
        rq, rs = kq.quantize_per_token(x.astype(np.float32), 8 if qmax == 127 else 4)
        assert _same(q, rq if qmax == 127 else kq.pack_kv_int4(rq))
        assert _same(s, rs.astype(np.float16))


@pytest.mark.parametrize("g,S", [(16, 128), (32, 128), (32, 70), (64, 128), (128, 128), (128, 100), (300, 700)])
def test_k_groupwise(llmik, cuda, g, S):
    # 128 channels of S tokens; every group's first token holds its maximum.
    rng = np.random.default_rng(g + S)
    x = np.concatenate([np.resize(_rows(128, 7, int(rng.integers(1 << 30)) + t).T, (min(g, S - t), 128))
                        for t in range(0, S, g)])[None, None]
    assert x.shape == (1, 1, S, 128)
    q, s = llmik.quantize_k_per_channel_groupwise_int4(torch.from_numpy(x).to(cuda), g)
    rq, rs = kq.quantize_per_channel_groupwise(x.astype(np.float32), 4, g)
    assert _same(q, kq.pack_kv_int4(rq))
    assert _same(s, rs.astype(np.float16))
