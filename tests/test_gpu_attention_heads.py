"""Decode attention with head counts that fill a workgroup's 8 rows, leave some
of them empty, or need several chunks per KV head.

The plan takes up to 8 query heads of a KV head into one workgroup (4 where
even one step per wave leaves CUs idle) and rounds 3 up to 4 and 5, 6 and 7 up
to 8; more than 8 run in chunks whose last may be shorter. Slab counts that do
not divide the CUs take plans of their own. Every head's output
is compared with the oracle on the (dequantised) cache, max-abs <= 2e-3 as in
the other attention tests, a repeated call returns the same bits, and values
next to the output stay untouched.
"""
from __future__ import annotations

import math

import numpy as np
import pytest
import torch

from oracle import attention as oa
from oracle import kv_quant as kq
from tests.helpers import kv_with_outliers, randn

TOL = 2e-3


def _dev(a, dev):
    return torch.from_numpy(np.ascontiguousarray(a)).to(dev)


# (fmt, B, Hkv, heads per KV head, L, live, group)
CASES = [
    ("fp16", 4, 8, 8, 2300, 2050, 0),    # one chunk of 8, 8 waves, a 2-token last tile
    ("fp16", 32, 8, 8, 333, -1, 0),      # 8 heads, no split, 4 waves
    ("fp16", 4, 8, 7, 2048, -1, 0),      # 7 of 8 rows
    ("fp16", 9, 8, 5, 1100, 1099, 0),
    ("fp16", 2, 4, 6, 700, 1, 0),        # one token; two chunks of 3
    ("fp16", 1, 4, 7, 300, -1, 0),       # chunks of 4 and 3
    ("fp16", 3, 8, 3, 2000, -1, 0),      # 3 of 4 rows
    ("fp16", 16, 4, 9, 1500, -1, 0),     # chunks of 5 and 4
    ("fp16", 16, 4, 16, 1030, -1, 0),    # two chunks of 8
    ("fp16", 8, 2, 17, 2000, 1999, 0),   # chunks of 6, 6 and 5
    ("int8", 8, 8, 8, 1500, 1487, 0),
    ("int8", 8, 8, 7, 1500, -1, 0),
    ("int8", 3, 8, 3, 500, -1, 0),
    ("int8", 40, 8, 5, 130, 129, 0),
    ("int4", 8, 8, 8, 1500, 1487, 128),
    ("int4", 8, 8, 6, 1500, -1, 32),
    ("int4", 12, 4, 12, 900, 899, 64),   # two chunks of 6
    ("int4", 2, 8, 3, 400, -1, 32),
    # slab counts that do not divide 256 CUs
    ("fp16", 12, 8, 4, 1111, 1100, 0),   # 2 splits of 8 waves instead of 3
    ("fp16", 17, 8, 4, 1281, -1, 0),     # 136 slabs: 3 splits of 4 waves
    ("fp16", 17, 8, 4, 1279, 1279, 0),   # unsplit
    ("fp16", 26, 8, 2, 700, 699, 0),     # 208 slabs, unsplit, 4 waves
    ("fp16", 34, 8, 1, 515, 513, 0),     # 272 slabs in 3 splits
    ("int8", 21, 8, 4, 1300, -1, 0),     # 168 slabs: 3 x 4 waves
    ("int8", 32, 8, 1, 700, 697, 0),     # 256 slabs: 8 waves
    ("int4", 21, 8, 4, 1300, 1299, 32),
    ("int4", 24, 8, 4, 600, -1, 128),    # 192 slabs: 8 waves
    ("int4", 33, 8, 1, 4100, 4097, 128),   # 264 slabs in 3 splits
    ("int4", 32, 8, 1, 2561, -1, 64),    # 256 slabs: 8 waves
    # short walks, unsplit
    ("fp16", 2, 8, 4, 300, 129, 0),
    ("fp16", 3, 8, 4, 224, -1, 0),
    ("fp16", 3, 8, 4, 225, -1, 0),       # the first that is split
    ("int8", 2, 8, 4, 384, 383, 0),
    ("int8", 2, 8, 4, 385, -1, 0),
    ("int4", 2, 8, 4, 256, 253, 32),
    ("int4", 2, 8, 4, 257, -1, 32),
    ("int4", 7, 8, 4, 384, 381, 64),
    ("int4", 4, 8, 8, 500, -1, 48),      # VALU kernel: chunks of 4
    ("int4", 4, 4, 7, 500, 499, 16),     # VALU kernel: one head per workgroup
]


@pytest.mark.gpu
@pytest.mark.parametrize("fmt,B,Hkv,gqa,L,live,gs", CASES,
                         ids=[f"{c[0]}-B{c[1]}-Hkv{c[2]}-x{c[3]}-L{c[4]}-live{c[5]}-g{c[6]}" for c in CASES])
def test_head_chunks_match_oracle(llmik, cuda, fmt, B, Hkv, gqa, L, live, gs):
    H = Hkv * gqa
    seed = 31 * B + L + gqa
    q = randn((B, H, 128), seed).astype(np.float16)
    k = (randn((B, Hkv, L, 128), seed + 1) if fmt == "fp16"
         else kv_with_outliers((B, Hkv, L, 128), seed + 1)).astype(np.float16)
    v = randn((B, Hkv, L, 128), seed + 2).astype(np.float16)
    scale = 1.0 / math.sqrt(128)
    qd = _dev(q, cuda)
    if fmt == "fp16":
        args = (llmik.decode_attention, (qd, _dev(k, cuda), _dev(v, cuda), scale, live))
        k_ref, v_ref = k, v
    elif fmt == "int8":
        kq_, ks = llmik.quantize_per_token(_dev(k, cuda))
        vq_, vs = llmik.quantize_per_token(_dev(v, cuda))
        args = (llmik.decode_attention_int8, (qd, kq_, ks, vq_, vs, scale, live))
        k_ref = kq.dequantize_per_token(kq_.cpu().numpy(), ks.cpu().numpy())
        v_ref = kq.dequantize_per_token(vq_.cpu().numpy(), vs.cpu().numpy())
    else:
        kq_, ks = llmik.quantize_k_per_channel_groupwise_int4(_dev(k, cuda), gs)
        vq_, vs = llmik.quantize_v_per_token_int4(_dev(v, cuda))
        args = (llmik.decode_attention_int4, (qd, kq_, ks, vq_, vs, gs, scale, live))
        k_ref = kq.dequantize_per_channel_groupwise(kq.unpack_kv_int4(kq_.cpu().numpy()), ks.cpu().numpy(), gs)
        v_ref = kq.dequantize_per_token(kq.unpack_kv_int4(vq_.cpu().numpy()), vs.cpu().numpy())
    out = args[0](*args[1])
    rows = sorted({0, B // 2, B - 1})
    ref = np.concatenate([oa.decode_attention(q[b:b + 1], k_ref[b:b + 1], v_ref[b:b + 1], scale,
                                              seqlen=None if live < 0 else live) for b in rows])
    assert float(np.abs(out[rows].float().cpu().numpy() - ref).max()) <= TOL
    assert torch.equal(args[0](*args[1]), out)


@pytest.mark.gpu
@pytest.mark.parametrize("form", [0, 1])
@pytest.mark.parametrize("gqa", [3, 7, 8])
def test_both_fp16_tile_forms(llmik, cuda, gqa, form):
    from llmik_cuda._lib import lib
    B, Hkv, S = 5, 8, 1543
    q = randn((B, Hkv * gqa, 128), 5).astype(np.float16)
    k = randn((B, Hkv, S, 128), 6).astype(np.float16)
    v = randn((B, Hkv, S, 128), 7).astype(np.float16)
    scale = 1.0 / math.sqrt(128)
    # The output is written into a slice of a larger buffer through the C entry point.
    guard = torch.full((B * Hkv * gqa * 128 + 256,), 7.0, dtype=torch.float16, device=cuda)
    out = guard[128:-128]
    need = lib.llmik_attention_workspace_size(B, Hkv * gqa, Hkv, S, 128)
    ws = torch.zeros(need, dtype=torch.uint8, device=cuda)
    qd, kd, vd = _dev(q, cuda), _dev(k, cuda), _dev(v, cuda)
    lib.llmik_attention_set_plan_override(form)
    try:
        rc = lib.llmik_decode_attention_f16(qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), out.data_ptr(), B,
                                            Hkv * gqa, Hkv, S, 128, S, scale, ws.data_ptr(), need,
                                            torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
    finally:
        lib.llmik_attention_set_plan_override(-1)
    assert rc == 0
    ref = oa.decode_attention(q, k, v, scale)
    got = out.view(B, Hkv * gqa, 128).float().cpu().numpy()
    assert float(np.abs(got - ref).max()) <= TOL
    assert float(guard[:128].min()) == float(guard[-128:].max()) == 7.0
    assert int(ws[:16384].count_nonzero()) == 0   # counters left zeroed


def test_workspace_fits_the_static_scratch():
    """Every plan's workspace fits the 2 MiB of the entry point that takes
    none, as it did with at most 4 heads per workgroup."""
    from llmik_cuda._lib import lib
    for gqa in (1, 2, 3, 4, 5, 7, 8, 12, 16):
        for slabs in (1, 3, 8, 16, 31, 32, 33, 63, 64, 65, 100, 127, 128, 129, 200, 255, 256, 300):
            for S in (1, 31, 256, 511, 1024, 2047, 4096, 33000, 131072):
                assert lib.llmik_attention_workspace_size(slabs, gqa, 1, S, 128) <= 2 << 20
