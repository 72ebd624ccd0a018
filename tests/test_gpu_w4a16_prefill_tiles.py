"""GPU parity: the 128 x 128-tile W4A16 GEMM of M > 128 (groups 32, 64, 128) at
the edges of its tiles, stages, groups and splits. Gate as in the other W4A16
tests: the fp32 output within 2e-3 of the float64 product, the fp16 output its
rounding bit for bit, a second call the same bits; values beside the output
stay untouched."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = 2e-3

# (M, K, N, group). 256 x 128 tiles over 85 (a third of 256 CUs) reach it.
CASES = [
    (256, 64, 11008, 64),      # one stage
    (256, 64, 11008, 32),
    (257, 128, 5632, 128),     # one group of two stages; last tile one row, its second half empty
    (384, 192, 5632, 64),      # three stages; the last tile half full
    (385, 320, 5632, 32),      # five stages
    (300, 384, 6400, 128),     # three groups of 128: two stages left after the unrolled four
    (511, 448, 5632, 64),      # seven stages
    (512, 640, 5632, 128),     # ten stages
    (256, 256, 11136, 128),    # 87 tiles: 2 K splits of two stages
    (260, 320, 11136, 64),     # 2 splits of 3 and 2 stages
    (300, 1152, 5760, 128),    # 90 tiles, 2 splits of 10 and 8 stages
    (770, 1024, 11008, 32),    # tiles past whole rounds split
    (1030, 512, 8192, 128),
    (129, 256, 11008, 128),    # from 129 rows: one row tile, 2 splits of two stages
    (255, 320, 11264, 64),
    (160, 1088, 11008, 32),    # 17 stages in 2 splits
    (300, 8192, 4096, 128),    # 64 tiles in 4 splits of 32 stages
    (500, 8256, 4096, 64),     # 129 stages: 33, 33, 33 and 30
    (900, 4096, 4224, 64),     # an odd number of column tiles
]


@pytest.mark.parametrize("M,K,N,gs", CASES, ids=["-".join(map(str, c)) for c in CASES])
def test_edges(llmik, cuda, M, K, N, gs):
    from llmik_cuda._lib import lib
    g = torch.Generator(device=cuda).manual_seed(M + K)
    w = torch.randint(-2 ** 31, 2 ** 31 - 1, (K // 8, N), generator=g, device=cuda, dtype=torch.int32)
    sc = (torch.rand((K // gs, N), generator=g, device=cuda) * 0.02 + 0.001).half()
    a = torch.randn((M, K), generator=g, device=cuda, dtype=torch.float16)
    shifts = torch.arange(0, 32, 4, device=cuda, dtype=torch.int32).view(1, 8, 1)
    codes = (w.unsqueeze(1) >> shifts) & 0xF
    codes = torch.where(codes >= 8, codes - 16, codes).reshape(K, N)
    ref = a.double() @ (codes.double() * sc.double().repeat_interleave(gs, dim=0))
    out32 = llmik.w4a16_gemm_f32out(a, w, sc, gs)
    assert float((out32.double() - ref).abs().max()) <= TOL
    out16 = llmik.w4a16_gemm(a, w, sc, gs)
    assert torch.equal(out16, out32.half())
    assert torch.equal(llmik.w4a16_gemm_f32out(a, w, sc, gs), out32)
    # an output 4 bytes off 16-byte alignment, between guard values
    need = lib.llmik_w4a16_workspace_size(M, N, K, gs)
    ws = torch.zeros(max(need, 1), dtype=torch.uint8, device=cuda)
    pad = torch.full((M * N + 128,), 5.0, dtype=torch.float16, device=cuda)
    dst = pad[66:66 + M * N]
    rc = lib.llmik_w4a16_gemm(a.data_ptr(), w.data_ptr(), sc.data_ptr(), dst.data_ptr(), M, N, K, gs,
                              ws.data_ptr() if need else None, need, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert rc == 0 and torch.equal(dst.view(M, N), out16)
    assert bool((pad[:66] == 5).all()) and bool((pad[66 + M * N:] == 5).all())
    assert int(ws[:min(need, 16384)].count_nonzero()) == 0


def test_capture_and_replay_split(llmik, cuda):
    M, K, N, gs = 300, 1152, 5760, 128
    g = torch.Generator(device=cuda).manual_seed(1)
    w = torch.randint(-2 ** 31, 2 ** 31 - 1, (K // 8, N), generator=g, device=cuda, dtype=torch.int32)
    sc = (torch.rand((K // gs, N), generator=g, device=cuda) * 0.02 + 0.001).half()
    a = torch.randn((M, K), generator=g, device=cuda, dtype=torch.float16)
    eager = llmik.w4a16_gemm(a, w, sc, gs)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        llmik.w4a16_gemm(a, w, sc, gs)
    s.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        out = llmik.w4a16_gemm(a, w, sc, gs)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)
        assert torch.equal(llmik.w4a16_gemm(a, w, sc, gs), eager)
