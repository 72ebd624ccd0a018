"""GPU parity: the LDS-staged W4A16 GEMM, which serves scale groups of 256 and
more from 256 rows, unsplit, with every tile split, and with only the tiles
past whole rounds of the CUs split (in 2, 3 and 4). Gates and guard values as
for the smaller groups' kernel; the number of split partials, from the
workspace size, says that each case runs the split it names."""
from __future__ import annotations

import pytest
import torch

from tests import test_gpu_w4a16_prefill_tiles as tiles

pytestmark = pytest.mark.gpu

# (M, K, N, group, 256 x 128 tiles that are split x splits on 256 CUs)
CASES = [
    (513, 256, 6144, 256, 0),          # the last tile one row; one group
    (352, 1024, 11008, 512, 0),
    (300, 512, 6400, 256, 100 * 2),
    (300, 1024, 6400, 512, 100 * 2),   # splits of one group each
    (768, 4096, 4096, 1024, 96 * 2),
    (768, 1024, 14336, 256, 80 * 2),   # 256 tiles whole, 80 split
    (768, 1024, 14336, 512, 80 * 3),   # 6, 6 and 4 stages: inside groups of 8
    (3072, 1024, 14336, 256, 64 * 4),
]


@pytest.mark.parametrize("M,K,N,gs,partials", CASES, ids=["-".join(map(str, c[:4])) for c in CASES])
def test_lds_staged(llmik, cuda, M, K, N, gs, partials):
    from llmik_cuda._lib import lib
    need = lib.llmik_w4a16_workspace_size(M, N, K, gs)
    if torch.cuda.get_device_properties(cuda).multi_processor_count == 256:
        assert need == (16384 + partials * 256 * 128 * 4 if partials else 0)
    tiles.test_edges(llmik, cuda, M, K, N, gs)
