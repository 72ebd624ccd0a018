"""GPU: rope's 16-byte form gives the bits of its one-pair-per-thread form (the
same rope_pair), which serves tensors that are not 16-byte aligned and head
dimensions that are no multiple of 16."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


def _rope(lib, x, c, s, out):
    B, H, S, D = x.shape
    rc = lib.llmik_rope(x.data_ptr(), c.data_ptr(), s.data_ptr(), out.data_ptr(), B, H, S, D,
                        torch.cuda.current_stream().cuda_stream)
    assert rc == 0


@pytest.mark.parametrize("B,H,S,D", [
    (1, 1, 1, 16), (2, 3, 5, 32), (1, 5, 33, 48), (3, 2, 31, 64), (1, 7, 257, 128), (2, 32, 130, 128),
    (1, 9, 900, 128),     # odd head count at two heads per thread, plain accesses
    (1, 33, 1100, 128),   # the same with non-temporal accesses
    (4, 1, 40, 256),
])
def test_vector_form_equals_scalar_form(llmik, cuda, B, H, S, D):
    from llmik_cuda._lib import lib
    g = torch.Generator(device=cuda).manual_seed(S)
    new = lambda *sh: torch.randn(sh, generator=g, device=cuda, dtype=torch.float16)   # noqa: E731
    x, c, s = new(B, H, S, D), new(B, S, D), new(B, S, D)
    pad = torch.full((x.numel() + 32,), 3.0, dtype=torch.float16, device=cuda)
    out = pad[16:-16].view(x.shape)
    _rope(lib, x, c, s, out)
    off = torch.empty(x.numel() + 1, dtype=torch.float16, device=cuda)   # 2 bytes off alignment
    xo = off[1:].view(x.shape)
    xo.copy_(x)
    want = torch.empty_like(x)
    _rope(lib, xo, c, s, want)
    assert torch.equal(out.view(torch.int16), want.view(torch.int16))
    assert bool((pad[:16] == 3).all()) and bool((pad[-16:] == 3).all())
    h = D // 2
    x1, x2 = x.double()[..., :h], x.double()[..., h:]
    cd, sd = c.double()[:, None], s.double()[:, None]
    ref = torch.cat([x1 * cd[..., :h] - x2 * sd[..., :h], x2 * cd[..., h:] + x1 * sd[..., h:]], dim=-1)
    # one fp16 rounding of an fp32 fma of fp16 products
    assert float(((out.double() - ref).abs() - ref.abs() * 2.0 ** -11).max()) <= 2.0 ** -20 + 1e-6


@pytest.mark.parametrize("n", [1, 7, 8, 2049, 1_223_338, 1_300_003])
def test_silu_mul_around_the_streaming_size(llmik, cuda, n):
    """6 bytes a value: non-temporal accesses from 7 MiB, 1,223,339 values."""
    g = torch.Generator(device=cuda).manual_seed(n)
    a = torch.randn(n, generator=g, device=cuda, dtype=torch.float16)
    b = torch.randn(n, generator=g, device=cuda, dtype=torch.float16)
    ref = torch.nn.functional.silu(a.double()) * b.double()
    out = llmik.silu_mul(a, b)
    assert float(((out.double() - ref).abs() - ref.abs() * 2.0 ** -11).max()) <= 1e-6
