"""CPU: the plans of decode attention (csrc/attention_plan.cpp, compiled here with
the host compiler) over the shapes that callers use: the workspace query covers
the plan of every cache format, the allocation-free entry point's scratch covers
every call, and the splits cover the sequence with none empty."""
from __future__ import annotations

import ctypes
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "llm-inference-kernels_amd" / "csrc"
HIP_INCLUDE = Path("/opt/rocm/include")
F16, I8, I4, VALU = range(4)

SHIM = r"""
#include "attention_plan.cpp"
using namespace llmik;
extern "C" void plan(int b, int h, int hkv, int s, int kind, int cus, long* out) {
    const AttnPlan p = plan_attention(b, h, hkv, s, (AttnKind)kind, cus);
    out[0] = p.n_splits; out[1] = p.chunk; out[2] = p.waves; out[3] = p.hpw; out[4] = p.n_hchunks;
    out[5] = p.heads_per_chunk; out[6] = (long)p.workspace_bytes; out[7] = p.n_slot_groups;
}
// First shape (b, h, hkv, s, kind) of the sweep that breaks a rule, with the
// rule's number in out[5]; returns the number of plans looked at.
extern "C" long sweep(int cus, const int* heads, int n_heads, const int* seqs, int n_seqs, int max_b, long* out) {
    long n = 0;
    for (int i = 0; i < n_heads; ++i)
        for (int b = 1; b <= max_b; b += b < 48 ? 1 : 7)
            for (int j = 0; j < n_seqs; ++j)
                for (int kind = 0; kind < 4; ++kind, ++n) {
                    const int h = heads[2 * i], hkv = heads[2 * i + 1], s = seqs[j];
                    const AttnPlan p = plan_attention(b, h, hkv, s, (AttnKind)kind, cus);
                    const int gqa = h / hkv;
                    long bad = 0;
                    if ((long)p.chunk * p.n_splits < s || (long)p.chunk * (p.n_splits - 1) >= s) bad = 1;
                    if (p.chunk % (kTile * p.waves) != 0) bad = 2;
                    if (p.heads_per_chunk > p.hpw || p.n_hchunks * p.heads_per_chunk < gqa ||
                        (p.n_hchunks - 1) * p.heads_per_chunk >= gqa) bad = 3;
                    if (p.workspace_bytes > LLMIK_NOALLOC_SCRATCH_BYTES) bad = 4;
                    if (p.n_splits > 1 && p.n_slot_groups > kMaxCounters) bad = 5;
                    if (bad) {
                        const long v[6] = {b, h, hkv, s, kind, bad};
                        for (int k = 0; k < 6; ++k) out[k] = v[k];
                        return n;
                    }
                }
    out[5] = 0;
    return n;
}
"""

HEADS = [(32, 8), (64, 8), (32, 32), (16, 8), (28, 4), (40, 8), (24, 8), (12, 4), (48, 8), (9, 1), (17, 1), (64, 4),
         (71, 1)]
SEQS = sorted({1, 31, 32, 33, 100, 127, 128, 129, 192, 224, 225, 256, 257, 300, 384, 385, 512, 600, 1024, 1279, 1280,
               1500, 2048, 2304, 2559, 2560, 2561, 2700, 3001, 4095, 4096, 5000, 8192, 16000, 32768, 131072}
              | set(range(64, 3000, 97)))


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    if shutil.which("g++") is None or not (HIP_INCLUDE / "hip" / "hip_runtime.h").exists():
        pytest.skip("no host compiler or no HIP headers")
    d = tmp_path_factory.mktemp("plan")
    (d / "shim.cpp").write_text(SHIM)
    so = d / "plan.so"
    res = subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__=1", f"-I{CSRC}",
                          f"-I{HIP_INCLUDE}", str(d / "shim.cpp"), "-o", str(so)], capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    return ctypes.CDLL(str(so))


def _plan(plans, b, h, hkv, s, kind, cus=256):
    out = (ctypes.c_long * 8)()
    plans.plan(b, h, hkv, s, kind, cus, out)
    names = ("n_splits", "chunk", "waves", "hpw", "n_hchunks", "heads_per_chunk", "workspace", "slabs")
    return dict(zip(names, out))


@pytest.mark.parametrize("cus", [256, 304, 128])
def test_plans_are_whole(plans, cus):
    heads = (ctypes.c_int * (2 * len(HEADS)))(*[x for p in HEADS for x in p])
    seqs = (ctypes.c_int * len(SEQS))(*SEQS)
    out = (ctypes.c_long * 6)()
    plans.sweep.restype = ctypes.c_long
    n = plans.sweep(cus, heads, len(HEADS), seqs, len(SEQS), 70, out)
    assert out[5] == 0, list(out)
    assert n > 100_000


def test_workspace_query_covers_every_format(plans):
    from llmik_cuda._lib import lib
    # the query plans for the current device, or for 256 CUs without one
    import torch
    cus = torch.cuda.get_device_properties(0).multi_processor_count if torch.cuda.is_available() else 256
    for h, hkv in HEADS:
        for b in (1, 2, 3, 5, 8, 12, 17, 21, 27, 33, 40, 64):
            for s in SEQS[::2]:
                need = lib.llmik_attention_workspace_size(b, h, hkv, s, 128)
                most = max(_plan(plans, b, h, hkv, s, kind, cus)["workspace"] for kind in (F16, I8, I4, VALU))
                assert need == most, (b, h, hkv, s)


@pytest.mark.parametrize("b,h,hkv,s,kind,chunks", [
    (1, 24, 8, 120, I4, 3), (8, 24, 8, 120, I4, 3), (11, 24, 8, 120, I4, 1),   # 264 workgroups: joint
    (1, 48, 8, 1145, I4, 3), (2, 40, 8, 300, I4, 5), (1, 48, 8, 2048, I4, 3), (1, 48, 8, 2049, I4, 2),
    (2, 24, 8, 400, I4, 3), (3, 24, 8, 400, I4, 1), (1, 28, 4, 120, I4, 2), (1, 24, 8, 120, F16, 1), (1, 24, 8, 120, I8, 1), (1, 24, 8, 120, VALU, 3),
    (1, 64, 8, 300, I4, 2), (1, 32, 8, 300, I4, 1),
])
def test_small_int4_calls_keep_dividing_chunks(plans, b, h, hkv, s, kind, chunks):
    assert _plan(plans, b, h, hkv, s, kind)["n_hchunks"] == chunks


@pytest.mark.parametrize("b,h,hkv,s,kind,splits", [
    (1, 24, 8, 2560, I4, 10), (1, 24, 8, 2561, I4, 6), (1, 24, 8, 5900, I4, 12), (2, 28, 4, 2700, I4, 6),
    (1, 24, 8, 9000, I4, 18),                            # 32 wanted of 36: two tiles per wave already
    (1, 32, 8, 5900, I4, 24),                            # heads that were not joined
    (1, 24, 8, 5900, F16, 24), (1, 24, 8, 5900, I8, 24), (4, 32, 8, 5900, I4, 8),
])
def test_int4_splits_of_one_tile_per_wave(plans, b, h, hkv, s, kind, splits):
    assert _plan(plans, b, h, hkv, s, kind)["n_splits"] == splits
