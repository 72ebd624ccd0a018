// Decode attention: how a call is divided over workgroups (head chunks, KV
// splits, waves). Host code of its own, without a kernel, so that the plans of
// every cache format can be checked over their shapes on the CPU.
#include <algorithm>

#include "llmik_internal.hpp"

namespace llmik {

namespace {

// Heads per workgroup, two ways. All query heads of a kv head together up to
// `most` (4 or 8) of them, more in equal chunks: the 16 rows of a matrix
// operand cost the same for 3 heads as for 4 and for 5 as for 8.
void joint_chunks(int gqa, int most, AttnPlan& pl) {
    pl.n_hchunks = (gqa + most - 1) / most;
    pl.heads_per_chunk = (gqa + pl.n_hchunks - 1) / pl.n_hchunks;
    pl.hpw = pl.heads_per_chunk > 4 ? 8 : pl.heads_per_chunk > 2 ? 4 : pl.heads_per_chunk;
}
// The power of two up to 4 that divides them: the VALU kernel, whose work grows
// with every head, and small INT4 calls.
int dividing_heads(int gqa) { return gqa % 4 == 0 ? 4 : gqa % 2 == 0 ? 2 : 1; }
void dividing_chunks(int gqa, AttnPlan& pl) {
    pl.hpw = pl.heads_per_chunk = dividing_heads(gqa);
    pl.n_hchunks = gqa / pl.hpw;
}

}  // namespace

// (split, slot group) pairs of one head that fit LLMIK_NOALLOC_SCRATCH_BYTES:
// 128 fp32 outputs and (m, l), after the counters and two alignments.
constexpr long kMaxScratchSlots =
    (long)((LLMIK_NOALLOC_SCRATCH_BYTES - kCounterBytes - 512) / ((kHeadDim + 2) * sizeof(float)));

AttnPlan plan_attention(int batch, int n_heads, int n_kv_heads, int seqlen, AttnKind kind, int cus) {
    AttnPlan pl{};
    const bool mfma = kind != AttnKind::Valu;
    const int gqa = n_heads / n_kv_heads;
    const long target = (long)kAttnWgsPerCu * cus;
    const long splits8 = ((long)seqlen + 8 * kTile - 1) / (8 * kTile);
    // One workgroup for up to 8 heads of a kv head reads its cache once; with
    // chunks of 4, 2 or 1 heads (the largest that divides the head count, the
    // rule before) every chunk read it again, through L2 at best. us, fp16:
    // H=64 Hkv=8 (4 + 4) B=12 S=3001 49.4 -> 35.7, B=32 S=2048 78.1 -> 40.1;
    // H=28 Hkv=4 (7 x 1) B=16 S=2000 64.0 -> 14.9; H=40 Hkv=8 (5 x 1) B=8
    // S=4096 118 -> 27.2; H=24 Hkv=8 (3 x 1) B=20 S=1500 51.9 -> 26.7. INT8
    // H=64 B=8 S=4096 23.8 -> 15.2, INT4 g128 B=32 S=4096 50.8 -> 32.3. If
    // even one step per wave would leave CUs idle, chunks of up to 4 heads
    // (twice the workgroups) finish sooner: INT4 H=64 B=2 S=2048 8.95 against
    // 8.35, INT8 B=1 S=2000 7.6 against 7.5.
    // INT4 calls whose dividing chunks, in steps of 8 waves (4 waves from 385
    // to 512 tokens, as split below), find a CU each keep those, up to 5 of a kv
    // head and 2048 tokens (longer walks are better off with fewer, longer
    // splits, below): a workgroup does a few tiles only, and its time is the
    // softmax and the merge of its own heads, not the cache, which the chunks
    // read again. us, joint -> dividing, caches read in turn from HBM: H=24
    // Hkv=8 (3 x 1) B=1 S=120 4.15 -> 3.81, S=400 5.83 -> 5.45, S=1145 7.17 ->
    // 6.76, B=4 S=256 4.96 -> 4.72; H=48 Hkv=8 (3 x 2) B=1 S=2000 8.24 -> 7.66;
    // H=40 Hkv=8 (5 x 1) B=1 S=400 5.96 -> 5.55. With more workgroups than CUs
    // (H=24 B=3 S=400) 6.02 -> 6.34. Not 7 chunks (H=28 Hkv=4 B=4 S=120 4.35 ->
    // 4.42, S=256 5.06 -> 5.27); fp16 and INT8 are even (B=4 S=120, H=24 Hkv=8:
    // 4.28, 4.26 and 3.71, 3.81).
    const long dividing = gqa / dividing_heads(gqa);
    const long small_splits = seqlen > 384 && seqlen <= 512 ? (seqlen + 4 * kTile - 1) / (4 * kTile) : splits8;
    if (!mfma || (kind == AttnKind::I4 && dividing <= 5 && splits8 <= 8 &&
                  (long)batch * n_kv_heads * dividing * small_splits <= target))
        dividing_chunks(gqa, pl);
    else
        joint_chunks(gqa, (long)batch * n_kv_heads * ((gqa + 7) / 8) * splits8 < target ? 4 : 8, pl);
    const long base_wgs = (long)batch * n_kv_heads * pl.n_hchunks;
    // Aim for kAttnWgsPerCu workgroups per CU. Calls that must split the
    // sequence to fill the chip use 8-wave workgroups (more loads in flight
    // per CU); otherwise 4 waves. Every split
    // gets at least one 32-token tile per wave.
    // A short sequence that 8-wave splits (one 256-token step each) cannot
    // spread over the chip runs 4-wave splits instead, as long as that keeps
    // the combine to at most 8 partials: at B=1, S=1024 the 8 splits took
    // 6.9 us against 9.0 us for 4; at B=1, S=4096 32 splits took 12.6 us
    // against 10.4 us for 16 (the combine grows with the split count).
    // (Not with more than half as many slabs as CUs: one unsplit round beats
    // both this and the thin splits below; us, B=27 S=200 fp16 / INT8 / INT4
    // 7.7 / 6.4 / 7.1 -> 6.2 / 5.0 / 5.2, B=20 S=300 8.0 / 6.5 / 7.0 -> 7.1 / 5.4 / 6.1.)
    const bool few = !mfma || 2 * base_wgs <= target;
    const bool short_seq = few && base_wgs * splits8 < target && 2 * splits8 <= 8;
    pl.waves = (base_wgs < target && !short_seq) ? 8 : 4;
    // Splits that would give each of 8 waves a single 32-token tile run as
    // 4-wave workgroups at twice the split count (two per CU), as long as the
    // combine stays at <= 8 partials: B=8, S=1024 11.36-11.40 -> 10.94-11.03
    // us; with more partials (B=4, S=1024; B=1, S=4096) it was slower.
    const bool thin = pl.waves == 8 && few && (long)seqlen * base_wgs <= target * 8 * kTile &&
                      2 * ((target + base_wgs - 1) / base_wgs) <= 8;
    if (thin) pl.waves = 4;
    long want = ((thin ? 2 : 1) * target + base_wgs - 1) / base_wgs;
    // Slab counts that do not divide the CUs. Rounding the split count up, as
    // before, put a second round of workgroups on a few CUs (12 x 8 slabs in
    // 3 splits: 288 workgroups, 32 of them alone at the end); the matrix-core
    // plans round down, so that one round covers the call. Where rounding down
    // leaves a third or more of the CUs idle (129-170 slabs on 256 CUs; below
    // 1280 tokens their extra combine costs more), and above one slab per CU
    // (257-341), where some CUs would do twice the work of others, 3 splits
    // of 4-wave workgroups even it out, as far as their partials fit the static
    // scratch (slot_cap, for every caller: at 4 heads per workgroup up to 325
    // slabs; at 8 heads 167-170 slabs take 2 splits and 257-341 none). us, H=32 Hkv=8, before -> now, fp16 |
    // INT8 | INT4 g128:
    //   B=9  S=6000  51 -> 38.5     | 28.3 -> 20.9 | 24.5 -> 16.0
    //   B=12 S=3000  33.5 -> 25.4   | 20.8 -> 15.7 | 19.7 -> 12.9
    //   B=17 S=4000  68.2 -> 49.3   | 35.5 -> 25.6 | 28.9 -> 19.6
    //   B=17 S=900   17.7 -> 14.3   | 12.4 -> 9.5  | 14.7 -> 8.9
    //   B=22 S=1500  27.0 -> 21.9   | 17.3 -> 13.4 | 18.3 -> 11.5
    //   B=40 S=5000  160.7 -> 130.4 | 76.6 -> 73.0 | 48.8 -> 45.7
    //   B=5 S=16000  74.7 -> 52.9   | 39.9 -> 27.8 | 31.8 -> 20.6
    // (129-170 slabs at S=900, unsplit against 3 splits: fp16 15.6, 15.5; INT8
    // 9.8, 11.0; INT4 9.2, 9.8. 257-341 slabs, INT8 / INT4 at S=1500: 22.5 /
    // 18.1 unsplit, 22.6 / 19.7 in 3.) Unsplit at one workgroup per CU, 4
    // waves against 8: fp16 B=24 S=3000 49.8, 52.0 but B=20 S=300 7.9, 7.3;
    // INT8 B=32 S=3000 37.8, 32.3, S=500 8.9, 8.1; INT4 B=24 S=1500 13.1,
    // 12.2, B=27 S=200 5.4, 6.0, and with every CU filled B=32 S=3000 23.3,
    // 20.9, S=2048 16.2, 16.7.
    // Short walks are not split at all: the hand-off (partials, counter,
    // combine: three memory round trips) costs more than one or two further
    // tiles per wave. us, split -> unsplit, B=1 / B=4 / B=12 (Hkv=8): fp16
    // S=192 5.3 / 5.5 / 5.7 -> 4.65 / 5.1 / 5.2, S=224 5.3 / 5.4 / 5.8 -> 4.9 /
    // 5.4 / 5.6, S=256 5.6 / 5.7 / 6.1 -> 5.1 / 5.85 / 6.3; INT8 S=256 5.45 /
    // 5.55 / 5.85 -> 4.7 / 4.9 / 5.1, S=384 5.5 / 5.8 / 6.6 -> 5.3 / 5.7 / 5.8,
    // S=448 5.5 / 6.0 / 7.1 -> 5.9 / 6.3 / 6.4; INT4 (4 waves) S=256 5.9 / 6.1
    // / 6.3 -> 5.1 / 5.3 / 5.4, (8 waves) S=320 5.9 / 6.2 / 7.3 -> 6.0 / 6.2 /
    // 6.3, S=384 6.0 / 6.2 / 7.7 -> 6.3 / 6.55 / 6.6.
    const int short_walk = kind == AttnKind::F16 ? 224 : kind == AttnKind::I8 || base_wgs >= 48 ? 384 : 256;
    const bool unsplit = mfma && few && seqlen > 4 * kTile && seqlen <= short_walk;
    if (unsplit) {
        want = 1;
        pl.waves = kind == AttnKind::I4 && seqlen <= 256 ? 4 : 8;
    }
    const long slot_cap = kMaxScratchSlots / pl.hpw / base_wgs;
    const bool short_ints = kind != AttnKind::F16 && seqlen < 4096;
    if (mfma && !unsplit && !thin && !short_seq && base_wgs <= target) {
        if (want * base_wgs > target) want = target / base_wgs;
        if (want == 1 && 3 * base_wgs <= 2 * target && seqlen >= 1280) {
            want = 3;
            pl.waves = 4;
        } else if (want == 1) {
            pl.waves = seqlen > 4 * kTile ? 8 : 4;
            if (kind == AttnKind::F16 && (base_wgs == target || seqlen >= 512)) pl.waves = 4;
            if (kind == AttnKind::I4 && seqlen < (base_wgs == target ? 2560 : 600)) pl.waves = 4;
        }
    } else if (mfma && base_wgs > target && 3 * base_wgs <= 4 * target && slot_cap >= 3 && seqlen >= 512 &&
               !short_ints) {
        want = 3;
    }
    const int step = kTile * pl.waves;
    const long max_useful = (seqlen + step - 1) / step;
    // INT4 heads that were joined leave fewer slabs for the same CUs, which
    // would be cut into more splits of one tile per wave: above 10 of those,
    // half as many of two tiles, as the combine's time grows with their
    // number. us, caches from HBM, H=24 Hkv=8: B=1 S=2700 8.26 -> 8.05, S=4500
    // 10.10 -> 8.94, S=7500 11.56 -> 9.59, B=2 S=3500 10.03 -> 8.92; H=28
    // Hkv=4 B=1 S=5900 10.70 -> 9.22; H=40 Hkv=8 B=1 S=3500 10.00 -> 8.91. At 8
    // splits it is even (B=1 S=2000 7.51, 7.50), with 4 slabs up to 4 % slower
    // below 3500 tokens (H=12 Hkv=4 S=2700 7.71 -> 7.94).
    if (kind == AttnKind::I4 && pl.n_hchunks < dividing && !unsplit && !thin && !short_seq && max_useful > 10 &&
        want >= max_useful)
        want = (max_useful + 1) / 2;
    if (want > max_useful) want = max_useful;
    if (want > kMaxAttnSplits) want = kMaxAttnSplits;
    if (base_wgs > kMaxCounters) want = 1;   // enough workgroups without splitting
    // Partials stay within the static scratch of the entry point that takes no
    // workspace, for the callers that bring one too (one plan, the same bits).
    if (mfma && slot_cap > 0) want = std::min(want, slot_cap);
    if (want < 1) want = 1;
    int chunk = (int)((seqlen + want - 1) / want);
    chunk = ((chunk + step - 1) / step) * step;
    if (chunk < step) chunk = step;
    pl.chunk = chunk;
    pl.n_splits = seqlen > 0 ? (seqlen + chunk - 1) / chunk : 1;
    pl.n_slot_groups = base_wgs;
    const size_t slots = (size_t)base_wgs * pl.n_splits * pl.hpw;
    const size_t ml = align_up(slots * 2 * sizeof(float), 256);
    const size_t po = align_up(slots * kHeadDim * sizeof(float), 256);
    pl.workspace_bytes = (pl.n_splits > 1) ? kCounterBytes + ml + po : 0;
    pl.off_ml = kCounterBytes;
    pl.off_o = kCounterBytes + ml;
    return pl;
}

}  // namespace llmik
