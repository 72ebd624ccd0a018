// Quantize-on-append KV-cache writers for gfx950, bit-exact with
// reference/kv_cache_ref.py applied to x.float():
//   scale = max(absmax / qmax, 1e-8)            (fp32, IEEE division)
//   q     = clamp(round_half_even(x / scale), -qmax, qmax)
//   scale stored as fp16 (round to nearest even)
// (kv_cache_ref.py:46-62 per token, :73-112 per channel groupwise.)
// Non-finite inputs follow torch: amax propagates NaN (kv_cache_ref.py:59-61)
// and clamp keeps it, so a row (or group channel) holding a NaN stores scale
// NaN and codes 0; one holding +-inf stores scale +inf, and every quotient is
// then 0 (finite / inf) or NaN (inf / inf), whose int8 conversion is 0.
// The reference CUDA writers multiply by an approximate reciprocal under
// fast-math (kernels/kv_cache/kv_compress.cu:50-58,128-129,200-201) and are
// only within +-1 code of the oracle; these kernels divide exactly.
//
// Layouts (one "row" per (batch, kv_head) pair):
//   x     [rows, src_len, 128] fp16; tokens [0, n_tok) of each row are read
//   int8  [rows, dst_len, 128] int8, scale [rows, dst_len] fp16
//   int4  [rows, dst_len, 64] packed (channel 2i -> low nibble of byte i),
//         scale as above
//   K groupwise int4: scale [rows, dst_groups, 128] fp16
// Token t of a row is written to cache position dst_off + t (K groupwise:
// dst_off is a multiple of group_size and group g goes to scale slot
// dst_off / group_size + g). The out-of-place ops are the identity map
// src_len = dst_len = n_tok, dst_off = 0.
#include <type_traits>

#include "device_common.hpp"
#include "llmik_internal.hpp"

namespace llmik {

constexpr int kWriterThreads = 256;   // 32 token groups of 8 lanes, or 16 rows of 16 lanes

// Token indexing of the writers: `flat` runs over the n_tok tokens of every
// (batch, kv_head) row; src / dst give the token's position in x and in the
// destination cache.
struct TokenMap {
    uint32_t n_tok;     // tokens per (batch, kv_head) row to quantise
    uint32_t src_len;   // token stride of x
    uint32_t dst_len;   // token stride of the destination cache
    uint32_t dst_off;   // cache position of token 0
    __device__ __forceinline__ long src(uint32_t flat) const {
        const uint32_t r = flat / n_tok;
        return (long)r * src_len + (flat - r * n_tok);
    }
    __device__ __forceinline__ long dst(uint32_t flat) const {
        const uint32_t r = flat / n_tok;
        return (long)r * dst_len + dst_off + (flat - r * n_tok);
    }
};

// Per token: 8 lanes per token; lane c of an 8-lane group owns channels
// 8c..8c+7 and 64+8c..64+8c+7, so each load instruction reads the first or
// the second half of its tokens' rows, contiguous. The per-token work (the
// 8-lane DPP max, the scale's division, the reciprocal, the addresses) is
// shared by 16 values per lane. The absmax runs on the fp16 bit patterns
// (sign masked, packed unsigned max), the same order as the fp32 magnitudes
// (NaN above +inf). A workgroup covers 32 groups x kTokensPerRow8
// consecutive tokens. Against 16 lanes per token with 8 values each (two
// tokens per lane group), same bits, on one box (us): INT8 B=8 S=4096 18.87
// -> 18.50, INT4 V 17.79 -> 16.25, INT8 / INT4 V B=64 131.8 / 120.7 ->
// 125.5 / 110.2, S=1000 6.62 / 6.48 -> 6.27 / 5.95; two tokens per group
// (64 per workgroup) was slower for INT8 (20.4) and at small shapes. With
// code_words: INT8 / INT4 V B=8 S=4096 18.1 / 15.4 -> 17.6 / 14.8, INT4 V
// B=64 108.8 -> 104.2, INT8 B=64 125.2 -> 125.8 (bound by the stream).
constexpr int kTokensPerRow8 = 1;

__device__ __forceinline__ uint32_t row8_umax(uint32_t v) {
    v = max(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, kDppQuadXor1, 0xF, 0xF, true));
    v = max(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, kDppQuadXor2, 0xF, 0xF, true));
    v = max(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, kDppRowHalfMirror, 0xF, 0xF, true));
    return v;
}

template <int QMAX, bool PACK4, bool MAPPED>
__global__ __launch_bounds__(kWriterThreads) void quantize_per_token_kernel(
    const uint16_t* __restrict__ x, int8_t* __restrict__ q, uint16_t* __restrict__ scale,
    long rows, TokenMap map) {
    constexpr int kGroups = kWriterThreads / 8;
    const long blk = (long)blockIdx.x * (kGroups * kTokensPerRow8);
    const int grp = threadIdx.x >> 3;
    const int c = threadIdx.x & 7;
    u32x4 raw[kTokensPerRow8][2];
#pragma unroll
    for (int i = 0; i < kTokensPerRow8; ++i) {
        // Tokens past the end take part in the DPP reduction on a clamped,
        // in-bounds token but store nothing.
        const long flat = min(blk + kGroups * i + grp, rows - 1);
        const long src = MAPPED ? map.src((uint32_t)flat) : flat;
        raw[i][0] = stream16(x + src * 128 + 8 * c);
        raw[i][1] = stream16(x + src * 128 + 64 + 8 * c);
    }
#pragma unroll
    for (int i = 0; i < kTokensPerRow8; ++i) {
        const long flat = blk + kGroups * i + grp;
        // |x| of the 16 fp16 values as bit patterns, packed max per half.
        uint32_t w[8], m = 0u;
#pragma unroll
        for (int d = 0; d < 8; ++d) {
            w[d] = raw[i][d >> 2][d & 3];
            m = max_abs2(m, w[d]);
        }
        const uint32_t m16 = max(m & 0xFFFFu, m >> 16);
        const uint32_t amax16 = row8_umax(m16);
        const float amax = h2f((uint16_t)amax16);   // exact; NaN stays NaN, inf stays inf
        const float sc = sym_scale(__float_as_uint(amax), (float)QMAX);
        const float s1[1] = {sc}, r1[1] = {recip_approx(sc)};
        uint32_t code[16];
        code_words<QMAX>(w, s1, r1, code);
        if (flat < rows) {
            const long row = MAPPED ? map.dst((uint32_t)flat) : flat;
            if constexpr (PACK4) {
                __builtin_nontemporal_store(pack_nibbles(code), reinterpret_cast<uint32_t*>(q + row * 64 + 4 * c));
                __builtin_nontemporal_store(pack_nibbles(code + 8), reinterpret_cast<uint32_t*>(q + row * 64 + 32 + 4 * c));
            } else {
                __builtin_nontemporal_store(u32x2{pack_bytes(code), pack_bytes(code + 4)},
                                            reinterpret_cast<u32x2*>(q + row * 128 + 8 * c));
                __builtin_nontemporal_store(u32x2{pack_bytes(code + 8), pack_bytes(code + 12)},
                                            reinterpret_cast<u32x2*>(q + row * 128 + 64 + 8 * c));
            }
            if (c == 0) scale[row] = f2h_bits(sc);
        }
    }
}

// The K writers' workgroup: NT / 16 rows of 16 lanes, lane c of a row owning
// channels 8c..8c+7. Merges the rows' packed absmax (fp16 bit patterns, m):
// the four rows of a wave by lane swaps, the waves through LDS; computes the
// 128 channels' scales and their reciprocals once, stores the fp16 scales and
// hands each lane its channels'.
template <int NT>
struct KScales {
    uint16_t maxes[NT / kWave][128];
    float scale[128], rcp[128];
};
template <int NT>
__device__ __forceinline__ void k_group_scales(KScales<NT>& l, uint32_t (&m)[4], uint16_t* __restrict__ scale,
                                               float (&sv)[8], float (&rv)[8]) {
    const int lane = threadIdx.x & (kWave - 1);
    const int c = threadIdx.x & 15;
    // Two copies of a value swap their 32-lane halves (16-lane rows): the two
    // results hold each half (row) in both places.
#pragma unroll
    for (int d = 0; d < 4; ++d) {
        const auto h = __builtin_amdgcn_permlane32_swap(m[d], m[d], false, false);
        m[d] = max_abs2(h[0], h[1]);
        const auto r = __builtin_amdgcn_permlane16_swap(m[d], m[d], false, false);
        m[d] = max_abs2(r[0], r[1]);
    }
    if (lane < 16) *reinterpret_cast<u32x4*>(&l.maxes[threadIdx.x / kWave][8 * c]) = u32x4{m[0], m[1], m[2], m[3]};
    __syncthreads();
    if (threadIdx.x < 128) {
        uint32_t a = 0u;
#pragma unroll
        for (int r = 0; r < NT / kWave; ++r) a = max(a, (uint32_t)l.maxes[r][threadIdx.x]);
        const float sc = sym_scale(__float_as_uint(h2f((uint16_t)a)), 7.0f);
        l.scale[threadIdx.x] = sc;
        l.rcp[threadIdx.x] = recip_approx(sc);
        scale[threadIdx.x] = f2h_bits(sc);
    }
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        sv[e] = l.scale[8 * c + e];
        rv[e] = l.rcp[8 * c + e];
    }
}

// Dynamic LDS that, beside the static part, admits four workgroups to a CU's 160 KiB.
constexpr size_t kWideGroupLds = 36 * 1024 - sizeof(KScales<kWriterThreads>);
static_assert(5 * (kWideGroupLds + sizeof(KScales<kWriterThreads>)) > 160 * 1024 && 4 * (kWideGroupLds + sizeof(KScales<kWriterThreads>)) <= 160 * 1024,
              "four workgroups, not five");

// K per channel, group-wise: one workgroup per (batch, kv_head, group). Row r
// holds the group's tokens r, r+16, ... (at most TPR of them, group_size <=
// 16 * TPR) in registers; the codes are formed from the registers: the input
// is read once. Bound by the read + write stream. With code_words, packed
// maxima and one reciprocal per channel (us, before -> now): B=8 Hkv=8 S=4096
// g128 17.5 -> 16.7, g64 16.1 -> 15.5, g32 17.0 -> 15.7; B=64 g32 116 -> 109.
// Groups of 97-128 tokens (7 or 8 real loads a lane) are held to 4 workgroups
// per CU by unused dynamic LDS (kWideGroupLds; the registers would admit 6)
// above 128 MiB of input, as more loads in flight then only lengthen the memory
// queues: g128 B=64 108 -> 105, against 113 with 6, 112 with 5 and 108.8 with 3.
// us, free -> held, g128 | g112: B=24 S=4096 41.8 -> 40.8 | 42.0 -> 41.3, B=16
// (128 MiB) 28.8 -> 28.6 | 28.6 -> 28.8, B=8 16.2 -> 16.8 | 16.2 -> 16.7; with
// fewer real loads it does not pay: g96 B=24 41.2 -> 42.5, g72 42.2 -> 47.6.
template <int TPR>
__global__ __launch_bounds__(kWriterThreads) void quantize_k_groupwise_int4_kernel(
    const uint16_t* __restrict__ x, int8_t* __restrict__ q, uint16_t* __restrict__ scale,
    int group_size, TokenMap map, int dst_groups) {
    const int seqlen = (int)map.n_tok;
    const int g = blockIdx.x;
    const long bh = blockIdx.y;   // batch * n_kv_heads + kv_head
    const int row = threadIdx.x >> 4;
    const int c = threadIdx.x & 15;
    const int t_start = g * group_size;
    const int t_end = min(t_start + group_size, seqlen);
    const long base = bh * map.src_len;                     // x row of token 0
    const long qbase = bh * map.dst_len + map.dst_off;      // cache row of token 0
    const long sslot = bh * dst_groups + map.dst_off / group_size + g;

    u32x4 raw[TPR];
#pragma unroll
    for (int i = 0; i < TPR; ++i) {
        const int t = min(t_start + row + 16 * i, t_end - 1);   // in bounds; duplicates do not move the max
        raw[i] = stream16(x + (base + t) * 128 + 8 * c);
    }
    uint32_t m[4] = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int i = 0; i < TPR; ++i)
#pragma unroll
        for (int d = 0; d < 4; ++d) m[d] = max_abs2(m[d], raw[i][d]);
    __shared__ __attribute__((aligned(16))) KScales<kWriterThreads> lds;
    float sv[8], rv[8];
    k_group_scales(lds, m, scale + sslot * 128, sv, rv);
#pragma unroll
    for (int i = 0; i < TPR; ++i) {
        const int t = t_start + row + 16 * i;
        const uint32_t w[4] = {raw[i][0], raw[i][1], raw[i][2], raw[i][3]};
        uint32_t code[8];
        code_words<7>(w, sv, rv, code);
        if (t < t_end)
            __builtin_nontemporal_store(pack_nibbles(code), reinterpret_cast<uint32_t*>(q + (qbase + t) * 64 + 4 * c));
    }
}

// Group sizes beyond 16 * 8 tokens: the group is walked twice (max, then
// codes); the second pass re-reads it from the caches.
__global__ __launch_bounds__(kWriterThreads) void quantize_k_groupwise_int4_large_kernel(
    const uint16_t* __restrict__ x, int8_t* __restrict__ q, uint16_t* __restrict__ scale,
    int group_size, TokenMap map, int dst_groups) {
    const int seqlen = (int)map.n_tok;
    const int g = blockIdx.x;
    const long bh = blockIdx.y;
    const int row = threadIdx.x >> 4;
    const int c = threadIdx.x & 15;
    const int t_start = g * group_size;
    const int t_end = min(t_start + group_size, seqlen);
    const long base = bh * map.src_len;                     // x row of token 0
    const long qbase = bh * map.dst_len + map.dst_off;      // cache row of token 0
    const long sslot = bh * dst_groups + map.dst_off / group_size + g;

    uint32_t m[4] = {0u, 0u, 0u, 0u};
    for (int t = t_start + row; t < t_end; t += 16) {
        const u32x4 v = load16(x + (base + t) * 128 + 8 * c);
#pragma unroll
        for (int d = 0; d < 4; ++d) m[d] = max_abs2(m[d], v[d]);
    }
    __shared__ __attribute__((aligned(16))) KScales<kWriterThreads> lds;
    float sv[8], rv[8];
    k_group_scales(lds, m, scale + sslot * 128, sv, rv);
    for (int t = t_start + row; t < t_end; t += 16) {
        const u32x4 v = load16(x + (base + t) * 128 + 8 * c);
        const uint32_t w[4] = {v[0], v[1], v[2], v[3]};
        uint32_t code[8];
        code_words<7>(w, sv, rv, code);
        *reinterpret_cast<uint32_t*>(q + (qbase + t) * 64 + 4 * c) = pack_nibbles(code);
    }
}

int launch_quantize_per_token(const void* x, void* q, void* scale, int rows, int n_tok,
                              int src_len, int dst_len, int dst_off, int qmax, bool pack4,
                              hipStream_t stream) {
    const long total = (long)rows * n_tok;
    if (total == 0) return LLMIK_OK;
    if (total > 0x7FFFFFFFL) return set_error(LLMIK_ERR_UNSUPPORTED, "too many tokens");
    const long rows_per_wg = (kWriterThreads / 8) * kTokensPerRow8;
    const long grid = (total + rows_per_wg - 1) / rows_per_wg;
    const TokenMap map{(uint32_t)n_tok, (uint32_t)src_len, (uint32_t)dst_len, (uint32_t)dst_off};
    auto xp = static_cast<const uint16_t*>(x);
    auto qp = static_cast<int8_t*>(q);
    auto sp = static_cast<uint16_t*>(scale);
    const bool mapped = !(src_len == n_tok && dst_len == n_tok && dst_off == 0);
    const dim3 g((unsigned)grid), b(kWriterThreads);
    if (qmax == 127 && !pack4) {
        if (mapped) hipLaunchKernelGGL((quantize_per_token_kernel<127, false, true>), g, b, 0, stream, xp, qp, sp, total, map);
        else hipLaunchKernelGGL((quantize_per_token_kernel<127, false, false>), g, b, 0, stream, xp, qp, sp, total, map);
    } else if (qmax == 7 && pack4) {
        if (mapped) hipLaunchKernelGGL((quantize_per_token_kernel<7, true, true>), g, b, 0, stream, xp, qp, sp, total, map);
        else hipLaunchKernelGGL((quantize_per_token_kernel<7, true, false>), g, b, 0, stream, xp, qp, sp, total, map);
    } else {
        return set_error(LLMIK_ERR_UNSUPPORTED, "unsupported per-token quantiser variant");
    }
    return check_launch();
}

int launch_quantize_k_groupwise_int4(const void* x, void* q, void* scale, int rows, int n_tok,
                                     int src_len, int dst_len, int dst_off, int dst_groups,
                                     int group_size, hipStream_t stream) {
    if (n_tok == 0 || rows == 0) return LLMIK_OK;
    if (rows > 65535) return set_error(LLMIK_ERR_UNSUPPORTED, "batch * n_kv_heads exceeds 65535");
    const int n_groups = (n_tok + group_size - 1) / group_size;
    const dim3 grid(n_groups, (unsigned)rows), blk(kWriterThreads);
    const TokenMap map{(uint32_t)n_tok, (uint32_t)src_len, (uint32_t)dst_len, (uint32_t)dst_off};
    auto xp = static_cast<const uint16_t*>(x);
    auto qp = static_cast<int8_t*>(q);
    auto sp = static_cast<uint16_t*>(scale);
    // Four workgroups per CU (see the kernel).
    const bool held = group_size > 96 && 256L * n_tok * rows > (128L << 20);
    if (group_size <= 16)
        hipLaunchKernelGGL(quantize_k_groupwise_int4_kernel<1>, grid, blk, 0, stream, xp, qp, sp, group_size, map, dst_groups);
    else if (group_size <= 32)
        hipLaunchKernelGGL(quantize_k_groupwise_int4_kernel<2>, grid, blk, 0, stream, xp, qp, sp, group_size, map, dst_groups);
    else if (group_size <= 64)
        hipLaunchKernelGGL(quantize_k_groupwise_int4_kernel<4>, grid, blk, 0, stream, xp, qp, sp, group_size, map, dst_groups);
    else if (group_size <= 128)
        hipLaunchKernelGGL(quantize_k_groupwise_int4_kernel<8>, grid, blk, held ? kWideGroupLds : 0, stream, xp, qp, sp, group_size, map, dst_groups);
    else
        hipLaunchKernelGGL(quantize_k_groupwise_int4_large_kernel, grid, blk, 0, stream, xp, qp, sp, group_size, map, dst_groups);
    return check_launch();
}

// One decode-step token appended to a KIVI INT4 cache in one launch, per
// (batch, kv_head) row (one workgroup each; the three launches of the
// general path, integration/kv_int4_cache.py:104-144 restated in place):
//   * V: the token quantised per token into v_q / v_scale at position pos;
//   * K: the token written after the open group's r fp16 tokens (k_open),
//     and the open group (tokens pos - r .. pos) re-quantised per channel
//     into its codes and its scale slot (pos - r) / group_size.
// The arithmetic is the per-token and group-wise writers' above, so the
// stored codes and scales are the same bits. group_size <= 16 * TPR.
template <int TPR>
__global__ __launch_bounds__(kWriterThreads) void kivi_append_token_kernel(
    const uint16_t* __restrict__ k_in, long k_stride, const uint16_t* __restrict__ v_in, long v_stride,
    uint16_t* __restrict__ k_open, int8_t* __restrict__ k_q, uint16_t* __restrict__ k_scale,
    int8_t* __restrict__ v_q, uint16_t* __restrict__ v_scale, int r, int pos, int group_size,
    int max_len, int n_groups) {
    const long bh = blockIdx.x;
    const int row = threadIdx.x >> 4;
    const int c = threadIdx.x & 15;
    const uint16_t* kin = k_in + bh * k_stride + 8 * c;
    uint16_t* kopen = k_open + bh * (long)group_size * 128 + 8 * c;

    // ---- K: tokens 0..r of the open group (r from k_in, the rest from k_open)
    const u32x4 knew = load16(kin);
    u32x4 raw[TPR];
#pragma unroll
    for (int i = 0; i < TPR; ++i) {
        const int t = min(row + 16 * i, r);   // past the group: a duplicate, which does not move the max
        raw[i] = (t == r) ? knew : load16(kopen + (long)t * 128);
    }
    if (row == (r & 15)) *reinterpret_cast<u32x4*>(kopen + (long)r * 128) = knew;

    uint32_t m[4] = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int i = 0; i < TPR; ++i)
#pragma unroll
        for (int d = 0; d < 4; ++d) m[d] = max_abs2(m[d], raw[i][d]);
    const int start = pos - r;
    __shared__ __attribute__((aligned(16))) KScales<kWriterThreads> lds;
    float sv[8], rv[8];
    k_group_scales(lds, m, k_scale + (bh * n_groups + start / group_size) * 128, sv, rv);
#pragma unroll
    for (int i = 0; i < TPR; ++i) {
        const int t = row + 16 * i;
        const uint32_t w[4] = {raw[i][0], raw[i][1], raw[i][2], raw[i][3]};
        uint32_t code[8];
        code_words<7>(w, sv, rv, code);
        if (t <= r) *reinterpret_cast<uint32_t*>(k_q + (bh * max_len + start + t) * 64 + 4 * c) = pack_nibbles(code);
    }

    // ---- V: the token per token (row 0's 16 lanes)
    if (row == 0) {
        const u32x4 vr = load16(v_in + bh * v_stride + 8 * c);
        const uint32_t w[4] = {vr[0], vr[1], vr[2], vr[3]};
        uint32_t mv = 0u;
#pragma unroll
        for (int d = 0; d < 4; ++d) mv = max_abs2(mv, w[d]);
        const uint32_t amax16 = row16_umax(max(mv & 0xFFFFu, mv >> 16));
        const float sc = sym_scale(__float_as_uint(h2f((uint16_t)amax16)), 7.0f);
        const float s1[1] = {sc}, r1[1] = {recip_approx(sc)};
        uint32_t code[8];
        code_words<7>(w, s1, r1, code);
        *reinterpret_cast<uint32_t*>(v_q + (bh * max_len + pos) * 64 + 4 * c) = pack_nibbles(code);
        if (c == 0) v_scale[bh * max_len + pos] = f2h_bits(sc);
    }
}

int launch_kivi_append_token(const void* k, long k_stride, const void* v, long v_stride, void* k_open,
                             void* k_q, void* k_scale, void* v_q, void* v_scale, int rows, int r,
                             int pos, int group_size, int max_len, int n_groups, hipStream_t stream) {
    if (rows == 0) return LLMIK_OK;
    const int tpr = (group_size + 15) / 16;
    auto go = [&](auto tag) {
        constexpr int T = decltype(tag)::value;
        hipLaunchKernelGGL((kivi_append_token_kernel<T>), dim3(rows), dim3(kWriterThreads), 0, stream,
                           static_cast<const uint16_t*>(k), k_stride, static_cast<const uint16_t*>(v),
                           v_stride, static_cast<uint16_t*>(k_open), static_cast<int8_t*>(k_q),
                           static_cast<uint16_t*>(k_scale), static_cast<int8_t*>(v_q),
                           static_cast<uint16_t*>(v_scale), r, pos, group_size, max_len, n_groups);
    };
    if (tpr <= 1) go(std::integral_constant<int, 1>{});
    else if (tpr <= 2) go(std::integral_constant<int, 2>{});
    else if (tpr <= 4) go(std::integral_constant<int, 4>{});
    else go(std::integral_constant<int, 8>{});
    return check_launch();
}

// Several tokens appended to a KIVI INT4 cache, and / or its fp16 view, one
// workgroup per (group of group_size tokens, (batch, kv_head) row). Replaces
// the V writer, the K writer of the whole groups, a copy of the open group and
// the K writer of the open group (four launches), and for the view unpacking,
// scaling and concatenating in torch (about 20 launches over 32-bit
// intermediates). A group's tokens are loaded once, K and V together:
//   * a group that gains tokens: K scale and codes over all its tokens (the
//     ones before `start` from k_open), V codes and scales of its new tokens;
//     its new K tokens go to k_open if it began before `start` or stays open,
//     its new V tokens to v_open if it stays open;
//   * view: fp16(code * scale) of a full group, the fp16 tokens of an open one
//     (the old ones from k_open / v_open); full groups before `start` are
//     read from the codes.
// k_open and v_open hold one group, so a launch that reads the tokens of a
// group begun before `start` must not also open another (launch_kivi_append
// splits the call there). Bound by the read + write stream (append of 3000
// tokens, B=4 Hkv=8 g32: 62 MB, 4.6 TB/s); us, before -> now: that append 21.9
// -> 13.5, B=8 n=4096 g128 33.8 -> 30.4, B=1 n=50 g32 9.8 -> 3.3; with the
// view, eager, B=1 n=2048 g32: 176-192 -> 7.8.
struct KiviAppend {
    const uint16_t* k;   // token t of row bh: k + bh * k_stride + (t - start) * 128
    const uint16_t* v;
    long k_stride, v_stride;
    uint16_t* k_open;    // [rows, group_size, 128]
    uint16_t* v_open;    // as k_open, or null
    int8_t* k_q;         // [rows, max_len, 64]
    uint16_t* k_scale;   // [rows, n_groups, 128]
    int8_t* v_q;
    uint16_t* v_scale;   // [rows, max_len]
    uint16_t* k_view;    // [rows, view_len, 128], or null
    uint16_t* v_view;
    int start, end;      // live length before and after
    int group0;          // group of workgroup 0
    int group_size, max_len, n_groups, view_len;
};

__device__ __forceinline__ uint32_t pack_f16(float a, float b) {
    return (uint32_t)f2h_bits(a) | ((uint32_t)f2h_bits(b) << 16);
}

template <int NT, int TPR, bool VIEW>
__global__ __launch_bounds__(NT) void kivi_append_kernel(KiviAppend p) {
    constexpr int kRows = NT / 16;   // token rows of the workgroup; kRows * TPR >= group_size
    const int grp = p.group0 + blockIdx.x;
    const long bh = blockIdx.y;
    const int row = threadIdx.x >> 4;
    const int c = threadIdx.x & 15;
    const int t0 = grp * p.group_size;
    const int t1 = min(t0 + p.group_size, p.end);   // t0 < end: the group has a token
    const bool full = t1 - t0 == p.group_size;
    const long qrow = bh * p.max_len;
    uint16_t* const sc_row = p.k_scale + (bh * p.n_groups + grp) * 128;
    uint16_t* const kopen = p.k_open + bh * (long)p.group_size * 128 + 8 * c;
    uint16_t* const vopen = (p.v_open ? p.v_open : p.k_open) + bh * (long)p.group_size * 128 + 8 * c;

    if (VIEW && full && t1 <= p.start) {   // a full group of the past: from its codes
        float sv[8];
        f16x8_to_f32(load16(sc_row + 8 * c), sv);
#pragma unroll
        for (int i = 0; i < TPR; ++i) {
            const int t = t0 + row + kRows * i;
            if (t >= t1) break;
            float kc[8], vc[8];
            i4x8_to_f32(load4(p.k_q + (qrow + t) * 64 + 4 * c), kc);
            i4x8_to_f32(load4(p.v_q + (qrow + t) * 64 + 4 * c), vc);
            const float vs = h2f(p.v_scale[qrow + t]);
            u32x4 ko, vo;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                ko[e] = pack_f16(kc[2 * e] * sv[2 * e], kc[2 * e + 1] * sv[2 * e + 1]);
                vo[e] = pack_f16(vc[2 * e] * vs, vc[2 * e + 1] * vs);
            }
            const long o = (bh * p.view_len + t) * 128 + 8 * c;
            *reinterpret_cast<u32x4*>(p.k_view + o) = ko;
            *reinterpret_cast<u32x4*>(p.v_view + o) = vo;
        }
        return;
    }

    // Tokens of this lane's row; past the group's end its last one again
    // (in bounds, does not move the maximum, nothing of it is stored).
    u32x4 kr[TPR], vr[TPR];
#pragma unroll
    for (int i = 0; i < TPR; ++i) {
        const int t = min(t0 + row + kRows * i, t1 - 1);
        const bool fresh = t >= p.start;
        kr[i] = fresh ? stream16(p.k + bh * p.k_stride + (long)(t - p.start) * 128 + 8 * c)
                      : load16(kopen + (long)(t - t0) * 128);
        // An old token's V is wanted for the view only.
        vr[i] = fresh ? stream16(p.v + bh * p.v_stride + (long)(t - p.start) * 128 + 8 * c)
                      : (VIEW ? load16(vopen + (long)(t - t0) * 128) : u32x4{0u, 0u, 0u, 0u});
    }
    if (VIEW && t1 <= p.start) {   // the open group, unchanged
#pragma unroll
        for (int i = 0; i < TPR; ++i) {
            const int t = t0 + row + kRows * i;
            if (t >= t1) break;
            const long o = (bh * p.view_len + t) * 128 + 8 * c;
            *reinterpret_cast<u32x4*>(p.k_view + o) = kr[i];
            *reinterpret_cast<u32x4*>(p.v_view + o) = vr[i];
        }
        return;
    }

    uint32_t m[4] = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int i = 0; i < TPR; ++i)
#pragma unroll
        for (int d = 0; d < 4; ++d) m[d] = max_abs2(m[d], kr[i][d]);
    __shared__ __attribute__((aligned(16))) KScales<NT> lds;
    float sv[8], rv[8];
    k_group_scales(lds, m, sc_row, sv, rv);
#pragma unroll
    for (int i = 0; i < TPR; ++i) {
        const int t = t0 + row + kRows * i;
        const bool ok = t < t1, fresh = ok && t >= p.start;
        const uint32_t kw[4] = {kr[i][0], kr[i][1], kr[i][2], kr[i][3]};
        uint32_t kc[8];
        code_words<7>(kw, sv, rv, kc);
        const uint32_t vw[4] = {vr[i][0], vr[i][1], vr[i][2], vr[i][3]};
        uint32_t mv = 0u;
#pragma unroll
        for (int d = 0; d < 4; ++d) mv = max_abs2(mv, vw[d]);
        const float vs = sym_scale(__float_as_uint(h2f((uint16_t)row16_umax(max(mv & 0xFFFFu, mv >> 16)))), 7.0f);
        const float s1[1] = {vs}, r1[1] = {recip_approx(vs)};
        uint32_t vc[8];
        code_words<7>(vw, s1, r1, vc);
        if (ok) __builtin_nontemporal_store(pack_nibbles(kc), reinterpret_cast<uint32_t*>(p.k_q + (qrow + t) * 64 + 4 * c));
        if (fresh) {
            __builtin_nontemporal_store(pack_nibbles(vc), reinterpret_cast<uint32_t*>(p.v_q + (qrow + t) * 64 + 4 * c));
            if (c == 0) p.v_scale[qrow + t] = f2h_bits(vs);
            if (t0 < p.start || !full) *reinterpret_cast<u32x4*>(kopen + (long)(t - t0) * 128) = kr[i];
            if (p.v_open && !full) *reinterpret_cast<u32x4*>(vopen + (long)(t - t0) * 128) = vr[i];
        }
        if constexpr (VIEW) {
            if (ok) {
                u32x4 ko = kr[i], vo = vr[i];
                if (full) {
                    // The code as a float is its word minus kCodeMagic, except
                    // that a NaN word stands for code 0; fp16(code * scale) is
                    // NaN in both, as that word's scale is NaN or inf.
                    const float v16 = h2f(f2h_bits(vs));
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        float kf[2], vf[2];
#pragma unroll
                        for (int u = 0; u < 2; ++u) {
                            kf[u] = (__uint_as_float(kc[2 * e + u]) - kCodeMagic) * h2f(f2h_bits(sv[2 * e + u]));
                            vf[u] = (__uint_as_float(vc[2 * e + u]) - kCodeMagic) * v16;
                        }
                        ko[e] = pack_f16(kf[0], kf[1]);
                        vo[e] = pack_f16(vf[0], vf[1]);
                    }
                }
                const long o = (bh * p.view_len + t) * 128 + 8 * c;
                *reinterpret_cast<u32x4*>(p.k_view + o) = ko;
                *reinterpret_cast<u32x4*>(p.v_view + o) = vo;
            }
        }
    }
}

int launch_kivi_append(const void* k, long k_stride, const void* v, long v_stride, void* k_open, void* v_open,
                       void* k_q, void* k_scale, void* v_q, void* v_scale, void* k_view, void* v_view, int rows,
                       int n, int length, int group_size, int max_len, int n_groups, hipStream_t stream) {
    if (rows == 0 || length + n == 0) return LLMIK_OK;
    if (rows > 65535) return set_error(LLMIK_ERR_UNSUPPORTED, "batch * n_kv_heads exceeds 65535");
    const bool view = k_view != nullptr;
    if (n == 0 && !view) return LLMIK_OK;
    KiviAppend p{};
    p.k = static_cast<const uint16_t*>(k);
    p.v = static_cast<const uint16_t*>(v);
    p.k_stride = k_stride;
    p.v_stride = v_stride;
    p.k_open = static_cast<uint16_t*>(k_open);
    p.v_open = static_cast<uint16_t*>(v_open);
    p.k_q = static_cast<int8_t*>(k_q);
    p.k_scale = static_cast<uint16_t*>(k_scale);
    p.v_q = static_cast<int8_t*>(v_q);
    p.v_scale = static_cast<uint16_t*>(v_scale);
    p.k_view = static_cast<uint16_t*>(k_view);
    p.v_view = static_cast<uint16_t*>(v_view);
    p.group_size = group_size;
    p.max_len = max_len;
    p.n_groups = n_groups;
    p.view_len = length + n;
    // Groups [first, the group of end - 1].
    auto go = [&](int first, int start, int end) {
        p.group0 = first;
        p.start = start;
        p.end = end;
        const dim3 grid((end - 1) / group_size - first + 1, rows);
        auto with = [&](auto nt, auto tpr) {
            constexpr int NT = decltype(nt)::value, T = decltype(tpr)::value;
            if (view) hipLaunchKernelGGL((kivi_append_kernel<NT, T, true>), grid, dim3(NT), 0, stream, p);
            else hipLaunchKernelGGL((kivi_append_kernel<NT, T, false>), grid, dim3(NT), 0, stream, p);
        };
        using std::integral_constant;
        // Threads x tokens per lane (us): g32 B=4 n=3000 256 x 2 13.5, 512 x 1
        // 14.0, 128 x 4 15.2; g64 B=2 n=10000 512 x 2 19.8, 256 x 4 21.2; g128
        // B=8 n=4096 512 x 4 30.4, 256 x 8 33.8, 1024 x 2 39.9, but with at
        // most one workgroup per CU (B=1 n=2048) 6.75, 9.8 and 5.9.
        if (group_size <= 16) with(integral_constant<int, 256>{}, integral_constant<int, 1>{});
        else if (group_size <= 32) with(integral_constant<int, 256>{}, integral_constant<int, 2>{});
        else if (group_size <= 64) with(integral_constant<int, 512>{}, integral_constant<int, 2>{});
        else if ((long)grid.x * rows > device_cu_count()) with(integral_constant<int, 512>{}, integral_constant<int, 4>{});
        else with(integral_constant<int, 1024>{}, integral_constant<int, 2>{});
    };
    const int first = view ? 0 : length / group_size;
    const int boundary = (length / group_size + 1) * group_size;   // end of the group begun before `length`
    const int end = length + n;
    if (length % group_size != 0 && end > boundary && end % group_size != 0) {
        // The open group is completed and another one opened: k_open / v_open
        // are read by the first launch and rewritten by the second.
        go(first, length, boundary);
        p.k += (long)(boundary - length) * 128;
        p.v += (long)(boundary - length) * 128;
        go(boundary / group_size, boundary, end);
    } else {
        go(first, length, end);
    }
    return check_launch();
}

}  // namespace llmik
