// Fused elementwise decode-path ops for gfx950: RMSNorm, SwiGLU, RoPE.
// Semantics follow kernels/fused/fused_ops.cu:31-86 of the reference
// (fp32 math, one fp16 rounding of each output).
#include "device_common.hpp"
#include "llmik_internal.hpp"

namespace llmik {

// Loads and stores of the elementwise kernels that move each byte once. STREAM
// (both non-temporal) from kStreamBytes of traffic, what the eight L2s hold
// together: with plain stores the next kernel also pays for writing the dirty
// lines back. us, plain -> STREAM: rmsnorm, rope of q and k and silu_mul in
// turn, T=2000, 32 + 8 heads, 14336 wide 54.2 -> 47.0, T=1000, 11008 wide 29.0
// -> 25.7, T=4096 97.6 -> 86.7. What reads the output finds less of it in L2:
// silu_mul and the down projection of [2000, 14336] 255 -> 258, [700, 8192] 50.1
// -> 51.7, but a layer's prefill without its attention takes the same (T=2000
// 918 and 920, T=700 305 and 305, T=1000 440 and 441, T=4096 1808 and 1802).
// Below, the output fits and the reader's loss is all there is: silu_mul and
// down of [170, 14336] 44.3 -> 45.9, rope [1, 32, 2000, 128] (31 MiB) alone 6.9
// -> 7.8 and with the K writer 12.5 -> 13.7.
constexpr long kStreamBytes = 32L << 20;
template <bool STREAM>
__device__ __forceinline__ u32x4 ew_load16(const void* p) {
    return STREAM ? stream16(p) : load16(p);
}
template <bool STREAM>
__device__ __forceinline__ void ew_store16(void* p, u32x4 v) {
    if constexpr (STREAM) __builtin_nontemporal_store(v, reinterpret_cast<u32x4*>(p));
    else *reinterpret_cast<u32x4*>(p) = v;
}

// One workgroup per row; 16-byte vectors when the row allows it.
__global__ __launch_bounds__(256) void rmsnorm_kernel(const uint16_t* __restrict__ x,
                                                      const uint16_t* __restrict__ w,
                                                      uint16_t* __restrict__ out, int hidden,
                                                      float eps) {
    const long row = blockIdx.x;
    const uint16_t* xr = x + row * hidden;
    uint16_t* orow = out + row * hidden;
    const bool vec = (hidden % 8) == 0;
    float ss = 0.0f;
    if (vec) {
        for (int i = threadIdx.x * 8; i < hidden; i += 256 * 8) {
            float v[8];
            f16x8_to_f32(load16(xr + i), v);
#pragma unroll
            for (int e = 0; e < 8; ++e) ss = fmaf(v[e], v[e], ss);
        }
    } else {
        for (int i = threadIdx.x; i < hidden; i += 256) {
            const float v = h2f(xr[i]);
            ss = fmaf(v, v, ss);
        }
    }
    // wave sum: 16-lane rows, then across the 4 rows via LDS
    ss = row16_sum(ss);
    __shared__ float s_red[16];
    if ((threadIdx.x & 15) == 0) s_red[threadIdx.x >> 4] = ss;
    __syncthreads();
    float tot = 0.0f;
#pragma unroll
    for (int r = 0; r < 16; ++r) tot += s_red[r];
    const float inv = 1.0f / sqrtf(tot / (float)hidden + eps);
    if (vec) {
        for (int i = threadIdx.x * 8; i < hidden; i += 256 * 8) {
            float v[8], g[8];
            f16x8_to_f32(load16(xr + i), v);
            f16x8_to_f32(load16(w + i), g);
            u32x4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e)
                o[e] = (uint32_t)f2h_bits(v[2 * e] * inv * g[2 * e]) |
                       ((uint32_t)f2h_bits(v[2 * e + 1] * inv * g[2 * e + 1]) << 16);
            *reinterpret_cast<u32x4*>(orow + i) = o;
        }
    } else {
        for (int i = threadIdx.x; i < hidden; i += 256)
            orow[i] = f2h_bits(h2f(xr[i]) * inv * h2f(w[i]));
    }
}

// Rows of up to 256 * 8 * NV fp16 (hidden % 8 == 0): the row and the weight
// are loaded once into registers, both before the reduction, so the kernel
// waits on memory once instead of twice.
template <int NV>
__global__ __launch_bounds__(256) void rmsnorm_regs_kernel(const uint16_t* __restrict__ x,
                                                           const uint16_t* __restrict__ w,
                                                           uint16_t* __restrict__ out, int hidden,
                                                           float eps) {
    const long row = blockIdx.x;
    const uint16_t* xr = x + row * hidden;
    uint16_t* orow = out + row * hidden;
    u32x4 xv[NV], wv[NV];
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        const int i = (threadIdx.x + 256 * k) * 8;
        const bool ok = i < hidden;
        xv[k] = ok ? load16(xr + i) : u32x4{0u, 0u, 0u, 0u};
        wv[k] = ok ? load16(w + i) : u32x4{0u, 0u, 0u, 0u};
    }
    float ss = 0.0f;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        float v[8];
        f16x8_to_f32(xv[k], v);
#pragma unroll
        for (int e = 0; e < 8; ++e) ss = fmaf(v[e], v[e], ss);
    }
    ss = row16_sum(ss);
    __shared__ float s_red[16];
    if ((threadIdx.x & 15) == 0) s_red[threadIdx.x >> 4] = ss;
    __syncthreads();
    float tot = 0.0f;
#pragma unroll
    for (int r = 0; r < 16; ++r) tot += s_red[r];
    const float inv = 1.0f / sqrtf(tot / (float)hidden + eps);
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        const int i = (threadIdx.x + 256 * k) * 8;
        if (i >= hidden) break;
        float v[8], g[8];
        f16x8_to_f32(xv[k], v);
        f16x8_to_f32(wv[k], g);
        u32x4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            o[e] = (uint32_t)f2h_bits(v[2 * e] * inv * g[2 * e]) |
                   ((uint32_t)f2h_bits(v[2 * e + 1] * inv * g[2 * e + 1]) << 16);
        *reinterpret_cast<u32x4*>(orow + i) = o;
    }
}


template <bool STREAM>
__global__ __launch_bounds__(256) void silu_mul_kernel(const uint16_t* __restrict__ g,
                                                       const uint16_t* __restrict__ u,
                                                       uint16_t* __restrict__ out, long n) {
    const long i8 = ((long)blockIdx.x * 256 + threadIdx.x) * 8;
    if (i8 + 8 <= n) {
        float gv[8], uv[8];
        f16x8_to_f32(ew_load16<STREAM>(g + i8), gv);
        f16x8_to_f32(ew_load16<STREAM>(u + i8), uv);
        u32x4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            o[e] = (uint32_t)f2h_bits(silu_mul1(gv[2 * e], uv[2 * e])) |
                   ((uint32_t)f2h_bits(silu_mul1(gv[2 * e + 1], uv[2 * e + 1])) << 16);
        ew_store16<STREAM>(out + i8, o);
    } else {
        for (long i = i8; i < n; ++i) out[i] = f2h_bits(silu_mul1(h2f(g[i]), h2f(u[i])));
    }
}

// One thread per (b, h, s, d) with d < D/2: it produces out[d] and
// out[d + D/2] from the pair (x[d], x[d + D/2]).
__global__ __launch_bounds__(256) void rope_kernel(const uint16_t* __restrict__ x,
                                                   const uint16_t* __restrict__ cs,
                                                   const uint16_t* __restrict__ sn,
                                                   uint16_t* __restrict__ out, int B, int H,
                                                   int S, int D) {
    const int half_d = D / 2;
    const long total = (long)B * H * S * half_d;
    const long idx = (long)blockIdx.x * 256 + threadIdx.x;
    if (idx >= total) return;
    const int d = (int)(idx % half_d);
    const long bhs = idx / half_d;
    const int s = (int)(bhs % S);
    const int b = (int)(bhs / ((long)S * H));
    const long xrow = bhs * D;
    const long crow = ((long)b * S + s) * D;
    rope_pair(h2f(x[xrow + d]), h2f(x[xrow + d + half_d]), h2f(cs[crow + d]), h2f(sn[crow + d]),
              h2f(cs[crow + d + half_d]), h2f(sn[crow + d + half_d]), out[xrow + d],
              out[xrow + d + half_d]);
}

// rope of kHeads heads per thread, 16-byte accesses (D % 16 == 0, 16-byte
// aligned tensors): thread (h0, b, s, j) takes dimensions 8j .. 8j + 7 and
// their partners + D / 2 of heads h0 .. h0 + kHeads - 1 at (b, s), so the
// position's cos and sin are read once for kHeads heads. One thread per pair
// of values moved 2 bytes per access and read 4 table values for 2 outputs.
// Bound by the read + write stream; us, before -> now: [1, 32, 2000, 128]
// 14.0 -> 7.1, [1, 8, 2000, 128] 5.5 -> 3.4, [1, 64, 4096, 128] 64 -> 24.
template <int kHeads, bool STREAM>
__global__ __launch_bounds__(256) void rope_vec_kernel(const uint16_t* __restrict__ x,
                                                       const uint16_t* __restrict__ cs,
                                                       const uint16_t* __restrict__ sn,
                                                       uint16_t* __restrict__ out, int H, int S, int D,
                                                       uint32_t units) {
    const uint32_t idx = blockIdx.x * 256u + threadIdx.x;   // over S * (D / 16) of one batch row
    if (idx >= units) return;
    const int h0 = blockIdx.y * kHeads;
    const int b = blockIdx.z;
    const uint32_t per_row = (uint32_t)D / 16u;
    const uint32_t s = idx / per_row;
    const int d = 8 * (int)(idx - s * per_row);
    const int half_d = D / 2;
    const long crow = ((long)b * S + s) * D + d;
    const u32x4 c1 = load16(cs + crow), c2 = load16(cs + crow + half_d);
    const u32x4 s1 = load16(sn + crow), s2 = load16(sn + crow + half_d);
    u32x4 x1[kHeads], x2[kHeads];
    const long row0 = (((long)b * H + h0) * S + s) * D + d;
    const long head = (long)S * D;
#pragma unroll
    for (int i = 0; i < kHeads; ++i) {
        const long r = row0 + min(i, H - 1 - h0) * head;
        x1[i] = ew_load16<STREAM>(x + r);
        x2[i] = ew_load16<STREAM>(x + r + half_d);
    }
    float c1f[8], c2f[8], s1f[8], s2f[8];
    f16x8_to_f32(c1, c1f);
    f16x8_to_f32(c2, c2f);
    f16x8_to_f32(s1, s1f);
    f16x8_to_f32(s2, s2f);
#pragma unroll
    for (int i = 0; i < kHeads; ++i) {
        if (h0 + i >= H) break;
        float a[8], e[8];
        f16x8_to_f32(x1[i], a);
        f16x8_to_f32(x2[i], e);
        u32x4 o1, o2;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            uint16_t lo1, lo2, hi1, hi2;
            rope_pair(a[2 * k], e[2 * k], c1f[2 * k], s1f[2 * k], c2f[2 * k], s2f[2 * k], lo1, lo2);
            rope_pair(a[2 * k + 1], e[2 * k + 1], c1f[2 * k + 1], s1f[2 * k + 1], c2f[2 * k + 1], s2f[2 * k + 1],
                      hi1, hi2);
            o1[k] = (uint32_t)lo1 | ((uint32_t)hi1 << 16);
            o2[k] = (uint32_t)lo2 | ((uint32_t)hi2 << 16);
        }
        const long r = row0 + i * head;
        ew_store16<STREAM>(out + r, o1);
        ew_store16<STREAM>(out + r + half_d, o2);
    }
}

// ---------------------------------------------------------------- decode step
// Kernels that merge consecutive ops of one decode step; each computes what
// the ops it replaces compute, in the same order, so the results are the
// same bits.

// rope of the q and k heads of a fused q|k|v projection row and the new
// token's K and V written into cache slot `pos`: one thread per (b, head,
// d < D/2) over the H + 2 Hkv heads of qkv [B, H + 2 Hkv, D]. cs / sn are
// the position's [D] row of the rotary tables.
__global__ __launch_bounds__(256) void rope_qkv_append_kernel(
    const uint16_t* __restrict__ qkv, const uint16_t* __restrict__ cs, const uint16_t* __restrict__ sn,
    uint16_t* __restrict__ q_out, uint16_t* __restrict__ kbuf, uint16_t* __restrict__ vbuf, int B, int H,
    int Hkv, int D, int max_len, int pos) {
    const int half_d = D / 2;
    const int NH = H + 2 * Hkv;
    const long idx = (long)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (long)B * NH * half_d) return;
    const int d = (int)(idx % half_d);
    const long bj = idx / half_d;
    const int j = (int)(bj % NH);
    const int b = (int)(bj / NH);
    const uint16_t* x = qkv + bj * D;
    if (j >= H + Hkv) {
        uint16_t* dst = vbuf + (((long)b * Hkv + (j - H - Hkv)) * max_len + pos) * D;
        dst[d] = x[d];
        dst[d + half_d] = x[d + half_d];
        return;
    }
    uint16_t* dst = j < H ? q_out + ((long)b * H + j) * D
                          : kbuf + (((long)b * Hkv + (j - H)) * max_len + pos) * D;
    rope_pair(h2f(x[d]), h2f(x[d + half_d]), h2f(cs[d]), h2f(sn[d]), h2f(cs[d + half_d]),
              h2f(sn[d + half_d]), dst[d], dst[d + half_d]);
}

// h = fp16(x + r) (torch's fp16 add: fp32 sum, one rounding) and
// out = rmsnorm(h) as rmsnorm_regs_kernel computes it, one workgroup per row,
// hidden % 8 == 0 and hidden <= 256 * 8 * NV.
template <int NV>
__global__ __launch_bounds__(256) void add_rmsnorm_kernel(const uint16_t* __restrict__ x,
                                                          const uint16_t* __restrict__ r,
                                                          const uint16_t* __restrict__ w,
                                                          uint16_t* __restrict__ h_out,
                                                          uint16_t* __restrict__ out, int hidden,
                                                          float eps) {
    const long row = blockIdx.x;
    // Every load is issued before any is used, so the kernel waits on memory
    // once (with the h stores between the loads of two rounds, the compiler
    // waited twice).
    u32x4 xa[NV], ra[NV], hv[NV], wv[NV];
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        const int i = (threadIdx.x + 256 * k) * 8;
        const bool ok = i < hidden;
        const u32x4 z{0u, 0u, 0u, 0u};
        xa[k] = ok ? load16(x + row * hidden + i) : z;
        ra[k] = ok ? load16(r + row * hidden + i) : z;
        wv[k] = ok ? load16(w + i) : z;
    }
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        const int i = (threadIdx.x + 256 * k) * 8;
        const bool ok = i < hidden;
        float a[8], c[8];
        f16x8_to_f32(xa[k], a);
        f16x8_to_f32(ra[k], c);
#pragma unroll
        for (int e = 0; e < 4; ++e)
            hv[k][e] = (uint32_t)f2h_bits(a[2 * e] + c[2 * e]) |
                       ((uint32_t)f2h_bits(a[2 * e + 1] + c[2 * e + 1]) << 16);
        if (ok) *reinterpret_cast<u32x4*>(h_out + row * hidden + i) = hv[k];
    }
    float ss = 0.0f;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        float v[8];
        f16x8_to_f32(hv[k], v);
#pragma unroll
        for (int e = 0; e < 8; ++e) ss = fmaf(v[e], v[e], ss);
    }
    ss = row16_sum(ss);
    __shared__ float s_red[16];
    if ((threadIdx.x & 15) == 0) s_red[threadIdx.x >> 4] = ss;
    __syncthreads();
    float tot = 0.0f;
#pragma unroll
    for (int q = 0; q < 16; ++q) tot += s_red[q];
    const float inv = 1.0f / sqrtf(tot / (float)hidden + eps);
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        const int i = (threadIdx.x + 256 * k) * 8;
        if (i >= hidden) break;
        float v[8], g[8];
        f16x8_to_f32(hv[k], v);
        f16x8_to_f32(wv[k], g);
        u32x4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            o[e] = (uint32_t)f2h_bits(v[2 * e] * inv * g[2 * e]) |
                   ((uint32_t)f2h_bits(v[2 * e + 1] * inv * g[2 * e + 1]) << 16);
        *reinterpret_cast<u32x4*>(out + row * hidden + i) = o;
    }
}

// out[r, c] = silu(gu[r, c]) * gu[r, cols + c] over a fused gate|up
// projection gu [rows, 2 cols], cols % 8 == 0.
__global__ __launch_bounds__(256) void silu_mul_halves_kernel(const uint16_t* __restrict__ gu,
                                                              uint16_t* __restrict__ out, long rows,
                                                              int cols) {
    const long i8 = ((long)blockIdx.x * 256 + threadIdx.x) * 8;
    if (i8 >= rows * cols) return;
    const long row = i8 / cols;
    const int col = (int)(i8 % cols);
    float gv[8], uv[8];
    f16x8_to_f32(load16(gu + row * 2 * cols + col), gv);
    f16x8_to_f32(load16(gu + row * 2 * cols + cols + col), uv);
    u32x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e)
        o[e] = (uint32_t)f2h_bits(silu_mul1(gv[2 * e], uv[2 * e])) |
               ((uint32_t)f2h_bits(silu_mul1(gv[2 * e + 1], uv[2 * e + 1])) << 16);
    *reinterpret_cast<u32x4*>(out + i8) = o;
}

int launch_rmsnorm(const void* x, const void* w, void* out, int rows, int hidden, float eps,
                   hipStream_t stream) {
    if (rows == 0 || hidden == 0) return LLMIK_OK;
    const uint16_t* xs = static_cast<const uint16_t*>(x);
    const uint16_t* ws = static_cast<const uint16_t*>(w);
    uint16_t* os = static_cast<uint16_t*>(out);
    if (hidden % 8 == 0 && hidden <= 256 * 8 * 4) {
        const int nv = (hidden + 256 * 8 - 1) / (256 * 8);
        if (nv == 1)
            hipLaunchKernelGGL(rmsnorm_regs_kernel<1>, dim3(rows), dim3(256), 0, stream, xs, ws, os, hidden, eps);
        else if (nv == 2)
            hipLaunchKernelGGL(rmsnorm_regs_kernel<2>, dim3(rows), dim3(256), 0, stream, xs, ws, os, hidden, eps);
        else
            hipLaunchKernelGGL(rmsnorm_regs_kernel<4>, dim3(rows), dim3(256), 0, stream, xs, ws, os, hidden, eps);
        return check_launch();
    }
    hipLaunchKernelGGL(rmsnorm_kernel, dim3(rows), dim3(256), 0, stream, xs, ws, os, hidden, eps);
    return check_launch();
}

int launch_silu_mul(const void* g, const void* u, void* out, long n, hipStream_t stream) {
    if (n == 0) return LLMIK_OK;
    const long blocks = (n + 256 * 8 - 1) / (256 * 8);
    const auto kernel = 6 * n >= kStreamBytes ? silu_mul_kernel<true> : silu_mul_kernel<false>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(256), 0, stream,
                       static_cast<const uint16_t*>(g), static_cast<const uint16_t*>(u),
                       static_cast<uint16_t*>(out), n);
    return check_launch();
}

int launch_rope(const void* x, const void* cs, const void* sn, void* out, int B, int H, int S,
                int D, hipStream_t stream) {
    const long total = (long)B * H * S * (D / 2);
    if (total == 0) return LLMIK_OK;
    const auto al16 = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
    const long units = (long)S * (D / 16);
    if (D % 16 == 0 && al16(x) && al16(cs) && al16(sn) && al16(out) && units <= 0x7FFFFFFFL && B <= 65535) {
        // Two heads per thread, or one where that leaves CUs without a
        // workgroup ([1, 64, 4096, 128], heads per thread 1 / 2 / 4 / 8: 24.9,
        // 24.1, 25.2, 24.2 us; at 2000 tokens and 32 heads, with non-temporal
        // accesses, 8.3, 8.0, 8.1, 8.3).
        const unsigned gx = (unsigned)((units + 255) / 256);
        const bool two = H >= 2 && (long)gx * ((H + 1) / 2) * B >= device_cu_count();
        const int ny = two ? (H + 1) / 2 : H;
        if (ny <= 65535) {
            const bool big = 8 * total >= kStreamBytes;
            const auto kernel = two ? (big ? rope_vec_kernel<2, true> : rope_vec_kernel<2, false>)
                                    : (big ? rope_vec_kernel<1, true> : rope_vec_kernel<1, false>);
            hipLaunchKernelGGL(kernel, dim3(gx, ny, B), dim3(256), 0, stream, static_cast<const uint16_t*>(x),
                               static_cast<const uint16_t*>(cs), static_cast<const uint16_t*>(sn),
                               static_cast<uint16_t*>(out), H, S, D, (uint32_t)units);
            return check_launch();
        }
    }
    const long blocks = (total + 255) / 256;
    hipLaunchKernelGGL(rope_kernel, dim3((unsigned)blocks), dim3(256), 0, stream,
                       static_cast<const uint16_t*>(x), static_cast<const uint16_t*>(cs),
                       static_cast<const uint16_t*>(sn), static_cast<uint16_t*>(out), B, H, S, D);
    return check_launch();
}

int launch_rope_qkv_append(const void* qkv, const void* cs, const void* sn, void* q_out, void* kbuf,
                           void* vbuf, int B, int H, int Hkv, int D, int max_len, int pos,
                           hipStream_t stream) {
    const long total = (long)B * (H + 2 * Hkv) * (D / 2);
    if (total == 0) return LLMIK_OK;
    hipLaunchKernelGGL(rope_qkv_append_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, stream,
                       static_cast<const uint16_t*>(qkv), static_cast<const uint16_t*>(cs),
                       static_cast<const uint16_t*>(sn), static_cast<uint16_t*>(q_out),
                       static_cast<uint16_t*>(kbuf), static_cast<uint16_t*>(vbuf), B, H, Hkv, D, max_len,
                       pos);
    return check_launch();
}

int launch_add_rmsnorm(const void* x, const void* r, const void* w, void* h_out, void* out, int rows,
                       int hidden, float eps, hipStream_t stream) {
    if (rows == 0 || hidden == 0) return LLMIK_OK;
    const uint16_t* xs = static_cast<const uint16_t*>(x);
    const uint16_t* rs = static_cast<const uint16_t*>(r);
    const uint16_t* ws = static_cast<const uint16_t*>(w);
    uint16_t* hs = static_cast<uint16_t*>(h_out);
    uint16_t* os = static_cast<uint16_t*>(out);
    const int nv = (hidden + 256 * 8 - 1) / (256 * 8);
    if (nv == 1)
        hipLaunchKernelGGL(add_rmsnorm_kernel<1>, dim3(rows), dim3(256), 0, stream, xs, rs, ws, hs, os, hidden, eps);
    else if (nv == 2)
        hipLaunchKernelGGL(add_rmsnorm_kernel<2>, dim3(rows), dim3(256), 0, stream, xs, rs, ws, hs, os, hidden, eps);
    else
        hipLaunchKernelGGL(add_rmsnorm_kernel<4>, dim3(rows), dim3(256), 0, stream, xs, rs, ws, hs, os, hidden, eps);
    return check_launch();
}

int launch_silu_mul_halves(const void* gu, void* out, long rows, int cols, hipStream_t stream) {
    const long n = rows * cols;
    if (n == 0) return LLMIK_OK;
    hipLaunchKernelGGL(silu_mul_halves_kernel, dim3((unsigned)((n + 256 * 8 - 1) / (256 * 8))), dim3(256), 0,
                       stream, static_cast<const uint16_t*>(gu), static_cast<uint16_t*>(out), rows, cols);
    return check_launch();
}

}  // namespace llmik
