// Row-wise and element-wise kernels: embedding gather, residual add + RMSNorm, rotary position
// encoding fused with the write into the paged cache, SiLU-multiply.
//
// The residual stream is float in every mode; the kernels that read or write activations take
// the storage type (float or bfloat16) as a template argument and compute in float.
#include "common.h"

#include <math.h>
#include <stdarg.h>
#include <stdio.h>

// ---- error reporting -----------------------------------------------------------------------
static thread_local char g_tl_error[512] = "";

int tl_fail(const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_tl_error, sizeof(g_tl_error), fmt, ap);
    va_end(ap);
    return 1;
}

extern "C" const char* tl_last_error() { return g_tl_error; }

extern "C" int tl_abi_version() { return 1; }

// ---- the matrix-core ordered copy of a matrix --------------------------------------------------
// out[tile][step][16 g + r] = row 16 tile + r of W from its 16-byte unit 4 step + g on, zero beyond N rows and `units` of a row: what a wave of
// the few-row products loads at once lies together.  Bound by memory; a work-group takes sixteen steps of a tile, a row's 1 KB.
// 152,064 x 3,584 in bfloat16 388 us (5.6 TB/s), where torch's copy of the permuted view took 538; 37,888 x 3,584 107 and 151, in float 198 and 213.
#define EW_ORDER_STEPS 16
__global__ __launch_bounds__(256) void order_weight_kernel(const uint4* __restrict__ W, uint4* __restrict__ out, int N, int units, int steps) {
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4, tile = blockIdx.y;
    const int s0 = blockIdx.x * EW_ORDER_STEPS + (threadIdx.x >> 6);
    const int row = tile * 16 + r;
    const uint4* from = W + (size_t)min(row, N - 1) * units;
    uint4* to = out + ((size_t)tile * steps + s0) * 64 + lane;
    uint4 x[EW_ORDER_STEPS / 4];
#pragma unroll
    for (int i = 0; i < EW_ORDER_STEPS / 4; ++i) {
        const int u = (s0 + 4 * i) * 4 + g;
        x[i] = make_uint4(0, 0, 0, 0);
        if (u < units && row < N) x[i] = from[u];
    }
#pragma unroll
    for (int i = 0; i < EW_ORDER_STEPS / 4; ++i)
        if (s0 + 4 * i < steps) to[i * 256] = x[i];
}

// W [N, units of 16 bytes] contiguous; out [ceil(N / 16), ceil(units / 4), 64 units], both 16-byte aligned.
extern "C" int tl_order_weight(const void* W, void* out, int N, int units, hipStream_t stream) {
    TL_CHECK_ARG(N > 0 && units > 0 && (uintptr_t)W % 16 == 0 && (uintptr_t)out % 16 == 0, "tl_order_weight: bad sizes N=%d units=%d, or unaligned", N, units);
    const int tiles = tl_ceil_div(N, 16), steps = tl_ceil_div(units, 4);
    for (int t = 0; t < tiles; t += 65535) {           // (a grid's second dimension has 16 bits)
        const int n = tiles - t < 65535 ? tiles - t : 65535;
        hipLaunchKernelGGL(order_weight_kernel, dim3(tl_ceil_div(steps, EW_ORDER_STEPS), n), dim3(256), 0, stream, (const uint4*)W + (size_t)t * 16 * units,
                           (uint4*)out + (size_t)t * steps * 64, N - t * 16, units, steps);
    }
    TL_CHECK_LAUNCH("tl_order_weight");
    return 0;
}

// ---- embedding gather ----------------------------------------------------------------------
// x[t, :] = float(table[ids[t], :]) * scale.  An id outside [0, V) gives a row of NaN instead of a fault;
// callers validate ids on the host.
template <typename T>
__global__ void embed_kernel(const int32_t* __restrict__ ids, const T* __restrict__ table,
                             float* __restrict__ x, int H, int V, float scale) {
    const int t = blockIdx.x;
    const int id = ids[t];
    float* xr = x + (size_t)t * H;
    if (id < 0 || id >= V) {
        for (int c = threadIdx.x; c < H; c += blockDim.x) xr[c] = NAN;
        return;
    }
    const T* row = table + (size_t)id * H;
    constexpr int V4 = 16 / sizeof(T);                       // a row is scattered memory: 16 bytes a thread, all of it on its way at once
    if (H % V4 == 0 && (uintptr_t)table % 16 == 0 && (uintptr_t)x % 16 == 0) {
        for (int c = threadIdx.x * V4; c < H; c += blockDim.x * V4) {
            const uint4 raw = *reinterpret_cast<const uint4*>(row + c);
            const T* e = reinterpret_cast<const T*>(&raw);
#pragma unroll
            for (int i = 0; i < V4; i += 4)
                *reinterpret_cast<float4*>(xr + c + i) = make_float4(tl_to_float(e[i]) * scale, tl_to_float(e[i + 1]) * scale,
                                                                     tl_to_float(e[i + 2]) * scale, tl_to_float(e[i + 3]) * scale);
        }
        return;
    }
    for (int c = threadIdx.x; c < H; c += blockDim.x) xr[c] = tl_to_float(row[c]) * scale;
}

extern "C" int tl_embed(const int32_t* ids, const void* table, int table_dtype, float* x, int T, int H, int V,
                        float scale, hipStream_t stream) {
    TL_CHECK_ARG(T >= 0 && H > 0 && V > 0, "tl_embed: bad sizes T=%d H=%d V=%d", T, H, V);
    if (T == 0) return 0;
    dim3 grid(T), block(H > 2048 ? 512 : 256);
    if (table_dtype == TL_F32)
        hipLaunchKernelGGL(embed_kernel<float>, grid, block, 0, stream, ids, (const float*)table, x, H, V, scale);
    else if (table_dtype == TL_BF16)
        hipLaunchKernelGGL(embed_kernel<bf16_t>, grid, block, 0, stream, ids, (const bf16_t*)table, x, H, V, scale);
    else
        return tl_fail("tl_embed: unknown dtype %d", table_dtype);
    TL_CHECK_LAUNCH("tl_embed");
    return 0;
}

// ---- embedding gather with a hashed bigram row added ------------------------------------------
// x[t, :] = float(table[ids[t], :]) + float(bigram[row, :]), row = (prev * mul_prev + ids[t] * mul_cur) mod
// buckets, where prev is the token ahead of t in its sequence: the row above in the step, or, for the
// sequence's first row of the step, what its state slot keeps (prev_kept[slot]); a sequence's first token
// (position 0) reads row `buckets`, the table's last.  The sum is float.
template <typename T>
__global__ void embed_bigram_kernel(const int32_t* __restrict__ ids, const int32_t* __restrict__ pos,
                                    const int32_t* __restrict__ seq_of_token, const int32_t* __restrict__ q_start,
                                    const int32_t* __restrict__ state_slots, const int32_t* __restrict__ prev_kept,
                                    long long kept_stride, const T* __restrict__ table, const T* __restrict__ bigram,
                                    float* __restrict__ x, int H, int V, long long buckets, long long mul_prev,
                                    long long mul_cur) {
    const int t = blockIdx.x;
    const int id = ids[t];
    float* xr = x + (size_t)t * H;
    if (id < 0 || id >= V) {
        for (int c = threadIdx.x; c < H; c += blockDim.x) xr[c] = NAN;
        return;
    }
    long long row = buckets;
    if (pos[t] > 0) {
        const int s = seq_of_token[t];
        const long long prev = t > q_start[s] ? ids[t - 1] : prev_kept[(size_t)state_slots[s] * kept_stride];
        row = (prev * mul_prev + (long long)id * mul_cur) % buckets;
        if (row < 0) row += buckets;
    }
    const T* er = table + (size_t)id * H;
    const T* br = bigram + (size_t)row * H;
    for (int c = threadIdx.x; c < H; c += blockDim.x) xr[c] = tl_to_float(er[c]) + tl_to_float(br[c]);
}

// A thread per sequence: the slot keeps the sequence's last token of the step.
__global__ void keep_last_token_kernel(const int32_t* __restrict__ ids, const int32_t* __restrict__ q_start,
                                       const int32_t* __restrict__ state_slots, int32_t* __restrict__ prev_kept,
                                       long long kept_stride, int S) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= S) return;
    const int r1 = q_start[s + 1];
    if (r1 > q_start[s]) prev_kept[(size_t)state_slots[s] * kept_stride] = ids[r1 - 1];
}

extern "C" int tl_embed_bigram(const int32_t* ids, const int32_t* pos, const int32_t* seq_of_token, const int32_t* q_start,
                               const int32_t* state_slots, int32_t* prev_kept, long long kept_stride, const void* table,
                               const void* bigram, int table_dtype, float* x, int T, int S, int H, int V, long long buckets,
                               long long mul_prev, long long mul_cur, hipStream_t stream) {
    TL_CHECK_ARG(T >= 0 && S >= 0 && H > 0 && V > 0 && buckets > 0 && kept_stride >= 1, "tl_embed_bigram: bad sizes T=%d H=%d V=%d", T, H, V);
    if (T == 0 || S == 0) return 0;
    dim3 grid(T), block(256);
    if (table_dtype == TL_F32)
        hipLaunchKernelGGL(embed_bigram_kernel<float>, grid, block, 0, stream, ids, pos, seq_of_token, q_start, state_slots,
                           prev_kept, kept_stride, (const float*)table, (const float*)bigram, x, H, V, buckets, mul_prev, mul_cur);
    else if (table_dtype == TL_BF16)
        hipLaunchKernelGGL(embed_bigram_kernel<bf16_t>, grid, block, 0, stream, ids, pos, seq_of_token, q_start, state_slots,
                           prev_kept, kept_stride, (const bf16_t*)table, (const bf16_t*)bigram, x, H, V, buckets, mul_prev, mul_cur);
    else
        return tl_fail("tl_embed_bigram: unknown dtype %d", table_dtype);
    TL_CHECK_LAUNCH("tl_embed_bigram");
    hipLaunchKernelGGL(keep_last_token_kernel, dim3(tl_ceil_div(S, 256)), dim3(256), 0, stream, ids, q_start, state_slots,
                       prev_kept, kept_stride, S);
    TL_CHECK_LAUNCH("tl_embed_bigram keep");
    return 0;
}

// ---- residual add + RMSNorm ----------------------------------------------------------------
// Without `rows`: x[r] += residual[r] (written back, float), out[r] = x[r] * rstd * w.
// With `rows`:    out[r] = norm(x[rows[r]] + residual[rows[r]]); x is left as it is.
// The residual may come in `parts` slices `pstride` elements apart (the K shares of a product):
// it is then their sum in ascending order, formed first and added to x as one number.
// The sum, the mean of squares and the scaling are float (reference: tensorline/fused.py:19-32).
template <typename R, typename O, bool HAS_RES, bool HAS_ROWS>
__global__ void add_rmsnorm_kernel(float* __restrict__ x, const R* __restrict__ res, const float* __restrict__ w,
                                   O* __restrict__ out, const int32_t* __restrict__ rows, int H, float eps, int parts,
                                   size_t pstride) {
    __shared__ float red[16];
    const int r = blockIdx.x;
    const size_t src = HAS_ROWS ? (size_t)rows[r] : (size_t)r;
    float* xr = x + src * H;
    const R* rr = HAS_RES ? res + src * H : nullptr;
    O* orow = out + (size_t)r * H;

    float ss = 0.f;
    for (int c = threadIdx.x; c < H; c += blockDim.x) {
        float v = xr[c];
        if (HAS_RES) {
            float b = tl_to_float(rr[c]);
            for (int p = 1; p < parts; ++p) b += tl_to_float(rr[c + p * pstride]);
            v += b;
            if (!HAS_ROWS) xr[c] = v;
        }
        ss += v * v;
    }
    ss = tl_block_sum(ss, red);
    const float rstd = 1.0f / sqrtf(ss / (float)H + eps);
    for (int c = threadIdx.x; c < H; c += blockDim.x) {
        float v = xr[c];
        if (HAS_RES && HAS_ROWS) {
            float b = tl_to_float(rr[c]);
            for (int p = 1; p < parts; ++p) b += tl_to_float(rr[c + p * pstride]);
            v += b;
        }
        orow[c] = tl_from_float<O>(v * rstd * w[c]);
    }
}

// The same for H a multiple of 4 and at most 16384: one pass, 16-byte accesses, the row kept in
// registers between the sum of squares and the scaling.
__device__ __forceinline__ float4 tl_load4(const float* p) { return *reinterpret_cast<const float4*>(p); }
__device__ __forceinline__ float4 tl_load4(const bf16_t* p) {
    const uint2 u = *reinterpret_cast<const uint2*>(p);
    return make_float4(__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xffff0000u), __uint_as_float(u.y << 16),
                       __uint_as_float(u.y & 0xffff0000u));
}
__device__ __forceinline__ void tl_store4(float* p, float4 v) { *reinterpret_cast<float4*>(p) = v; }
__device__ __forceinline__ void tl_store4(bf16_t* p, float4 v) {
    uint2 u;
    u.x = tl_pack_bf16(v.x, v.y);
    u.y = tl_pack_bf16(v.z, v.w);
    *reinterpret_cast<uint2*>(p) = u;
}

#define NORM_VPT 4   // float4 per thread at most
template <typename R, typename O, bool HAS_RES, bool HAS_ROWS>
__global__ __launch_bounds__(1024) void add_rmsnorm_vec_kernel(float* __restrict__ x, const R* __restrict__ res,
                                                               const float* __restrict__ w, O* __restrict__ out,
                                                               const int32_t* __restrict__ rows, int H, float eps,
                                                               int parts, size_t pstride) {
    __shared__ float red[16];
    const int r = blockIdx.x;
    const size_t src = HAS_ROWS ? (size_t)rows[r] : (size_t)r;
    float* xr = x + src * H;
    const R* rr = HAS_RES ? res + src * H : nullptr;
    O* orow = out + (size_t)r * H;
    const int n4 = H >> 2;
    float4 v[NORM_VPT], gw[NORM_VPT];
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < NORM_VPT; ++i) {
        const int c4 = threadIdx.x + i * blockDim.x;
        if (c4 < n4) {
            float4 a = tl_load4(xr + 4 * c4);
            gw[i] = tl_load4(w + 4 * c4);                    // used at the end
            if (HAS_RES) {
                float4 b = tl_load4(rr + 4 * c4);
                for (int p = 1; p < parts; p += 4) {         // four shares are asked for before they are added
                    float4 e[4];
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                        if (p + k < parts) e[k] = tl_load4(rr + 4 * c4 + (p + k) * pstride);
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                        if (p + k < parts) b.x += e[k].x, b.y += e[k].y, b.z += e[k].z, b.w += e[k].w;
                }
                a.x += b.x;
                a.y += b.y;
                a.z += b.z;
                a.w += b.w;
                if (!HAS_ROWS) tl_store4(xr + 4 * c4, a);
            }
            v[i] = a;
            ss += a.x * a.x;
            ss += a.y * a.y;
            ss += a.z * a.z;
            ss += a.w * a.w;
        }
    }
    ss = tl_block_sum(ss, red);
    const float rstd = 1.0f / sqrtf(ss / (float)H + eps);
#pragma unroll
    for (int i = 0; i < NORM_VPT; ++i) {
        const int c4 = threadIdx.x + i * blockDim.x;
        if (c4 < n4) {
            float4 o;
            o.x = v[i].x * rstd * gw[i].x;
            o.y = v[i].y * rstd * gw[i].y;
            o.z = v[i].z * rstd * gw[i].z;
            o.w = v[i].w * rstd * gw[i].w;
            tl_store4(orow + 4 * c4, o);
        }
    }
}

// ---- a normed branch added to the stream, and the next norm -------------------------------------
// A residual branch whose output y is RMS-normed before it joins the stream:
//   x[r] += mult * y[r] / sqrt(mean(y[r]^2) + eps_b) * wb
// and, with w, the norm that reads the stream next, out[r] = x[r] / sqrt(mean(x[r]^2) + eps) * w, in the
// same pass.  With `rows`: out only, for x[rows[r]] and y[rows[r]]; x is left as it is.  Float sums.
template <typename O, bool HAS_ROWS>
__global__ __launch_bounds__(1024) void branch_norm_add_kernel(float* __restrict__ x, const float* __restrict__ y,
                                                               const float* __restrict__ wb, float mult, float eps_b,
                                                               const float* __restrict__ w, float eps, O* __restrict__ out,
                                                               const int32_t* __restrict__ rows, int H) {
    __shared__ float red[16];
    const int r = blockIdx.x;
    const size_t src = HAS_ROWS ? (size_t)rows[r] : (size_t)r;
    float* xr = x + src * H;
    const float* yr = y + src * H;
    float ss = 0.f;
    for (int c = threadIdx.x; c < H; c += blockDim.x) ss += yr[c] * yr[c];
    ss = tl_block_sum(ss, red);
    const float f = mult / sqrtf(ss / (float)H + eps_b);
    float sx = 0.f;
    for (int c = threadIdx.x; c < H; c += blockDim.x) {
        const float v = xr[c] + yr[c] * f * wb[c];
        if (!HAS_ROWS) xr[c] = v;
        sx += v * v;
    }
    if (!w) return;
    sx = tl_block_sum(sx, red);
    const float rstd = 1.0f / sqrtf(sx / (float)H + eps);
    O* orow = out + (size_t)r * H;
    for (int c = threadIdx.x; c < H; c += blockDim.x) {
        const float v = HAS_ROWS ? xr[c] + yr[c] * f * wb[c] : xr[c];
        orow[c] = tl_from_float<O>(v * rstd * w[c]);
    }
}

// The same for H a multiple of 4 and at most 16384: one pass over memory, 16-byte accesses, the rows of y and of
// the new x kept in registers between the sums and the scalings.
template <typename O, bool HAS_ROWS>
__global__ __launch_bounds__(1024) void branch_norm_add_vec_kernel(float* __restrict__ x, const float* __restrict__ y,
                                                                   const float* __restrict__ wb, float mult, float eps_b,
                                                                   const float* __restrict__ w, float eps, O* __restrict__ out,
                                                                   const int32_t* __restrict__ rows, int H) {
    __shared__ float red[16];
    const int r = blockIdx.x;
    const size_t src = HAS_ROWS ? (size_t)rows[r] : (size_t)r;
    float* xr = x + src * H;
    const float* yr = y + src * H;
    const int n4 = H >> 2;
    float4 v[NORM_VPT];
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < NORM_VPT; ++i) {
        const int c4 = threadIdx.x + i * blockDim.x;
        if (c4 < n4) {
            v[i] = tl_load4(yr + 4 * c4);
            ss += v[i].x * v[i].x;
            ss += v[i].y * v[i].y;
            ss += v[i].z * v[i].z;
            ss += v[i].w * v[i].w;
        }
    }
    ss = tl_block_sum(ss, red);
    const float f = mult / sqrtf(ss / (float)H + eps_b);
    float sx = 0.f;
#pragma unroll
    for (int i = 0; i < NORM_VPT; ++i) {
        const int c4 = threadIdx.x + i * blockDim.x;
        if (c4 < n4) {
            const float4 a = tl_load4(xr + 4 * c4), g = tl_load4(wb + 4 * c4);
            float4 n;
            n.x = a.x + v[i].x * f * g.x;
            n.y = a.y + v[i].y * f * g.y;
            n.z = a.z + v[i].z * f * g.z;
            n.w = a.w + v[i].w * f * g.w;
            if (!HAS_ROWS) tl_store4(xr + 4 * c4, n);
            v[i] = n;
            sx += n.x * n.x;
            sx += n.y * n.y;
            sx += n.z * n.z;
            sx += n.w * n.w;
        }
    }
    if (!w) return;
    sx = tl_block_sum(sx, red);
    const float rstd = 1.0f / sqrtf(sx / (float)H + eps);
    O* orow = out + (size_t)r * H;
#pragma unroll
    for (int i = 0; i < NORM_VPT; ++i) {
        const int c4 = threadIdx.x + i * blockDim.x;
        if (c4 < n4) {
            const float4 g = tl_load4(w + 4 * c4);
            float4 o;
            o.x = v[i].x * rstd * g.x;
            o.y = v[i].y * rstd * g.y;
            o.z = v[i].z * rstd * g.z;
            o.w = v[i].w * rstd * g.w;
            tl_store4(orow + 4 * c4, o);
        }
    }
}

extern "C" int tl_branch_norm_add(float* x, const float* y, const float* wb, float mult, float eps_b, const float* w, float eps,
                                  void* out, int out_dtype, const int32_t* rows, int n_rows, int H, hipStream_t stream) {
    TL_CHECK_ARG(n_rows >= 0 && H > 0 && eps >= 0.f && eps_b >= 0.f, "tl_branch_norm_add: bad sizes rows=%d H=%d", n_rows, H);
    TL_CHECK_ARG((w == nullptr) == (out == nullptr) && (rows == nullptr || w != nullptr), "tl_branch_norm_add: a norm needs its output, and rows a norm");
    if (n_rows == 0) return 0;
    const bool vec = H % 4 == 0 && H <= 1024 * 4 * NORM_VPT;
    int threads = (((vec ? H / 4 : H) + 63) / 64) * 64;
    if (threads > 1024) threads = 1024;
    dim3 grid(n_rows), block(threads);
#define TL_BRANCH_VEC(OT)                                                                                                            \
    do {                                                                                                                             \
        if (rows)                                                                                                                    \
            hipLaunchKernelGGL((branch_norm_add_vec_kernel<OT, true>), grid, block, 0, stream, x, y, wb, mult, eps_b, w, eps, (OT*)out, \
                               rows, H);                                                                                             \
        else                                                                                                                         \
            hipLaunchKernelGGL((branch_norm_add_vec_kernel<OT, false>), grid, block, 0, stream, x, y, wb, mult, eps_b, w, eps,          \
                               (OT*)out, rows, H);                                                                                   \
    } while (0)
    if (vec && (out_dtype == TL_BF16 || out_dtype == TL_F32)) {
        if (out_dtype == TL_BF16) TL_BRANCH_VEC(bf16_t);
        else TL_BRANCH_VEC(float);
        TL_CHECK_LAUNCH("tl_branch_norm_add");
        return 0;
    }
#undef TL_BRANCH_VEC
#define TL_BRANCH_CASE(OT)                                                                                                       \
    do {                                                                                                                         \
        if (rows)                                                                                                                \
            hipLaunchKernelGGL((branch_norm_add_kernel<OT, true>), grid, block, 0, stream, x, y, wb, mult, eps_b, w, eps, (OT*)out, \
                               rows, H);                                                                                         \
        else                                                                                                                     \
            hipLaunchKernelGGL((branch_norm_add_kernel<OT, false>), grid, block, 0, stream, x, y, wb, mult, eps_b, w, eps,          \
                               (OT*)out, rows, H);                                                                               \
    } while (0)
    if (out_dtype == TL_BF16) TL_BRANCH_CASE(bf16_t);
    else if (out_dtype == TL_F32) TL_BRANCH_CASE(float);
    else return tl_fail("tl_branch_norm_add: unknown dtype %d", out_dtype);
#undef TL_BRANCH_CASE
    TL_CHECK_LAUNCH("tl_branch_norm_add");
    return 0;
}

template <typename R, typename O>
static void launch_add_rmsnorm(float* x, const R* res, const float* w, O* out, const int32_t* rows, int n_rows,
                               int H, float eps, int parts, size_t pstride, hipStream_t stream) {
    if (H % 4 == 0 && H <= 1024 * 4 * NORM_VPT && pstride % 4 == 0) {
        int threads = ((H / 4 + 63) / 64) * 64;
        if (threads > 1024) threads = 1024;
        dim3 grid(n_rows), block(threads);
        if (res && rows)
            hipLaunchKernelGGL((add_rmsnorm_vec_kernel<R, O, true, true>), grid, block, 0, stream, x, res, w, out, rows, H, eps, parts, pstride);
        else if (res)
            hipLaunchKernelGGL((add_rmsnorm_vec_kernel<R, O, true, false>), grid, block, 0, stream, x, res, w, out, rows, H, eps, parts, pstride);
        else if (rows)
            hipLaunchKernelGGL((add_rmsnorm_vec_kernel<R, O, false, true>), grid, block, 0, stream, x, res, w, out, rows, H, eps, parts, pstride);
        else
            hipLaunchKernelGGL((add_rmsnorm_vec_kernel<R, O, false, false>), grid, block, 0, stream, x, res, w, out, rows, H, eps, parts, pstride);
        return;
    }
    dim3 grid(n_rows), block(H >= 2048 ? 512 : 256);
    if (res && rows)
        hipLaunchKernelGGL((add_rmsnorm_kernel<R, O, true, true>), grid, block, 0, stream, x, res, w, out, rows, H, eps, parts, pstride);
    else if (res)
        hipLaunchKernelGGL((add_rmsnorm_kernel<R, O, true, false>), grid, block, 0, stream, x, res, w, out, rows, H, eps, parts, pstride);
    else if (rows)
        hipLaunchKernelGGL((add_rmsnorm_kernel<R, O, false, true>), grid, block, 0, stream, x, res, w, out, rows, H, eps, parts, pstride);
    else
        hipLaunchKernelGGL((add_rmsnorm_kernel<R, O, false, false>), grid, block, 0, stream, x, res, w, out, rows, H, eps, parts, pstride);
}

extern "C" int tl_add_rmsnorm(float* x, const void* residual, int res_dtype, int res_parts, long long res_part_stride,
                              const float* w, void* out, int out_dtype, const int32_t* rows, int n_rows, int H,
                              float eps, hipStream_t stream) {
    TL_CHECK_ARG(n_rows >= 0 && H > 0, "tl_add_rmsnorm: bad sizes rows=%d H=%d", n_rows, H);
    TL_CHECK_ARG(res_parts >= 1 && res_parts <= 64 && (res_parts == 1 || (residual && res_part_stride > 0)),
                 "tl_add_rmsnorm: bad residual parts %d (stride %lld)", res_parts, res_part_stride);
    TL_CHECK_ARG(eps >= 0.f, "tl_add_rmsnorm: eps must be >= 0");
    if (n_rows == 0) return 0;
    if (!residual) res_dtype = TL_F32;
#define TL_NORM_CASE(RD, RT, OD, OT)                                                                     \
    if (res_dtype == RD && out_dtype == OD) {                                                            \
        launch_add_rmsnorm<RT, OT>(x, (const RT*)residual, w, (OT*)out, rows, n_rows, H, eps, res_parts, \
                                   (size_t)res_part_stride, stream);                                     \
        TL_CHECK_LAUNCH("tl_add_rmsnorm");                                                               \
        return 0;                                                                                        \
    }
    TL_NORM_CASE(TL_F32, float, TL_F32, float)
    TL_NORM_CASE(TL_F32, float, TL_BF16, bf16_t)
    TL_NORM_CASE(TL_BF16, bf16_t, TL_F32, float)
    TL_NORM_CASE(TL_BF16, bf16_t, TL_BF16, bf16_t)
#undef TL_NORM_CASE
    return tl_fail("tl_add_rmsnorm: unknown dtypes residual=%d out=%d", res_dtype, out_dtype);
}

// ---- rotary position encoding + cache write ------------------------------------------------
// qkv: [T, (nq + 2 nkv) * d] as the fused projection leaves it.  Query heads are rotated in place;
// key heads are rotated and written to k_cache at the token's slot; value heads are copied to
// v_cache, which is transposed within a page so that the keys of one page are contiguous for each
// head dim (what the matrix cores want for the P*V product).  Rotate-half layout over the first
// `rot` dims of a head (reference: fused.py:34-51):
//   out[i]         = a*cos(theta_i) - b*sin(theta_i)       a = x[i], b = x[i + rot/2]
//   out[i + rot/2] = b*cos(theta_i) + a*sin(theta_i)       theta_i = pos * inv_freq[i]
// The angle, sine and cosine are float.  A negative slot skips the cache write of that token.
// k_cache is [pages, page, nkv, d] (addressed as [slot, nkv, d]); v_cache is [pages, nkv, d, page].
// One work-group a token.  In a step of a few hundred tokens it is a chain of waits (801 tokens of 12 + 2 + 2 heads of 128
// are 6.6 MB): a thread asks for its first pairs and their bias ahead of the angles, the waves that have no angle copy the values
// meanwhile, and a head's number is a multiplication by the reciprocal ceil(2^32 / pairs a head).
// bfloat16, 12 + 2 + 2 heads of 128, us: 160 tokens 4.0 -> 3.0, 801 tokens 5.5 -> 4.3; 28 + 4 + 4 heads, 2,048 tokens 12.5 -> 10.4 (3.6 TB/s);
// float32 8 tokens 5.0 -> 2.8.  A thread has one group of pairs wherever 1,024 threads are enough: with two the second was asked for
// behind the angles (float32, 2,048 tokens of 28 + 4 + 4 heads 20.8 against 19.4).
template <typename T>
__global__ __launch_bounds__(1024) void rope_store_kernel(T* __restrict__ qkv, const int32_t* __restrict__ pos,
                                                         const float* __restrict__ inv_freq, T* __restrict__ k_cache, T* __restrict__ v_cache,
                                                         const int32_t* __restrict__ slots, int nq, int nkv, int d, int rot, int write_kv,
                                                         int bs, const float* __restrict__ bias, int vec, uint32_t per_head_rcp, int values_last) {
    constexpr int V = 16 / sizeof(T);               // pairs to a thread where the sizes allow 16-byte accesses (vec)
    struct __attribute__((aligned(4))) Quad { float v[4]; };
    __shared__ __attribute__((aligned(16))) float cs_s[256], sn_s[256];          // one sine and cosine per rotated pair of the token
    const int t = blockIdx.x, half = rot / 2;
    T* row = qkv + (size_t)t * (nq + 2 * nkv) * d;
    const int nrot = nq + nkv;  // heads that are rotated: q then k
    const int per_head = vec ? half / V : half, items = nrot * per_head;
    const auto head_of = [&](int idx) {             // (the product with the rounded reciprocal is one too many at most)
        const uint32_t q = per_head_rcp ? __umulhi((uint32_t)idx, per_head_rcp) : (uint32_t)idx;
        return (int)(q - (q * (uint32_t)per_head > (uint32_t)idx));
    };
    uint4 lo, hi;
    Quad blo[V / 4], bhi[V / 4];
    const auto ask = [&](int h, int i) {
        const T* hp = row + (size_t)h * d + i;
        lo = *reinterpret_cast<const uint4*>(hp), hi = *reinterpret_cast<const uint4*>(hp + half);
        if (bias) {
#pragma unroll
            for (int k = 0; k < V / 4; ++k) {
                blo[k] = *reinterpret_cast<const Quad*>(bias + (size_t)h * d + i + 4 * k);
                bhi[k] = *reinterpret_cast<const Quad*>(bias + (size_t)h * d + i + half + 4 * k);
            }
        }
    };
    int h = 0, i = 0;
    if (vec) {
        const int idx = min((int)threadIdx.x, items - 1);
        h = head_of(idx), i = (idx - h * per_head) * V;
        ask(h, i);
    }
    const int slot = write_kv ? slots[t] : -1;
    const float p = (float)pos[t];
    const int busy = (half + 63) & ~63, spare = busy < (int)blockDim.x ? busy : 0;   // threads in waves with angles
    for (int k = threadIdx.x; k < half; k += blockDim.x) sincosf(p * inv_freq[k], &sn_s[k], &cs_s[k]);
    const auto values = [&](int from) {             // by the threads from `from` on
        const T* vrow = row + (size_t)nrot * d;
        const float* vbias = bias ? bias + (size_t)nrot * d : nullptr;
        const int page = slot / bs, off = slot - page * bs;
        T* vdst = v_cache + (size_t)page * nkv * d * bs + off;
        for (int idx = threadIdx.x - from; idx < nkv * d; idx += blockDim.x - from)
            vdst[(size_t)idx * bs] = vbias ? tl_from_float<T>(tl_to_float(vrow[idx]) + vbias[idx]) : vrow[idx];
    };
    if (!values_last && slot >= 0 && (int)threadIdx.x >= spare) values(spare);
    __syncthreads();
    if (vec) {
        for (int idx = threadIdx.x; idx < items; idx += blockDim.x) {
            if (idx != (int)threadIdx.x) h = head_of(idx), i = (idx - h * per_head) * V, ask(h, i);
            T* dst = h < nq ? row + (size_t)h * d : k_cache + ((size_t)slot * nkv + (h - nq)) * d;
            if (h >= nq && slot < 0) continue;
            float cs[V], sn[V], o1[V], o2[V];
#pragma unroll
            for (int k = 0; k < V; k += 4) {
                *reinterpret_cast<float4*>(cs + k) = *reinterpret_cast<const float4*>(cs_s + i + k);
                *reinterpret_cast<float4*>(sn + k) = *reinterpret_cast<const float4*>(sn_s + i + k);
            }
            const uint32_t lw[4] = {lo.x, lo.y, lo.z, lo.w}, hw[4] = {hi.x, hi.y, hi.z, hi.w};
#pragma unroll
            for (int k = 0; k < V; ++k) {
                float a, b;
                if constexpr (sizeof(T) == 2) {
                    a = __uint_as_float(k & 1 ? lw[k / 2] & 0xffff0000u : lw[k / 2] << 16);
                    b = __uint_as_float(k & 1 ? hw[k / 2] & 0xffff0000u : hw[k / 2] << 16);
                } else {
                    a = __uint_as_float(lw[k]), b = __uint_as_float(hw[k]);
                }
                if (bias) a += blo[k / 4].v[k % 4], b += bhi[k / 4].v[k % 4];
                o1[k] = a * cs[k] - b * sn[k];
                o2[k] = b * cs[k] + a * sn[k];
            }
            if constexpr (sizeof(T) == 2) {
                *reinterpret_cast<uint4*>(dst + i) =
                    make_uint4(tl_pack_bf16(o1[0], o1[1]), tl_pack_bf16(o1[2], o1[3]), tl_pack_bf16(o1[4], o1[5]), tl_pack_bf16(o1[6], o1[7]));
                *reinterpret_cast<uint4*>(dst + i + half) =
                    make_uint4(tl_pack_bf16(o2[0], o2[1]), tl_pack_bf16(o2[2], o2[3]), tl_pack_bf16(o2[4], o2[5]), tl_pack_bf16(o2[6], o2[7]));
            } else {
                *reinterpret_cast<float4*>(dst + i) = make_float4(o1[0], o1[1], o1[2], o1[3]);
                *reinterpret_cast<float4*>(dst + i + half) = make_float4(o2[0], o2[1], o2[2], o2[3]);
            }
        }
    } else
    for (int idx = threadIdx.x; idx < items; idx += blockDim.x) {
        const int h = head_of(idx), i = idx - h * half;
        const float sn = sn_s[i], cs = cs_s[i];
        T* hp = row + (size_t)h * d;
        float a = tl_to_float(hp[i]), b = tl_to_float(hp[i + half]);
        if (bias) {
            a += bias[h * d + i];
            b += bias[h * d + i + half];
        }
        const T o1 = tl_from_float<T>(a * cs - b * sn);
        const T o2 = tl_from_float<T>(b * cs + a * sn);
        if (h < nq) {
            hp[i] = o1;
            hp[i + half] = o2;
        } else if (slot >= 0) {
            T* kp = k_cache + ((size_t)slot * nkv + (h - nq)) * d;
            kp[i] = o1;
            kp[i + half] = o2;
        }
    }
    // dims beyond the rotated part pass through: query dims only change when a bias is owed
    const int tail = d - rot;
    if (tail && bias) {
        for (int idx = threadIdx.x; idx < nq * tail; idx += blockDim.x) {
            const int h = idx / tail, i = rot + (idx - h * tail);
            row[(size_t)h * d + i] = tl_from_float<T>(tl_to_float(row[(size_t)h * d + i]) + bias[h * d + i]);
        }
    }
    if (slot < 0) return;
    for (int idx = threadIdx.x; idx < nkv * tail; idx += blockDim.x) {
        const int h = idx / tail, i = rot + (idx - h * tail);
        const T v = row[(size_t)(nq + h) * d + i];
        k_cache[((size_t)slot * nkv + h) * d + i] = bias ? tl_from_float<T>(tl_to_float(v) + bias[(nq + h) * d + i]) : v;
    }
    if (values_last) values(0);
}

extern "C" int tl_rope_store(void* qkv, int dtype, const int32_t* pos, const float* inv_freq, void* k_cache,
                             void* v_cache, const int32_t* slots, int T, int nq, int nkv, int d, int rot,
                             int write_kv, int bs, const float* bias, hipStream_t stream) {
    TL_CHECK_ARG(T >= 0 && nq > 0 && nkv >= 0 && d > 0, "tl_rope_store: bad sizes T=%d nq=%d nkv=%d d=%d", T, nq, nkv, d);
    TL_CHECK_ARG(rot >= 0 && rot <= d && rot % 2 == 0, "tl_rope_store: rotary width %d must be even and <= head size %d", rot, d);
    TL_CHECK_ARG(rot <= 512, "tl_rope_store: rotary width %d is above the supported 512", rot);
    TL_CHECK_ARG(!write_kv || (k_cache && v_cache && slots && bs > 0), "tl_rope_store: cache write asked for without a cache");
    if (T == 0) return 0;
    dim3 grid(T);
    // 16-byte accesses: every head and both halves of the rotated part start at a multiple of 8 (float: 4) values
    const int V = dtype == TL_BF16 ? 8 : 4;
    const int vec = d % V == 0 && rot % (2 * V) == 0 && rot > 0 && ((uintptr_t)qkv % 16) == 0 &&
                    (!write_kv || ((uintptr_t)k_cache % 16) == 0);
    const int per_head = rot ? (vec ? rot / 2 / V : rot / 2) : 1;
    const uint32_t rcp = (uint32_t)(((1ull << 32) + per_head - 1) / per_head);      // 0: one a head
    const int items = (nq + nkv) * per_head;
    // One item a thread: the first is asked for ahead.  Steps of many tokens hide a work-group's waits behind the others and are bound by
    // memory, where small work-groups, or values behind the keys, are better (us, as for few tokens and as here):
    // - bfloat16 pairs one by one: 32 + 32 + 32 heads of 24, 700, 2,048, 4,000 tokens 7.1, 13.9, 23.7 and 6.6, 11.6, 18.8 (but 500 5.6 and 6.1);
    // - values last, float32 28 + 4 + 4 heads of 128, 2,048 tokens 20.2 and 18.8 (12 + 2 + 2, 17 MB, 9.2 and 9.7), bfloat16 with half of 128 rotated,
    //   32 + 8 + 8 heads 15.3 and 14.8; fully rotated bfloat16 loses (12 + 2 + 2, 4,000 tokens 9.7 and 10.7);
    // - without rotation there is less to hide: float32, 14 + 2 + 2 heads of 256, 631 tokens 11.0 and 9.8, 8 + 8 + 8 of 64, 1,500 tokens (9 MB) 9.9 and 10.1.
    const double bytes = (double)T * (nq + 2 * nkv) * d * (dtype == TL_F32 ? 4 : 2);
    const int values_last = bytes >= (rot ? 24e6 : 10e6) && (vec || !rot) && (dtype == TL_F32 || rot < d);
    const bool small = vec ? values_last && dtype == TL_F32 && items % 256 == 0 && items <= 512 : dtype == TL_BF16 && T > 512;
    const dim3 block(small || items <= 256 ? 256 : items <= 512 ? 512 : 1024);
    if (dtype == TL_F32)
        hipLaunchKernelGGL(rope_store_kernel<float>, grid, block, 0, stream, (float*)qkv, pos, inv_freq,
                           (float*)k_cache, (float*)v_cache, slots, nq, nkv, d, rot, write_kv, bs, bias, vec, rcp, values_last);
    else if (dtype == TL_BF16)
        hipLaunchKernelGGL(rope_store_kernel<bf16_t>, grid, block, 0, stream, (bf16_t*)qkv, pos, inv_freq,
                           (bf16_t*)k_cache, (bf16_t*)v_cache, slots, nq, nkv, d, rot, write_kv, bs, bias, vec, rcp, values_last);
    else
        return tl_fail("tl_rope_store: unknown dtype %d", dtype);
    TL_CHECK_LAUNCH("tl_rope_store");
    return 0;
}

// ---- SiLU(gate) * up ------------------------------------------------------------------------
// gu: [T, 2 I] with the gate in the first I columns and the up projection in the last I.
template <typename T>
__global__ void silu_mul_kernel(const T* __restrict__ gu, T* __restrict__ out, int I) {
    const int t = blockIdx.y;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= I) return;
    const T* row = gu + (size_t)t * 2 * I;
    const float g = tl_to_float(row[i]), u = tl_to_float(row[I + i]);
    out[(size_t)t * I + i] = tl_from_float<T>(g / (1.0f + expf(-g)) * u);
}

// 16 bytes of gate and of up per thread (I a multiple of 8 bfloat16 or 4 floats).  Bound by memory once the gates of a wave of middling
// numbers take half the instructions: 2,048 x 18,944, us, bfloat16 38.4 -> 36.7, float32 98 -> 79.5 (5.9 TB/s; by 4 bytes before).
template <typename T>
__global__ void silu_mul_vec_kernel(const T* __restrict__ gu, T* __restrict__ out, int I) {
    constexpr int V = 16 / sizeof(T);
    const int t = blockIdx.y;
    const int i = (blockIdx.x * blockDim.x + threadIdx.x) * V;
    if (i >= I) return;
    const T* row = gu + (size_t)t * 2 * I + i;
    const uint4 gv = *reinterpret_cast<const uint4*>(row), uv = *reinterpret_cast<const uint4*>(row + I);
    const uint32_t gw[4] = {gv.x, gv.y, gv.z, gv.w}, uw[4] = {uv.x, uv.y, uv.z, uv.w};
    float g[V], u[V];
    TlMagnitudes size;
#pragma unroll
    for (int k = 0; k < V; ++k) {
        if constexpr (sizeof(T) == 2) {
            g[k] = __uint_as_float(k & 1 ? gw[k / 2] & 0xffff0000u : gw[k / 2] << 16);
            u[k] = __uint_as_float(k & 1 ? uw[k / 2] & 0xffff0000u : uw[k / 2] << 16);
        } else {
            g[k] = __uint_as_float(gw[k]), u[k] = __uint_as_float(uw[k]);
        }
        size.take(g[k]);
    }
    if (size.mid_silu()) {
#pragma unroll
        for (int k = 0; k < V; ++k) g[k] = tl_silu_mid(g[k]) * u[k];
    } else {
#pragma unroll
        for (int k = 0; k < V; ++k) g[k] = g[k] / (1.0f + expf(-g[k])) * u[k];
    }
    T* dst = out + (size_t)t * I + i;
    if constexpr (sizeof(T) == 2)
        *reinterpret_cast<uint4*>(dst) = make_uint4(tl_pack_bf16(g[0], g[1]), tl_pack_bf16(g[2], g[3]), tl_pack_bf16(g[4], g[5]), tl_pack_bf16(g[6], g[7]));
    else
        *reinterpret_cast<float4*>(dst) = make_float4(g[0], g[1], g[2], g[3]);
}

// The two forms of the gates (common.h) over the floats whose bits are first, first + 1, ..: counts[0] and [1] take how many have another SiLU
// and another 1 / (1 + e^-x), [2] and [3] how many were of middling size for each.  For tests.
__global__ __launch_bounds__(256) void gate_forms_kernel(uint32_t first, uint64_t n, uint32_t* __restrict__ counts) {
    uint32_t silu = 0, sigmoid = 0, mid_silu = 0, mid_sigmoid = 0;
    for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (uint64_t)gridDim.x * 256) {
        const float v = __uint_as_float(first + (uint32_t)i);
        TlMagnitudes size;
        size.take(v);
        if (!size.beyond_silu()) ++mid_silu, silu += __float_as_uint(tl_silu_mid(v)) != __float_as_uint(v / (1.0f + expf(-v)));
        if (!size.beyond_sigmoid()) ++mid_sigmoid, sigmoid += __float_as_uint(tl_sigmoid_mid(v)) != __float_as_uint(1.0f / (1.0f + expf(-v)));
    }
    if (silu) atomicAdd(counts, silu);
    if (sigmoid) atomicAdd(counts + 1, sigmoid);
    if (mid_silu) atomicAdd(counts + 2, mid_silu);
    if (mid_sigmoid) atomicAdd(counts + 3, mid_sigmoid);
}

extern "C" int tl_gate_forms_differ(uint32_t first, long long n, uint32_t* counts, hipStream_t stream) {
    TL_CHECK_ARG(n > 0 && n <= 1ll << 32 && counts, "tl_gate_forms_differ: bad range of %lld floats", n);
    const long long blocks = (n + 255) / 256;
    hipLaunchKernelGGL(gate_forms_kernel, dim3((unsigned)(blocks < 8192 ? blocks : 8192)), dim3(256), 0, stream, first, (uint64_t)n, counts);
    TL_CHECK_LAUNCH("tl_gate_forms_differ");
    return 0;
}

extern "C" int tl_silu_mul(const void* gu, void* out, int dtype, int T, int I, hipStream_t stream) {
    TL_CHECK_ARG(T >= 0 && I > 0, "tl_silu_mul: bad sizes T=%d I=%d", T, I);
    TL_CHECK_ARG(T <= 65535 * 64, "tl_silu_mul: too many rows %d", T);
    if (T == 0) return 0;
    // grid.y is limited to 65535: rows beyond that are covered by repeated launches.
    for (int t0 = 0; t0 < T; t0 += 65535) {
        const int tn = (T - t0 < 65535) ? T - t0 : 65535;
        dim3 grid(tl_ceil_div(I, 256), tn), block(256);
        const int V = dtype == TL_BF16 ? 8 : 4;
        if (I % V == 0 && ((uintptr_t)gu % 16) == 0 && ((uintptr_t)out % 16) == 0 && (dtype == TL_BF16 || dtype == TL_F32)) {
            const dim3 vgrid(tl_ceil_div(I / V, 256), tn);
            if (dtype == TL_BF16)
                hipLaunchKernelGGL(silu_mul_vec_kernel<bf16_t>, vgrid, block, 0, stream, (const bf16_t*)gu + (size_t)t0 * 2 * I, (bf16_t*)out + (size_t)t0 * I, I);
            else
                hipLaunchKernelGGL(silu_mul_vec_kernel<float>, vgrid, block, 0, stream, (const float*)gu + (size_t)t0 * 2 * I, (float*)out + (size_t)t0 * I, I);
            continue;
        }
        if (dtype == TL_F32)
            hipLaunchKernelGGL(silu_mul_kernel<float>, grid, block, 0, stream, (const float*)gu + (size_t)t0 * 2 * I,
                               (float*)out + (size_t)t0 * I, I);
        else if (dtype == TL_BF16)
            hipLaunchKernelGGL(silu_mul_kernel<bf16_t>, grid, block, 0, stream, (const bf16_t*)gu + (size_t)t0 * 2 * I,
                               (bf16_t*)out + (size_t)t0 * I, I);
        else
            return tl_fail("tl_silu_mul: unknown dtype %d", dtype);
    }
    TL_CHECK_LAUNCH("tl_silu_mul");
    return 0;
}
