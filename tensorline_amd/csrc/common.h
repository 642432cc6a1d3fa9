// Shared device helpers for the gfx950 kernels: storage types, wave and block reductions,
// error reporting of the C entry points.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#define TL_WAVE 64

// ---- storage types -------------------------------------------------------------------------
// bfloat16 is handled as raw 16 bits; conversion is a shift one way and round-to-nearest-even
// the other.  All arithmetic is done in float.
struct bf16_t {
    uint16_t bits;
};

__device__ __forceinline__ float tl_to_float(float v) { return v; }
__device__ __forceinline__ float tl_to_float(bf16_t v) { return __uint_as_float(((uint32_t)v.bits) << 16); }

// round to nearest even by the conversion instruction: for every one of the 2^32 floats, NaN included, the bits that adding 0x7fff and
// the last kept bit gives, in one instruction for two of them where that takes a dozen
__device__ __forceinline__ uint16_t tl_f2bf_bits(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }
__device__ __forceinline__ uint32_t tl_pack_bf16(float lo, float hi) {
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{lo, hi}), bf16x2));
}

// 16 bytes that are read once and not again soon (the weights of a decode step's products): a
// non-temporal load.  Such data then does not displace what the caches hold for reuse, and the long
// products of a decode step stream 5 to 10% faster (lm_head of a 7B model at 8 rows: 195 -> 176 us,
// 6.2 TB/s).  Decode attention gains nothing from it for its keys and values (batch 64) or loses
// (batch 8: 16.4 -> 17.6 us per layer) and reads them with plain loads.
typedef unsigned tl_u32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ uint4 tl_load_stream(const uint4* p) {
    return __builtin_bit_cast(uint4, __builtin_nontemporal_load(reinterpret_cast<const tl_u32x4*>(p)));
}

template <typename T> __device__ __forceinline__ T tl_from_float(float v);
template <> __device__ __forceinline__ float tl_from_float<float>(float v) { return v; }
template <> __device__ __forceinline__ bf16_t tl_from_float<bf16_t>(float v) {
    bf16_t r;
    r.bits = tl_f2bf_bits(v);
    return r;
}

// the sum over the lanes up to and with the lane's own
__device__ __forceinline__ int tl_wave_scan(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);       // within rows of 16: from 1, 2, 4, 8 lanes below
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);      // rows 1 and 3: the last lane of the row below
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);      // the upper half: lane 31
    return v;
}

// ---- reductions ----------------------------------------------------------------------------
// Over a wave with all its lanes active, lane i with lane i ^ 32, then ^ 16, ^ 8, ^ 4, ^ 2, ^ 1, without trips through LDS: the halves of 32 and 16
// lanes by register swaps, the rest by rotations within a row of 16 (after the step of 8 the values repeat every 8 lanes, so the
// lane 4 further holds what lane ^ 4 holds, and so on).  Six shuffles in a row take a wave 0.3 us, these 0.05.
typedef unsigned int tl_u32x2 __attribute__((ext_vector_type(2)));
template <typename Op>
__device__ __forceinline__ float tl_row_all(float v, Op op) {
#define TL_ROTATED(N) __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x120 + N, 0xf, 0xf, true))
    v = op(v, TL_ROTATED(8));
    v = op(v, TL_ROTATED(4));
    v = op(v, TL_ROTATED(2));
    v = op(v, TL_ROTATED(1));
#undef TL_ROTATED
    return v;
}
template <typename Op>
__device__ __forceinline__ float tl_wave_all(float v, Op op) {
    tl_u32x2 sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = op(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
    sw = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = op(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
    return tl_row_all(v, op);
}
__device__ __forceinline__ float tl_wave_sum(float v) {
    return tl_wave_all(v, [](float a, float b) { return a + b; });
}

__device__ __forceinline__ float tl_row_sum(float v) {       // of 16 lanes
    return tl_row_all(v, [](float a, float b) { return a + b; });
}

__device__ __forceinline__ float tl_wave_max(float v) {
    return tl_wave_all(v, [](float a, float b) { return fmaxf(a, b); });
}

// The sum over aligned groups of 2^log2 lanes, lane i with i ^ 1, then ^ 2, ^ 4, ..: within a row of 16 by permutations of quads and mirrors (after
// the step of 2 a quad holds one value, so the mirror within eight lanes brings what lane ^ 4 holds, and so on).
__device__ __forceinline__ float tl_group_sum(float v, int log2) {
#define TL_MOVED(CTRL) __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true))
    if (log2 > 0) v += TL_MOVED(0xB1);                   // quad_perm 1, 0, 3, 2
    if (log2 > 1) v += TL_MOVED(0x4E);                   // quad_perm 2, 3, 0, 1
    if (log2 > 2) v += TL_MOVED(0x141);                  // row_half_mirror
    if (log2 > 3) v += TL_MOVED(0x140);                  // row_mirror
#undef TL_MOVED
    if (log2 > 4) {
        const tl_u32x2 sw = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
        v = __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
    }
    if (log2 > 5) {
        const tl_u32x2 sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
        v = __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
    }
    return v;
}

// Block-wide reductions for blocks of up to 1024 threads (16 waves).  `scratch` is LDS with room
// for 16 floats.  The value is returned to every thread; the combination order is fixed, so the
// result does not depend on timing.  Both end with a barrier, so `scratch` can be reused at once.
__device__ __forceinline__ float tl_block_sum(float v, float* scratch) {
    const int lane = threadIdx.x & (TL_WAVE - 1), wave = threadIdx.x / TL_WAVE;
    const int nwaves = (blockDim.x + TL_WAVE - 1) / TL_WAVE;
    v = tl_wave_sum(v);
    if (lane == 0) scratch[wave] = v;
    __syncthreads();
    float r = 0.f;
#pragma unroll
    for (int w0 = 0; w0 < 16; w0 += 4) {                 // four at a time are read before they are added
        if (w0 >= nwaves) break;
        const float s0 = scratch[w0], s1 = scratch[w0 + 1], s2 = scratch[w0 + 2], s3 = scratch[w0 + 3];
        r += s0;
        if (w0 + 1 < nwaves) r += s1;
        if (w0 + 2 < nwaves) r += s2;
        if (w0 + 3 < nwaves) r += s3;
    }
    __syncthreads();
    return r;
}

__device__ __forceinline__ float tl_block_max(float v, float* scratch) {
    const int lane = threadIdx.x & (TL_WAVE - 1), wave = threadIdx.x / TL_WAVE;
    const int nwaves = (blockDim.x + TL_WAVE - 1) / TL_WAVE;
    v = tl_wave_max(v);
    if (lane == 0) scratch[wave] = v;
    __syncthreads();
    float r = -INFINITY;
    for (int w = 0; w < nwaves; ++w) r = fmaxf(r, scratch[w]);
    __syncthreads();
    return r;
}

// What a matrix product does for the RMS norms around it (gemm_skinny.hip, gemm_rows64.hip);
// bfloat16 activations.  Passed by the caller as a pointer (null: nothing).
struct TlNormArgs {
    // owed normalisation of A's rows (null: none): ss_in [ss_n, ss_ld] holds ss_n partial sums per
    // row, row m in column m (a wave reads four partials of all rows from one stretch of memory)
    const float* ss_in;
    int ss_ld, ss_n;
    float dim, eps;            // result rows are scaled by 1/sqrt(sum / dim + eps)
    // residual add and next norm's input (MODE_PLAIN; null: none)
    float* resid;              // [M, resid_ld] float, updated in place
    int resid_ld;
    const float* next_weight;  // [N]
    bf16_t* a_out;             // [M, a_ld] = resid * next_weight
    int a_ld;
    float* ss_out;             // [work-groups, ss_out_ld]: a row gets its work-group's sums of resid^2, one per row of A
    int ss_out_ld;
    // activation of a plain product's output, after the bias (the few-row kernel; no sink with it):
    // 0 none, 1 the square of relu; 2, in the gated forms of both kernels only: the tanh form of GELU passes
    // the gate instead of SiLU
    int act;
};

// ---- which keys a token sees -------------------------------------------------------------------
// Beside the causal rule (key <= p) a token at position p sees the keys from lo(p) on, and the first
// `first` keys of its sequence wherever lo(p) lies:
//   window > 0: lo = p - window + 1 (itself and the window - 1 keys before it);
//   chunk > 0:  lo = the last multiple of chunk at or below p (positions count from the start of the
//               sequence, not from where a step begins);
//   both 0:     lo = 0.
// lo never decreases with p.  Where lo(p) <= first the two ranges touch and lo is given as 0, so that a
// gap between the kept first keys and lo exists exactly where lo > 0 and first > 0.
struct TlMask {
    int window, chunk, first;
};
__host__ __device__ __forceinline__ int tl_mask_lo(const TlMask& k, int p) {
    int lo = 0;
    if (k.window > 0 && p - k.window + 1 > lo) lo = p - k.window + 1;
    if (k.chunk > 0) {
        const int c = (p / k.chunk) * k.chunk;
        lo = c > lo ? c : lo;
    }
    return lo <= k.first ? 0 : lo;
}
// a key below lo is hidden unless it is one of the kept first keys
__device__ __forceinline__ bool tl_mask_hides(const TlMask& k, int key, int lo) { return key < lo && key >= k.first; }

// ---- v / (1 + e^-v) and 1 / (1 + e^-x) of numbers of middling size ---------------------------------
// expf and the division spend half their instructions on ends of the range that a product's results seldom reach (26 for the gate of SiLU where
// these take 14, and a tile's end has 64 of them a lane).  A wave asks TlMagnitudes for its values and takes these steps or expf and the
// division, so for |x| <= TL_MID (and a v of 2^-60 and more) both must give the same bits, or a row's would depend on its neighbours':
// tl_gate_forms_differ counts the floats of the range where they do not (none).  Hence the exponent's steps are those that expf has in
// ROCm's device library (ocml, open source) between its checks: x log2 e in two floats, the second by fused multiply-adds, the nearest
// whole number of it as an exponent, the rest by the instruction.  The quotient is that of the rounded reciprocal, corrected once by its
// remainder (P. Markstein, IBM Journal of Research and Development 34, 1990).
#define TL_MID 40.0f
__device__ __forceinline__ float tl_exp_mid(float x) {
    const float ph = x * 0x1.715476p+0f, e = __builtin_rintf(ph);
    const float pl = __builtin_fmaf(x, 0x1.4ae0bep-26f, __builtin_fmaf(x, 0x1.715476p+0f, -ph));
    return __builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f((ph - e) + pl), (int)e);
}
__device__ __forceinline__ float tl_silu_mid(float v) {
    const float d = 1.0f + tl_exp_mid(-v), r = __builtin_amdgcn_rcpf(d), q = v * r;
    return __builtin_fmaf(__builtin_fmaf(-d, q, v), r, q);
}
__device__ __forceinline__ float tl_sigmoid_mid(float x) {
    const float d = 1.0f + tl_exp_mid(-x), r = __builtin_amdgcn_rcpf(d);
    return __builtin_fmaf(__builtin_fmaf(-d, r, 1.0f), r, r);
}
// the least and largest magnitudes of a lane's values (as bits without the sign), and whether all of a wave's are of middling size
struct TlMagnitudes {
    uint32_t least = 0xffffffffu, most = 0;
    __device__ __forceinline__ void take(float v) {
        const uint32_t u = __float_as_uint(v) << 1;
        least = min(least, u), most = max(most, u);
    }
    __device__ __forceinline__ bool beyond_silu() const { return most > __float_as_uint(TL_MID) << 1 || least < __float_as_uint(0x1p-60f) << 1; }
    __device__ __forceinline__ bool beyond_sigmoid() const { return most > __float_as_uint(TL_MID) << 1; }
    __device__ __forceinline__ bool mid_silu() const { return !__any(beyond_silu()); }
    __device__ __forceinline__ bool mid_sigmoid() const { return !__any(beyond_sigmoid()); }
};

// ---- scores bent by a cap ------------------------------------------------------------------------
// cap * tanh(score / cap), in the units the caller keeps scores in: raw is the bare product of query and
// key, to_exp = 2 log2(e) * scale / cap turns it into the exponent of e^(2 score / cap) = 2^(raw to_exp), and
// cap_out is the cap in the caller's units (times log2 e where scores are exponents of two).  tanh(y) =
// 1 - 2 / (1 + e^(2 y)): one exponential and one reciprocal, exact limits at both ends (an infinite or zero
// exponential gives cap_out and -cap_out), an absolute error of the order of cap times the float's precision.
__device__ __forceinline__ float tl_capped(float raw, float to_exp, float cap_out) {
    const float e = __builtin_amdgcn_exp2f(raw * to_exp);
    return __builtin_fmaf(-2.0f * cap_out, __builtin_amdgcn_rcpf(1.0f + e), cap_out);
}

// ---- a bias by distance ----------------------------------------------------------------------------
// A learned number per query head and distance n = position of the query - position of the key, added to a score after
// scale and cap: table [nq, reach + 1], the last column for every distance of `reach` and more; null: none.
struct TlBias {
    const float* table;
    int reach;
};
__device__ __forceinline__ int tl_bias_at(int distance, int reach) {
    return distance < 0 ? 0 : distance < reach ? distance : reach;      // (a key ahead of the query is masked anyway)
}

// A score in the base-2 domain from the bare product of query and key.  MODE 0: raw * scale2; 1: capped (tl_capped, scale2
// its factor into the exponent, cap2 the cap in the base-2 domain); 2: capped where cap2 > 0, and `add` (in the base-2
// domain) on top.
template <int MODE>
__device__ __forceinline__ float tl_score2(float raw, float scale2, float cap2, float add) {
    if (MODE == 0) return raw * scale2;
    if (MODE == 1) return tl_capped(raw, scale2, cap2);
    if (cap2 > 0.f) {
        const float e = __builtin_amdgcn_exp2f(raw * scale2);
        return __builtin_fmaf(-2.0f * cap2, __builtin_amdgcn_rcpf(1.0f + e), cap2 + add);
    }
    return __builtin_fmaf(raw, scale2, add);
}

// 16 bytes per lane from memory straight into LDS at lds_base + 16 * lane (lds_base, an LDS address, is the same for the whole
// wave).  Written as assembly so that the compiler does not make every later LDS read wait for it: a kernel waits with
// s_waitcnt vmcnt where it needs the data.  M0 holds the LDS base for the instruction and is put back.
__device__ __forceinline__ void tl_load_to_lds(const void* g, uint32_t lds_base) {
    uint32_t saved;
    asm volatile(
        "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, off\n\ts_mov_b32 m0, %0"
        : "=&s"(saved)
        : "s"(lds_base), "v"(g)
        : "memory");
}
__device__ __forceinline__ uint32_t tl_lds_address(void* p) { return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)p; }

// ---- host side -----------------------------------------------------------------------------
// Every C entry point returns 0 on success.  On failure it returns a non-zero code and leaves a
// message that tl_last_error() hands out; nothing is launched in that case.
int tl_fail(const char* fmt, ...);

#define TL_CHECK_ARG(cond, ...)                  \
    do {                                         \
        if (!(cond)) return tl_fail(__VA_ARGS__); \
    } while (0)

#define TL_CHECK_LAUNCH(name)                                                              \
    do {                                                                                   \
        hipError_t e__ = hipGetLastError();                                                \
        if (e__ != hipSuccess) return tl_fail("%s: launch failed: %s", name, hipGetErrorString(e__)); \
    } while (0)

enum TlDtype { TL_F32 = 0, TL_BF16 = 1 };

static inline int tl_ceil_div(int a, int b) { return (a + b - 1) / b; }
