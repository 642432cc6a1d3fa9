// Float attention of steps with prompt portions (the 32-bit path's prefill): head sizes 64 and 128, pages of a power of two of at
// least four tokens, no cap and no bias.  Products on v_mfma_f32_32x32x16_bf16, every float as the exact sum of three bfloat16 numbers
// (8 + 8 + 8 significant bits, each the rest of the one before; Dekker, Numerische Mathematik 18, 1971).  Of the nine partial products of
// two floats six are taken, each exact, with sums in float; the three left out (second by third part, third by second and by third) are at most 2^-24 of the
// product they belong to.  Off 64 bits by 3.4e-7 in the 2-norm where the float instruction was by 4.5e-7 (2,048 tokens, 28 / 4 heads of 128).
//
// A work-group of four waves takes 128 columns, (token, query head) pairs of one sequence and key/value head in the order of the
// tokens, a wave 32 of them; keys go by tiles of 32 at absolute multiples of 32.  A tile's keys, then its values, go from the cache
// into registers ahead of their use, are split there, and are left in LDS in the order in which fragments are read (16 bytes a
// lane, lane after lane).  Scores are computed transposed, keys along the result's rows: a lane holds sixteen keys of one
// column, so the softmax crosses lanes once, and the weights are the second operand of the product with the values where they
// are, if the values' fragments have their keys in the same order, which the split sees to.
//
// A tile that holds infinities, NaN or numbers beyond 2^60, or none above 2^-40 but zeros, or of values one below 2^-110, goes to the float instruction
// (v_mfma_f32_32x32x2_f32) instead, from the cache, for the same result layout; so does a column whose query does, and its neighbours stay as they are.
// (Weights below 2^-110 of a column's largest so far keep fewer bits, off by 2^-134 of that one.)
// A column's bits do not depend on how its sequence is cut, then, unless a key or value behind its own position makes its tile such a one.
//
// What bounds it: a tile is a chain of some 4 us for a wave that has its SIMD to itself, 1.6 of them 96 matrix instructions, 0.9 some 430 vector
// instructions (the splits of keys, values and weights 260 of them), the rest waits for values, fragments and the two barriers, which a second
// work-group on the CU fills in part; and the longest walk of a fresh prompt.  us a layer, here and on v_mfma_f32_16x16x4_f32
// (attention_generic_kernel.h, 0.19 of whose peak that form reached): 2,048 tokens of 28 / 4 heads of 128 290 and 644, of 14 / 2 of 64 153
// and 243; 9 prompts of 21 to 157 tokens, 12 / 2 of 128, 28 and 38; 489 tokens behind 3,072 beside 24 decoded ones 560 and 785;
// 64 behind 3,000 380 and 504.  The last parts of the queries are in LDS for want of registers at a head size of 128 (all in registers: 320 us).
#pragma once
#include "attention_generic_kernel.h"

typedef __bf16 aft_bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 aft_bf16x2 __attribute__((ext_vector_type(2)));
typedef float aft_f32x2 __attribute__((ext_vector_type(2)));
typedef float aft_f32x16 __attribute__((ext_vector_type(16)));

#define AFT_WAVES 4
#define AFT_COLUMNS (32 * AFT_WAVES)
#define AFT_KT 32

// two floats as two bfloat16, rounded to nearest even, and what is left of each
__device__ __forceinline__ uint32_t aft_take(float& a, float& b) {
    const uint32_t p = __builtin_bit_cast(uint32_t, __builtin_convertvector((aft_f32x2{a, b}), aft_bf16x2));
    a -= __uint_as_float(p << 16);
    b -= __uint_as_float(p & 0xffff0000u);
    return p;
}
__device__ __forceinline__ uint32_t aft_rest(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((aft_f32x2{a, b}), aft_bf16x2));
}
__device__ __forceinline__ void aft_split(float (&x)[8], uint4 (&to)[3]) {
    to[0] = make_uint4(aft_take(x[0], x[1]), aft_take(x[2], x[3]), aft_take(x[4], x[5]), aft_take(x[6], x[7]));
    to[1] = make_uint4(aft_take(x[0], x[1]), aft_take(x[2], x[3]), aft_take(x[4], x[5]), aft_take(x[6], x[7]));
    to[2] = make_uint4(aft_rest(x[0], x[1]), aft_rest(x[2], x[3]), aft_rest(x[4], x[5]), aft_rest(x[6], x[7]));
}
// the sum of squares shows infinities, NaN and numbers past 2^60, and that those that are not zero are below 2^-40 (below 2^-75 it does not, but
// three parts hold numbers down to 2^-110, and keys below that give scores of nothing with any query that has parts)
__device__ __forceinline__ void aft_squares(const float (&x)[8], float& z) {
#pragma unroll
    for (int i = 0; i < 8; ++i) z = __builtin_fmaf(x[i], x[i], z);
}
__device__ __forceinline__ bool aft_odd(float z) { return __any(!(z < 0x1p120f)) || (__any(z > 0.f) && !__any(z >= 0x1p-80f)); }

// A value below 2^-110 that is not zero: a head dimension may have no others, and the third part no longer holds its last bits (up to 6e-3 of a
// value of 2^-126).  The smallest of twice a number's bits less one, in which zero comes last.
__device__ __forceinline__ void aft_least(const float (&x)[8], uint32_t& least) {
#pragma unroll
    for (int i = 0; i < 8; ++i) least = min(least, (__float_as_uint(x[i]) << 1) - 1u);
}
__device__ __forceinline__ bool aft_tiny(uint32_t least) { return __any(least < (__float_as_uint(0x1p-110f) << 1) - 1u); }

#define AFT_MUL(ACC, A_, B_) \
    ACC = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(aft_bf16x8, A_), __builtin_bit_cast(aft_bf16x8, B_), ACC, 0, 0, 0)

template <int D>
__global__ __launch_bounds__(AFT_WAVES * 64, 2) void attn_float_tile_kernel(
    const float* __restrict__ q, int q_stride, const float* __restrict__ k_cache, const float* __restrict__ v_cache,
    const int32_t* __restrict__ tables, int NB, const int32_t* __restrict__ q_start, const int32_t* __restrict__ pos,
    float* __restrict__ out, int out_stride, int tiles_per_seq, int nq, int nkv, int bs, int bs_shift, TlMask mask, float scale,
    const float* __restrict__ sinks, int vec) {
    constexpr int KS = D / 16, DB = D / 32;              // steps of 16 head dimensions, blocks of 32
    constexpr int KU = KS / AFT_WAVES, VU = 2 * DB / AFT_WAVES;      // units of a wave: a step of the keys, a block and 16 keys of the values
    __shared__ uint4 kparts[KS * 3 * 64], vparts[DB * 2 * 3 * 64];
    constexpr int QL = D == 128 ? KS - 1 : 0;            // steps whose queries' last parts lie in LDS: what registers do not hold
    __shared__ uint4 qparts[QL ? AFT_WAVES * QL * 64 : 1];
    __shared__ int odd_keys[AFT_WAVES], odd_values[AFT_WAVES], range[2][AFT_WAVES];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), h = lane >> 5;
    const int s = blockIdx.x / tiles_per_seq, ti = tiles_per_seq - 1 - (int)(blockIdx.x - s * tiles_per_seq);     // the longest walks first
    const int kvh = blockIdx.y, G = nq / nkv;
    const int t0 = q_start[s], columns = (q_start[s + 1] - t0) * G;
    if (ti * AFT_COLUMNS >= columns) return;
    const int32_t* table = tables + (size_t)s * NB;

    const int column = ti * AFT_COLUMNS + wave * 32 + (lane & 31);
    const bool real = column < columns;
    const int p = real ? pos[t0 + column / G] : 0x7fffffff, lo = real ? tl_mask_lo(mask, p) : 0;
    // the keys this wave's columns see, [w_lo, w_hi), and the work-group's
    auto wave_most = [&](int v) {
#pragma unroll
        for (int o = 32; o; o >>= 1) v = max(v, __shfl_xor(v, o));
        return __builtin_amdgcn_readfirstlane(v);
    };
    const int w_hi = wave_most(real ? p + 1 : 0), w_lo = -wave_most(real ? -lo : -0x7fffffff);
    const int p_least = -wave_most(-p), lo_most = wave_most(lo);
    if (lane == 0) range[0][wave] = w_hi, range[1][wave] = w_lo;
    const float sign = scale < 0.f ? -1.f : 1.f, to_exp = fabsf(scale) * 1.44269504088896340736f;

    uint4 qf[KS][3];
    bool odd_query;                                      // this lane's column
    {
        const float* qrow = q + (size_t)(t0 + (real ? column / G : 0)) * q_stride + (size_t)(kvh * G + (real ? column % G : 0)) * D + 8 * h;
        float z = 0.f;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            float x[8];
            if (vec) {
                const float4 a = *reinterpret_cast<const float4*>(qrow + 16 * ks), b = *reinterpret_cast<const float4*>(qrow + 16 * ks + 4);
                x[0] = a.x, x[1] = a.y, x[2] = a.z, x[3] = a.w, x[4] = b.x, x[5] = b.y, x[6] = b.z, x[7] = b.w;
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) x[e] = qrow[16 * ks + e];
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) x[e] = real ? x[e] * sign : 0.f;
            aft_squares(x, z);
            aft_split(x, qf[ks]);
            if (ks < QL) qparts[(wave * QL + ks) * 64 + lane] = qf[ks][2];
        }
        const tl_u32x2 sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(z), __float_as_uint(z), false, false);
        z = __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
        odd_query = !(z < 0x1p120f) || (z > 0.f && z < 0x1p-80f);
    }
    const bool odd_queries = __any(odd_query);
    __syncthreads();
    int k_hi = 0, k_lo = 0x7fffffff;
#pragma unroll
    for (int w = 0; w < AFT_WAVES; ++w) k_hi = max(k_hi, range[0][w]), k_lo = min(k_lo, range[1][w]);
    const int k_main = k_lo / AFT_KT * AFT_KT;
    int head_end = 0;                                    // the tiles of the kept first keys, where those do not touch the rest
    if (mask.first > 0 && k_main > 0) head_end = min((mask.first + AFT_KT - 1) / AFT_KT * AFT_KT, k_main);
    auto tile_after = [&](int k0) {
        const int n = k0 + AFT_KT;
        return n >= head_end && n < k_main ? k_main : n;
    };

    // Where this lane reads of a tile: a key's head dimensions (key lane % 32), and four keys of head dimension lane % 32 of a block twice,
    // keys 4 h and 8 + 4 h of a unit's sixteen.  Keys beyond the last one are that one again and zero once split.
    // Pages are looked up a tile before they are read from.
    auto last = [&](int key) { return min(key, k_hi - 1); };
    auto page_of = [&](int key) { return table[last(key) >> bs_shift]; };
    auto key_at = [&](int page, int k0) {
        return k_cache + ((size_t)page * bs + (last(k0 + (lane & 31)) & (bs - 1))) * nkv * D + (size_t)kvh * D + 8 * h;
    };
    auto value_key = [&](int k0, int x) { return k0 + 16 * ((wave * VU + x / 2) & 1) + 8 * (x & 1) + 4 * h; };       // piece x of this wave's
    auto value_at = [&](int page, int k0, int x) {
        return v_cache + (((size_t)page * nkv + kvh) * D + 32 * ((wave * VU + x / 2) >> 1) + (lane & 31)) * bs + (last(value_key(k0, x)) & (bs - 1) & ~3);
    };
    auto from_two = [](const float4& a, const float4& b, float (&x)[8]) {
        x[0] = a.x, x[1] = a.y, x[2] = a.z, x[3] = a.w, x[4] = b.x, x[5] = b.y, x[6] = b.z, x[7] = b.w;
    };
    aft_f32x16 o[DB];
    float m = -INFINITY, l = 0.f;
#pragma unroll
    for (int i = 0; i < DB; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[i][r] = 0.f;

    const int k_first = head_end > 0 ? 0 : k_main;
    float4 kreg[KU][2];
    int kpage = page_of(k_first + (lane & 31)), vpage[2 * VU];
#pragma unroll
    for (int x = 0; x < 2 * VU; ++x) vpage[x] = page_of(value_key(k_first, x));
    auto ask_keys = [&](int k0) {
        const float* kp = key_at(kpage, k0) + 16 * wave;
#pragma unroll
        for (int u = 0; u < KU; ++u) {
            kreg[u][0] = *reinterpret_cast<const float4*>(kp + 16 * AFT_WAVES * u);
            kreg[u][1] = *reinterpret_cast<const float4*>(kp + 16 * AFT_WAVES * u + 4);
        }
    };
    ask_keys(k_first);
    kpage = page_of(tile_after(k_first) + (lane & 31));
    for (int k0 = k_first; k0 < k_hi; k0 = tile_after(k0)) {
        const int next = tile_after(k0);
        {
            float z = 0.f;
#pragma unroll
            for (int u = 0; u < KU; ++u) {
                float x[8];
                from_two(kreg[u][0], kreg[u][1], x);
                if (k0 + AFT_KT > k_hi) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) x[e] = k0 + (lane & 31) < k_hi ? x[e] : 0.f;
                }
                aft_squares(x, z);
                uint4 parts[3];
                aft_split(x, parts);
#pragma unroll
                for (int t = 0; t < 3; ++t) kparts[((wave + u * AFT_WAVES) * 3 + t) * 64 + lane] = parts[t];
            }
            const bool odd = aft_odd(z);
            if (lane == 0) odd_keys[wave] = odd;
        }
        __syncthreads();                                 // the keys are there, and nobody reads the values before
        const bool sees = k0 < w_hi && (k0 + AFT_KT > w_lo || k0 < mask.first);
        aft_f32x16 sc, sc2;
        if (sees) {
            int slow = 0;
#pragma unroll
            for (int w = 0; w < AFT_WAVES; ++w) slow |= odd_keys[w];
            slow = __builtin_amdgcn_readfirstlane(slow);
            if (slow == 0) {
#pragma unroll
                for (int r = 0; r < 16; ++r) sc[r] = sc2[r] = 0.f;
                uint4 a[2][3];
                auto keys_of = [&](int ks) {
#pragma unroll
                    for (int t = 0; t < 3; ++t) a[ks & 1][t] = kparts[(ks * 3 + t) * 64 + lane];
                };
                keys_of(0);
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) {
                    if (ks + 1 < KS) keys_of(ks + 1);
#define AFT_ONE(ACC, TA, TB) AFT_MUL(ACC, a[ks & 1][TA], qf[ks][TB]);
                    uint4 ql = qf[ks][2];
                    if (ks < QL) ql = qparts[(wave * QL + ks) * 64 + lane];
                    AFT_ONE(sc, 2, 0)
                    AFT_MUL(sc2, a[ks & 1][0], ql);
                    AFT_ONE(sc, 1, 1)
                    AFT_ONE(sc2, 1, 0) AFT_ONE(sc, 0, 1) AFT_ONE(sc2, 0, 0)
#undef AFT_ONE
                    __builtin_amdgcn_sched_barrier(0);
                }
#pragma unroll
                for (int r = 0; r < 16; ++r) sc[r] += sc2[r];
            }
            if (slow || odd_queries) {
#pragma unroll
                for (int r = 0; r < 16; ++r) sc2[r] = 0.f;
                int here = lane & 31;
                asm volatile("" : "+v"(here));           // nothing of this is made ahead of the loop
                const bool there = k0 + here < k_hi;
                const int c = ti * AFT_COLUMNS + wave * 32 + here;
                const float* kp = k_cache + ((size_t)page_of(k0 + here) * bs + (last(k0 + here) & (bs - 1))) * nkv * D + (size_t)kvh * D + h;
                const float* qp = q + (size_t)(t0 + (c < columns ? c / G : 0)) * q_stride + (size_t)(kvh * G + (c < columns ? c % G : 0)) * D + h;
                for (int kk = 0; kk < D / 2; ++kk)       // head dimension 2 kk + h
                    sc2 = __builtin_amdgcn_mfma_f32_32x32x2f32(there ? kp[2 * kk] : 0.f, c < columns ? qp[2 * kk] * sign : 0.f, sc2, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 16; ++r) sc[r] = slow || odd_query ? sc2[r] : sc[r];
            }
        }
        // this tile's values, asked for as late as there is something to do until they come (registers)
        float4 vreg[VU][2];
#pragma unroll
        for (int x = 0; x < 2 * VU; ++x) {
            vreg[x / 2][x & 1] = *reinterpret_cast<const float4*>(value_at(vpage[x], k0, x));
            vpage[x] = page_of(value_key(next, x));
        }
        if (sees) {
            // ---- softmax: register r is key k0 + 8 (r / 4) + 4 h + r % 4 ----
            const bool edge = k0 + AFT_KT - 1 > p_least || k0 < lo_most;
            float most = -INFINITY;
#pragma unroll
            for (int r = 0; r < 16; ++r) sc[r] *= to_exp;
            if (edge) {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int key = k0 + 8 * (r >> 2) + 4 * h + (r & 3);
                    sc[r] = key <= p && (key >= lo || key < mask.first) ? sc[r] : -INFINITY;
                }
            }
#pragma unroll
            for (int r = 0; r < 16; ++r) most = fmaxf(most, sc[r]);
            const tl_u32x2 sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(most), __float_as_uint(most), false, false);
            const float m_new = fmaxf(m, fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1])));
            const float from = m_new == -INFINITY ? 0.f : m_new;         // (no key seen yet)
            const float alpha = __builtin_amdgcn_exp2f(m - from);
            float sum = 0.f;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                sc[r] = __builtin_amdgcn_exp2f(sc[r] - from);
                sum += sc[r];
            }
            l = __builtin_fmaf(l, alpha, sum);           // of this lane's keys: the halves are added at the end
            m = m_new;
            if (__any(alpha != 1.f)) {
#pragma unroll
                for (int i = 0; i < DB; ++i)
#pragma unroll
                    for (int r = 0; r < 16; ++r) o[i][r] *= alpha;
            }
        }
        {
            float z = 0.f;
            uint32_t least = ~0u;
#pragma unroll
            for (int u = 0; u < VU; ++u) {
                const int unit = wave * VU + u;
                float x[8];
                from_two(vreg[u][0], vreg[u][1], x);
                if (k0 + AFT_KT > k_hi) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) x[e] = k0 + 16 * (unit & 1) + 8 * (e >> 2) + 4 * h + (e & 3) < k_hi ? x[e] : 0.f;
                }
                aft_squares(x, z);
                aft_least(x, least);
                uint4 parts[3];
                aft_split(x, parts);
#pragma unroll
                for (int t = 0; t < 3; ++t) vparts[(unit * 3 + t) * 64 + lane] = parts[t];
            }
            const bool odd = aft_odd(z) || aft_tiny(least);
            if (lane == 0) odd_values[wave] = odd;
        }
        // the next tile's keys
        ask_keys(next);
        kpage = page_of(tile_after(next) + (lane & 31));
        __syncthreads();                                 // the values are there, and nobody reads the keys before
        if (sees) {
            int slow = 0;
#pragma unroll
            for (int w = 0; w < AFT_WAVES; ++w) slow |= odd_values[w];
            if (__builtin_amdgcn_readfirstlane(slow) == 0) {
#pragma unroll
                for (int half = 0; half < 2; ++half) {
                    float x[8];
#pragma unroll
                    for (int e = 0; e < 8; ++e) x[e] = sc[8 * half + e];
                    uint4 w[3];
                    aft_split(x, w);
#pragma unroll
                    for (int i = 0; i < DB; i += 2) {
                        uint4 a[2][3];
#pragma unroll
                        for (int u = 0; u < 2; ++u)
#pragma unroll
                            for (int t = 0; t < 3; ++t) a[u][t] = vparts[(((i + u) * 2 + half) * 3 + t) * 64 + lane];
#define AFT_BOTH(TA, TB)                  \
    AFT_MUL(o[i], a[0][TA], w[TB]);       \
    AFT_MUL(o[i + 1], a[1][TA], w[TB]);
                        AFT_BOTH(2, 0) AFT_BOTH(0, 2) AFT_BOTH(1, 1) AFT_BOTH(1, 0) AFT_BOTH(0, 1) AFT_BOTH(0, 0)
#undef AFT_BOTH
                    }
                }
            } else {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    int key = k0 + 8 * (r >> 2) + 4 * h + (r & 3);
                    asm volatile("" : "+v"(key));
                    const float* v = v_cache + (((size_t)page_of(key) * nkv + kvh) * D + (lane & 31)) * bs + (last(key) & (bs - 1));
#pragma unroll
                    for (int i = 0; i < DB; ++i) o[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(key < k_hi ? v[(size_t)32 * i * bs] : 0.f, sc[r], o[i], 0, 0, 0);
                }
            }
        }
    }
    const tl_u32x2 sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(l), __float_as_uint(l), false, false);
    l = __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
    int c = ti * AFT_COLUMNS + wave * 32 + (lane & 31);
    asm volatile("" : "+v"(c));
    if (c >= columns) return;
    const int token = t0 + c / G, head = kvh * G + c % G;
    // the head's sink: a key that has no value
    const float inv = l > 0.f ? 1.f / (sinks ? l + __builtin_amdgcn_exp2f(sinks[head] * 1.44269504088896340736f - m) : l) : 0.f;
    float* to = out + (size_t)token * out_stride + (size_t)head * D + 4 * h;
#pragma unroll
    for (int i = 0; i < DB; ++i)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            float* t = to + 32 * i + 8 * g;
            if (vec) *reinterpret_cast<float4*>(t) = make_float4(o[i][4 * g] * inv, o[i][4 * g + 1] * inv, o[i][4 * g + 2] * inv, o[i][4 * g + 3] * inv);
            else
#pragma unroll
                for (int r = 0; r < 4; ++r) t[r] = o[i][4 * g + r] * inv;
        }
}

// Whether a float launch runs on the kernel above.
static bool aft_takes(const AgLaunch& a) {
    return !a.keys_over_waves && a.nsplit == 1 && (a.d == 64 || a.d == 128) && a.bs >= 4 && a.bs_shift >= 0 && a.softcap == 0.f && !a.bias.table &&
           (uintptr_t)a.k_cache % 16 == 0 && (uintptr_t)a.v_cache % 16 == 0;
}

static void aft_launch(const AgLaunch& a, int S, int max_query_len) {
    const int G = a.nq / a.nkv, tiles = (int)(((long long)max_query_len * G + AFT_COLUMNS - 1) / AFT_COLUMNS);
    const int vec = a.q_stride % 4 == 0 && a.out_stride % 4 == 0 && (uintptr_t)a.q % 16 == 0 && (uintptr_t)a.out % 16 == 0 ? 1 : 0;
#define AFT_GO(D)                                                                                                                 \
    hipLaunchKernelGGL(attn_float_tile_kernel<D>, dim3((unsigned)(S * tiles), a.nkv), dim3(AFT_WAVES * 64), 0, a.stream, (const float*)a.q,   \
                       a.q_stride, (const float*)a.k_cache, (const float*)a.v_cache, a.tables, a.NB, a.q_start, a.pos, (float*)a.out, \
                       a.out_stride, tiles, a.nq, a.nkv, a.bs, a.bs_shift, a.mask, a.scale, a.sinks, vec)
    if (a.d == 64) AFT_GO(64);
    else AFT_GO(128);
#undef AFT_GO
}
