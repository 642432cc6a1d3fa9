// C[M, N] = A[M, K] * W[N, K]^T (+ bias[N]):  the any-shape matrix product.
//
// Float inputs, float products and sums on the matrix cores' float instruction v_mfma_f32_16x16x4_f32: the true 32-bit
// path's product of up to 16 rows, of a K below 64 and of weights without a matrix-core ordered copy (with one, 17 rows and
// more go to gemm_float.hip: 4.84 against 2.79 ms at 2,048 rows of 37,888 x 3,584), and the any-shape fallback for bfloat16 inputs
// (converted to float on the way into LDS, which is exact).  Any M, N and K, any row strides.
//
// One output element is summed over k in one fixed order: steps of 16 from k = 0 upwards, four
// products per step, the lanes' k within a step fixed by the operand layout.  The order does not
// depend on M or on which tile shape the launch picked, so cutting a batch differently does not
// change a bit of a result, and neither does the number of rows that come along (from 17 rows on;
// up to 16 rows have an order of their own, see gemm_fewrows_kernel).
//
// Tiles: four waves compute BM x BN outputs, a wave MB x NB blocks of 16 x 16; 128 x 128 for many
// rows, 64 x 128 and 32 x 64 for few (more work-groups stream the weights then); at most 16 rows
// have a kernel of their own (gemm_fewrows_kernel), which sums K in segments.  A k-step's rows
// of A and W go from memory into registers while the step before is computed, then as float into
// LDS [row][16 + 4] (the padding keeps the 16-byte operand reads off each other's banks).
//
// Operand layout of the 16x16x4 product D = A B + C: lane l gives A[l % 16][l / 16] and
// B[l / 16][l % 16]; it holds D[4 (l / 16) + v][l % 16] in register v.  Lane group g = l / 16 feeds
// k = 4 g + v of the step to the v-th of its four products, for A and B alike, so a lane's four
// operands are one 16-byte read.
#include "common.h"

#define GG_THREADS 256
#define GG_KS 16              // k per step
#define GG_LD (GG_KS + 4)     // LDS row stride in floats

typedef float gg_f32x4 __attribute__((ext_vector_type(4)));

// Four consecutive k of one row as floats; zero where the row or k is outside the matrix.
template <typename T>
__device__ __forceinline__ float4 gg_load4(const T* __restrict__ base, bool row_ok, int k, int K, bool vec_ok);

template <>
__device__ __forceinline__ float4 gg_load4<float>(const float* __restrict__ base, bool row_ok, int k, int K, bool vec_ok) {
    if (!row_ok || k >= K) return make_float4(0.f, 0.f, 0.f, 0.f);
    if (vec_ok && k + 3 < K) return *reinterpret_cast<const float4*>(base + k);
    float4 r;
    r.x = base[k];
    r.y = (k + 1 < K) ? base[k + 1] : 0.f;
    r.z = (k + 2 < K) ? base[k + 2] : 0.f;
    r.w = (k + 3 < K) ? base[k + 3] : 0.f;
    return r;
}

template <>
__device__ __forceinline__ float4 gg_load4<bf16_t>(const bf16_t* __restrict__ base, bool row_ok, int k, int K, bool vec_ok) {
    if (!row_ok || k >= K) return make_float4(0.f, 0.f, 0.f, 0.f);
    if (vec_ok && k + 3 < K) {
        const uint2 raw = *reinterpret_cast<const uint2*>(base + k);
        return make_float4(__uint_as_float(raw.x << 16), __uint_as_float(raw.x & 0xffff0000u),
                           __uint_as_float(raw.y << 16), __uint_as_float(raw.y & 0xffff0000u));
    }
    float4 r;
    r.x = tl_to_float(base[k]);
    r.y = (k + 1 < K) ? tl_to_float(base[k + 1]) : 0.f;
    r.z = (k + 2 < K) ? tl_to_float(base[k + 2]) : 0.f;
    r.w = (k + 3 < K) ? tl_to_float(base[k + 3]) : 0.f;
    return r;
}

// The same four k with nothing to check: the caller knows that the row exists, that all four k do
// and that the piece is aligned.
template <typename T>
__device__ __forceinline__ float4 gg_load4_whole(const T* __restrict__ p);
template <>
__device__ __forceinline__ float4 gg_load4_whole<float>(const float* __restrict__ p) {
    return *reinterpret_cast<const float4*>(p);
}
template <>
__device__ __forceinline__ float4 gg_load4_whole<bf16_t>(const bf16_t* __restrict__ p) {
    const uint2 raw = *reinterpret_cast<const uint2*>(p);
    return make_float4(__uint_as_float(raw.x << 16), __uint_as_float(raw.x & 0xffff0000u), __uint_as_float(raw.y << 16),
                       __uint_as_float(raw.y & 0xffff0000u));
}

// WM x WN waves (WM * WN == 4), each MB x NB blocks of 16 x 16.
template <typename TA, typename TW, typename TO, int WM, int WN, int MB, int NB>
__global__ __launch_bounds__(GG_THREADS) void gemm_generic_kernel(const TA* __restrict__ A, const TW* __restrict__ W,
                                                                 const float* __restrict__ bias, TO* __restrict__ C,
                                                                 int M, int N, int K, int lda, int ldc, int a_vec,
                                                                 int w_vec, long long a_bs, long long w_bs, long long c_bs) {
    constexpr int BM = WM * MB * 16, BN = WN * NB * 16;
    A += (size_t)blockIdx.z * a_bs;          // a batch of products: one per blockIdx.z, operands a stride apart
    W += (size_t)blockIdx.z * w_bs;
    C += (size_t)blockIdx.z * c_bs;
    constexpr int A_PIECES = BM * 4, W_PIECES = BN * 4;                 // 16-byte (four k) pieces per step
    constexpr int A_PER = (A_PIECES + GG_THREADS - 1) / GG_THREADS, W_PER = (W_PIECES + GG_THREADS - 1) / GG_THREADS;
    __shared__ float As[2][BM * GG_LD];
    __shared__ float Ws[2][BN * GG_LD];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int li = lane & 15, lg = lane >> 4;
    const int wm = wave / WN, wn = wave - wm * WN;
    const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;

    gg_f32x4 acc[MB][NB];
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] = (gg_f32x4){0.f, 0.f, 0.f, 0.f};

    float4 areg[A_PER], wreg[W_PER];
    auto fetch = [&](int k0) {
#pragma unroll
        for (int it = 0; it < A_PER; ++it) {
            const int p = tid + it * GG_THREADS;
            const int r = p >> 2, c4 = p & 3;
            areg[it] = gg_load4<TA>(A + (size_t)(m0 + r) * lda, p < A_PIECES && m0 + r < M, k0 + 4 * c4, K, a_vec != 0);
        }
#pragma unroll
        for (int it = 0; it < W_PER; ++it) {
            const int p = tid + it * GG_THREADS;
            const int r = p >> 2, c4 = p & 3;
            wreg[it] = gg_load4<TW>(W + (size_t)(n0 + r) * K, p < W_PIECES && n0 + r < N, k0 + 4 * c4, K, w_vec != 0);
        }
    };
    auto to_lds = [&](int buf) {
#pragma unroll
        for (int it = 0; it < A_PER; ++it) {
            const int p = tid + it * GG_THREADS;
            if (p < A_PIECES) *reinterpret_cast<float4*>(&As[buf][(p >> 2) * GG_LD + 4 * (p & 3)]) = areg[it];
        }
#pragma unroll
        for (int it = 0; it < W_PER; ++it) {
            const int p = tid + it * GG_THREADS;
            if (p < W_PIECES) *reinterpret_cast<float4*>(&Ws[buf][(p >> 2) * GG_LD + 4 * (p & 3)]) = wreg[it];
        }
    };

    fetch(0);
    to_lds(0);
    __syncthreads();
    int buf = 0;
    for (int k0 = 0; k0 < K; k0 += GG_KS) {
        const bool more = k0 + GG_KS < K;
        if (more) fetch(k0 + GG_KS);
        float4 af[MB], wf[NB];
#pragma unroll
        for (int i = 0; i < MB; ++i)
            af[i] = *reinterpret_cast<const float4*>(&As[buf][((wm * MB + i) * 16 + li) * GG_LD + 4 * lg]);
#pragma unroll
        for (int j = 0; j < NB; ++j)
            wf[j] = *reinterpret_cast<const float4*>(&Ws[buf][((wn * NB + j) * 16 + li) * GG_LD + 4 * lg]);
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int j = 0; j < NB; ++j) {
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(af[i].x, wf[j].x, acc[i][j], 0, 0, 0);
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(af[i].y, wf[j].y, acc[i][j], 0, 0, 0);
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(af[i].z, wf[j].z, acc[i][j], 0, 0, 0);
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(af[i].w, wf[j].w, acc[i][j], 0, 0, 0);
            }
        if (more) {
            to_lds(buf ^ 1);          // the other buffer: nobody reads it during this step
            __syncthreads();
            buf ^= 1;
        }
    }

    // this lane holds rows 4 lg + v and column li of each block
#pragma unroll
    for (int j = 0; j < NB; ++j) {
        const int n = n0 + (wn * NB + j) * 16 + li;
        if (n >= N) continue;
        const float b = bias ? bias[n] : 0.f;
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int m = m0 + (wm * MB + i) * 16 + 4 * lg + v;
                if (m < M) C[(size_t)m * ldc + n] = tl_from_float<TO>(acc[i][j][v] + b);
            }
    }
}

// At most 16 rows (a decode step of few sequences): the work is streaming W once, and a tile of the
// kernel above would leave most of the GPU without work (56 work-groups for 3,584 columns) with one
// k-step in flight each.  Here a work-group owns 16 columns and its waves share K: K is cut into
// segments of GF_SEG at absolute k, wave w sums segments w, w + waves, ... each in the order above
// (steps of 16 upwards, four products per step), with the next GF_RING - 1 steps' operands on their
// way in a ring of registers, and the segments' sums are added in ascending order at the end.  So
// one output element is again summed in one fixed order that depends on K alone, not on M (1 to 16),
// on the number of waves or on timing; it is not the order of the kernel above, whose results differ
// from this one's by rounding.
// Sixteen waves and segments of 256: a product with fewer tiles than the GPU has CUs (the down projection
// of a 7B model: 224) has one work-group per CU, and what streams its weights is the loads that
// group keeps in flight (eight waves: 2.5 TB/s for the float down projection, sixteen: 3.4), and how
// evenly the segments deal out over the waves (74 segments of 256 over 16 waves: 5 at most, 4.6 on
// average; 37 of 512: 3 against 2.3).  A deeper ring pays only where nothing stands between its loads (GF_AHEAD).
#define GF_SEG 256
#define GF_RING 4
#define GF_AHEAD 8
#define GF_WAVES 16
#define GF_MAX_SEGMENTS 128   // 128 KB of LDS for the segments' sums: K up to 32,768 (beyond: the kernel above)

// The waves of a work-group: all sixteen where the tiles are about as many as the CUs, eight where
// every CU holds several work-groups anyway (their loads in flight add up, and a wave with more steps
// fills its ring less often: gate/up of a 7B model 120 against 125 us).  The result does not depend on it.
static inline int gf_waves(int nseg, int tiles) {
    const int most = tiles >= 512 ? GF_WAVES / 2 : GF_WAVES;
    return nseg < most ? nseg : most;
}

// SHUF: W is the matrix-core ordered copy of a float matrix, [ceil(N/16) tiles][ceil(K/16) steps][64
// lanes][4 values], lane 16 lg + li holding row li of the tile at k = 16 step + 4 lg .. + 4, zero
// where it pads: a step's load of a wave is 1 KB of consecutive memory (from the row-major matrix it
// is 16 pieces of 64 bytes, which streams at about two thirds of the rate), and needs no check.
template <typename TA, typename TW, typename TO, bool SHUF>
__global__ __launch_bounds__(GF_WAVES * 64) void gemm_fewrows_kernel(const TA* __restrict__ A, const TW* __restrict__ W,
                                                           const float* __restrict__ bias, TO* __restrict__ C, int M,
                                                           int N, int K, int lda, int ldc, int a_vec, int w_vec,
                                                           long long a_bs, long long w_bs, long long c_bs) {
    extern __shared__ float gf_part[];
    A += (size_t)blockIdx.y * a_bs;          // a batch of products: one per blockIdx.y
    W += (size_t)blockIdx.y * w_bs;
    C += (size_t)blockIdx.y * c_bs;                       // [segment][register v][lane]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nwaves = blockDim.x >> 6;
    const int li = lane & 15, lg = lane >> 4;
    const int n0 = blockIdx.x * 16;
    const int nseg = (K + GF_SEG - 1) / GF_SEG;
    constexpr int SPS = GF_SEG / GG_KS;                      // steps per segment
    const TW* wrow = W + (size_t)(n0 + li) * K;
    const TA* arow = A + (size_t)li * lda;
    const bool w_ok = n0 + li < N, a_ok = li < M;
    // Whole steps (all 16 k inside K, aligned pieces) load without a condition, so that the loads of
    // the steps ahead stay in flight: a row that does not exist is read from one that does (what it
    // brings only reaches outputs that are not written).
    const TW* wrow_any = W + (size_t)(w_ok ? n0 + li : N - 1) * K;
    const TA* arow_any = A + (size_t)(a_ok ? li : 0) * lda;
    const bool pieces_whole = a_vec != 0 && w_vec != 0;
    const float4* wtile = reinterpret_cast<const float4*>(W) + (size_t)blockIdx.x * ((K + GG_KS - 1) / GG_KS) * 64 + lane;
    auto load_step = [&](int k0, float4& wv, float4& av) {
        if (SHUF) {
            if (k0 >= K) {                                      // past the last segment's end: the copy ends with K
                wv = av = make_float4(0.f, 0.f, 0.f, 0.f);
            } else {
                wv = __builtin_bit_cast(float4, tl_load_stream(reinterpret_cast<const uint4*>(wtile + (size_t)(k0 / GG_KS) * 64)));
                if (a_vec != 0 && k0 + GG_KS <= K) av = gg_load4_whole<TA>(arow_any + k0 + 4 * lg);
                else av = gg_load4<TA>(arow, a_ok, k0 + 4 * lg, K, a_vec != 0);
            }
        } else if (pieces_whole && k0 + GG_KS <= K) {           // the same for the whole wave
            wv = gg_load4_whole<TW>(wrow_any + k0 + 4 * lg);
            av = gg_load4_whole<TA>(arow_any + k0 + 4 * lg);
        } else {                                              // past K (the last segment's end): zeros
            wv = gg_load4<TW>(wrow, w_ok, k0 + 4 * lg, K, w_vec != 0);
            av = gg_load4<TA>(arow, a_ok, k0 + 4 * lg, K, a_vec != 0);
        }
    };
    // this wave's steps, numbered through its segments: step j is step j % SPS of segment wave + (j / SPS) * nwaves
    const int my_segs = (nseg - wave + nwaves - 1) / nwaves;   // 0 for a wave beyond the segments
    const int nsteps = my_segs * SPS;
    auto k_of = [&](int j) { return (wave + (j / SPS) * nwaves) * GF_SEG + (j % SPS) * GG_KS; };
    // as in the kernel above: the lane gives row li of A and row li of the W tile at k = k0 + 4 lg + v to the v-th product
    // and holds C[4 lg + v][n0 + li]
    gg_f32x4 acc = (gg_f32x4){0.f, 0.f, 0.f, 0.f};
    auto multiply = [&](const float4& av, const float4& wv) {
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(av.x, wv.x, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(av.y, wv.y, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(av.z, wv.z, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(av.w, wv.w, acc, 0, 0, 0);
    };
    auto end_segment = [&](int j) {                               // step j was the segment's last one
        const int seg = wave + (j / SPS) * nwaves;
#pragma unroll
        for (int v = 0; v < 4; ++v) gf_part[(seg * 4 + v) * 64 + lane] = acc[v];
        acc = (gg_f32x4){0.f, 0.f, 0.f, 0.f};
    };
    if (SHUF && a_vec != 0 && K % GG_KS == 0) {
        // Whole steps only, and of those that lie in K alone (a wave's first ones): the loop asks without a condition, so that
        // the loads of GF_AHEAD steps stay on their way.  With conditions around them a product waited for nearly all that
        // was on its way (8 rows, us: 37,888 x 3,584 108 -> 95, 152,064 x 3,584 387 -> 355, 3,584 x 18,944 68 -> 53).
        static_assert(SPS % GF_AHEAD == 0, "segments end with a round of the ring");
        const bool ends = (nseg - 1 - wave) % nwaves == 0;        // this wave has the last segment
        const int mine = ends ? nsteps - SPS + (K - (nseg - 1) * GF_SEG) / GG_KS : nsteps;
        float4 wr[GF_AHEAD], ar[GF_AHEAD];
        auto ask = [&](int j, int r) {
            const int k0 = k_of(j);
            wr[r] = __builtin_bit_cast(float4, tl_load_stream(reinterpret_cast<const uint4*>(wtile + (size_t)(k0 / GG_KS) * 64)));
            ar[r] = gg_load4_whole<TA>(arow_any + k0 + 4 * lg);
        };
#pragma unroll
        for (int r = 0; r < GF_AHEAD; ++r) ask(r < mine ? r : mine - 1, r);
        int j = 0;
        for (; j + 2 * GF_AHEAD <= mine; j += GF_AHEAD) {
#pragma unroll
            for (int r = 0; r < GF_AHEAD; ++r) {
                multiply(ar[r], wr[r]);
                __builtin_amdgcn_sched_barrier(0);
                ask(j + r + GF_AHEAD, r);
                __builtin_amdgcn_sched_barrier(0);
            }
            if ((j + GF_AHEAD) % SPS == 0) end_segment(j + GF_AHEAD - 1);
        }
#pragma unroll
        for (int r = 0; r < 2 * GF_AHEAD; ++r) {
            const int t = j + r;
            if (t >= mine) break;
            multiply(ar[r % GF_AHEAD], wr[r % GF_AHEAD]);
            if (t + GF_AHEAD < mine) ask(t + GF_AHEAD, r % GF_AHEAD);
            if ((t + 1) % SPS == 0 || t + 1 == mine) end_segment(t);
        }
    } else {
        float4 wreg[GF_RING], areg[GF_RING];
#pragma unroll
        for (int r = 0; r < GF_RING - 1; ++r) {
            if (r < nsteps) load_step(k_of(r), wreg[r], areg[r]);
        }
        for (int jb = 0; jb < nsteps; jb += GF_RING) {
#pragma unroll
            for (int r = 0; r < GF_RING; ++r) {
                const int j = jb + r;
                if (j < nsteps) {                                 // the same for the whole wave
                    const int ahead = j + GF_RING - 1;
                    if (ahead < nsteps) load_step(k_of(ahead), wreg[(r + GF_RING - 1) % GF_RING], areg[(r + GF_RING - 1) % GF_RING]);
                    multiply(areg[r], wreg[r]);
                    if (j % SPS == SPS - 1) end_segment(j);
                }
            }
        }
    }
    __syncthreads();
    // element (v, lane): row m = 4 lg + v, column n0 + li; segments in ascending order
    for (int e = tid; e < 256; e += blockDim.x) {
        const int l = e & 63, v = e >> 6;
        const int m = 4 * (l >> 4) + v, n = n0 + (l & 15);
        if (m >= M || n >= N) continue;
        float sum = 0.f;
        for (int seg = 0; seg < nseg; ++seg) sum += gf_part[(seg * 4 + v) * 64 + l];
        C[(size_t)m * ldc + n] = tl_from_float<TO>(sum + (bias ? bias[n] : 0.f));
    }
}

template <typename TA, typename TW, typename TO>
static int gg_launch(const void* A, const void* W, const float* bias, void* C, int M, int N, int K, int lda, int ldc,
                     hipStream_t stream, int batch = 1, long long a_bs = 0, long long w_bs = 0, long long c_bs = 0) {
    // whole 16-byte (8-byte for bfloat16) pieces can be read where rows start aligned
    const int a_vec = ((uintptr_t)A % (4 * sizeof(TA)) == 0 && lda % 4 == 0 && a_bs % 4 == 0) ? 1 : 0;
    const int w_vec = ((uintptr_t)W % (4 * sizeof(TW)) == 0 && K % 4 == 0 && w_bs % 4 == 0) ? 1 : 0;
#define GG_GO(WM, WN, MB, NB)                                                                                    \
    do {                                                                                                         \
        constexpr int BM = WM * MB * 16, BN = WN * NB * 16;                                                      \
        const long long gy = tl_ceil_div(M, BM);                                                                 \
        if (gy > 65535) return tl_fail("tl_gemm_generic: %d rows are too many for one launch", M);               \
        dim3 grid(tl_ceil_div(N, BN), (unsigned)gy, batch), block(GG_THREADS);                                   \
        hipLaunchKernelGGL((gemm_generic_kernel<TA, TW, TO, WM, WN, MB, NB>), grid, block, 0, stream,            \
                           (const TA*)A, (const TW*)W, bias, (TO*)C, M, N, K, lda, ldc, a_vec, w_vec, a_bs, w_bs, c_bs); \
    } while (0)
    const int nseg = tl_ceil_div(K, GF_SEG);
    if (M <= 16 && nseg <= GF_MAX_SEGMENTS) {
        const int waves = gf_waves(nseg, tl_ceil_div(N, 16));
        const size_t lds = (size_t)nseg * 4 * 64 * sizeof(float);
        hipLaunchKernelGGL((gemm_fewrows_kernel<TA, TW, TO, false>), dim3(tl_ceil_div(N, 16), batch), dim3(64 * waves), lds, stream,
                           (const TA*)A, (const TW*)W, bias, (TO*)C, M, N, K, lda, ldc, a_vec, w_vec, a_bs, w_bs, c_bs);
    } else if (M <= 32)
        GG_GO(1, 4, 2, 1);        // 32 x 64
    else if (M <= 64)
        GG_GO(1, 4, 4, 2);        // 64 x 128
    else
        GG_GO(2, 2, 4, 4);        // 128 x 128
#undef GG_GO
    return 0;
}

// Whether the few-row kernel takes a product of this K (the segments' sums must fit its LDS).
extern "C" int tl_gemm_fewrows_takes(int K) { return K > 0 && tl_ceil_div(K, GF_SEG) <= GF_MAX_SEGMENTS ? 1 : 0; }

// The float product for at most 16 rows from the matrix-core ordered copy of W (see gemm_fewrows_kernel,
// SHUF): A float [M, K] with row stride lda, Ws float [ceil(N/16), ceil(K/16), 64, 4], C float [M, N].
// The same sums in the same order as tl_gemm_generic gives for these rows.
extern "C" int tl_gemm_fewrows_shuffled(const float* A, const float* Ws, const float* bias, float* C, int M, int N, int K,
                                        int lda, int ldc, hipStream_t stream) {
    TL_CHECK_ARG(M >= 0 && M <= 16 && N > 0 && K > 0, "tl_gemm_fewrows_shuffled: bad sizes M=%d N=%d K=%d", M, N, K);
    TL_CHECK_ARG(lda >= K && ldc >= N, "tl_gemm_fewrows_shuffled: row strides lda=%d ldc=%d too small for K=%d N=%d", lda, ldc, K, N);
    TL_CHECK_ARG(tl_gemm_fewrows_takes(K), "tl_gemm_fewrows_shuffled: K=%d is too long for the segments' sums", K);
    TL_CHECK_ARG(((uintptr_t)Ws % 16) == 0, "tl_gemm_fewrows_shuffled: the weight copy must be 16-byte aligned");
    if (M == 0) return 0;
    const int a_vec = ((uintptr_t)A % 16 == 0 && lda % 4 == 0) ? 1 : 0;
    const int nseg = tl_ceil_div(K, GF_SEG);
    const int waves = gf_waves(nseg, tl_ceil_div(N, 16));
    const size_t lds = (size_t)nseg * 4 * 64 * sizeof(float);
    hipLaunchKernelGGL((gemm_fewrows_kernel<float, float, float, true>), dim3(tl_ceil_div(N, 16)), dim3(64 * waves), lds, stream,
                       A, Ws, bias, C, M, N, K, lda, ldc, a_vec, 1, 0LL, 0LL, 0LL);
    TL_CHECK_LAUNCH("tl_gemm_fewrows_shuffled");
    return 0;
}

// A: [M, K] with row stride lda; W: [N, K] contiguous; C: [M, N] with row stride ldc.
extern "C" int tl_gemm_generic(const void* A, int a_dtype, const void* W, int w_dtype, const float* bias, void* C,
                               int c_dtype, int M, int N, int K, int lda, int ldc, hipStream_t stream) {
    TL_CHECK_ARG(M >= 0 && N > 0 && K > 0, "tl_gemm_generic: bad sizes M=%d N=%d K=%d", M, N, K);
    TL_CHECK_ARG(lda >= K && ldc >= N, "tl_gemm_generic: row strides lda=%d ldc=%d too small for K=%d N=%d", lda, ldc, K, N);
    if (M == 0) return 0;
    int rc;
    if (a_dtype == TL_F32 && w_dtype == TL_F32 && c_dtype == TL_F32)
        rc = gg_launch<float, float, float>(A, W, bias, C, M, N, K, lda, ldc, stream);
    else if (a_dtype == TL_BF16 && w_dtype == TL_BF16 && c_dtype == TL_BF16)
        rc = gg_launch<bf16_t, bf16_t, bf16_t>(A, W, bias, C, M, N, K, lda, ldc, stream);
    else if (a_dtype == TL_BF16 && w_dtype == TL_BF16 && c_dtype == TL_F32)
        rc = gg_launch<bf16_t, bf16_t, float>(A, W, bias, C, M, N, K, lda, ldc, stream);
    else if (a_dtype == TL_F32 && w_dtype == TL_BF16 && c_dtype == TL_F32)
        rc = gg_launch<float, bf16_t, float>(A, W, bias, C, M, N, K, lda, ldc, stream);
    else
        return tl_fail("tl_gemm_generic: unsupported dtypes a=%d w=%d c=%d", a_dtype, w_dtype, c_dtype);
    if (rc) return rc;
    TL_CHECK_LAUNCH("tl_gemm_generic");
    return 0;
}

// A batch of bfloat16 products on v_mfma_f32_16x16x32_bf16 (products exact, sums in float), for the small matrices that are
// applied per head (a latent's: 192 x 128): a wave has 32 or 64 rows of A by 64 of W and takes its fragments straight from memory
// (lane 16 g + c: row c, eight k from 8 g on), the four waves of a work-group the same 64 rows of W, which an L1 then holds.
// What a head's matrix is read from is L2 (48 KB a head), what bounds it is A, C and the reading of W by every wave again: 2,048 rows of 32
// heads take 22 us for 192 x 128 and 19 for 128 x 192 with 64 rows a wave and results by 16 bytes (ROWS), where they took 25 and 24 with 32 rows and
// two bytes (200 rows of 16 times 1,024 x 1,024 46 -> 31), and 86 and 55 on the float instruction through LDS.  One order of summation per element whatever the rows: k in steps of 32 from 0 up.
typedef __bf16 gg_bf16x8 __attribute__((ext_vector_type(8)));
template <int MB, bool ROWS>
__global__ __launch_bounds__(GG_THREADS) void gemm_batched_bf16_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W,
                                                                      bf16_t* __restrict__ C, int M, int N, int K, int lda, int ldc,
                                                                      long long a_bs, long long w_bs, long long c_bs) {
    A += (size_t)blockIdx.z * a_bs;
    W += (size_t)blockIdx.z * w_bs;
    C += (size_t)blockIdx.z * c_bs;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c = lane & 15, g = lane >> 4;
    const int m0 = (blockIdx.y * 4 + wave) * 16 * MB, n0 = blockIdx.x * 64;
    if (m0 >= M) return;
    const bf16_t* ap[MB];
    const bf16_t* wp[4];
#pragma unroll
    for (int i = 0; i < MB; ++i) ap[i] = A + (size_t)min(m0 + i * 16 + c, M - 1) * lda + 8 * g;    // a row that is not there: the
#pragma unroll
    for (int j = 0; j < 4; ++j) wp[j] = W + (size_t)min(n0 + (ROWS ? (c >> 2) * 16 + j * 4 + (c & 3) : j * 16 + c), N - 1) * K + 8 * g;   // last one, not written back
    gg_f32x4 acc[MB][4];
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = (gg_f32x4){0.f, 0.f, 0.f, 0.f};
    auto step = [&](int k0, bool here) {
        uint4 a[MB], w[4];
        const uint4 zero = make_uint4(0, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < MB; ++i) a[i] = here ? *reinterpret_cast<const uint4*>(ap[i] + k0) : zero;
#pragma unroll
        for (int j = 0; j < 4; ++j) w[j] = here ? *reinterpret_cast<const uint4*>(wp[j] + k0) : zero;
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(gg_bf16x8, ROWS ? w[j] : a[i]),
                                                                    __builtin_bit_cast(gg_bf16x8, ROWS ? a[i] : w[j]), acc[i][j], 0, 0, 0);
    };
    const int whole = K / 32 * 32;
#pragma unroll 4
    for (int k0 = 0; k0 < whole; k0 += 32) step(k0, true);
    if (whole < K) step(whole, whole + 8 * g < K);           // K is a multiple of eight: a lane's piece is there or not
    if constexpr (ROWS) {              // a lane has row c of a block of rows and the sixteen columns from n0 + 16 g on, four of each block j
        const int n = n0 + 16 * g;
#pragma unroll
        for (int i = 0; i < MB; ++i) {
            const int m = m0 + i * 16 + c;
            if (m >= M || n >= N) continue;
#pragma unroll
            for (int j = 0; j < 4; j += 2)
                *reinterpret_cast<uint4*>(C + (size_t)m * ldc + n + 4 * j) =
                    make_uint4(tl_pack_bf16(acc[i][j][0], acc[i][j][1]), tl_pack_bf16(acc[i][j][2], acc[i][j][3]),
                               tl_pack_bf16(acc[i][j + 1][0], acc[i][j + 1][1]), tl_pack_bf16(acc[i][j + 1][2], acc[i][j + 1][3]));
        }
    } else {
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int m = m0 + i * 16 + 4 * g + v;
                if (m >= M) continue;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int n = n0 + j * 16 + c;
                    if (n < N) C[(size_t)m * ldc + n] = tl_from_float<bf16_t>(acc[i][j][v]);
                }
            }
    }
}

// Whether a wave of such a product has 64 rows: where that leaves enough waves, which a short K needs more of (600 rows of 32 heads of 192 x
// 128 10.0 and 11.9 us with 32 and 64 rows a wave, 2,048 23.5 and 22.1; 900 of 128 x 192 12.8 and 9.6), and where the rows fill them: 16 of 1,024 x
// 1,024 take 16.6 and 20.8 us for 17 rows, 19.0 and 22.2 for 64, 22 and 23 for 96, 27 and 23 for 128; 257 to 384 rows are three
// work-groups or two with a wave or two in the second, level in time (60 and 61 us) unless the two are one round of the GPU (4 of 2,048 x 1,024 46 and 32).
extern "C" int tl_gemm_batched_tall(int M, int N, int K, int batch) {
    const double groups = (double)tl_ceil_div(N, 64) * tl_ceil_div(M, 256) * batch;
    return M >= 128 && groups >= (K >= 192 ? 256 : 512) && (tl_ceil_div(M, 128) != 3 || groups <= 256) ? 1 : 0;
}

// `batch` products of the same shape in one launch: product b reads A + b * a_bs (row stride lda),
// W + b * w_bs ([N, K] contiguous) and writes C + b * c_bs (row stride ldc); strides in elements.
// Each is summed as tl_gemm_generic sums it, or (aligned bfloat16) in steps of 32 k from 0 upwards on the bfloat16
// instruction.  (A head's share of a projection that is applied per
// head: the operands are column blocks of wider matrices, a stride of one head apart.)
extern "C" int tl_gemm_generic_batched(const void* A, int a_dtype, const void* W, int w_dtype, void* C, int c_dtype, int M,
                                       int N, int K, int lda, int ldc, int batch, long long a_bs, long long w_bs,
                                       long long c_bs, hipStream_t stream) {
    TL_CHECK_ARG(M >= 0 && N > 0 && K > 0 && batch > 0 && batch <= 65535, "tl_gemm_generic_batched: bad sizes M=%d N=%d K=%d batch=%d", M, N, K, batch);
    TL_CHECK_ARG(lda >= K && ldc >= N, "tl_gemm_generic_batched: row strides lda=%d ldc=%d too small for K=%d N=%d", lda, ldc, K, N);
    if (M == 0) return 0;
    int rc;
    // Aligned bfloat16 operands, us on the kernels below and on the one without LDS (8 products of N x K): 17 rows of 64 x 64 4.8
    // and 3.9, 512 x 512 20.7 and 8.0, 1,024 x 1,024 44 and 17; 2,048 rows 19 and 5.8, 109 and 49, 451 and 175.  At most 16 rows
    // go to the few-row kernel behind K = 512, whose waves share K where one wave walks it here: 8 rows of 128 x 256 7.7 and
    // 5.4, x 448 7.3 and 7.1, x 512 7.4 and 7.7, x 640 7.6 and 8.8, 64 x 1,024 7.7 and 12.2.
    if (a_dtype == TL_BF16 && w_dtype == TL_BF16 && c_dtype == TL_BF16 && K % 8 == 0 && K <= (M <= 16 ? 512 : 1024) && lda % 8 == 0 && a_bs % 8 == 0 &&
        w_bs % 8 == 0 && (uintptr_t)A % 16 == 0 && (uintptr_t)W % 16 == 0 && tl_ceil_div(M, 128) <= 65535) {
        // whole aligned sixteens of columns
        const bool rows = N % 16 == 0 && (uintptr_t)C % 16 == 0 && ldc % 8 == 0 && c_bs % 8 == 0;
        const bool tall = rows && tl_gemm_batched_tall(M, N, K, batch);
#define GO(MB, ROWS)                                                                                                                  \
    hipLaunchKernelGGL((gemm_batched_bf16_kernel<MB, ROWS>), dim3(tl_ceil_div(N, 64), tl_ceil_div(M, 64 * MB), batch), dim3(GG_THREADS), 0, \
                       stream, (const bf16_t*)A, (const bf16_t*)W, (bf16_t*)C, M, N, K, lda, ldc, a_bs, w_bs, c_bs)
        if (tall) GO(4, true);
        else if (rows) GO(2, true);
        else GO(2, false);
#undef GO
        TL_CHECK_LAUNCH("tl_gemm_generic_batched");
        return 0;
    }
    if (a_dtype == TL_F32 && w_dtype == TL_F32 && c_dtype == TL_F32)
        rc = gg_launch<float, float, float>(A, W, nullptr, C, M, N, K, lda, ldc, stream, batch, a_bs, w_bs, c_bs);
    else if (a_dtype == TL_BF16 && w_dtype == TL_BF16 && c_dtype == TL_BF16)
        rc = gg_launch<bf16_t, bf16_t, bf16_t>(A, W, nullptr, C, M, N, K, lda, ldc, stream, batch, a_bs, w_bs, c_bs);
    else
        return tl_fail("tl_gemm_generic_batched: unsupported dtypes a=%d w=%d c=%d", a_dtype, w_dtype, c_dtype);
    if (rc) return rc;
    TL_CHECK_LAUNCH("tl_gemm_generic_batched");
    return 0;
}
