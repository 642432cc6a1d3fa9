// C[M, N] = A[M, K] * W[N, K]^T (+ bias[N]) in float for more than 16 rows, on the bfloat16 matrix
// instruction (v_mfma_f32_32x32x16_bf16): the 32-bit path's product of prompts and large batches.
//
// A float times 2^24 is exactly the sum of three bfloat16 numbers (8 + 8 + 8 significant bits; each is the rest of the
// one before, rounded to nearest, so the rests have either sign; splitting floats into shorter ones so that products
// are exact is Dekker's, Numerische Mathematik 18, 1971).  The factor keeps the last part of the smallest
// float a normal bfloat16: without it floats below 2^-110 lost their rests (4.6e-4 of a value of 1e-37).  It comes out
// again as 2^-48 of a segment's sum, and costs 1 to 3% (2,048 rows of 37,888 x 3,584: 2.79 ms against 2.75).
//
// Of the nine partial products of two such sums the six with a first part in them and the product of the two second parts
// are taken, small ones first, each exact; the three left out come to at most 2^-24 of the product they
// belong to (a second part is up to 2^-8 of its float, a third up to 2^-17) and 1e-8 of it on average, and a sum of K
// products takes roundings of that size at every step whatever the instruction.  What the result is off the exact one,
// 2-norm, 256 rows, six products here / eight of the nine / v_mfma_f32_16x16x4_f32:
//                                    K = 16                  896                     3,584                   18,944
//   normal numbers                   3.4e-8 3.3e-8 7.3e-8    4.6e-7 4.6e-7 5.4e-7    6.7e-7 6.7e-7 1.1e-6    7.6e-7 7.6e-7 2.5e-6
//   positive (uniform in [0, 1))     3.3e-8 3.3e-8 6.2e-8    2.9e-7 2.9e-7 4.2e-7    2.8e-7 2.8e-7 8.4e-7    1.4e-7 1.4e-7 2.1e-6
//   one column 3,000 times the rest  5.9e-8 5.9e-8 8.4e-8    3.9e-7 3.9e-7 6.2e-7    4.6e-7 4.6e-7 1.3e-6    6.9e-7 6.9e-7 2.9e-6
// The two more products cost 20% (gate/up of 2,048 rows 2.74 -> 3.34 ms) and change nothing from K = 16 on; below, where a
// result is a handful of products, the matrix instruction's own last addition is the error (K = 1: 3.4e-8 with six or eight,
// 2.6e-8 on the float instruction), and products of a K below 64 go to the float instruction.  Six bfloat16 products take 6 / 16 of the
// matrix cores' time of one on the float instruction (2.5 PFLOP/s against 157 TFLOP/s).
//
// What is split where: the rows of A once, by a pass of its own, into the order in which the product reads
// them (fs_split_kernel: 4 bytes read and 6 written per value); W, which may be most of the GPU's memory,
// stays float and is split in registers by the wave that owns its columns, from the matrix-core ordered copy
// that the few-row product streams as well.  A wave owns 32 or 64 columns and all the rows of its work-group
// (up to 128): 52 vector instructions per 32 columns beside 6 matrix instructions per 32 x 32 block and 16 k.
//
// Per step of 16 k a work-group holds 3 KB of A per 32 rows and 2 KB of W per 32 columns of a wave in LDS, in the
// layout the fragments are read in (a fragment is 1 KB, lane after lane: no bank conflicts), fetched one or two
// steps ahead by global_load_lds; one barrier per step.  What bounds it: the matrix cores are busy half of the time
// (200 TFLOP/s are 1.2 PFLOP/s of bfloat16 products), the rest is the splitting of W, which does not overlap with them,
// and LDS reads (a fragment of A feeds six products of a column block).
//
// One output element is summed in one fixed order whatever the number of rows or the tile: k in segments of
// FS_SEG at absolute k, within a segment steps of 16 upwards with the six partial products of a step in one
// order, the segments' sums added in ascending order.  Few tiles (few rows of a narrow matrix) are spread
// over the GPU by segments, whose sums a second kernel adds in the same order.
//
// Values that are not finite, and those of 2^104 and more, which the factor takes past the largest bfloat16, make the
// split itself infinity minus infinity, and sums of 2^80 and more pass the largest float where the sums themselves do
// not: an element whose segment does not come out finite is computed again on the float instruction, so infinities,
// NaN and sums of any size give what they give there.  (A wave takes its blocks of 32 x 32 in
// turn: 2.5 ms for 2,048 rows of 4,608 x 3,584 with an infinity in every row, 0.4 without.)
#include "common.h"

typedef __bf16 fs_bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 fs_bf16x2 __attribute__((ext_vector_type(2)));
typedef float fs_f32x2 __attribute__((ext_vector_type(2)));
typedef float fs_f32x16 __attribute__((ext_vector_type(16)));

#define FS_STEP 16
#define FS_SEG 2048                      // k per segment
#define FS_SEG_STEPS (FS_SEG / FS_STEP)
#define FS_WAVES 4
#define FS_CUS 256
#define FS_MOST_SUMS (512LL << 18)       // floats at most of the segments' sums (512 MB): beyond, K stays whole
#define FS_UP 0x1p24f                    // factor of both operands
#define FS_DOWN 0x1p-48f
#define FS_RAW_K 2048                    // at most 32 aligned rows of a K up to this are split where they are used (RAW)
#define FS_RAW_GROUP 4                   // steps whose weights a wave asks for together
#define FS_RAW_CHUNK 24                  // steps whose rows are in LDS at a time

// two floats as two bfloat16, rounded to nearest even, and what is left of each
__device__ __forceinline__ uint32_t fs_take(float& a, float& b) {
    const fs_f32x2 v = {a, b};
    const uint32_t p = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, fs_bf16x2));
    a -= __uint_as_float(p << 16);
    b -= __uint_as_float(p & 0xffff0000u);
    return p;
}
// floats times FS_UP as three times as many bfloat16
__device__ __forceinline__ void fs_split4(float4 x, uint2& hi, uint2& mid, uint2& lo) {
    x.x *= FS_UP, x.y *= FS_UP, x.z *= FS_UP, x.w *= FS_UP;
    hi = make_uint2(fs_take(x.x, x.y), fs_take(x.z, x.w));
    mid = make_uint2(fs_take(x.x, x.y), fs_take(x.z, x.w));
    lo = make_uint2(fs_take(x.x, x.y), fs_take(x.z, x.w));
}
__device__ __forceinline__ void fs_split8(float4 x, float4 y, uint4& hi, uint4& mid, uint4& lo) {
    x.x *= FS_UP, x.y *= FS_UP, x.z *= FS_UP, x.w *= FS_UP, y.x *= FS_UP, y.y *= FS_UP, y.z *= FS_UP, y.w *= FS_UP;
    hi = make_uint4(fs_take(x.x, x.y), fs_take(x.z, x.w), fs_take(y.x, y.y), fs_take(y.z, y.w));
    mid = make_uint4(fs_take(x.x, x.y), fs_take(x.z, x.w), fs_take(y.x, y.y), fs_take(y.z, y.w));
    lo = make_uint4(fs_take(x.x, x.y), fs_take(x.z, x.w), fs_take(y.x, y.y), fs_take(y.z, y.w));
}

// A as the product reads it: [ceil(M/32) blocks][ceil(K/16) steps][3 parts][64 lanes][8 values], lane l the row
// l % 32 of the block at k = 16 step + 8 (l / 32) .. + 8; zero beyond M and K.  A wave per (block, step).
__global__ __launch_bounds__(256) void fs_split_kernel(const float* __restrict__ A, uint4* __restrict__ out, int M, int K, int lda,
                                                       int steps, int vec) {
    const int lane = threadIdx.x & 63, step = blockIdx.x * 4 + (threadIdx.x >> 6), block = blockIdx.y;
    if (step >= steps) return;
    const int row = block * 32 + (lane & 31), k = step * FS_STEP + 8 * (lane >> 5);
    float4 x = make_float4(0.f, 0.f, 0.f, 0.f), y = x;
    if (row < M) {
        const float* p = A + (size_t)row * lda + k;
        if (vec && k + 8 <= K) {
            x = *reinterpret_cast<const float4*>(p);
            y = *reinterpret_cast<const float4*>(p + 4);
        } else {
            x.x = k < K ? p[0] : 0.f;
            x.y = k + 1 < K ? p[1] : 0.f;
            x.z = k + 2 < K ? p[2] : 0.f;
            x.w = k + 3 < K ? p[3] : 0.f;
            y.x = k + 4 < K ? p[4] : 0.f;
            y.y = k + 5 < K ? p[5] : 0.f;
            y.z = k + 6 < K ? p[6] : 0.f;
            y.w = k + 7 < K ? p[7] : 0.f;
        }
    }
    uint4 hi, mid, lo;
    fs_split8(x, y, hi, mid, lo);
    uint4* o = out + ((size_t)block * steps + step) * 192 + lane;
    o[0] = hi;
    o[64] = mid;
    o[128] = lo;
}

// tl_load_to_lds, the address made a scalar; waited for where FS_LANDED says so
__device__ __forceinline__ void fs_load_to_lds(const void* g, void* lds_base) {
    tl_load_to_lds(g, (uint32_t)__builtin_amdgcn_readfirstlane((int)tl_lds_address(lds_base)));
}
// at most N of this wave's loads are still on their way, and its LDS reads are done
#define FS_LANDED(N) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory")

#define FS_MUL_ONE(ACC, A_, W_)                                                                                              \
    ACC = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(fs_bf16x8, A_), __builtin_bit_cast(fs_bf16x8, W_), ACC, 0, 0, 0);

// MB blocks of 32 rows, FS_WAVES waves side by side with NB blocks of 32 columns each.  PARTS: blockIdx.y is a segment
// of K and C the workspace [segments][M][N]; else the whole K, C holding the sum of the segments so far (a lane reads
// and writes its own elements only).
// Work-groups of one XCD (every eighth in the order of their ids) take the row tiles of one column tile in turn, so
// that W is fetched into an L2 once and the rows are what its work-groups share at a time.
// RAW (17 to 32 rows, 16-byte aligned, K a multiple of four and one segment): one launch, the rows split by the work-group that
// uses them.  What bounds such a product is the chain of one element's products, six a step that wait for each other (0.25 us a
// step with what lies between), and ahead of it a launch and two waits for memory.  So a wave's eight rows come by whole lines
// of 128 bytes, a chunk of 24 steps at a time with the next one on its way, and go to LDS as parts once; the weights go from memory to
// registers, three groups of four steps ahead, and the next step's are split between a step's products, where nothing else would
// run; a barrier per chunk.  17 and 32 rows of 1,152 x K, us: parts beforehand / here / the float instruction: K = 64 7.2, 7.9 /
// 5.3, 5.9 / 4.8, 5.1; 128 8.6, 9.4 / 6.2, 6.8 / 6.4, 6.7; 256 11.7, 12.4 / 8.1, 8.7 / 9.7, 10.1; 896 26, 27 / 18, 19 / 26, 27;
// 2,048 52, 53 / 35, 36 / 56, 56.  (Waves that fetched and split 16 k at a time between barriers: 64 5.2, 128 7.1, 256 11.1; left to
// the compiler, the splitting ran ahead of the products: 2,048 40.)
template <int MB, int NB, int STAGES, bool PARTS, bool RAW>
__global__ __launch_bounds__(FS_WAVES * 64, MB * NB > 8 ? 1 : 2) void fs_gemm_kernel(
    const uint4* __restrict__ As, const float* __restrict__ A, const float* __restrict__ Ws, const float* __restrict__ bias,
    float* __restrict__ C, int M, int N, int K, int lda, int ldc, int steps) {
    extern __shared__ uint4 fs_lds[];
    static_assert(!RAW || (MB == 1 && NB == 1 && !PARTS), "unsplit rows come in one block, with the whole of a short K");
    static_assert(FS_RAW_K <= FS_SEG && FS_RAW_CHUNK % (3 * FS_RAW_GROUP) == 0 && FS_RAW_CHUNK % 2 == 0, "RAW: one segment, whole turns of three groups");
    constexpr int CHUNKS = MB * 3, LA = (CHUNKS + FS_WAVES - 1) / FS_WAVES, LW = NB * 2, STAGE = (CHUNKS + FS_WAVES * LW) * 64;
    constexpr int BN = FS_WAVES * NB * 32;
    const int blocks = (M + 31) / 32, mtiles = (blocks + MB - 1) / MB, ntiles = (N + BN - 1) / BN;
    const int local = blockIdx.x >> 3;
    const int nt = (local / mtiles) * 8 + (blockIdx.x & 7), mt = local % mtiles;
    if (nt >= ntiles) return;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int b0 = mt * MB, n0 = (nt * FS_WAVES + wave) * NB * 32;
    const int first = PARTS ? blockIdx.y * FS_SEG_STEPS : 0;
    const int last = PARTS ? min(first + FS_SEG_STEPS, steps) : steps;

    const uint4* ap[LA];
    const uint4* wp[LW];
#pragma unroll
    for (int i = 0; i < LA; ++i) {
        const int c = min(wave + i * FS_WAVES, CHUNKS - 1);            // a wave without a piece of its own repeats the last one
        ap[i] = As + ((size_t)min(b0 + c / 3, blocks - 1) * steps + first) * 192 + (c % 3) * 64 + lane;
    }
#pragma unroll
    for (int j = 0; j < LW; ++j)
        wp[j] = reinterpret_cast<const uint4*>(Ws) + ((size_t)min(n0 / 16 + j, (N + 15) / 16 - 1) * steps + first) * 64 + lane;
    int ahead = first;                   // the step that is fetched next; the last one again at the end
    auto fetch = [&](int buf) {
        uint4* stage = fs_lds + buf * STAGE;
#pragma unroll
        for (int i = 0; i < LA; ++i) fs_load_to_lds(ap[i], stage + min(wave + i * FS_WAVES, CHUNKS - 1) * 64);
#pragma unroll
        for (int j = 0; j < LW; ++j) fs_load_to_lds(wp[j], stage + (CHUNKS + wave * LW + j) * 64);
        if (++ahead < last) {
#pragma unroll
            for (int i = 0; i < LA; ++i) ap[i] += 192;
#pragma unroll
            for (int j = 0; j < LW; ++j) wp[j] += 64;
        }
    };
    fs_f32x16 acc[MB][NB];
    auto clear = [&]() {
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int j = 0; j < NB; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
    };
    // this lane holds rows 8 (r / 4) + 4 (lane / 32) + r % 4 of a block and one column
    float* out = PARTS ? C + (size_t)blockIdx.y * M * N : C;
    const size_t ld = PARTS ? N : ldc;
    const int row0 = b0 * 32 + 4 * (lane >> 5);
    auto store = [&](int s0, int s1) {       // the sums over steps [s0, s1), a segment
        const bool first_seg = s0 == 0, last_seg = s1 == steps;
        const bool inside = RAW && M == MB * 32 && n0 + NB * 32 <= N;      // no element's place is looked at
        int row = row0, col = n0 + (lane & 31);
        asm volatile("" : "+v"(row), "+v"(col));       // addresses and bounds are made here, not kept through the loop over k
        uint32_t again[(MB * NB + 1) / 2];             // elements to compute again: sixteen bits per block
#pragma unroll
        for (int u = 0; u < (MB * NB + 1) / 2; ++u) again[u] = 0;
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            const int n = col + j * 32;
            const float b = !PARTS && bias && last_seg && n < N ? bias[n] : 0.f;
            float* o = out + (size_t)row * ld + n;
#pragma unroll
            for (int i = 0; i < MB; ++i)
#pragma unroll
                for (int q = 0; q < 4; ++q) {          // four rows at a time: a few addresses and sums in registers
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const float v = acc[i][j][4 * q + r] * FS_DOWN;
                        if (inside || (n < N && row + i * 32 + 8 * q + r < M)) {
                            const bool fine = fabsf(v) < INFINITY;         // else the sum so far stays where it is
                            again[(i * NB + j) / 2] |= fine ? 0u : 1u << (((i * NB + j) & 1) * 16 + 4 * q + r);
                            const float so_far = !PARTS && !first_seg ? o[r * ld] : 0.f;
                            o[r * ld] = fine ? (!PARTS && !first_seg ? so_far + v : v) + b : so_far;
                        }
                    }
                    o += 8 * ld;
                    asm volatile("" ::: "memory");
                }
        }
        bool any = false;
#pragma unroll
        for (int u = 0; u < (MB * NB + 1) / 2; ++u) any |= again[u] != 0;
        if (!__any(any)) return;
        // the marked elements from the values themselves
        for (int block = 0; block < MB * NB; ++block) {
            uint32_t marks = 0;
#pragma unroll
            for (int u = 0; u < (MB * NB + 1) / 2; ++u) marks = block >> 1 == u ? again[u] : marks;
            marks = marks >> (block & 1) * 16 & 0xffffu;
            if (!__any(marks != 0)) continue;
            int here = lane;
            asm volatile("" : "+v"(here));             // nothing of this is made ahead of the loop over k
            const int i = block / NB, n = n0 + block % NB * 32 + (here & 31), half = here >> 5;
            const float* a = A + (size_t)min((b0 + i) * 32 + (here & 31), M - 1) * lda + half;        // rows and columns that
            const float* w = Ws + ((size_t)min(n >> 4, (N + 15) / 16 - 1) * steps * 64 + (n & 15)) * 4 + half;   // are not there: others
            fs_f32x16 sum;
#pragma unroll
            for (int r = 0; r < 16; ++r) sum[r] = 0.f;
            for (int s = s0; s < s1; ++s) {
                float av[8], wv[8];                    // k = 16 s + 2 t + half
#pragma unroll
                for (int t = 0; t < 8; ++t) {
                    av[t] = s * FS_STEP + 2 * t + half < K ? a[s * FS_STEP + 2 * t] : 0.f;
                    wv[t] = w[(size_t)s * 256 + (t >> 1) * 64 + (t & 1) * 2];
                }
#pragma unroll
                for (int t = 0; t < 8; ++t) sum = __builtin_amdgcn_mfma_f32_32x32x2f32(av[t], wv[t], sum, 0, 0, 0);
            }
            const float b = !PARTS && bias && last_seg && n < N ? bias[n] : 0.f;
#pragma unroll
            for (int r = 0; r < 16; ++r)
                if (marks >> r & 1) {
                    float* o = out + (size_t)((b0 + i) * 32 + 4 * half + 8 * (r >> 2) + (r & 3)) * ld + n;
                    *o = (!PARTS && !first_seg ? *o + sum[r] : sum[r]) + b;
                }
        }
    };
    clear();
    if constexpr (RAW) {
        const float4* wl = reinterpret_cast<const float4*>(Ws) + (size_t)min(n0 / 16 + (lane >> 4 & 1), (N + 15) / 16 - 1) * steps * 64 +
                           (lane >> 5) * 32 + (lane & 15);
        const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
        float4 w[3][FS_RAW_GROUP][2];                                // three groups of steps on their way
        auto ask = [&](float4 (&to)[FS_RAW_GROUP][2], int s) {       // a step past the last one: the last one again, not used
            if (s >= steps) return;
#pragma unroll
            for (int u = 0; u < FS_RAW_GROUP; ++u) {
                const size_t at = (size_t)min(s + u, steps - 1) * 64;
                to[u][0] = wl[at];
                to[u][1] = wl[at + 16];
            }
        };
        // One step's products, each of which waits for the one before, and between them the splitting of the next step's weights.
        uint4 x[3];
        auto step = [&](const uint4* rows_of, const float4 (&next)[2]) {
            uint4 a[3];
#pragma unroll
            for (int p = 0; p < 3; ++p) a[p] = rows_of[p * 64];
            float f[8] = {next[0].x, next[0].y, next[0].z, next[0].w, next[1].x, next[1].y, next[1].z, next[1].w};
            uint32_t y[12];
            auto take = [&](int t) { y[t] = fs_take(f[2 * (t & 3)], f[2 * (t & 3) + 1]); };
#define FS_AMONG(PA, PW, ...)                   \
    FS_MUL_ONE(acc[0][0], a[PA], x[PW])         \
    __VA_ARGS__;                                \
    __builtin_amdgcn_sched_barrier(0);
            FS_AMONG(0, 2, _Pragma("unroll") for (int i = 0; i < 8; ++i) f[i] *= FS_UP; take(0))
            FS_AMONG(2, 0, take(1); take(2))
            FS_AMONG(1, 1, take(3); take(4))
            FS_AMONG(0, 1, take(5); take(6))
            FS_AMONG(1, 0, take(7); take(8))
            FS_AMONG(0, 0, take(9); take(10); take(11))
#undef FS_AMONG
#pragma unroll
            for (int p = 0; p < 3; ++p) x[p] = make_uint4(y[4 * p], y[4 * p + 1], y[4 * p + 2], y[4 * p + 3]);
        };
        auto multiply = [&](float4 (&from)[FS_RAW_GROUP][2], const float4 (&then)[FS_RAW_GROUP][2], int s, int c0) {
            const uint4* rows_of = fs_lds + (s - c0) * 192 + lane;
#pragma unroll
            for (int u = 0; u < FS_RAW_GROUP; ++u)
                if (s + u < steps) step(rows_of + u * 192, u + 1 < FS_RAW_GROUP ? from[u + 1 < FS_RAW_GROUP ? u + 1 : 0] : then[0]);
            ask(from, s + 3 * FS_RAW_GROUP);
        };
        // Rows: a wave has eight of them, a lane 16 bytes of one in a line of 128 (two steps), so that no line is asked for twice.
        constexpr int LINES = FS_RAW_CHUNK / 2;
        const int row = wave * 8 + (lane >> 3), unit = 4 * (lane & 7);
        const float* al = A + (size_t)min(row, M - 1) * lda;
        uint2* part = reinterpret_cast<uint2*>(fs_lds) + ((lane >> 2 & 1) * 192 + (lane >> 1 & 1) * 32 + row) * 2 + (lane & 1);
        float4 rows[LINES];
        auto ask_rows = [&](int c0) {
#pragma unroll
            for (int i = 0; i < LINES; ++i)
                if (c0 + 2 * i < steps) rows[i] = *reinterpret_cast<const float4*>(al + min((c0 + 2 * i) * FS_STEP + unit, K - 4));
        };
#pragma unroll
        for (int i = 0; i < LINES; ++i) rows[i] = zero;
        ask_rows(0);
#pragma unroll
        for (int g = 0; g < 3; ++g) {
#pragma unroll
            for (int u = 0; u < FS_RAW_GROUP; ++u) w[g][u][0] = w[g][u][1] = zero;
            ask(w[g], g * FS_RAW_GROUP);
        }
        for (int c0 = 0; c0 < steps; c0 += FS_RAW_CHUNK) {
            const int here = min(steps - c0, FS_RAW_CHUNK);
            if (c0) __syncthreads();                     // every wave has read the rows before
#pragma unroll
            for (int i = 0; i < LINES; ++i)
                if (2 * i < here) {
                    uint2 hi, mid, lo;
                    fs_split4((c0 + 2 * i) * FS_STEP + unit < K ? rows[i] : zero, hi, mid, lo);
                    uint2* to = part + i * 768;
                    to[0] = hi;
                    to[128] = mid;
                    to[256] = lo;
                }
            if (c0 + FS_RAW_CHUNK < steps) ask_rows(c0 + FS_RAW_CHUNK);
            if (c0 == 0) fs_split8(w[0][0][0], w[0][0][1], x[0], x[1], x[2]);
            __syncthreads();
            for (int s = c0; s < c0 + here; s += 3 * FS_RAW_GROUP) {
                multiply(w[0], w[1], s, c0);
                if (s + FS_RAW_GROUP < c0 + here) multiply(w[1], w[2], s + FS_RAW_GROUP, c0);
                if (s + 2 * FS_RAW_GROUP < c0 + here) multiply(w[2], w[0], s + 2 * FS_RAW_GROUP, c0);
            }
        }
        store(0, steps);
        return;
    }
    for (int i = 0; i < STAGES - 1; ++i) fetch(i);
    int buf = 0;
    const int wfrag = (CHUNKS + wave * LW) * 64 + ((lane >> 4) & 1) * 64 + (lane >> 5) * 32 + (lane & 15);
    for (int s = first; s < last; ++s) {
        FS_LANDED((STAGES - 2) * (LA + LW));   // step s is here; later ones may be on their way
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        fetch(buf == 0 ? STAGES - 1 : buf - 1);   // the buffer of step s - 1, which every wave has read
        const uint4* stage = fs_lds + buf * STAGE;
        uint4 w[NB][3];
#pragma unroll
        for (int j = 0; j < NB; ++j)
            fs_split8(__builtin_bit_cast(float4, stage[wfrag + j * 128]), __builtin_bit_cast(float4, stage[wfrag + j * 128 + 16]),
                      w[j][0], w[j][1], w[j][2]);
        // two blocks' products in turn, so that none waits for the one before it
        constexpr int IB = NB > 1 || MB == 1 ? 1 : 2;
#pragma unroll
        for (int i = 0; i < MB; i += IB) {
            uint4 a[IB][3];
#pragma unroll
            for (int b = 0; b < IB; ++b)
#pragma unroll
                for (int p = 0; p < 3; ++p) a[b][p] = stage[((i + b) * 3 + p) * 64 + lane];
#define FS_MUL(PA, PW)                                                                                                       \
    _Pragma("unroll") for (int b = 0; b < IB; ++b) _Pragma("unroll") for (int j = 0; j < NB; ++j) FS_MUL_ONE(acc[i + b][j], a[b][PA], w[j][PW])
            FS_MUL(0, 2)
            FS_MUL(2, 0)
            FS_MUL(1, 1)
            FS_MUL(0, 1)
            FS_MUL(1, 0)
            FS_MUL(0, 0)
#undef FS_MUL
        }
        if (!PARTS && (s + 1) % FS_SEG_STEPS == 0 && s + 1 < last) {
            store(s + 1 - FS_SEG_STEPS, s + 1);
            clear();
        }
        buf = buf == STAGES - 1 ? 0 : buf + 1;
    }
    FS_LANDED(0);                        // nothing may land in LDS that is no longer this work-group's
    store(PARTS ? first : (last - 1) / FS_SEG_STEPS * FS_SEG_STEPS, last);
}

// The segments' sums in ascending order, as the product adds them where it has the whole K.  VEC: four columns a
// thread (N and ldc multiples of four, everything aligned).
template <bool VEC>
__global__ __launch_bounds__(256) void fs_add_kernel(const float* __restrict__ parts, const float* __restrict__ bias,
                                                     float* __restrict__ C, int M, int N, int ldc, int nseg) {
    const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * (VEC ? 4 : 1), all = (size_t)M * N;
    if (i >= all) return;
    const int m = (int)(i / N), n = (int)(i - (size_t)m * N);
    if (VEC) {
        float4 sum = *reinterpret_cast<const float4*>(parts + i);
        for (int g = 1; g < nseg; ++g) {
            const float4 p = *reinterpret_cast<const float4*>(parts + (size_t)g * all + i);
            sum.x += p.x, sum.y += p.y, sum.z += p.z, sum.w += p.w;
        }
        if (bias) sum.x += bias[n], sum.y += bias[n + 1], sum.z += bias[n + 2], sum.w += bias[n + 3];
        *reinterpret_cast<float4*>(C + (size_t)m * ldc + n) = sum;
    } else {
        float sum = parts[i];
        for (int g = 1; g < nseg; ++g) sum += parts[(size_t)g * all + i];
        C[(size_t)m * ldc + n] = sum + (bias ? bias[n] : 0.f);
    }
}

// The tiles (row blocks and column blocks of a wave) with what was measured on the products of 7B and 0.5B models: a step of
// 16 k takes a work-group `alone` us when its CU has nothing else (the chain barrier - reads - products), and a CU gets
// through one in `shared` us when it holds as many as fit.  The tile, and whether K is dealt out by segments, is the
// least estimate; e.g. at 2,048 rows gate/up (37,888 x 3,584) 2.8 ms in tiles of 128 x 256 (200 TFLOP/s; tiles of 256 rows
// 3.1, of 128 x 128 3.0), down (3,584 x 18,944) 1.55 ms with K dealt out (1.66 against 1.72 when both were tried), where the float
// instruction takes 4.8 and 2.8; at 40 rows down takes 93 us dealt out (97 against 480).
struct FsTile {
    int mb, nb, fit;
    double alone, shared;
};
static const FsTile fs_tiles[] = {{4, 2, 2, 1.90, 1.36}, {4, 1, 2, 0.95, 0.71}, {2, 1, 3, 0.56, 0.41}, {1, 1, 4, 0.43, 0.26}};

static int fs_choose(int M, int N, int K, bool* parts) {
    const int blocks = tl_ceil_div(M, 32), steps = tl_ceil_div(K, FS_STEP), nseg = tl_ceil_div(K, FS_SEG);
    int best = 3;
    double cost = 1e300;
    for (int t = 0; t < 4; ++t) {
        const FsTile& z = fs_tiles[t];
        if (z.mb > 1 && z.mb / 2 >= blocks) continue;                  // half of it holds all the rows
        const double tiles = (double)tl_ceil_div(blocks, z.mb) * tl_ceil_div(N, FS_WAVES * 32 * z.nb);
        for (int cut = 0; cut < (nseg > 1 && nseg <= 65535 && (long long)M * N <= FS_MOST_SUMS / nseg ? 2 : 1); ++cut) {
            const double each = tiles * (cut ? nseg : 1) / FS_CUS, whole = (double)(long long)(each + 0.999999);
            const double on_a_cu = whole < 4 ? whole : each + 0.5, turns = (double)(long long)((whole + z.fit - 1) / z.fit);
            const double step = turns * z.alone > on_a_cu * z.shared ? turns * z.alone : on_a_cu * z.shared;
            const double us = step * steps / (cut ? nseg : 1) + (cut ? 4.0 + 8.0 * M * N * nseg / 6e6 : 0.0);
            if (us < cost) cost = us, best = t, *parts = cut != 0;
        }
    }
    return best;
}

// The tile that tl_gemm_float_split takes (an index of fs_tiles), plus 4 where K is dealt out by segments.
extern "C" int tl_gemm_float_split_tile(int M, int N, int K) {
    bool parts = false;
    const int tile = fs_choose(M, N, K, &parts);
    return tile + (parts ? 4 : 0);
}

// Whether rows that start 16-byte aligned are split where they are used and need no workspace for their parts: where every
// work-group of 128 columns has a CU of its own, and, for a K that leaves little else to do, where two share one (32 rows, us,
// parts beforehand and not: 32,768 x 512 20.1 and 20.3, x 2,048 67 and 65; 37,888 x 128 10.6 and 9.9, x 160 11.7 and 11.9, x 512 21.6
// and 22.3, where more columns' work-groups split the rows again than there are CUs).
extern "C" int tl_gemm_float_split_takes_rows(int M, int N, int K, int lda) {
    const int groups = tl_ceil_div(N, FS_WAVES * 32);
    return M <= 32 && K >= FS_STEP && K <= FS_RAW_K && K % 4 == 0 && lda % 4 == 0 &&
                   (groups <= FS_CUS || (K < 160 && groups <= 2 * FS_CUS)) ? 1 : 0;
}

// Floats of workspace that tl_gemm_float_split needs for the segments' sums (0: none).
extern "C" long long tl_gemm_float_split_workspace(int M, int N, int K) {
    if (M <= 0 || N <= 0 || K <= 0) return 0;
    bool parts = false;
    fs_choose(M, N, K, &parts);
    return parts ? (long long)tl_ceil_div(K, FS_SEG) * M * N : 0;
}

// A float [M, K] with row stride lda; Ws float [ceil(N/16), ceil(K/16), 64, 4] (the matrix-core ordered copy of W, zero
// where it pads); split: workspace of ceil(M/32) * ceil(K/16) * 3 KB, or null where
// tl_gemm_float_split_takes_rows says that the rows are split where they are used; ws: tl_gemm_float_split_workspace floats.
extern "C" int tl_gemm_float_split(const float* A, const float* Ws, const float* bias, float* C, void* split, float* ws, int M,
                                   int N, int K, int lda, int ldc, hipStream_t stream) {
    TL_CHECK_ARG(M >= 0 && N > 0 && K > 0, "tl_gemm_float_split: bad sizes M=%d N=%d K=%d", M, N, K);
    TL_CHECK_ARG(lda >= K && ldc >= N, "tl_gemm_float_split: row strides lda=%d ldc=%d too small for K=%d N=%d", lda, ldc, K, N);
    TL_CHECK_ARG((uintptr_t)Ws % 16 == 0 && (uintptr_t)split % 16 == 0, "tl_gemm_float_split: the weight copy and the workspace must be 16-byte aligned");
    if (M == 0) return 0;
    const int steps = tl_ceil_div(K, FS_STEP), blocks = tl_ceil_div(M, 32), nseg = tl_ceil_div(K, FS_SEG);
    TL_CHECK_ARG(blocks <= 65535, "tl_gemm_float_split: %d rows are too many for one launch", M);
    bool parts = false;
    const int tile = fs_choose(M, N, K, &parts);
    const int mtiles = tl_ceil_div(blocks, fs_tiles[tile].mb), ntiles = tl_ceil_div(N, FS_WAVES * 32 * fs_tiles[tile].nb);
    const long long grid = (long long)mtiles * tl_ceil_div(ntiles, 8) * 8;
    TL_CHECK_ARG(grid < (1ll << 31), "tl_gemm_float_split: M=%d N=%d are too many tiles for one launch", M, N);
    TL_CHECK_ARG(!parts || ws, "tl_gemm_float_split: no workspace for the segments' sums");
    const int vec = ((uintptr_t)A % 16 == 0 && lda % 4 == 0) ? 1 : 0;
    TL_CHECK_ARG(split || (tl_gemm_float_split_takes_rows(M, N, K, lda) && vec && tile == 3 && !parts),
                 "tl_gemm_float_split: M=%d K=%d lda=%d need a workspace for the rows' parts", M, K, lda);
    if (split)
        hipLaunchKernelGGL(fs_split_kernel, dim3(tl_ceil_div(steps, 4), blocks), dim3(256), 0, stream, A, (uint4*)split, M, K, lda, steps, vec);
#define FS_GO(MB, NB, ST, P, RAW, LDS)                                                                                           \
    hipLaunchKernelGGL((fs_gemm_kernel<MB, NB, ST, P, RAW>), dim3((unsigned)grid, P ? nseg : 1), dim3(FS_WAVES * 64), LDS, stream, \
                       (const uint4*)split, A, Ws, bias, P ? ws : C, M, N, K, lda, ldc, steps)
#define FS_GO_P(MB, NB, ST)                                                               \
    if (parts) FS_GO(MB, NB, ST, true, false, ST * (MB * 3 + FS_WAVES * NB * 2) * 1024); \
    else FS_GO(MB, NB, ST, false, false, ST * (MB * 3 + FS_WAVES * NB * 2) * 1024)
    if (tile == 0) {
        FS_GO_P(4, 2, 2);
    } else if (tile == 1) {
        FS_GO_P(4, 1, 3);
    } else if (tile == 2) {
        FS_GO_P(2, 1, 3);
    } else if (split) {
        FS_GO_P(1, 1, 3);
    } else {
        FS_GO(1, 1, 1, false, true, (steps < FS_RAW_CHUNK ? (steps + 1) / 2 * 2 : FS_RAW_CHUNK) * 3072);
    }
#undef FS_GO_P
#undef FS_GO
    if (parts) {
        const long long all = (long long)M * N;
        TL_CHECK_ARG((all + 255) / 256 < (1ll << 31), "tl_gemm_float_split: M=%d N=%d are too many sums for one launch", M, N);
        if (N % 4 == 0 && ldc % 4 == 0 && (uintptr_t)C % 16 == 0 && (uintptr_t)ws % 16 == 0)
            hipLaunchKernelGGL(fs_add_kernel<true>, dim3((unsigned)((all / 4 + 255) / 256)), dim3(256), 0, stream, ws, bias, C, M, N, ldc, nseg);
        else
            hipLaunchKernelGGL(fs_add_kernel<false>, dim3((unsigned)((all + 255) / 256)), dim3(256), 0, stream, ws, bias, C, M, N, ldc, nseg);
    }
    TL_CHECK_LAUNCH("tl_gemm_float_split");
    return 0;
}
