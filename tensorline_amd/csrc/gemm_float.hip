// C[M, N] = A[M, K] * W[N, K]^T (+ bias[N]) in float for more than 16 rows, on the half-precision matrix
// instruction (v_mfma_f32_32x32x16_f16): the 32-bit path's product of prompts and large batches.
//
// A float is the sum of two halves of 11 significant bits, each rounded to nearest, the second the rest of the first (splitting floats
// into shorter ones so that products are exact is Dekker's, Numerische Mathematik 18, 1971): 22 to 23 bits with the second one's
// sign, off by 4e-8 of the float in the mean.  Halves reach from 2^-24 to 2^16, so the values of a segment of a row (FS_SEG k) are
// multiplied by a power of two that brings its largest into [2^14, 2^15), which comes out again of the segment's sum.  Of the four
// partial products the three with a first part in them are taken, small ones first, each exact; the one left out comes to 2^-22 of the
// product at most, 4e-8 in the mean.  What the result is off the exact one, 2-norm, 256 rows, here / three bfloat16 parts and six products
// on v_mfma_f32_32x32x16_bf16, as it was before / v_mfma_f32_16x16x4_f32, in 1e-7:
//                                    K = 64              128                 896                 3,584               18,944
//   normal numbers                   1.13 1.09 1.44      1.44 1.64 2.05      3.36 4.52 5.36      4.79 6.67 10.7      5.24 7.61 24.5
//   positive (uniform in [0, 1))     0.65 0.83 1.14      0.92 1.24 1.58      2.57 2.93 4.20      2.66 2.75 8.43      1.42 1.43 20.8
//   one column 3,000 times the rest  1.35 1.06 1.64      1.64 1.51 2.34      3.87 3.88 6.16      4.61 4.57 12.3      6.74 6.85 28.3
//   fifth powers of normal numbers   1.22 1.25 1.56      1.53 1.60 2.09      3.43 4.13 5.12      4.81 5.80 10.2      5.24 6.49 23.1
// Half the products are half the roundings of the sums, which is more than the parts lose from K = 896 on.  Products of a K below
// 64 go to the float instruction.
//
// Values below 2^-18 of their segment's largest lose bits of the second half: it is off by up to 2^-25 after scaling, 2^-40 of the
// largest.  Beside the sum of the other products that is nothing, unless those cancel or vanish (a column that is zero where the row
// is large).  So a result below FS_SMALL sqrt(length of the segment), which is 2^20 times what such values can be off by in the worst
// case and 2^23 times what they usually are, is computed again from the floats, one at a time: some 2 in 100,000 of normal
// numbers' products; results of segments that are all zero are not.
//
// What is split where: the rows of A once, by a pass of its own, into the order in which the product reads
// them (fs_split_kernel); W, which may be most of the GPU's memory, stays float and is split in registers by the wave that owns its
// columns, from the matrix-core ordered copy that the few-row product streams as well.  The powers of two of W's rows are asked for
// beforehand (tl_gemm_float_ranges), once for a matrix that is kept.  A wave owns 32 columns and all the rows of its work-group
// (up to 256): 40 vector instructions beside 3 matrix instructions per 32 x 32 block and 16 k.
//
// Per step of 16 k a work-group holds 2 KB of A per 32 rows and 8 KB of W in LDS, in the layout the fragments are read in (a fragment is
// 1 KB, lane after lane: no bank conflicts), fetched two or three steps ahead by global_load_lds; one barrier per step.  A step's weights are
// split, and its first rows read, between the products of the step before.
// What bounds it at thousands of rows: the power that products of random halves take; 2,048 rows of 37,888 x 3,584 1.85 ms (300 TFLOP/s,
// 0.9 PFLOP/s of half products; three bfloat16 parts 2.80), all ones 1.55, halves that are bfloat16 numbers 1.67.  With W split ahead by a pass of
// its own and both operands straight from LDS, tiles of 256 x 256, the products alone take 1.53, with the pass and its 0.5 GB of
// workspace 1.74: not kept.  At a few hundred rows: the chain barrier - reads - products of a step, and rounds that do not come out even (513 rows of
// 17,920 x 1,536 225 -> 147 us, 256 of 3,584 x 18,944 270 -> 168, 33 of 2,048 x 1,536 43 -> 28).
//
// One output element is summed in one fixed order whatever the number of rows or the tile: k in segments of
// FS_SEG at absolute k, within a segment steps of 16 upwards with the three partial products of a step in one
// order, the segments' sums added in ascending order.  Few tiles (few rows of a narrow matrix) are spread
// over the GPU by segments, whose sums a second kernel adds in the same order.
//
// Values that are not finite make the split itself infinity minus infinity, and sums may pass the largest float: an element whose segment does
// not come out finite is computed again on the float instruction, so infinities, NaN and sums of any size give what they give
// there.  (A wave takes its blocks of 32 x 32 in turn: 2.5 ms for 2,048 rows of 4,608 x 3,584 with an infinity in every row, 0.4 without.)
#include "common.h"

#include <type_traits>

typedef _Float16 fs_half8 __attribute__((ext_vector_type(8)));
typedef _Float16 fs_half2 __attribute__((ext_vector_type(2)));
typedef float fs_f32x2 __attribute__((ext_vector_type(2)));
typedef float fs_f32x16 __attribute__((ext_vector_type(16)));

#define FS_STEP 16
#define FS_SEG 2048                      // k per segment
#define FS_SEG_STEPS (FS_SEG / FS_STEP)
#define FS_WAVES 4
#define FS_CUS 256
#define FS_MOST_SUMS (512LL << 18)       // floats at most of the segments' sums (512 MB): beyond, K stays whole
#define FS_TOP 14                        // a segment's largest value is brought to [2^14, 2^15)
#define FS_MOST_UP 126                   // by a factor that is a normal float
#define FS_SMALL 0x1.6ap9f               // times the root of a segment's length: results below are computed again
#define FS_RAW_K 2048                    // at most 32 aligned rows of a K up to this are split where they are used (RAW)
#define FS_RAW_GROUP 4                   // steps whose weights a wave asks for together
#define FS_RAW_CHUNK 24                  // steps whose rows are in LDS at a time

// The exponent of a segment's factor; FS_ZERO where all its values are zero.
#define FS_ZERO 127
__device__ __forceinline__ int fs_up(float most) {       // (what lies below 2^-112 takes the largest factor)
    return most == 0.f ? FS_ZERO : min(FS_TOP + 127 - (int)(__float_as_uint(most) >> 23 & 255u), FS_MOST_UP);
}
__device__ __forceinline__ float fs_factor(int up) { return __uint_as_float((uint32_t)(up + 127) << 23); }

// over the eight lanes that have a row (lanes 8 r .. 8 r + 7), without trips through LDS
#define FS_MOVED(V, CTRL) __builtin_amdgcn_update_dpp(0, (int)(V), CTRL, 0xf, 0xf, true)
__device__ __forceinline__ float fs_group_most(float v) {
    v = fmaxf(v, __int_as_float(FS_MOVED(__float_as_int(v), 0xB1)));       // quad_perm 1, 0, 3, 2
    v = fmaxf(v, __int_as_float(FS_MOVED(__float_as_int(v), 0x4E)));       // quad_perm 2, 3, 0, 1
    return fmaxf(v, __int_as_float(FS_MOVED(__float_as_int(v), 0x141)));   // row_half_mirror
}

// two floats as two halves, rounded to nearest even, and what is left of each
__device__ __forceinline__ uint32_t fs_take(float& a, float& b) {
    const fs_f32x2 v = {a, b};
    const fs_half2 h = __builtin_convertvector(v, fs_half2);
    const uint32_t bits = __builtin_bit_cast(uint32_t, h);
    // a - h, exact; the compiler makes a conversion and a subtraction of it
    asm("v_fma_mix_f32 %0, %1, -1.0, %0 op_sel_hi:[1,0,0]" : "+v"(a) : "v"(bits));
    asm("v_fma_mix_f32 %0, %1, -1.0, %0 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "+v"(b) : "v"(bits));
    return bits;
}
__device__ __forceinline__ uint32_t fs_rest(float a, float b) {
    const fs_f32x2 v = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, fs_half2));
}
// floats, their factor applied, as twice as many halves
__device__ __forceinline__ void fs_split4(float4 x, uint2& hi, uint2& lo) {
    hi = make_uint2(fs_take(x.x, x.y), fs_take(x.z, x.w));
    lo = make_uint2(fs_rest(x.x, x.y), fs_rest(x.z, x.w));
}
__device__ __forceinline__ void fs_split8(float4 x, float4 y, uint4& hi, uint4& lo) {
    hi = make_uint4(fs_take(x.x, x.y), fs_take(x.z, x.w), fs_take(y.x, y.y), fs_take(y.z, y.w));
    lo = make_uint4(fs_rest(x.x, x.y), fs_rest(x.z, x.w), fs_rest(y.x, y.y), fs_rest(y.z, y.w));
}
__device__ __forceinline__ void fs_times(float4& x, float f) { x.x *= f, x.y *= f, x.z *= f, x.w *= f; }
__device__ __forceinline__ float fs_most(float4 x) { return fmaxf(fmaxf(fabsf(x.x), fabsf(x.y)), fmaxf(fabsf(x.z), fabsf(x.w))); }

// A as the product reads it: [ceil(M/32) blocks][ceil(K/16) steps][2 parts][64 lanes][8 values], lane l the row
// l % 32 of the block at k = 16 step + 8 (l / 32) .. + 8; zero beyond M and K; and the rows' ranges [segments][32 ceil(M/32)].
// A work-group per eight rows and segment, whose values wait in registers until their rows' largest is known: a wave has 64 k of
// each row (every fourth 64), a lane eight.
#define FS_SPLIT_WAVES 4
__global__ __launch_bounds__(FS_SPLIT_WAVES * 64) void fs_split_kernel(const float* __restrict__ A, uint4* __restrict__ out,
                                                                     int* __restrict__ ranges, int M, int K, int lda, int steps,
                                                                     int vec) {
    constexpr int EACH = FS_SEG / 64 / FS_SPLIT_WAVES;
    __shared__ float most_of[FS_SPLIT_WAVES][8];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane >> 3, unit = lane & 7;
    const int seg = blockIdx.x, row = blockIdx.y * 8 + r, s1 = min((seg + 1) * FS_SEG_STEPS, steps);
    const int s0 = seg * FS_SEG_STEPS + wave * 4 + (unit >> 1);         // this lane's steps: s0, s0 + 16, ..
    float4 x[EACH], y[EACH];
    const float* line = A + (size_t)min(row, M - 1) * lda;
#pragma unroll
    for (int i = 0; i < EACH; ++i) {
        const int k = (s0 + i * 4 * FS_SPLIT_WAVES) * FS_STEP + 8 * (unit & 1);
        x[i] = y[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (row < M && s0 + i * 4 * FS_SPLIT_WAVES < s1) {
            const float* p = line + k;
            if (vec && k + 8 <= K) {
                x[i] = *reinterpret_cast<const float4*>(p);
                y[i] = *reinterpret_cast<const float4*>(p + 4);
            } else {
                x[i].x = k < K ? p[0] : 0.f;
                x[i].y = k + 1 < K ? p[1] : 0.f;
                x[i].z = k + 2 < K ? p[2] : 0.f;
                x[i].w = k + 3 < K ? p[3] : 0.f;
                y[i].x = k + 4 < K ? p[4] : 0.f;
                y[i].y = k + 5 < K ? p[5] : 0.f;
                y[i].z = k + 6 < K ? p[6] : 0.f;
                y[i].w = k + 7 < K ? p[7] : 0.f;
            }
        }
    }
    float most = 0.f;
#pragma unroll
    for (int i = 0; i < EACH; ++i) most = fmaxf(most, fmaxf(fs_most(x[i]), fs_most(y[i])));
    most = fs_group_most(most);
    if (unit == 0) most_of[wave][r] = most;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < FS_SPLIT_WAVES; ++w) most = fmaxf(most, most_of[w][r]);
    const int up = fs_up(most);
    const float f = fs_factor(up);
    if (threadIdx.x < 64 && unit == 0) ranges[(size_t)seg * gridDim.y * 8 + row] = up;
    uint4* to = out + (size_t)(row >> 5) * steps * 128 + (unit & 1) * 32 + (row & 31);
#pragma unroll
    for (int i = 0; i < EACH; ++i) {
        fs_times(x[i], f);
        fs_times(y[i], f);
        if (s0 + i * 4 * FS_SPLIT_WAVES < s1) {
            uint4 hi, lo;
            fs_split8(x[i], y[i], hi, lo);
            uint4* o = to + (size_t)(s0 + i * 4 * FS_SPLIT_WAVES) * 128;
            o[0] = hi;
            o[64] = lo;
        }
    }
}

// The ranges of a matrix, [segments][16 ceil(N/16)], from its ordered copy, or (ORDER: from W [N, 4 units], aligned) with that copy, which is then
// one pass over W and not another one behind it: 37,888 x 3,584 229 us where the copy alone takes 198 and the ranges from it 103.
// A work-group per 16 rows and segment.
#define FS_RANGE_WAVES 8
template <bool ORDER>
__global__ __launch_bounds__(FS_RANGE_WAVES * 64) void fs_ranges_kernel(const float4* __restrict__ W, float4* __restrict__ Ws, int* __restrict__ ranges,
                                                                      int N, int units, int tiles, int steps) {
    constexpr int EACH = FS_SEG_STEPS / FS_RANGE_WAVES;
    __shared__ float most_of[FS_RANGE_WAVES][16];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, tile = blockIdx.x, seg = blockIdx.y;
    const int s0 = seg * FS_SEG_STEPS + wave, s1 = min((seg + 1) * FS_SEG_STEPS, steps);
    float4 x[EACH];
#pragma unroll
    for (int i = 0; i < EACH; ++i) {
        const int s = s0 + i * FS_RANGE_WAVES, u = s * 4 + (lane >> 4);
        x[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        if constexpr (ORDER) {
            if (s < s1 && u < units && tile * 16 + r < N) x[i] = W[(size_t)(tile * 16 + r) * units + u];
        } else {
            if (s < s1) x[i] = Ws[((size_t)tile * steps + s) * 64 + lane];
        }
    }
    if constexpr (ORDER) {
#pragma unroll
        for (int i = 0; i < EACH; ++i)
            if (s0 + i * FS_RANGE_WAVES < s1) Ws[((size_t)tile * steps + s0 + i * FS_RANGE_WAVES) * 64 + lane] = x[i];
    }
    float most = 0.f;
#pragma unroll
    for (int i = 0; i < EACH; ++i) most = fmaxf(most, fs_most(x[i]));
    most = fmaxf(most, __shfl_xor(most, 16));
    most = fmaxf(most, __shfl_xor(most, 32));
    if (lane < 16) most_of[wave][r] = most;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < FS_RANGE_WAVES; ++w) most = fmaxf(most, most_of[w][r]);
    if (threadIdx.x < 16) ranges[((size_t)seg * tiles + tile) * 16 + r] = fs_up(most);
}

// tl_load_to_lds, the address made a scalar; waited for where FS_LANDED says so
__device__ __forceinline__ void fs_load_to_lds(const void* g, void* lds_base) {
    tl_load_to_lds(g, (uint32_t)__builtin_amdgcn_readfirstlane((int)tl_lds_address(lds_base)));
}
// at most N of this wave's loads are still on their way, and its LDS reads are done
#define FS_LANDED(N) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory")

#define FS_MUL_ONE(ACC, A_, W_)                                                                                              \
    ACC = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(fs_half8, A_), __builtin_bit_cast(fs_half8, W_), ACC, 0, 0, 0);

// MB blocks of 32 rows, FS_WAVES waves side by side with 32 columns each.  PARTS: blockIdx.y is a segment
// of K and C the workspace [segments][M][N]; else the whole K, C holding the sum of the segments so far (a lane reads
// and writes its own elements only).
// Work-groups of one XCD (every eighth in the order of their ids) take the row tiles of one column tile in turn, so
// that W is fetched into an L2 once and the rows are what its work-groups share at a time.
// RAW (17 to 32 rows, 16-byte aligned, K a multiple of four and one segment): one launch, the rows split by the work-group that
// uses them.  What bounds such a product is the chain of one element's products, three a step that wait for each other, and ahead of it
// waits for memory: the rows once for their largest values, and again by chunks.  A wave's eight rows come by whole lines
// of 128 bytes, a chunk of 24 steps at a time with the next one on its way, and go to LDS as parts once; the weights go from memory to
// registers, three groups of four steps ahead, and the next step's are split between a step's products, where nothing else would
// run; a barrier per chunk.  17 and 32 rows, us, parts beforehand / here / three bfloat16 parts: 1,152 x 896 23, 24 / 17, 18 / 17, 18;
// 2,048 x 1,536 34, 35 / 26, 27 / 26, 27; 17,920 x 1,536 37, 38 / 33, 34 / 32, 33; 9,728 x 896 26, 27 / 21, 22 / 19, 20; 1,024 x 64 9, 10 / 5.5, 5.9 / 4.7,
// 5.1.  (All chunks' loads at once: slower, 46 us at 17,920 x 1,536.)
template <int MB, int STAGES, bool PARTS, bool RAW>
__global__ __launch_bounds__(FS_WAVES * 64, 2) void fs_gemm_kernel(
    const uint4* __restrict__ As, const int* __restrict__ row_ranges, const float* __restrict__ A, const float* __restrict__ Ws,
    const int* __restrict__ column_ranges, const float* __restrict__ bias, float* __restrict__ C, int M, int N, int K, int lda, int ldc,
    int steps) {
    extern __shared__ uint4 fs_lds[];
    __shared__ int raw_ranges[RAW ? 32 : 1];
    static_assert(!RAW || (MB == 1 && !PARTS), "unsplit rows come in one block, with the whole of a short K");
    static_assert(FS_RAW_K <= FS_SEG && FS_RAW_CHUNK % (3 * FS_RAW_GROUP) == 0 && FS_RAW_CHUNK % 2 == 0, "RAW: one segment, whole turns of three groups");
    constexpr int CHUNKS = MB * 2, LA = (CHUNKS + FS_WAVES - 1) / FS_WAVES, LW = 2, STAGE = (CHUNKS + FS_WAVES * LW) * 64;
    constexpr int BN = FS_WAVES * 32;
    const int blocks = (M + 31) / 32, mtiles = (blocks + MB - 1) / MB, ntiles = (N + BN - 1) / BN;
    const int local = blockIdx.x >> 3;
    const int nt = (local / mtiles) * 8 + (blockIdx.x & 7), mt = local % mtiles;
    if (nt >= ntiles) return;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int b0 = mt * MB, n0 = (nt * FS_WAVES + wave) * 32;
    const int first = PARTS ? blockIdx.y * FS_SEG_STEPS : 0;
    const int last = PARTS ? min(first + FS_SEG_STEPS, steps) : steps;

    const uint4* ap[LA];
    const uint4* wp[LW];
#pragma unroll
    for (int i = 0; i < LA; ++i) {
        const int c = min(wave + i * FS_WAVES, CHUNKS - 1);            // a wave without a piece of its own repeats the last one
        ap[i] = As + ((size_t)min(b0 + c / 2, blocks - 1) * steps + first) * 128 + (c % 2) * 64 + lane;
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
            for (int i = 0; i < LA; ++i) ap[i] += 128;
#pragma unroll
            for (int j = 0; j < LW; ++j) wp[j] += 64;
        }
    };
    // this lane's column's range of the segment of step s; its factor is applied as the weights are split
    auto column_of = [&](int s) { return column_ranges[(size_t)(s / FS_SEG_STEPS) * ((N + 15) / 16 * 16) + min(n0 + (lane & 31), N - 1)]; };
    int column = column_of(first);
    float factor = fs_factor(column);
    fs_f32x16 acc[MB];
    auto clear = [&]() {
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][r] = 0.f;
    };
    // this lane holds rows 8 (r / 4) + 4 (lane / 32) + r % 4 of a block and one column
    float* out = PARTS ? C + (size_t)blockIdx.y * M * N : C;
    const size_t ld = PARTS ? N : ldc;
    const int row0 = b0 * 32 + 4 * (lane >> 5);
    auto store = [&](int s0, int s1) {       // the sums over steps [s0, s1), a segment
        const bool first_seg = s0 == 0, last_seg = s1 == steps;
        const bool inside = RAW && M == MB * 32 && n0 + 32 <= N;           // no element's place is looked at
        int row = row0, n = n0 + (lane & 31);
        asm volatile("" : "+v"(row), "+v"(n));         // addresses and bounds are made here, not kept through the loop over k
        const int* ranges = RAW ? raw_ranges + row : row_ranges + (size_t)(s0 / FS_SEG_STEPS) * blocks * 32 + row;
        const float b = !PARTS && bias && last_seg && n < N ? bias[n] : 0.f;
        // elements to compute again, sixteen bits per block: those that are not finite, and those so small that what the
        // halves lose of the smallest values could show (but where all of a row or column is zero)
        const float least = column == FS_ZERO ? 0.f : FS_SMALL * __builtin_amdgcn_sqrtf((float)min(FS_SEG, K - s0 * FS_STEP));
        uint32_t again[(MB + 1) / 2], small[(MB + 1) / 2];
#pragma unroll
        for (int u = 0; u < (MB + 1) / 2; ++u) again[u] = small[u] = 0;
        int rows[2][16];                               // of a block's rows, asked for a block ahead
        auto ranges_of = [&](int i) {
#pragma unroll
            for (int r = 0; r < 16; ++r) rows[i & 1][r] = ranges[(RAW || b0 + i < blocks ? i : 0) * 32 + 8 * (r >> 2) + (r & 3)];
        };
        ranges_of(0);
#pragma unroll
        for (int i = 0; i < MB; ++i) {
            if (!RAW && b0 + i >= blocks) break;
            if (i + 1 < MB) ranges_of(i + 1);
            asm volatile("" ::: "memory");
#pragma unroll
            for (int q = 0; q < 4; ++q) {              // four rows at a time: a few addresses and sums in registers
                float* o = out + (size_t)(row + i * 32 + 8 * q) * ld + n;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int up = rows[i & 1][4 * q + r];
                    const float sum = acc[i][4 * q + r], v = __builtin_amdgcn_ldexpf(sum, -(up + column));
                    if (inside || (n < N && row + i * 32 + 8 * q + r < M)) {
                        const bool finite = fabsf(v) < INFINITY, low = finite && fabsf(sum) < least && up != FS_ZERO;
                        const bool fine = finite && !low;                  // else the sum so far stays where it is
                        const uint32_t bit = 1u << ((i & 1) * 16 + 4 * q + r);
                        again[i / 2] |= finite ? 0u : bit;
                        small[i / 2] |= low ? bit : 0u;
                        const float so_far = !PARTS && !first_seg ? o[r * ld] : 0.f;
                        o[r * ld] = fine ? (!PARTS && !first_seg ? so_far + v : v) + b : so_far;
                    }
                }
                asm volatile("" ::: "memory");
            }
        }
        // the small ones, one at a time: a lane every 64th k
        for (int i = 0; i < MB; ++i) {
            uint32_t marks = 0;
#pragma unroll
            for (int u = 0; u < (MB + 1) / 2; ++u) marks = i >> 1 == u ? small[u] : marks;
            marks = marks >> (i & 1) * 16 & 0xffffu;
            for (uint64_t holders = __ballot(marks != 0); holders; holders = __ballot(marks != 0)) {
                const int holder = __builtin_ctzll(holders), r = __builtin_ctz(__builtin_amdgcn_readlane((int)marks, holder));
                const int m = (b0 + i) * 32 + 4 * (holder >> 5) + 8 * (r >> 2) + (r & 3), col = n0 + (holder & 31);
                const float* a = A + (size_t)m * lda;
                const float* w = Ws + ((size_t)(col >> 4) * steps * 64 + (col & 15)) * 4;
                const int end = min(s1 * FS_STEP, K);
                float v = 0.f;
#pragma unroll 8
                for (int k = s0 * FS_STEP + lane; k < end; k += 64)
                    v = __builtin_fmaf(a[k], w[(size_t)(k >> 4) * 256 + (k >> 2 & 3) * 64 + (k & 3)], v);
                v = tl_wave_sum(v);
                if (lane == holder) {
                    float* o = out + (size_t)m * ld + col;
                    *o = (!PARTS && !first_seg ? *o + v : v) + b;
                    marks &= marks - 1;
                }
            }
        }
        bool any = false;
#pragma unroll
        for (int u = 0; u < (MB + 1) / 2; ++u) any |= again[u] != 0;
        if (!__any(any)) return;
        // those that are not finite from the values themselves, on the float instruction
        for (int i = 0; i < MB; ++i) {
            uint32_t marks = 0;
#pragma unroll
            for (int u = 0; u < (MB + 1) / 2; ++u) marks = i >> 1 == u ? again[u] : marks;
            marks = marks >> (i & 1) * 16 & 0xffffu;
            if (!__any(marks != 0)) continue;
            int here = lane;
            asm volatile("" : "+v"(here));             // nothing of this is made ahead of the loop over k
            const int n = n0 + (here & 31), half = here >> 5;
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
        // One step's products, each of which waits for the one before; between them the next step's rows are read and its weights split.
        uint4 x[2], a[2];
        auto step = [&](const uint4* next_rows, const float4 (&next)[2]) {
            uint4 b[2];
#pragma unroll
            for (int p = 0; p < 2; ++p) b[p] = next_rows[p * 64];
            float f[8] = {next[0].x, next[0].y, next[0].z, next[0].w, next[1].x, next[1].y, next[1].z, next[1].w};
            uint32_t y[8];
            auto take = [&](int t) { y[t] = t < 4 ? fs_take(f[2 * t], f[2 * t + 1]) : fs_rest(f[2 * (t & 3)], f[2 * (t & 3) + 1]); };
#define FS_AMONG(PA, PW, ...)                   \
    FS_MUL_ONE(acc[0], a[PA], x[PW])            \
    __VA_ARGS__;                                \
    __builtin_amdgcn_sched_barrier(0);
            FS_AMONG(0, 1, _Pragma("unroll") for (int i = 0; i < 8; ++i) f[i] *= factor; take(0); take(1))
            FS_AMONG(1, 0, take(2); take(3); take(4))
            FS_AMONG(0, 0, take(5); take(6); take(7))
#undef FS_AMONG
#pragma unroll
            for (int p = 0; p < 2; ++p) x[p] = make_uint4(y[4 * p], y[4 * p + 1], y[4 * p + 2], y[4 * p + 3]), a[p] = b[p];
        };
        // (behind a chunk's last step lie rows of the chunk before, or nothing: read and not used)
        auto multiply = [&](float4 (&from)[FS_RAW_GROUP][2], const float4 (&then)[FS_RAW_GROUP][2], int s, int c0) {
            const uint4* rows_of = fs_lds + (s - c0) * 128 + lane;
#pragma unroll
            for (int u = 0; u < FS_RAW_GROUP; ++u)
                if (s + u < steps)
                    step(rows_of + (s + u - c0 + 1 < FS_RAW_CHUNK && s + u + 1 < steps ? (u + 1) * 128 : 0),
                         u + 1 < FS_RAW_GROUP ? from[u + 1 < FS_RAW_GROUP ? u + 1 : 0] : then[0]);
            ask(from, s + 3 * FS_RAW_GROUP);
        };
        // Rows: a wave has eight of them, a lane 16 bytes of one in a line of 128 (two steps), so that no line is asked for twice.
        constexpr int LINES = FS_RAW_CHUNK / 2;
        const int row = wave * 8 + (lane >> 3), unit = 4 * (lane & 7);
        const float* al = A + (size_t)min(row, M - 1) * lda;
        uint2* part = reinterpret_cast<uint2*>(fs_lds) + ((lane >> 2 & 1) * 128 + (lane >> 1 & 1) * 32 + row) * 2 + (lane & 1);
        float4 rows[LINES];
        auto ask_rows = [&](float4 (&to)[LINES], int c0) {
#pragma unroll
            for (int i = 0; i < LINES; ++i)
                if (c0 + 2 * i < steps) to[i] = *reinterpret_cast<const float4*>(al + min((c0 + 2 * i) * FS_STEP + unit, K - 4));
        };
        auto ask_first = [&]() {
#pragma unroll
            for (int g = 0; g < 3; ++g) {
#pragma unroll
                for (int u = 0; u < FS_RAW_GROUP; ++u) w[g][u][0] = w[g][u][1] = zero;
                ask(w[g], g * FS_RAW_GROUP);
            }
        };
        // the rows' largest values first: the chunks from the last to the first, which stays
        float most = 0.f;
        auto most_of = [&](const float4 (&of)[LINES], int c0) {
#pragma unroll
            for (int i = 0; i < LINES; ++i)
                if ((c0 + 2 * i) * FS_STEP + unit < K) most = fmaxf(most, fs_most(of[i]));
        };
        for (int c0 = (steps - 1) / FS_RAW_CHUNK * FS_RAW_CHUNK; c0 > 0; c0 -= FS_RAW_CHUNK) {
            ask_rows(rows, c0);
            most_of(rows, c0);
        }
        ask_rows(rows, 0);
        ask_first();
        most_of(rows, 0);
        most = fs_group_most(most);
        const int up = fs_up(most);
        const float row_factor = fs_factor(up);
        if ((lane & 7) == 0) raw_ranges[row] = up;       // (behind barriers by the time it is read)
        for (int c0 = 0; c0 < steps; c0 += FS_RAW_CHUNK) {
            const int here = min(steps - c0, FS_RAW_CHUNK);
            if (c0) __syncthreads();                     // every wave has read the rows before
#pragma unroll
            for (int i = 0; i < LINES; ++i)
                if (2 * i < here) {
                    float4 f = (c0 + 2 * i) * FS_STEP + unit < K && row < M ? rows[i] : zero;
                    fs_times(f, row_factor);
                    uint2 hi, lo;
                    fs_split4(f, hi, lo);
                    uint2* to = part + i * 512;
                    to[0] = hi;
                    to[128] = lo;
                }
            if (c0 + FS_RAW_CHUNK < steps) ask_rows(rows, c0 + FS_RAW_CHUNK);
            if (c0 == 0) {
                fs_times(w[0][0][0], factor);
                fs_times(w[0][0][1], factor);
                fs_split8(w[0][0][0], w[0][0][1], x[0], x[1]);
            }
            __syncthreads();
#pragma unroll
            for (int p = 0; p < 2; ++p) a[p] = fs_lds[p * 64 + lane];
            for (int s = c0; s < c0 + here; s += 3 * FS_RAW_GROUP) {
                multiply(w[0], w[1], s, c0);
                if (s + FS_RAW_GROUP < c0 + here) multiply(w[1], w[2], s + FS_RAW_GROUP, c0);
                if (s + 2 * FS_RAW_GROUP < c0 + here) multiply(w[2], w[0], s + 2 * FS_RAW_GROUP, c0);
            }
        }
        store(0, steps);
        return;
    }
    // A step's weights are split, and its first rows read, while the step before is multiplied; within a step the next rows are read
    // while some are multiplied, two blocks in turn where there are two, so that a product does not wait for the one before it.
    constexpr int IB = MB == 1 ? 1 : 2, GROUPS = MB / IB;
    for (int i = 0; i < STAGES - 1; ++i) fetch(i);
    const int wfrag = (CHUNKS + wave * LW) * 64 + ((lane >> 4) & 1) * 64 + (lane >> 5) * 32 + (lane & 15);
    auto rows_of = [&](int buf, int g, uint4 (&to)[IB][2]) {
#pragma unroll
        for (int b = 0; b < IB; ++b)
#pragma unroll
            for (int p = 0; p < 2; ++p) to[b][p] = fs_lds[buf * STAGE + ((g * IB + b) * 2 + p) * 64 + lane];
    };
    uint4 a[2][IB][2], w[2][2];
    FS_LANDED((STAGES - 2) * (LA + LW));
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    {
        float4 x = __builtin_bit_cast(float4, fs_lds[wfrag]), y = __builtin_bit_cast(float4, fs_lds[wfrag + 16]);
        fs_times(x, factor);
        fs_times(y, factor);
        fs_split8(x, y, w[0][0], w[0][1]);
        rows_of(0, 0, a[0]);
    }
    int buf = 0;
    auto step = [&](auto parity, float factor) {       // factor: the next step's
        constexpr int S = decltype(parity)::value, A0 = GROUPS & 1 ? S : 0;     // which registers the step's first rows are in
        FS_LANDED((STAGES - 3) * (LA + LW));       // step s + 1 is here; later ones may be on their way
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        const int next = buf == STAGES - 1 ? 0 : buf + 1;
        float4 x = __builtin_bit_cast(float4, fs_lds[next * STAGE + wfrag]), y = __builtin_bit_cast(float4, fs_lds[next * STAGE + wfrag + 16]);
        fetch(buf == 0 ? STAGES - 1 : buf - 1);   // the buffer of step s - 1, which every wave has read
        float f[8] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
        uint32_t u[8];
        auto take = [&](int t) { u[t] = t < 4 ? fs_take(f[2 * t], f[2 * t + 1]) : fs_rest(f[2 * (t & 3)], f[2 * (t & 3) + 1]); };
#pragma unroll
        for (int g = 0; g < GROUPS; ++g) {
            if (g + 1 < GROUPS) rows_of(buf, g + 1, a[(A0 + g + 1) & 1]);
            else rows_of(next, 0, a[(A0 + g + 1) & 1]);
            const uint4 (&rows)[IB][2] = a[(A0 + g) & 1];
#define FS_MUL(T, PA, PW)                                                                                                    \
    _Pragma("unroll") for (int b = 0; b < IB; ++b) FS_MUL_ONE(acc[g * IB + b], rows[b][PA], w[S][PW])                         \
    if (g == 0 && T == 0) { _Pragma("unroll") for (int i = 0; i < 8; ++i) f[i] *= factor; }                                   \
    _Pragma("unroll") for (int t = (g * 3 + T) * 8 / (GROUPS * 3); t < (g * 3 + T + 1) * 8 / (GROUPS * 3); ++t) take(t);       \
    __builtin_amdgcn_sched_barrier(0);
            FS_MUL(0, 0, 1)
            FS_MUL(1, 1, 0)
            FS_MUL(2, 0, 0)
#undef FS_MUL
        }
#pragma unroll
        for (int p = 0; p < 2; ++p) w[S ^ 1][p] = make_uint4(u[4 * p], u[4 * p + 1], u[4 * p + 2], u[4 * p + 3]);
        buf = next;
    };
    int s = first;
    auto steps_to = [&](int end, float then) __attribute__((always_inline)) {          // then: the factor behind them
        for (; s + 2 <= end; s += 2) {
            step(std::integral_constant<int, 0>(), factor);
            step(std::integral_constant<int, 1>(), s + 2 < end ? factor : then);
        }
        if (s < end) {                   // (an odd segment is the last)
            step(std::integral_constant<int, 0>(), factor);
            ++s;
        }
    };
    if constexpr (PARTS) {
        steps_to(last, factor);
        FS_LANDED(0);                    // nothing may land in LDS that is no longer this work-group's
        store(first, last);
        return;
    }
    while (s < last) {                   // a segment at a time
        const int s0 = s, s1 = min(s + FS_SEG_STEPS, last), next = s1 < last ? column_of(s1) : column;
        asm volatile("" ::"v"(next));    // here before the loop, where a wait for it would wait for the steps on their way
        steps_to(s1, fs_factor(next));
        if (s == last) FS_LANDED(0);
        store(s0, s);
        if (s < last) {
            clear();
            column = next;
            factor = fs_factor(next);
        }
    }
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

// The tiles (row blocks of a wave) as a fitted time: a step of 16 k takes a work-group `alone` us when its CU has nothing else (the
// chain barrier - reads - products), and a CU gets through one in `shared` us when it holds as many as fit.  The tile, and whether K is
// dealt out by segments, is the least estimate: 2.8% longer than the best choice in the mean over eleven matrices of 64 to 18,944 k x
// nineteen row counts, 25% at most (1,700 rows of 3,584 x 3,584).  E.g. at 2,048 rows down (3,584 x 18,944) takes 0.96 ms with K dealt
// out, 1.46 without; at 40 rows 74 to 86 us and 440 to 920.
struct FsTile {
    int mb, fit;
    double alone, shared;
};
static const FsTile fs_tiles[] = {{8, 2, 1.30, 0.83}, {4, 2, 0.70, 0.48}, {2, 3, 0.55, 0.25}, {1, 4, 0.29, 0.18}};

static int fs_choose(int M, int N, int K, bool* parts) {
    const int blocks = tl_ceil_div(M, 32), steps = tl_ceil_div(K, FS_STEP), nseg = tl_ceil_div(K, FS_SEG);
    int best = 3;
    double cost = 1e300;
    for (int t = 0; t < 4; ++t) {
        const FsTile& z = fs_tiles[t];
        if (z.mb > 1 && z.mb / 2 >= blocks) continue;                  // half of it holds all the rows
        const double tiles = (double)tl_ceil_div(blocks, z.mb) * tl_ceil_div(N, FS_WAVES * 32);
        for (int cut = 0; cut < (nseg > 1 && nseg <= 65535 && (long long)M * N <= FS_MOST_SUMS / nseg ? 2 : 1); ++cut) {
            const double each = tiles * (cut ? nseg : 1) / FS_CUS, whole = (double)(long long)(each + 0.999999);
            const double on_a_cu = whole < 4 ? whole : each + 0.5, turns = (double)(long long)((whole + z.fit - 1) / z.fit);
            const double step = turns * z.alone > on_a_cu * z.shared ? turns * z.alone : on_a_cu * z.shared;
            const double us = step * steps / (cut ? nseg : 1) + (cut ? 4.7 + 8.0 * M * N * nseg / 6e6 : 0.0);
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

// 32-bit numbers of the ranges of a matrix [N, K], and the ranges from its ordered copy.
extern "C" long long tl_gemm_float_ranges_size(int N, int K) {
    return N > 0 && K > 0 ? (long long)tl_ceil_div(K, FS_SEG) * tl_ceil_div(N, 16) * 16 : 0;
}
extern "C" int tl_gemm_float_ranges(const float* Ws, void* ranges, int N, int K, hipStream_t stream) {
    TL_CHECK_ARG(N > 0 && K > 0 && tl_ceil_div(K, FS_SEG) <= 65535, "tl_gemm_float_ranges: bad sizes N=%d K=%d", N, K);
    TL_CHECK_ARG((uintptr_t)Ws % 16 == 0 && (uintptr_t)ranges % 4 == 0, "tl_gemm_float_ranges: the weight copy must be 16-byte aligned");
    hipLaunchKernelGGL(fs_ranges_kernel<false>, dim3(tl_ceil_div(N, 16), tl_ceil_div(K, FS_SEG)), dim3(FS_RANGE_WAVES * 64), 0, stream, nullptr,
                       (float4*)Ws, (int*)ranges, N, 0, tl_ceil_div(N, 16), tl_ceil_div(K, FS_STEP));
    TL_CHECK_LAUNCH("tl_gemm_float_ranges");
    return 0;
}
// The ordered copy Ws of W [N, K] (contiguous, K a multiple of four), and its ranges.
extern "C" int tl_gemm_float_order(const float* W, float* Ws, void* ranges, int N, int K, hipStream_t stream) {
    TL_CHECK_ARG(N > 0 && K > 0 && K % 4 == 0 && tl_ceil_div(K, FS_SEG) <= 65535, "tl_gemm_float_order: bad sizes N=%d K=%d", N, K);
    TL_CHECK_ARG((uintptr_t)W % 16 == 0 && (uintptr_t)Ws % 16 == 0 && (uintptr_t)ranges % 4 == 0, "tl_gemm_float_order: the matrix and its copy must be 16-byte aligned");
    hipLaunchKernelGGL(fs_ranges_kernel<true>, dim3(tl_ceil_div(N, 16), tl_ceil_div(K, FS_SEG)), dim3(FS_RANGE_WAVES * 64), 0, stream,
                       (const float4*)W, (float4*)Ws, (int*)ranges, N, K / 4, tl_ceil_div(N, 16), tl_ceil_div(K, FS_STEP));
    TL_CHECK_LAUNCH("tl_gemm_float_order");
    return 0;
}

// Bytes of `split` for M rows of K.
extern "C" long long tl_gemm_float_split_bytes(int M, int K) {
    return M > 0 && K > 0 ? (long long)tl_ceil_div(M, 32) * (tl_ceil_div(K, FS_STEP) * 2048ll + tl_ceil_div(K, FS_SEG) * 128ll) : 0;
}

// A float [M, K] with row stride lda; Ws float [ceil(N/16), ceil(K/16), 64, 4] (the matrix-core ordered copy of W, zero
// where it pads); ranges: tl_gemm_float_ranges of it; split: workspace of tl_gemm_float_split_bytes, or null where
// tl_gemm_float_split_takes_rows says that the rows are split where they are used; ws: tl_gemm_float_split_workspace floats.
extern "C" int tl_gemm_float_split(const float* A, const float* Ws, const void* ranges, const float* bias, float* C, void* split, float* ws,
                                   int M, int N, int K, int lda, int ldc, hipStream_t stream) {
    TL_CHECK_ARG(M >= 0 && N > 0 && K > 0, "tl_gemm_float_split: bad sizes M=%d N=%d K=%d", M, N, K);
    TL_CHECK_ARG(lda >= K && ldc >= N, "tl_gemm_float_split: row strides lda=%d ldc=%d too small for K=%d N=%d", lda, ldc, K, N);
    TL_CHECK_ARG((uintptr_t)Ws % 16 == 0 && (uintptr_t)split % 16 == 0, "tl_gemm_float_split: the weight copy and the workspace must be 16-byte aligned");
    if (M == 0) return 0;
    const int steps = tl_ceil_div(K, FS_STEP), blocks = tl_ceil_div(M, 32), nseg = tl_ceil_div(K, FS_SEG);
    TL_CHECK_ARG(blocks <= 65535, "tl_gemm_float_split: %d rows are too many for one launch", M);
    bool parts = false;
    const int tile = fs_choose(M, N, K, &parts);
    const int mtiles = tl_ceil_div(blocks, fs_tiles[tile].mb), ntiles = tl_ceil_div(N, FS_WAVES * 32);
    const long long grid = (long long)mtiles * tl_ceil_div(ntiles, 8) * 8;
    TL_CHECK_ARG(grid < (1ll << 31), "tl_gemm_float_split: M=%d N=%d are too many tiles for one launch", M, N);
    TL_CHECK_ARG(!parts || ws, "tl_gemm_float_split: no workspace for the segments' sums");
    const int vec = ((uintptr_t)A % 16 == 0 && lda % 4 == 0) ? 1 : 0;
    TL_CHECK_ARG(split || (tl_gemm_float_split_takes_rows(M, N, K, lda) && vec && tile == 3 && !parts),
                 "tl_gemm_float_split: M=%d K=%d lda=%d need a workspace for the rows' parts", M, K, lda);
    TL_CHECK_ARG(ranges && (uintptr_t)ranges % 4 == 0, "tl_gemm_float_split: no ranges of the matrix");
    int* rows = split ? (int*)((uint4*)split + (size_t)blocks * steps * 128) : nullptr;
    if (split)
        hipLaunchKernelGGL(fs_split_kernel, dim3(nseg, blocks * 4), dim3(FS_SPLIT_WAVES * 64), 0, stream, A, (uint4*)split, rows, M, K, lda, steps,
                           vec);
#define FS_GO(MB, ST, P, RAW, LDS)                                                                                           \
    hipLaunchKernelGGL((fs_gemm_kernel<MB, ST, P, RAW>), dim3((unsigned)grid, P ? nseg : 1), dim3(FS_WAVES * 64), LDS, stream, \
                       (const uint4*)split, rows, A, Ws, (const int*)ranges, bias, P ? ws : C, M, N, K, lda, ldc, steps)
#define FS_GO_P(MB, ST)                                                               \
    if (parts) FS_GO(MB, ST, true, false, ST * (MB * 2 + FS_WAVES * 2) * 1024); \
    else FS_GO(MB, ST, false, false, ST * (MB * 2 + FS_WAVES * 2) * 1024)
    if (tile == 0) {
        FS_GO_P(8, 3);
    } else if (tile == 1) {
        FS_GO_P(4, 4);
    } else if (tile == 2) {
        FS_GO_P(2, 4);
    } else if (split) {
        FS_GO_P(1, 4);
    } else {
        FS_GO(1, 1, false, true, (steps < FS_RAW_CHUNK ? (steps + 1) / 2 * 2 : FS_RAW_CHUNK) * 2048);
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
