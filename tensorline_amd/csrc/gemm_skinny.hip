// C[M, N] = A[M, K] * W[N, K]^T (+ bias) for few rows (M <= 16), bfloat16 inputs: the matrix
// products of a decode step.  The work is streaming W once from HBM.
//
// W is read from a copy laid out for the matrix cores ("shuffled", made once when the weights are
// loaded): [N/16 tiles][K/32 chunks][64 lanes][8 values], where lane l = 16*g + r holds row r of
// the tile and the 8 consecutive k values starting at 32*chunk + 8*g.  That is exactly the first
// operand of v_mfma_f32_16x16x32_bf16, so one load instruction of a wave reads 1 KB of contiguous
// memory and a wave walks straight through memory along K.  (Loading the same fragments from a
// row-major W touches 16 rows x 64 bytes per instruction: 64 cache-line lookups per KB instead of
// 8, which limits the rate well below HBM's.)
//
// A work-group owns one tile of 16 output columns and all M rows of A; its waves split K among
// themselves and add their partial sums through LDS in a fixed order, so a result never depends
// on timing.  Each wave brings its slice of A in with row-contiguous loads, 128 k at a time, into
// a private LDS region laid out [8-k unit][row] (+1 row of padding per unit, conflict-free both
// ways) and reads the second MFMA operand from there: lane l = 16*g + r reads row m = r of A at
// the k values of unit 4*chunk + g.  No barrier is needed for that: a wave's LDS operations
// complete in order.  The accumulator of lane l, register i, is C[m = l % 16][n = 4*(l / 16) + i].
//
// Two tiles per work-group (MODE_SWIGLU, MODE_QKV), sharing the A fragments:
//  * MODE_SWIGLU owns tile t of the first I/16 tiles and tile t of the next I/16 of a fused
//    [2I, K] gate/up matrix and writes silu(first) * second.
//  * MODE_QKV owns, in head h of a fused q/k/v projection, tiles j and j + d/32: the two halves
//    that rotate-half RoPE pairs.  Its epilogue adds the bias, rotates query and key heads by the
//    token's position (angle pos * inv_freq[i] in float, as tl_rope_store does), writes queries to
//    a [M, nq*d] matrix and keys and values straight into the paged cache at the token's slot:
//    the projection, the position encoding and the cache write of a decode step in one kernel.
//
// RMS normalisation around the products (NormArgs), so that a decode step needs no kernel of its
// own for a norm.  y = W (h * g / rms(h)) equals (W (h * g)) / rms(h): a product may take rows
// A = h * g whose division is still owed, with partial sums of h^2 per row, and scale its results
// by 1/sqrt(sum / dim + eps) in float.  And a plain product that ends a residual branch may do
// the add and prepare the next norm: resid += result (float), a_out = resid * next_weight, and
// the sum of resid^2 over the tile's 16 columns as one partial per row.  Sums of squares are
// added in a fixed order that depends on the shapes only.
#include "common.h"

#include <type_traits>

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

#define MODE_PLAIN 0
#define MODE_SWIGLU 1
#define MODE_QKV 2

// what MODE_QKV needs beyond the product
struct QkvArgs {
    const int32_t* pos;        // [M] positions
    const float* inv_freq;     // [d/2]
    const int32_t* slots;      // [M] cache rows (negative: do not store)
    bf16_t* q_out;             // [M, nq*d]
    bf16_t* k_cache;           // [pages, page, nkv, d]
    bf16_t* v_cache;           // [pages, nkv, d, page]
    int nq, nkv, d, bs;
};


#define SK_MAX_LDS (80 * 1024)          // LDS of a work-group; a CU has 160 KB
#define SK_SC 128                    // k values staged per step (4 chunks of 32)
#define SK_UNITS (SK_SC / 8)         // 16-byte units per row of a step
#define SK_ROWPAD 17                 // rows per unit in LDS: 16 + 1 of padding

__device__ __forceinline__ bf16x8 as_frag(uint4 v) { return __builtin_bit_cast(bf16x8, v); }

// Keeps the compiler from moving a wave's LDS reads above its earlier LDS writes (and the other
// way round) without waiting for anything: the hardware completes a wave's LDS operations in
// order, and the global loads in flight (the next step's W fragments) must stay in flight.
__device__ __forceinline__ void wave_lds_order() {
    __builtin_amdgcn_wave_barrier();
    asm volatile("" ::: "memory");
}

// SPLIT 2 (plain products): a work-group owns half a tile, eight columns, so that twice as many CUs stream a narrow matrix.  A load
// of a wave still brings 1 KB: the half's rows of two chunks of 32 k, lanes r < 8 of the first, r >= 8 of the second.  Two
// products per load, one with each chunk's activations, of which the rows 0..7 and the rows 8..15 are kept; the two
// halves are added at the end.
template <int MT, int MODE, typename TO, int SPLIT>
__global__ __launch_bounds__(MODE == MODE_SWIGLU ? 256 : 512) void gemm_skinny_kernel(
    const bf16_t* __restrict__ A, const uint4* __restrict__ Ws, const float* __restrict__ bias, TO* __restrict__ C,
    int M, int n_out, int K, int K32, int lda, int ldc, int second_tile, QkvArgs qa, TlNormArgs na) {
    extern __shared__ uint4 smem[];
    __shared__ float sh_part[64 * 16];               // [part][row] partial sums of squares
    __shared__ float sh_rstd[16];
    __shared__ float sh_sq[16 * 17];                 // [row][column of the tile] squares of the new residual
    constexpr bool DUAL = MODE != MODE_PLAIN;
    constexpr int NACC = MT * (DUAL ? 2 : 1);
    constexpr int COLS = 16 / SPLIT;                           // columns of a work-group
    static_assert(SPLIT == 1 || (MT == 1 && MODE == MODE_PLAIN), "half tiles come with one tile of rows and one stream of weights");
    constexpr int XS_PER_WAVE = MT * SPLIT * SK_UNITS * SK_ROWPAD;     // in uint4
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nwaves = blockDim.x >> 6;
    const int r = lane & 15, g = lane >> 4;
    const int unit = blockIdx.x / SPLIT, col0 = (blockIdx.x - unit * SPLIT) * COLS;      // tile (pair), first column in it
    int tile = unit, tile2 = second_tile + unit;
    if (MODE == MODE_QKV) {
        const int pph = qa.d / 32;                   // tile pairs per head
        const int head = unit / pph, j = unit - head * pph;
        tile = head * (qa.d / 16) + j;
        tile2 = tile + pph;
    }
    // within a chunk: this lane's 16 bytes (SPLIT 2: row col0 + r % 8 of k group g), and which of the load's chunks it reads
    const int in_chunk = SPLIT == 1 ? lane : 16 * g + col0 + (r & 7), sub = SPLIT == 1 ? 0 : r >> 3;
    const uint4* w1 = Ws + (size_t)tile * K32 * 64 + in_chunk;
    const uint4* w2 = DUAL ? Ws + (size_t)tile2 * K32 * 64 + in_chunk : nullptr;
    uint4* xs = smem + (size_t)wave * XS_PER_WAVE;
    const uint4 zero = make_uint4(0, 0, 0, 0);

    f32x4 acc[NACC * SPLIT];                         // [s * NACC + a]: the products with chunk s of a load
#pragma unroll
    for (int i = 0; i < NACC * SPLIT; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};

    // What the epilogue needs from memory is asked for now, so that it has arrived when the sums
    // are done: this thread's partial sums of squares (thread (row, part) owns every nparts-th
    // partial of its row; the first SS_PRE of them are fetched here) and, with a residual sink,
    // the residual, norm weight and bias of the thread's first output element.  Addresses are
    // clamped; what a clamped load brings is not used.
    const bool owed = na.ss_in != nullptr;
    const bool sink = MODE == MODE_PLAIN && na.resid != nullptr;
    const int ss_row = threadIdx.x & 15, ss_part = threadIdx.x >> 4, ss_nparts = blockDim.x >> 4;
    // groups of few waves (gate/up) have many partials per thread, wide groups have few
    constexpr int SS_PRE = (MODE == MODE_SWIGLU) ? 16 : 4;
    float ssv[SS_PRE];
    if (owed) {
        const float* sp = na.ss_in + (ss_row < M ? ss_row : 0);
#pragma unroll
        for (int k = 0; k < SS_PRE; ++k) {
            const int t = ss_part + k * ss_nparts;
            ssv[k] = sp[(size_t)(t < na.ss_n ? t : 0) * na.ss_ld];
        }
    }
    float pre_resid = 0.f, pre_weight = 0.f, pre_bias = 0.f;
    if (sink && threadIdx.x < 256 / SPLIT) {
        const int l = threadIdx.x & (64 / SPLIT - 1), i = threadIdx.x / (64 / SPLIT) & 3;
        const int m = l & 15, n = tile * 16 + col0 + 4 * (l >> 4) + i;
        const int mc = m < M ? m : 0, nc = n < n_out ? n : 0;
        pre_resid = na.resid[(size_t)mc * na.resid_ld + nc];
        pre_weight = na.next_weight[nc];
        if (bias) pre_bias = bias[nc];
    }

    const int nsc = (K32 + 4 * SPLIT - 1) / (4 * SPLIT);     // steps of 128 k (SPLIT 2: 256)
    const int per = (nsc + nwaves - 1) / nwaves;
    const int s0 = wave * per;
    const int s1 = (s0 + per < nsc) ? s0 + per : nsc;

    // Software pipeline, one step (128 k) deep: while a step is multiplied, the A rows and the W
    // fragments of the next one are in flight.  Loads retire in issue order, so within a step the
    // A rows (needed first, for the LDS write) are requested before the W fragments.  Every load is
    // unconditional: an address past the end is clamped to a valid one, and what it brings is
    // either never used (rows of A past M feed output rows that are not written) or replaced by zero (k past K).
    uint4 wf[4], uf[4], wn[4], un[4], xr[SPLIT][MT * 4];
    const int xrow0 = lane >> 4, xunit = lane & 15;
    const bf16_t* xp[MT * 4];
#pragma unroll
    for (int i = 0; i < MT * 4; ++i) {
        const int row = xrow0 + 4 * i;
        xp[i] = A + (size_t)(row < M ? row : 0) * lda;       // the row's start: the unit is part of the k offset
    }
    const int last_c = K32 - 1;
    {
        const int sc = (s0 < s1) ? s0 : 0;
#pragma unroll
        for (int h = 0; h < SPLIT; ++h) {
            const int kx = (sc * SPLIT + h) * SK_SC + xunit * 8;
            const int kxc = (kx < K) ? kx : 0;           // past K: the row's first unit, inside the row whatever K is
#pragma unroll
            for (int i = 0; i < MT * 4; ++i) xr[h][i] = *reinterpret_cast<const uint4*>(xp[i] + kxc);
            if (kx >= K) {
#pragma unroll
                for (int i = 0; i < MT * 4; ++i) xr[h][i] = zero;
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            int c = (sc * 4 + i) * SPLIT + sub;
            if (c > last_c) c = last_c;
            wf[i] = tl_load_stream(w1 + (size_t)c * 64);
            if (DUAL) uf[i] = tl_load_stream(w2 + (size_t)c * 64);
        }
    }
    // A rows of a step: registers -> LDS, lane (row = lane/16 + 4i, unit = lane%16)
    auto stage = [&]() {
#pragma unroll
        for (int h = 0; h < SPLIT; ++h)
#pragma unroll
            for (int i = 0; i < MT * 4; ++i) {
                const int row = xrow0 + 4 * i;
                xs[(((row >> 4) * SPLIT + h) * SK_UNITS + xunit) * SK_ROWPAD + (row & 15)] = xr[h][i];
            }
        wave_lds_order();
    };
    auto multiply = [&](int sc, const uint4 (&w)[4], const uint4 (&u)[4]) {
        // chunks past K32 of the last step read a clamped chunk: they must count as zero
        const int cbase = sc * 4 * SPLIT;
#pragma unroll
        for (int cc = 0; cc < 4; ++cc) {
#pragma unroll
            for (int h = 0; h < SPLIT; ++h) {
                const bool live = cbase + cc * SPLIT + h <= last_c;
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) {
                    uint4 xf = xs[(mt * SPLIT * SK_UNITS + (cc * SPLIT + h) * 4 + g) * SK_ROWPAD + r];
                    if (!live) xf = zero;
                    f32x4& a = acc[h * NACC + mt];
                    a = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_frag(w[cc]), as_frag(xf), a, 0, 0, 0);
                    if (DUAL)
                        acc[MT + mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_frag(u[cc]), as_frag(xf), acc[MT + mt], 0, 0, 0);
                }
            }
        }
        wave_lds_order();
    };
    // step sn's A rows (k past K zero when they are stored) and W fragments
    auto request = [&](int sn, uint4 (&w)[4], uint4 (&u)[4]) {
#pragma unroll
        for (int h = 0; h < SPLIT; ++h) {
            const int kxn = (sn * SPLIT + h) * SK_SC + xunit * 8;
            const int kxnc = (kxn < K) ? kxn : 0;
#pragma unroll
            for (int i = 0; i < MT * 4; ++i) xr[h][i] = *reinterpret_cast<const uint4*>(xp[i] + kxnc);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            int c = (sn * 4 + i) * SPLIT + sub;
            if (c > last_c) c = last_c;
            w[i] = tl_load_stream(w1 + (size_t)c * 64);
            if (DUAL) u[i] = tl_load_stream(w2 + (size_t)c * 64);
        }
    };
    auto clear_past = [&](int sn) {
#pragma unroll
        for (int h = 0; h < SPLIT; ++h)
            if ((sn * SPLIT + h) * SK_SC + xunit * 8 >= K) {
#pragma unroll
                for (int i = 0; i < MT * 4; ++i) xr[h][i] = zero;
            }
    };
    // two sets of W fragments in turn, so that nothing is moved between registers
    int sc = s0;
    for (; sc + 2 < s1; sc += 2) {
        stage();
        request(sc + 1, wn, un);
        multiply(sc, wf, uf);
        clear_past(sc + 1);
        stage();
        request(sc + 2, wf, uf);
        multiply(sc + 1, wn, un);
        clear_past(sc + 2);
    }
    // The last step asks for nothing: a wave of a narrow matrix has one to four steps, and a step asked for once more (to
    // keep the loop one body) was waited for at its end: a decode step of 28 layers of 3,584 at 8 rows 3,390 -> 3,242 us, of 24 layers of 896 at one 904 -> 877.
    if (sc + 1 < s1) {
        stage();
        request(sc + 1, wn, un);
        multiply(sc, wf, uf);
        clear_past(sc + 1);
        stage();
        multiply(sc + 1, wn, un);
    } else if (sc < s1) {
        stage();
        multiply(sc, wf, uf);
    }

    // Owed normalisation: thread (row, part) adds its partials in ascending order, then one thread
    // per row adds the parts in order.  (MT is 1 wherever this is used: rows 0..15.)
    if (owed) {
        float ssum = 0.f;
        if (ss_row < M) {
#pragma unroll
            for (int k = 0; k < SS_PRE; ++k)
                if (ss_part + k * ss_nparts < na.ss_n) ssum += ssv[k];
            // the rest, eight loads at a time so that they overlap
            for (int t0 = ss_part + SS_PRE * ss_nparts; t0 < na.ss_n; t0 += 8 * ss_nparts) {
                float more[8];
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    const int t = t0 + k * ss_nparts;
                    more[k] = na.ss_in[(size_t)(t < na.ss_n ? t : 0) * na.ss_ld + ss_row];
                }
#pragma unroll
                for (int k = 0; k < 8; ++k)
                    if (t0 + k * ss_nparts < na.ss_n) ssum += more[k];
            }
        }
        sh_part[ss_part * 16 + ss_row] = ssum;
    }
    if (sink)
        for (int e = threadIdx.x; e < 16 * 17; e += blockDim.x) sh_sq[e] = 0.f;
    // partial sums of the waves -> LDS (the staging regions are done with), then a fixed-order sum
    __syncthreads();
    float* red = reinterpret_cast<float*>(smem);     // [nwaves][NACC*4][64]
#pragma unroll
    for (int a = 0; a < NACC; ++a)
#pragma unroll
        for (int i = 0; i < 4; ++i)          // SPLIT 2: rows 0..7 (g < 2) of the first chunks' products, 8..15 of the second's
            red[((size_t)wave * NACC * 4 + a * 4 + i) * 64 + lane] = SPLIT == 2 && g >= 2 ? acc[(SPLIT - 1) * NACC + a][i] : acc[a][i];
    if (owed && threadIdx.x < 16) {
        const int nparts = blockDim.x >> 4;
        float ssum = 0.f;
        for (int p2 = 0; p2 < nparts; ++p2) ssum += sh_part[p2 * 16 + threadIdx.x];
        sh_rstd[threadIdx.x] = 1.0f / sqrtf(ssum / na.dim + na.eps);
    }
    __syncthreads();
    const int n0 = tile * 16 + col0;
    // element e = (mt, i, l): C[m = mt*16 + l % 16][n = n0 + 4*(l / 16) + i]; SPLIT 2: l < 32, its other half in lane l + 32
    for (int e = threadIdx.x; e < MT * 4 * 64 / SPLIT; e += blockDim.x) {
        const int l = e & (64 / SPLIT - 1), i = e / (64 / SPLIT) & 3, mt = SPLIT == 1 ? e >> 8 : 0;
        const int m = mt * 16 + (l & 15), n = n0 + 4 * (l >> 4) + i;
        if (m >= M || n >= n_out) continue;
        float v = 0.f, u = 0.f;
        for (int w = 0; w < nwaves; ++w) {
            v += red[((size_t)w * NACC * 4 + mt * 4 + i) * 64 + l];
            if (DUAL) u += red[((size_t)w * NACC * 4 + (MT + mt) * 4 + i) * 64 + l];
            if (SPLIT == 2) v += red[((size_t)w * NACC * 4 + mt * 4 + i) * 64 + l + 32];
        }
        if (owed) {
            const float rs = sh_rstd[m & 15];
            v *= rs;
            if (DUAL) u *= rs;
        }
        if (MODE == MODE_QKV) {
            // v, u: dims idx and idx + d/2 of head `head` for token m
            const int d = qa.d, half = d / 2;
            const int head = n / d, idx = n - head * d;
            if (bias) {
                v += bias[n];
                u += bias[n + half];
            }
            const int slot = qa.slots[m];
            if (head < qa.nq + qa.nkv) {
                float sn, cs;
                sincosf((float)qa.pos[m] * qa.inv_freq[idx], &sn, &cs);
                const float o1 = v * cs - u * sn, o2 = u * cs + v * sn;
                if (head < qa.nq) {
                    bf16_t* qp = qa.q_out + (size_t)m * qa.nq * d + (size_t)head * d + idx;
                    qp[0] = tl_from_float<bf16_t>(o1);
                    qp[half] = tl_from_float<bf16_t>(o2);
                } else if (slot >= 0) {
                    bf16_t* kp = qa.k_cache + ((size_t)slot * qa.nkv + (head - qa.nq)) * d + idx;
                    kp[0] = tl_from_float<bf16_t>(o1);
                    kp[half] = tl_from_float<bf16_t>(o2);
                }
            } else if (slot >= 0) {
                const int page = slot / qa.bs, off = slot - page * qa.bs;
                bf16_t* vp = qa.v_cache + (((size_t)page * qa.nkv + (head - qa.nq - qa.nkv)) * d + idx) * qa.bs + off;
                vp[0] = tl_from_float<bf16_t>(v);
                vp[(size_t)half * qa.bs] = tl_from_float<bf16_t>(u);
            }
            continue;
        }
        if (sink) {
            const bool first = e < (int)blockDim.x;      // the element whose operands were fetched at the start
            if (bias) v += first ? pre_bias : bias[n];
            float* rp = na.resid + (size_t)m * na.resid_ld + n;
            const float h = (first ? pre_resid : *rp) + v;
            *rp = h;
            na.a_out[(size_t)m * na.a_ld + n] = tl_from_float<bf16_t>(h * (first ? pre_weight : na.next_weight[n]));
            sh_sq[(m & 15) * 17 + (n - n0)] = h * h;
            continue;
        }
        if (MODE == MODE_SWIGLU) {
            if (na.act == 2)                             // the tanh form of GELU passes the gate instead of SiLU
                v = 0.5f * v * (1.0f + tanhf(0.7978845608028654f * (v + 0.044715f * v * v * v))) * u;
            else
                v = v / (1.0f + expf(-v)) * u;
        } else if (bias) {
            v += bias[n];
        }
        if (MODE == MODE_PLAIN && na.act == 1) {
            const float p = fmaxf(v, 0.f);
            v = p * p;
        }
        C[(size_t)m * ldc + n] = tl_from_float<TO>(v);
    }
    if (sink) {
        __syncthreads();
        if ((int)threadIdx.x < M && threadIdx.x < 16 && n0 < n_out) {       // (the last tile's second half may have no column)
            float ssum = 0.f;
            for (int c = 0; c < COLS; ++c) ssum += sh_sq[threadIdx.x * 17 + c];
            na.ss_out[(size_t)blockIdx.x * na.ss_out_ld + threadIdx.x] = ssum;
        }
    }
}

// ---- few steps a wave -------------------------------------------------------------------------------------------
// The same product where a wave's share of K is at most four steps, which is the products of narrow and of small models: every wave asks for all it
// reads before it waits for anything.  What bounds such a product is not memory but the instructions in a row: a vector
// instruction takes a wave 5 cycles and one that needs the result before it 8 (3.4 ns; measured), so the nine hundred instructions a
// wave of the kernel above goes through are 2 to 3 us beside 1.6 us that an empty kernel takes.  Hence: addresses in scalar registers
// (buffer loads: a lane's offset once, the steps in the scalar offset), whole steps only, so that nothing is clamped or
// cleared, sums of squares and rotations worked out while the weights are on their way, and an epilogue of one wave whose
// lanes hold four columns in a row.  Waves, shares of K and the order of every sum are those of the kernel above: the
// same bits.
//
// us before and now, weights from memory, M = 1 / 8 / 16: with a sink 896 x 896 3.9, 2.9 / 4.0, 3.2 / 4.1, 3.3; 896 x 4,864 7.0, 4.8 / 7.2, 5.8 / 8.1,
// 6.6; 2,048 x 6,144 9.1, 6.5 / 9.3, 7.5 / 9.9, 9.3; 3,584 x 3,584 7.7, 6.4 / 8.0, 7.0 / 8.8, 7.7; plain 1,024 x 1,024 3.6, 2.5 / 3.6, 2.6 / 3.6, 3.0; gate/up
// 9,728 x 896 7.2, 5.9 / 7.1, 6.3 / 7.5, 6.6; 12,288 x 2,048 12.2, 10.4 / 12.7, 12.6 / 13.6, 13.6; q/k/v 1,152 x 896 5.0, 3.6 / 4.7, 3.9 / 5.0, 4.2; 3,072 x 2,048 7.2,
// 5.3 / 7.2, 5.8 / 7.3, 6.3.  A decode step of 24 layers of 896 at one row 845 -> 676.  Above 640 tiles, or pairs of tiles
// (1,280 work-groups in halves), the rate of the stream counts and not the latency, and the kernel above has more waves to a CU: 32,000 x 2,048
// in this form 26.7 for 23.7.
typedef int sk_i32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ __amdgpu_buffer_rsrc_t sk_rsrc(const void* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, 0x00027000);
}
__device__ __forceinline__ sk_i32x4 sk_load(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
    return __builtin_bit_cast(sk_i32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)voff, (int)soff, 0));
}
__device__ __forceinline__ sk_i32x4 sk_load_stream(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
    return __builtin_bit_cast(sk_i32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)voff, (int)soff, 2));
}
__device__ __forceinline__ sk_i32x4 sk_swap8(sk_i32x4 v) {     // lanes 0..7 and 8..15 of every row of 16 change places
    sk_i32x4 r;
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = __builtin_amdgcn_update_dpp(0, v[i], 0x128, 0xf, 0xf, true);      // row_ror:8
    return r;
}
// a barrier of the work-group that waits for LDS only: loads stay on their way
__device__ __forceinline__ void sk_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}
__device__ __forceinline__ void sk_store4(float* p, f32x4 v) { *reinterpret_cast<f32x4*>(p) = v; }
__device__ __forceinline__ void sk_store4(bf16_t* p, f32x4 v) {
    *reinterpret_cast<uint2*>(p) = make_uint2(tl_pack_bf16(v[0], v[1]), tl_pack_bf16(v[2], v[3]));
}

// NW waves with shares of STEPS steps (the last ones of fewer or none) and one more that puts their sums together: it has nothing of the matrix to wait
// for, so the owed norm's factor, the angles and the residual are ready when the sums are.  K a whole number of steps, N of
// tiles, up to 4 RG rows.  The grid: plain tiles * SPLIT, gated pairs of tiles, q/k/v (pairs of a head, heads).
template <int MODE, typename TO, int SPLIT, bool NARROW, int STEPS, int NW, int RG>
__global__ __launch_bounds__(64 * (NW + (MODE == MODE_QKV ? 2 : 1))) void gemm_few_kernel(const uint4* __restrict__ Ws, const bf16_t* __restrict__ A, int K32, int lda, int M,
                                                                 int second_tile, const float* __restrict__ bias, TO* __restrict__ C, int ldc,
                                                                 QkvArgs qa, TlNormArgs na) {
    constexpr bool DUAL = MODE != MODE_PLAIN;
    constexpr int NACC = DUAL ? 2 : 1, NPARTS = 4 * NW;
    static_assert(SPLIT == 1 || (MODE == MODE_PLAIN && !NARROW), "half tiles come with one stream of weights");
    constexpr bool HALF = SPLIT == 2 || NARROW;                // eight columns of a tile
    constexpr int XS = SPLIT * SK_UNITS * SK_ROWPAD;           // a wave's region of LDS, in units of 16 bytes: its rows, then its sums
    __shared__ uint4 lds[NW * XS];
    __shared__ float sh_part[NPARTS * 16];                     // [part][row] partial sums of squares
    __shared__ float2 sh_rot[MODE == MODE_QKV ? 256 : 1];      // sine and cosine for column i of lane l at 64 i + l
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int c = lane & 15, g = lane >> 4;
    const int unit = HALF ? blockIdx.x >> 1 : blockIdx.x, col0 = HALF ? (blockIdx.x & 1) * 8 : 0;
    int tile = unit, tile2 = second_tile + unit;
    if (MODE == MODE_QKV) {
        const int pph = HALF ? gridDim.x >> 1 : gridDim.x;     // tile pairs per head
        tile = blockIdx.y * 2 * pph + unit, tile2 = tile + pph;
    }
    if (wave < NW) {
        const int s0 = wave * STEPS, mine = (K32 / (4 * SPLIT)) - s0;      // steps of this wave: min(mine, STEPS)
        f32x4 acc[NACC * SPLIT];                               // [h * NACC + a]: the products with chunk h of a load
#pragma unroll
        for (int i = 0; i < NACC * SPLIT; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
        uint4* xs = lds + wave * XS;
        if (mine > 0) {
            const uint32_t tile_bytes = (uint32_t)K32 * 1024u;
            const __amdgpu_buffer_rsrc_t w1 = sk_rsrc((const char*)Ws + (size_t)tile * tile_bytes, tile_bytes);
            const __amdgpu_buffer_rsrc_t w2 = sk_rsrc((const char*)Ws + (size_t)tile2 * tile_bytes, tile_bytes);
            // rows past M lie past the end of the buffer: they come as zeros and feed rows that are not written
            const __amdgpu_buffer_rsrc_t rows = sk_rsrc(A, ((uint32_t)(M - 1) * lda + (uint32_t)K32 * 32u) * 2u);
            const uint32_t in_chunk = !HALF ? lane * 16u : (16 * g + col0 + (c & 7)) * 16u + (c >> 3) * 1024u;
            uint32_t xoff[RG];
#pragma unroll
            for (int i = 0; i < RG; ++i) xoff[i] = (uint32_t)(g + 4 * i) * lda * 2u + c * 16u;
            auto share = [&](auto n) {                         // a share of N steps (in one block: no branch that a load could be moved behind)
                constexpr int N = decltype(n)::value;
                constexpr int NL = NARROW ? 2 : 4;             // loads of a step and tile (NARROW, SPLIT 2: two chunks each)
                sk_i32x4 wv[N][NL], uv[N][NL], xr[N][SPLIT][RG];
#pragma unroll
                for (int st = 0; st < N; ++st) {
                    const uint32_t s = s0 + st;
#pragma unroll
                    for (int h = 0; h < SPLIT; ++h)
#pragma unroll
                        for (int i = 0; i < RG; ++i) xr[st][h][i] = sk_load(rows, xoff[i] + 256 * h, s * 256 * SPLIT);
#pragma unroll
                    for (int i = 0; i < NL; ++i) {
                        const int at = i * (HALF ? 2048 : 1024);
                        wv[st][i] = sk_load_stream(w1, in_chunk + (at & 4095), s * 4096 * SPLIT + (at & ~4095));
                        if (DUAL) uv[st][i] = sk_load_stream(w2, in_chunk + at, s * 4096);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);             // (the compiler would move the loads down to their uses)
#pragma unroll
                for (int st = 0; st < N; ++st) {
                    // rows to LDS, 16 bytes a lane (row g + 4 i, unit c), and back as the product's second operand
#pragma unroll
                    for (int h = 0; h < SPLIT; ++h)
#pragma unroll
                        for (int i = 0; i < RG; ++i) xs[(h * SK_UNITS + c) * SK_ROWPAD + g + 4 * i] = __builtin_bit_cast(uint4, xr[st][h][i]);
                    wave_lds_order();
#pragma unroll
                    for (int cc = 0; cc < 4; ++cc)
#pragma unroll
                        for (int h = 0; h < SPLIT; ++h) {
                            const bf16x8 xf = as_frag(xs[((cc * SPLIT + h) * 4 + g) * SK_ROWPAD + c]);
                            f32x4& a = acc[h * NACC];
                            // NARROW: the odd chunk's columns lie in the lanes of the upper eight and are brought down; what the upper eight
                            // rows of the result add up belongs to no column
                            const sk_i32x4 w = !NARROW ? wv[st][cc] : cc & 1 ? sk_swap8(wv[st][cc >> 1]) : wv[st][cc >> 1];
                            a = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w), xf, a, 0, 0, 0);
                            if (DUAL) {
                                const sk_i32x4 u = !NARROW ? uv[st][cc] : cc & 1 ? sk_swap8(uv[st][cc >> 1]) : uv[st][cc >> 1];
                                acc[1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, u), xf, acc[1], 0, 0, 0);
                            }
                        }
                    wave_lds_order();
                }
            };
            if (mine >= STEPS) share(std::integral_constant<int, STEPS>());
            else if (STEPS > 3 && mine == 3) share(std::integral_constant<int, 3>());
            else if (STEPS > 2 && mine == 2) share(std::integral_constant<int, 2>());
            else share(std::integral_constant<int, 1>());
        }
        // SPLIT 2: rows 0..7 (g < 2) of the first chunks' products, 8..15 of the second's
        f32x4* red = reinterpret_cast<f32x4*>(xs);
#pragma unroll
        for (int a = 0; a < NACC; ++a) {
            f32x4 r = acc[a];
#pragma unroll
            for (int i = 0; i < 4; ++i) r[i] = SPLIT == 2 && g >= 2 ? acc[SPLIT - 1][i] : r[i];
            red[a * 64 + lane] = r;
        }
        sk_barrier();
        return;
    }

    if (MODE == MODE_QKV && wave == NW + 1) {                  // this one works out the angles
        if ((int)blockIdx.y < qa.nq + qa.nkv) {
            const float at = (float)qa.pos[c < M ? c : 0];
            const float* freq = qa.inv_freq + unit * 16 + col0 + 4 * (HALF ? g & 1 : g);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float sn, cs;
                sincosf(at * freq[i], &sn, &cs);
                sh_rot[i * 64 + lane] = make_float2(sn, cs);
            }
        }
        sk_barrier();
        return;
    }

    // the wave that puts the sums together: a lane has row c and the columns n0 .. n0 + 3
    const int n0 = tile * 16 + col0 + 4 * g;
    const bool writes = c < M && (!HALF || g < 2);
    const bool owed = na.ss_in != nullptr, sink = MODE == MODE_PLAIN && na.resid != nullptr;
    f32x4 pre_resid = {0.f, 0.f, 0.f, 0.f}, pre_weight = pre_resid, pre_bias = pre_resid, pre_bias2 = pre_resid;
    int head = 0, idx = 0, slot = 0;
    float rstd = 1.f;
    if (owed) {
        // sums of squares: NPARTS running sums of every NPARTS-th partial of the row, NS of them in a lane; past the last one come
        // zeros.  A load brings 64 / R partials of R rows.
        constexpr int R = 4 * RG, LANES = 64 / R, NS = NPARTS / LANES;
        const int row = lane & (R - 1), q = lane / R;
        const __amdgpu_buffer_rsrc_t ss = sk_rsrc(na.ss_in, (uint32_t)na.ss_n * na.ss_ld * 4u);
        float sum[NS];
#pragma unroll
        for (int p = 0; p < NS; ++p) sum[p] = 0.f;
        const uint32_t hop = (uint32_t)LANES * na.ss_ld * 4u;
        uint32_t off = ((uint32_t)q * na.ss_ld + row) * 4u;
        for (int t = 0; t < na.ss_n; t += 4 * NPARTS) {
            float more[4][NS];
#pragma unroll
            for (int k = 0; k < 4; ++k)
#pragma unroll
                for (int p = 0; p < NS; ++p, off += hop) {
                    more[k][p] = 0.f;
                    if (t + k * NPARTS < na.ss_n) more[k][p] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(ss, (int)off, 0, 0));
                }
#pragma unroll
            for (int k = 0; k < 4; ++k)
#pragma unroll
                for (int p = 0; p < NS; ++p) sum[p] += more[k][p];
        }
#pragma unroll
        for (int p = 0; p < NS; ++p) sh_part[(LANES * p + q) * 16 + row] = sum[p];
    }
    if (writes) {
        if (sink) {
            pre_resid = *reinterpret_cast<const f32x4*>(na.resid + (size_t)c * na.resid_ld + n0);
            pre_weight = *reinterpret_cast<const f32x4*>(na.next_weight + n0);
        }
        if (MODE != MODE_SWIGLU && bias) {
            pre_bias = *reinterpret_cast<const f32x4*>(bias + n0);
            if (MODE == MODE_QKV) pre_bias2 = *reinterpret_cast<const f32x4*>(bias + n0 + qa.d / 2);
        }
        if (MODE == MODE_QKV) slot = qa.slots[c];
    }
    if (MODE == MODE_QKV) head = blockIdx.y, idx = unit * 16 + col0 + 4 * g;
    if (owed) {
        wave_lds_order();
        float parts[NPARTS], ssum = 0.f;
#pragma unroll
        for (int p = 0; p < NPARTS; ++p) parts[p] = sh_part[p * 16 + (c & (4 * RG - 1))];
#pragma unroll
        for (int p = 0; p < NPARTS; ++p) ssum += parts[p];
        rstd = 1.0f / sqrtf(ssum / na.dim + na.eps);
    }
    sk_barrier();
    f32x4 part[NW][NACC * SPLIT];
#pragma unroll
    for (int w = 0; w < NW; ++w) {
        const f32x4* from = reinterpret_cast<const f32x4*>(lds + w * XS);
#pragma unroll
        for (int a = 0; a < NACC; ++a) part[w][a] = from[a * 64 + lane];
        if (SPLIT == 2) part[w][1] = from[(lane + 32) & 63];
    }
    f32x4 v = {0.f, 0.f, 0.f, 0.f}, u = v;
#pragma unroll
    for (int w = 0; w < NW; ++w)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v[i] += part[w][0][i];
            if (DUAL) u[i] += part[w][1][i];
            if (SPLIT == 2) v[i] += part[w][1][i];
        }
    if (owed) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v[i] *= rstd;
            if (DUAL) u[i] *= rstd;
        }
    }
    if (MODE == MODE_QKV) {
        // v, u: dims idx .. idx + 3 and the same + d / 2 of head `head` for token c
        if (!writes) return;
        const int d = qa.d, half = d / 2;
        if (bias) {
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] += pre_bias[i], u[i] += pre_bias2[i];
        }
        if (head < qa.nq + qa.nkv) {
            f32x4 o1, o2;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float2 r = sh_rot[i * 64 + lane];
                o1[i] = v[i] * r.y - u[i] * r.x, o2[i] = u[i] * r.y + v[i] * r.x;
            }
            bf16_t* p = head < qa.nq ? qa.q_out + ((size_t)c * qa.nq + head) * d + idx : qa.k_cache + ((size_t)slot * qa.nkv + (head - qa.nq)) * d + idx;
            if (head < qa.nq || slot >= 0) sk_store4(p, o1), sk_store4(p + half, o2);
        } else if (slot >= 0) {
            const int page = slot / qa.bs, off = slot - page * qa.bs;
            bf16_t* vp = qa.v_cache + (((size_t)page * qa.nkv + (head - qa.nq - qa.nkv)) * d + idx) * qa.bs + off;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                vp[(size_t)i * qa.bs] = tl_from_float<bf16_t>(v[i]);
                vp[(size_t)(i + half) * qa.bs] = tl_from_float<bf16_t>(u[i]);
            }
        }
        return;
    }
    if (MODE == MODE_SWIGLU) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (na.act == 2)                                   // the tanh form of GELU passes the gate instead of SiLU
                v[i] = 0.5f * v[i] * (1.0f + tanhf(0.7978845608028654f * (v[i] + 0.044715f * v[i] * v[i] * v[i]))) * u[i];
            else
                v[i] = v[i] / (1.0f + expf(-v[i])) * u[i];
        }
    } else if (bias) {
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] += pre_bias[i];
    }
    if (sink) {
        float sq[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v[i] = pre_resid[i] + v[i];
            sq[i] = v[i] * v[i];
            pre_weight[i] = v[i] * pre_weight[i];
        }
        if (writes) {
            sk_store4(na.resid + (size_t)c * na.resid_ld + n0, v);
            sk_store4(na.a_out + (size_t)c * na.a_ld + n0, pre_weight);
        }
        // the columns' squares in ascending order: on from the four columns of the lanes before
        float ssum = 0.f;
#pragma unroll
        for (int q = 0; q < 4 / SPLIT; ++q) {
            float t = q == 0 ? 0.f : __shfl_up(ssum, 16, 64);
#pragma unroll
            for (int i = 0; i < 4; ++i) t += sq[i];
            ssum = t;
        }
        if (writes && g == 4 / SPLIT - 1) na.ss_out[(size_t)blockIdx.x * na.ss_out_ld + c] = ssum;
        return;
    }
    if (MODE == MODE_PLAIN && na.act == 1) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float p = fmaxf(v[i], 0.f);
            v[i] = p * p;
        }
    }
    if (writes) sk_store4(C + (size_t)c * ldc + n0, v);
}

static size_t lds_per_wave(int MT, int nacc, int split = 1) {
    const size_t stage = (size_t)MT * split * SK_UNITS * SK_ROWPAD * sizeof(uint4);
    const size_t red = (size_t)nacc * 4 * 64 * sizeof(float);
    return stage > red ? stage : red;
}

static int pick_waves(int tiles, int nsc, int MT, int nacc, int max_waves, int split) {
    // enough waves in flight to cover HBM latency on 256 CUs; K is split among the waves of a group
    int w = 1;
    while (w < max_waves && tiles * w < 4096 && nsc >= 2 * w) w <<= 1;
    while (w > 1 && (size_t)w * lds_per_wave(MT, nacc, split) > SK_MAX_LDS) w >>= 1;
    return w;
}

// Whether a plain product gives half a tile to a work-group: where whole tiles leave half of the CUs without one.  Measured with 1, 8
// and 16 rows, time of half tiles over whole ones: 49 to 128 tiles K = 640 1.07 to 0.96, 776 1.10 to 0.97 and 864 1.11 to 0.99 (two
// waves with an uneven share), 896 0.95 to 0.88, 1,024 0.93 to 0.83, 1,056 1.04 to 0.97, 2,048 1.02 to 0.95, 4,096 1.02 to 0.94, 8,192 0.93 to 0.85; from 136 tiles on
// (more than a half-tile group per CU) 1.04 to 1.46; 16 to 40 tiles 0.9 at K = 1,024 and 8,192 but up to 1.06 at 2,048, and left
// whole.  With a residual sink the next product reads twice as many partial sums, in every work-group: only for a K of more than
// twice the columns, which ends a feed-forward and goes before a narrow q/k/v product, and not one that goes before a wide gate/up.  The two
// products together, half over whole: 1,152 columns next, 96 tiles K = 2,304 0.96 to 0.93, 4,864 0.95 to 0.93, 56 tiles 1.00 to 0.98
// and 0.96 (2,048 1.02 to 1.00); 9,728 columns next, 72 to 128 tiles K = 2,048 1.01 to 1.10, 4,864 1.00 to 1.07.  By the matrix and
// its use, not by the rows.
static int sk_split(int N, int K, bool sink) {
    const int tiles = tl_ceil_div(N, 16);
    return tiles > 48 && tiles <= 128 && (sink ? K >= 2048 && K > 2 * N : K >= 896) ? 2 : 1;
}

// Whether the kernel of few steps takes a product (of these waves and steps a wave), and its launch.  Whole steps and tiles, rows of the
// epilogue's operands on whole quads of columns.
// Pairs of tiles in halves (the same bits): where whole pairs leave half of the CUs without one, or, of up to four rows, where there are
// more pairs than CUs.  us, whole and halves, M = 1 / 8 / 16: q/k/v 1,152 x 896 (36 pairs) 4.5, 3.6 / 4.9, 3.9 / 5.1, 4.2; 3,072 x 2,048 (96) 7.0,
// 5.3 / 7.5, 5.8 / 7.5, 6.3; 4,608 x 3,584 (144) 10.8, 10.8 / 11.2, 12.2 / 11.8, 14.9; gate/up 2,816 x 2,048 (88) 6.9, 4.8 / 7.0, 5.5 / 7.3,
// 6.1; 4,096 x 1,024 (128) 4.2, 4.0 / 4.4, 4.0 / 4.7, 4.5; 6,144 x 1,024 (192) 4.6, 4.9 / 4.8, 5.3 / 5.1, 6.1; 9,728 x 896 (304) 5.9, 5.7 / 6.1, 6.2 /
// 6.7, 6.9; 12,288 x 2,048 (384) 12.1, 10.4 / 12.5, 12.1 / 13.6, 14.7; 17,920 x 1,536 (560) 12.1, 11.4 / 12.7, 13.1 / 15.0, 16.4.
static bool few_narrow(int pairs, int M) { return pairs <= 128 || (M <= 4 && pairs > 256); }
static bool few_aligned(const void* p, int bytes, int ld) { return (uintptr_t)p % bytes == 0 && ld % 4 == 0; }
template <int MODE, typename TO, int SPLIT, bool NARROW>
static bool launch_few(const bf16_t* A, const uint4* Ws, const float* bias, TO* C, int M, int N, int K, int lda, int ldc, int second_tile,
                       hipStream_t stream, const TlNormArgs& na, const QkvArgs& qa, int nwaves, int steps) {
    if (steps > 4 || nwaves < 4 || N > 16 * 640 * (MODE == MODE_QKV ? 2 : 1) || K % (SK_SC * SPLIT) || N % 16 || K >= 1 << 26 || (double)M * lda * 2 >= 2e9) return false;
    if (SPLIT == 2 ? steps == 4 : MODE != MODE_PLAIN && !NARROW && steps == 4) return false;       // (more registers than such a group has)
    if (bias && (uintptr_t)bias % 16) return false;
    if (na.ss_in && (double)na.ss_n * na.ss_ld * 4 >= 2e9) return false;
    if (na.resid && !(few_aligned(na.resid, 16, na.resid_ld) && few_aligned(na.a_out, 8, na.a_ld) && (uintptr_t)na.next_weight % 16 == 0)) return false;
    if (MODE == MODE_QKV ? !(few_aligned(qa.q_out, 8, 0) && few_aligned(qa.k_cache, 8, 0)) : !na.resid && !few_aligned(C, 4 * sizeof(TO), ldc)) return false;
    constexpr int H = NARROW || SPLIT == 2 ? 2 : 1, EXTRA = MODE == MODE_QKV ? 128 : 64;
    const dim3 grid = MODE == MODE_QKV ? dim3(qa.d / 32 * H, qa.nq + 2 * qa.nkv) : dim3(N / 16 * H);
#define GO(STEPS, NW, RG)                                                                                                                      \
    hipLaunchKernelGGL((gemm_few_kernel<MODE, TO, SPLIT, NARROW, STEPS, NW, RG>), grid, dim3(64 * NW + EXTRA), 0, stream, Ws, A, K / 32, lda, M,       \
                       second_tile, bias, C, ldc, qa, na)
#define ROWS(STEPS, NW)               \
    if (M <= 4) GO(STEPS, NW, 1);     \
    else if (M <= 8) GO(STEPS, NW, 2); \
    else GO(STEPS, NW, 4)
#define STEP(STEPS)                                             \
    case STEPS:                                                 \
        if (MODE == MODE_SWIGLU || nwaves == 4) {               \
            ROWS(STEPS, 4);                                     \
        } else {                                                \
            ROWS(STEPS, (MODE == MODE_SWIGLU ? 4 : 8));         \
        }                                                       \
        return true
    switch (steps) {
        STEP(1);
        STEP(2);
        STEP(3);
        default:
            if constexpr (SPLIT == 1 && (MODE == MODE_PLAIN || NARROW)) switch (steps) { STEP(4); }
    }
#undef STEP
#undef ROWS
#undef GO
    return false;
}

template <int MT, int MODE, typename TO, int SPLIT>
static void launch_skinny(const bf16_t* A, const uint4* Ws, const float* bias, TO* C, int M, int n_out, int K, int K32,
                          int lda, int ldc, int second_tile, hipStream_t stream, const TlNormArgs& na,
                          QkvArgs qa = QkvArgs()) {
    // the grid: one group per tile, or per pair of tiles in the two-tile modes
    const int groups = ((MODE == MODE_QKV) ? tl_ceil_div(n_out, 32) : tl_ceil_div(n_out, 16)) * SPLIT;
    const int nacc = MT * (MODE != MODE_PLAIN ? 2 : 1);
    // at most 8 waves to a group (4 in the gate/up form): measured at the 7B shapes, 16 waves stream
    // the down projection in 30.9 us and 8 in 28.0, the fused q/k/v projection in 12.1 and 11.3
    const int nsc = tl_ceil_div(K32, 4 * SPLIT), nwaves = pick_waves(groups, nsc, MT, nacc, MODE == MODE_SWIGLU ? 4 : 8, SPLIT);
    const int steps = tl_ceil_div(nsc, nwaves);
    if (MODE != MODE_PLAIN && few_narrow(groups, M)) {
        if (launch_few<MODE, TO, SPLIT, MODE != MODE_PLAIN>(A, Ws, bias, C, M, n_out, K, lda, ldc, second_tile, stream, na, qa, nwaves, steps)) return;
    } else if (launch_few<MODE, TO, SPLIT, false>(A, Ws, bias, C, M, n_out, K, lda, ldc, second_tile, stream, na, qa, nwaves, steps)) {
        return;
    }
    const size_t smem = (size_t)nwaves * lds_per_wave(MT, nacc, SPLIT);
    hipLaunchKernelGGL((gemm_skinny_kernel<MT, MODE, TO, SPLIT>), dim3(groups), dim3(nwaves * 64), smem, stream, A, Ws, bias, C,
                       M, n_out, K, K32, lda, ldc, second_tile, qa, na);
}

template <int DUAL, typename TO>
static int dispatch_skinny(const bf16_t* A, const uint4* Ws, const float* bias, TO* C, int M, int n_out, int K, int K32,
                           int lda, int ldc, int second_tile, hipStream_t stream, const TlNormArgs& na) {
    // one 16-row MFMA tile of A; more rows go to gemm_rows64.hip
    if (DUAL == MODE_PLAIN && sk_split(n_out, K, na.resid != nullptr) == 2)
        launch_skinny<1, DUAL, TO, DUAL == MODE_PLAIN ? 2 : 1>(A, Ws, bias, C, M, n_out, K, K32, lda, ldc, second_tile, stream, na);
    else
        launch_skinny<1, DUAL, TO, 1>(A, Ws, bias, C, M, n_out, K, K32, lda, ldc, second_tile, stream, na);
    TL_CHECK_LAUNCH("tl_gemm_skinny");
    return 0;
}

// `norm` as the entry points take it: null for none.  A sink needs MODE_PLAIN (checked by the caller).
static int check_norm(const TlNormArgs* norm, TlNormArgs* na, int M, int N, bool sink_allowed, bool gated = false) {
    *na = TlNormArgs();
    if (!norm) return 0;
    *na = *norm;
    if (na->ss_in)
        TL_CHECK_ARG(na->ss_n > 0 && na->ss_ld >= M && na->dim > 0.f && na->eps >= 0.f,
                     "tl_gemm_skinny: bad owed-norm arguments (partials %d, stride %d)", na->ss_n, na->ss_ld);
    TL_CHECK_ARG(na->act == 0 || (na->act == 1 && sink_allowed && !na->resid) || (na->act == 2 && gated),
                 "tl_gemm_skinny: activation %d is not one a plain product without a sink applies", na->act);
    if (na->resid) {
        TL_CHECK_ARG(sink_allowed, "tl_gemm_skinny: only a plain product can add into the residual");
        TL_CHECK_ARG(na->next_weight && na->a_out && na->ss_out && na->resid_ld >= N && na->a_ld >= N &&
                         na->ss_out_ld >= M && M <= 16,
                     "tl_gemm_skinny: bad residual-sink arguments for M=%d N=%d", M, N);
    }
    return 0;
}

static int check_skinny(const void* A, const void* Ws, const void* C, int M, int N, int K, int lda, int ldc) {
    TL_CHECK_ARG(M >= 0 && M <= 16, "tl_gemm_skinny: M=%d is outside [0, 16]", M);
    TL_CHECK_ARG(N > 0 && K > 0, "tl_gemm_skinny: bad sizes N=%d K=%d", N, K);
    TL_CHECK_ARG(K % 8 == 0 && lda % 8 == 0, "tl_gemm_skinny: K=%d and the row stride %d must be multiples of 8", K, lda);
    TL_CHECK_ARG(((uintptr_t)A % 16) == 0 && ((uintptr_t)Ws % 16) == 0, "tl_gemm_skinny: operands must be 16-byte aligned");
    TL_CHECK_ARG(lda >= K && ldc > 0, "tl_gemm_skinny: bad strides");
    return 0;
}

// Columns per partial sum of squares that a plain product with a residual sink leaves (a work-group's columns).
extern "C" int tl_gemm_skinny_columns(int N, int K) { return 16 / sk_split(N, K, true); }

// bfloat16 A [M, K] (row stride lda); Ws: the shuffled copy of W [N, K], ceil(N/16) * ceil(K/32) * 512
// values, zero where it pads; C [M, N] float or bfloat16 (row stride ldc).
// norm: null, or what the product does for the norms around it (TlNormArgs); with a residual sink
// C is not written and may be null.
extern "C" int tl_gemm_skinny(const void* A, const void* Ws, const float* bias, void* C, int c_dtype, int M, int N, int K,
                              int lda, int ldc, const TlNormArgs* norm, hipStream_t stream) {
    if (int rc = check_skinny(A, Ws, C, M, N, K, lda, ldc)) return rc;
    TlNormArgs na;
    if (int rc = check_norm(norm, &na, M, N, true)) return rc;
    TL_CHECK_ARG(na.resid || (C && ldc >= N), "tl_gemm_skinny: output row stride %d < N=%d, or no output", ldc, N);
    if (M == 0) return 0;
    const int K32 = tl_ceil_div(K, 32);
    if (c_dtype == TL_F32)
        return dispatch_skinny<MODE_PLAIN, float>((const bf16_t*)A, (const uint4*)Ws, bias, (float*)C, M, N, K, K32, lda, ldc, 0, stream, na);
    if (c_dtype == TL_BF16)
        return dispatch_skinny<MODE_PLAIN, bf16_t>((const bf16_t*)A, (const uint4*)Ws, bias, (bf16_t*)C, M, N, K, K32, lda, ldc, 0, stream, na);
    return tl_fail("tl_gemm_skinny: unknown output dtype %d", c_dtype);
}

// Ws: the shuffled copy of a [2I, K] matrix, rows [0, I) the gate and rows [I, 2I) the up projection;
// I is a multiple of 16.  C [M, I] = silu(A Wg^T) * (A Wu^T), bfloat16 (norm->act == 2: the tanh form of GELU
// in place of SiLU).
extern "C" int tl_gemm_skinny_swiglu(const void* A, const void* Ws, void* C, int M, int I, int K, int lda, int ldc,
                                     const TlNormArgs* norm, hipStream_t stream) {
    if (int rc = check_skinny(A, Ws, C, M, 2 * I, K, lda, ldc)) return rc;
    TlNormArgs na;
    if (int rc = check_norm(norm, &na, M, 2 * I, false, true)) return rc;
    TL_CHECK_ARG(I % 16 == 0, "tl_gemm_skinny_swiglu: I=%d must be a multiple of 16", I);
    TL_CHECK_ARG(C && ldc >= I, "tl_gemm_skinny_swiglu: output row stride %d < I=%d", ldc, I);
    if (M == 0) return 0;
    return dispatch_skinny<MODE_SWIGLU, bf16_t>((const bf16_t*)A, (const uint4*)Ws, nullptr, (bf16_t*)C, M, I, K,
                                         tl_ceil_div(K, 32), lda, ldc, I / 16, stream, na);
}

// The fused q/k/v projection of a decode step: Ws is the shuffled copy of the [(nq + 2 nkv) d, K]
// matrix, bias float [(nq + 2 nkv) d] or null.  Writes rotated queries to q_out [M, nq*d] and rotated
// keys and the values into the cache at slots[m] (k_cache [pages, page, nkv, d], v_cache
// [pages, nkv, d, page]).  Full-width rotate-half RoPE only: inv_freq holds d/2 values.
extern "C" int tl_gemm_skinny_qkv_rope(const void* A, const void* Ws, const float* bias, const int32_t* pos,
                                       const float* inv_freq, const int32_t* slots, void* q_out, void* k_cache,
                                       void* v_cache, int M, int K, int lda, int nq, int nkv, int d, int bs,
                                       const TlNormArgs* norm, hipStream_t stream) {
    const int N = (nq + 2 * nkv) * d;
    if (int rc = check_skinny(A, Ws, q_out, M, N, K, lda, 1)) return rc;
    TlNormArgs na;
    if (int rc = check_norm(norm, &na, M, N, false)) return rc;
    TL_CHECK_ARG(M <= 16, "tl_gemm_skinny_qkv_rope: M=%d is above 16", M);
    TL_CHECK_ARG(d % 32 == 0 && d > 0 && nq > 0 && nkv > 0 && bs > 0, "tl_gemm_skinny_qkv_rope: bad sizes d=%d nq=%d nkv=%d page=%d", d, nq, nkv, bs);
    TL_CHECK_ARG(pos && inv_freq && slots && q_out && k_cache && v_cache, "tl_gemm_skinny_qkv_rope: missing argument");
    if (M == 0) return 0;
    QkvArgs qa;
    qa.pos = pos;
    qa.inv_freq = inv_freq;
    qa.slots = slots;
    qa.q_out = (bf16_t*)q_out;
    qa.k_cache = (bf16_t*)k_cache;
    qa.v_cache = (bf16_t*)v_cache;
    qa.nq = nq;
    qa.nkv = nkv;
    qa.d = d;
    qa.bs = bs;
    launch_skinny<1, MODE_QKV, bf16_t, 1>((const bf16_t*)A, (const uint4*)Ws, bias, (bf16_t*)nullptr, M, N, K,
                                          tl_ceil_div(K, 32), lda, N, 0, stream, na, qa);
    TL_CHECK_LAUNCH("tl_gemm_skinny_qkv_rope");
    return 0;
}
