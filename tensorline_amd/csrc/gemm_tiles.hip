// bfloat16 products of more than 64 rows (prompts, portions, large decode batches): C = A W^T, W from its matrix-core ordered
// copy (1 KB pieces: 16 columns x 32 k, lane 16 g + r holding column r at k = 8 g .. + 8), sums in float on
// v_mfma_f32_16x16x32_bf16.
//
// What bounds it: at 2,048 rows the matrix cores at the clock this load runs at (products alone 1.5 to 1.7 PFLOP/s, with the
// fragment reads 1.4 to 1.6, with the loads 1.2 to 1.4), at a few hundred rows the start and end of a work-group's walk and
// how evenly the tiles fill the CUs.  tile_walk.h has the walk over k and why its loads never drain.
//
// WM x WN waves.  Eight waves hold 128 accumulators each at 256 x 256; four waves with 256 each took 1.6 times as long (the
// compiler moves accumulators back and forth).  The rows of A (128 bytes a step) have their eight 16-byte units at
// unit ^ (row / 2) % 8, so that the sixteen lanes that are served together hit all banks; W's pieces are read as they lie.
//
// Tile 7 has W's fragments go from memory into registers (four waves of 128 x 64, 232 registers, two work-groups to a CU): only the rows pass
// through LDS, 96 KB of a step's traffic there for the 176 KB of tile 2, and one work-group's start and end pass beside the other's
// products.  It is the gated form's, whose results of some thousand columns are many tiles.
//
// Tiles are dealt to the XCDs in runs (work-group id modulo 8), rows fastest within panels of 2,048 rows: an XCD walks a few
// tiles of W against all rows and its L2 holds both.
//
// K may be cut into shares (whole steps); the partial products go to a float workspace and are added in order, by whoever
// takes them or by gt_add_kernel.
//
// us, here and in the library with its own choice of kernel (gate/up with the SiLU pass it needs; weights from memory), of sizes that
// are taken (tl_gemm_tiles_plan): 2,048 rows of 17,920 x 1,536 gate/up 106 and 141, of 9,728 x 896 43 and 66, of 1,536 x 8,960 52 and 90;
// 801 rows of 17,920 x 1,536 gate/up 47 and 69, of 1,536 x 8,960 30 and 44, of 2,048 x 1,536 15 and 18; 192 rows of the same 27
// and 33, 16 and 38, 11 and 11; 128 rows of 37,888 x 3,584 gate/up 70 and 74, of 3,584 x 18,944 37 and 54, of 3,584 x 3,584 17 and 25.
// Alone, plain products of 2^20 to 2^23 results and a K of 2,048 to 4,096 are 4% slower here in the mean, 20% at most (640 rows of
// 2,048 x 2,816 23 and 20; 1,521 of 1,024 x 3,072 25 and 21); in whole steps the library is level there, and slower where the host
// queues the step (1,500 tokens of four layers of 1,024 769 us here, 889 with these products in the library).
#include "tile_walk.h"

#include <math.h>

#define GT_KT 64
#define GT_CUS 256

struct GtOut {
    void* C;                   // [M, ldc], or shares x [M, N] float
    int ldc;
    const float* bias;         // [N] or null
    int act;                   // plain: 1 the square of relu; gated: 0 SiLU, 2 the tanh form of GELU passes the gate
};

// GLU: W has the N / 2 gate rows, then the N / 2 up rows, and C = act(gate) * up [M, N / 2]; a wave's first NB / 2 blocks are gate
// columns, the others the up columns of the same places.
template <int WM, int WN, int MB, int NB, int AST, int BST, bool GLU, typename TO>
__global__ __launch_bounds__(64 * WM * WN, MB * NB >= 16 || !BST ? 2 : 4) void gemm_tiles_kernel(const bf16_t* __restrict__ A, int lda, const bf16_t* __restrict__ W,
                                                                                  GtOut out, int M, int N, int K, int mtiles, int ntiles, int shares) {
    constexpr int WAVES = WM * WN, BM = 16 * WM * MB, BN = 16 * WN * NB;
    constexpr int A_UNITS = BM * 8, B_UNITS = BN * 8;                  // 16-byte units of a stage
    constexpr int LA = BM / 8 / WAVES, LB = BN / 8 / WAVES;            // loads per wave and step
    static_assert(LA * 8 * WAVES == BM && LB * 8 * WAVES == BN, "the loads of a step do not divide among the waves");
    constexpr int PANEL = 2048 / BM;
    extern __shared__ uint4 gt_lds[];
    uint4 *lds_a = gt_lds, *lds_b = gt_lds + AST * A_UNITS;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave / WN, wn = wave % WN, c = lane & 15, g = lane >> 4;

    const int plane = mtiles * ntiles, total = plane * shares, per = (total + 7) >> 3;
    const int id = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
    if (id >= total) return;                                           // (the grid is 8 * per)
    const int share = id / plane, in = id - share * plane;
    const int panel = in / (PANEL * ntiles), rows_of = min(PANEL, mtiles - panel * PANEL), q = in - panel * PANEL * ntiles;
    const int nt = q / rows_of, m0 = (panel * PANEL + q % rows_of) * BM;
    const int steps = K / GT_KT, s0 = (int)((long)steps * share / shares), nsteps = (int)((long)steps * (share + 1) / shares) - s0;
    const int ctiles = (N + 15) >> 4, chunks = K >> 5, half = ctiles >> 1;
    const int tile0 = nt * (GLU ? WN * NB / 2 : WN * NB);              // of 16 columns

    // where this lane reads: rows and column tiles that the matrix does not have are its last one again
    uint32_t aoff[LA], boff[LB];
#pragma unroll
    for (int i = 0; i < LA; ++i) {
        const int x = wave * LA + i, r = min(m0 + x * 8 + (lane >> 3), M - 1) - m0;
        aoff[i] = (uint32_t)r * (uint32_t)lda * 2u + 16u * ((lane & 7) ^ ((x & 1) * 4 + (lane >> 4)));
    }
#pragma unroll
    for (int i = 0; i < LB; ++i) {
        const int f = wave * LB + i, t = f >> 1, w = t / NB, j = t % NB;
        const int tile = GLU ? min(tile0 + w * (NB / 2) + j % (NB / 2), half - 1) + (j >= NB / 2 ? half : 0) : min(tile0 + t, ctiles - 1);
        boff[i] = ((uint32_t)(tile - tile0) * (uint32_t)chunks + (f & 1)) * 1024u + lane * 16u;
    }
    const char* ab = (const char*)(A + (size_t)m0 * lda + (size_t)s0 * GT_KT);
    const char* bb = (const char*)W + ((size_t)tile0 * chunks + 2 * s0) * 1024;
    const uint32_t la = (uint32_t)__builtin_amdgcn_readfirstlane((int)tl_lds_address(lds_a)) + wave * LA * 1024;
    const uint32_t lb = (uint32_t)__builtin_amdgcn_readfirstlane((int)tl_lds_address(lds_b)) + wave * LB * 1024;
    const int afrag = (wm * MB * 16 + c) * 8 + (g ^ (c >> 1)), bfrag = wn * NB * 128 + lane;
    int na = 0, nb = 0;
    tw_f32x4 acc[MB][NB];
    if constexpr (BST == 0) {
        static_assert(WM == 1 && AST == 4, "W from memory into registers");
        // (voff is the lane's place in a piece; the scalar offsets are those of the wave's column tiles)
        const __amdgpu_buffer_rsrc_t w = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(W), 0, (int)((uint32_t)ctiles * (uint32_t)chunks * 1024u), 0x00027000);
        uint32_t toff[NB];
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            const int tile = GLU ? min(tile0 + wn * (NB / 2) + j % (NB / 2), half - 1) + (j >= NB / 2 ? half : 0) : min(tile0 + wn * NB + j, ctiles - 1);
            toff[j] = ((uint32_t)tile * (uint32_t)chunks + 2 * s0) * 1024u;
        }
        tile_walk_direct<MB, NB, LA>(
            nsteps, acc, lane * 16u, [&](int buf, int i, uint32_t& token) { tw_load_token(aoff[i], ab, la + buf * (A_UNITS * 16) + i * 1024, token); },
            [&](int x, uint32_t token) {
                return __builtin_bit_cast(tw_bf16x8, __builtin_amdgcn_raw_buffer_load_b128(w, (int)(token + x / NB * 1024), (int)toff[x % NB], 0));
            },
            [&]() { if (++na < nsteps) ab += GT_KT * 2; },
            [&]() {
                const uint32_t on = ++nb < nsteps ? 2048u : 0u;
#pragma unroll
                for (int j = 0; j < NB; ++j) toff[j] += on;
            },
            [&](int buf, int h, int i) { return __builtin_bit_cast(tw_bf16x8, lds_a[buf * A_UNITS + (afrag ^ (4 * h)) + i * 128]); });
    } else
    tile_walk<MB, NB, AST, BST, LA, LB>(
        nsteps, acc, [&](int buf, int i) { tw_load(aoff[i], ab, la + buf * (A_UNITS * 16) + i * 1024); },
        [&](int buf, int i) { tw_load(boff[i], bb, lb + buf * (B_UNITS * 16) + i * 1024); }, [&]() { if (++na < nsteps) ab += GT_KT * 2; },
        [&]() { if (++nb < nsteps) bb += 2048; },
        [&](int buf, int h, int i) { return __builtin_bit_cast(tw_bf16x8, lds_a[buf * A_UNITS + ((afrag + i * 128) ^ (4 * h))]); },
        [&](int buf, int h, int j) { return __builtin_bit_cast(tw_bf16x8, lds_b[buf * B_UNITS + bfrag + j * 128 + h * 64]); });

    // this lane holds row c and the columns 4 g .. 4 g + 3 of each block (N, or N / 2, is a multiple of 4 or of 16: whole quads)
    TO* C = reinterpret_cast<TO*>(out.C);
    if constexpr (GLU) {
        const auto store = [&](auto gate) {
#pragma unroll
            for (int i = 0; i < MB; ++i) {
                const int m = m0 + (wm * MB + i) * 16 + c;
                if (m >= M) continue;
                TO* row = C + (size_t)m * out.ldc;
#pragma unroll
                for (int j = 0; j < NB / 2; ++j) {
                    const int n = (tile0 + wn * (NB / 2) + j) * 16 + 4 * g;
                    if (2 * n >= N) continue;
                    tw_f32x4 o;
#pragma unroll
                    for (int v = 0; v < 4; ++v) o[v] = gate(acc[i][j][v]) * acc[i][NB / 2 + j][v];
                    tw_store4(row + n, o);
                }
            }
        };
        TlMagnitudes size;
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int j = 0; j < NB / 2; ++j)
#pragma unroll
                for (int v = 0; v < 4; ++v) size.take(acc[i][j][v]);
        if (out.act == 2) store([](float v) { return 0.5f * v * (1.0f + tanhf(0.7978845608028654f * (v + 0.044715f * v * v * v))); });
        else if (size.mid_silu()) store([](float v) { return tl_silu_mid(v); });
        else store([](float v) { return v / (1.0f + expf(-v)); });
        return;
    }
#pragma unroll
    for (int i = 0; i < MB; ++i) {
        const int m = m0 + (wm * MB + i) * 16 + c;
        if (m >= M) continue;
        TO* row = C + ((size_t)share * M + m) * out.ldc;
        {
#pragma unroll
            for (int j = 0; j < NB; ++j) {
                const int n = (tile0 + wn * NB + j) * 16 + 4 * g;
                if (n >= N) continue;
                tw_f32x4 o = acc[i][j];
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    if (out.bias) o[v] += out.bias[n + v];
                    if (out.act == 1) o[v] = fmaxf(o[v], 0.f) * fmaxf(o[v], 0.f);
                }
                tw_store4(row + n, o);
            }
        }
    }
}

// The shares' sum in order, with what the product itself does to its result.  Bound by memory; four columns a thread.
template <typename TO>
__global__ __launch_bounds__(256) void gt_add_kernel(const float* __restrict__ parts, int shares, GtOut out, int M, int N) {
    const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 4, plane = (size_t)M * N;
    if (i >= plane) return;
    const int m = (int)(i / N), n = (int)(i - (size_t)m * N);
    tw_f32x4 o = *reinterpret_cast<const tw_f32x4*>(parts + i);
    for (int s = 1; s < shares; ++s) {
        const tw_f32x4 p = *reinterpret_cast<const tw_f32x4*>(parts + s * plane + i);
#pragma unroll
        for (int v = 0; v < 4; ++v) o[v] += p[v];
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        if (out.bias) o[v] += out.bias[n + v];
        if (out.act == 1) o[v] = fmaxf(o[v], 0.f) * fmaxf(o[v], 0.f);
    }
    tw_store4(reinterpret_cast<TO*>(out.C) + (size_t)m * out.ldc + n, o);
}

// ---- which tile ------------------------------------------------------------------------------------------------
// The tiles, and what a step of 64 k takes a work-group: alone on its CU, beside a second one, and its start and end (us).  The
// figures, and those of gt_time, are a fit to 24 matrices (896 x 896 to 37,888 x 3,584) at 65 to 2,048 rows in every tile and
// 1 to 12 shares, with weights from memory (those that the last-level cache holds give other times and other choices): half of the
// 3,600 times are within 5%, and the choice by them takes 0.8% longer than the best one in the mean (0.75 of the library's time; at
// worst, 192 rows of 4,096 x 12,288, 38 us where the best takes 34 and the library 32).
//    id  waves  blocks stages (0: registers); where each has a CU of its own, from so many steps on; a CU holds  step alone, beside a second; start and end
// A grid that leaves every work-group a CU of its own has room for more stages: what bounds a 128 x 128 or 64 x 128 tile there is how much is
// on its way (32 or 24 KB a step, 40 to 50 KB ahead: 55 to 60 bytes a ns and CU), and 64 or 72 KB ahead bring a step in 0.42 us
// where it took 0.58.  The same products in the same order.  us before and after, weights from memory, 801 rows of 3,072 x 2,048 24.3 and
// 19.0; 1,521 of 2,048 x 2,048 24.6 and 21.5; 200 of 12,288 x 2,048 gate/up 25.4 and 21.9; 200 of 4,608 x
// 3,584 22.9 and 20.6; 801 of 2,048 x 2,048 (64 x 128) 17.1 and 16.3.  45 such products in tile 3: 1.13 times as fast in the mean, 1.02 to
// 1.29.  Tile 4 gains 1.02 to 1.11 from some 20 steps on and loses up to 4% below, where filling the stages is a part of the walk; tile 5's
// five stages are enough (nine: 0.97).
#define GT_TILES(X)                                         \
    X(0, 2, 4, 8, 4, 2, 3, 0, 0, 1, 1.072, 1.072, 4.22)     \
    X(1, 2, 4, 8, 3, 2, 3, 0, 0, 1, 0.854, 0.854, 3.94)     \
    X(2, 2, 4, 4, 4, 3, 3, 0, 0, 1, 0.735, 0.735, 3.29)     \
    X(3, 2, 4, 4, 2, 2, 3, 4, 1, 2, 0.584, 0.785, 1.46)     \
    X(4, 2, 4, 2, 2, 3, 3, 5, 20, 2, 0.407, 0.649, 0.95)    \
    X(5, 4, 2, 1, 2, 5, 5, 0, 0, 2, 0.224, 0.406, 0.99)     \
    X(6, 2, 4, 6, 4, 2, 3, 0, 0, 1, 0.931, 0.931, 3.72)     \
    X(7, 1, 4, 8, 4, 4, 0, 0, 0, 2, 0.670, 1.153, 3.72)
struct GtTile {
    int bm, bn, lds, per_cu;
    int alone_lds, alone_from;           // of the form for work-groups with a CU of their own (0: none)
    bool pairs, direct;        // the gated form: whole blocks of gate and of up columns in a wave; W straight into registers
    double step1, step2, ends;
};
#define X(ID, WM, WN, MB, NB, AST, BST, DEEP, FROM, CU, T1, T2, ENDS) \
    {16 * WM * MB, 16 * WN * NB, (16 * WM * MB * AST + 16 * WN * NB * BST) * 128, CU, (16 * WM * MB + 16 * WN * NB) * DEEP * 128, FROM, NB % 2 == 0, BST == 0, T1, T2, ENDS},
static const GtTile gt_tiles[] = {GT_TILES(X)};
#undef X
#define GT_TILE_COUNT 8
#define GT_DIRECT 7
#define GT_MAX_SHARES 12

static int gt_ntiles(const GtTile& t, int N, bool gated) { return gated ? tl_ceil_div(N / 2, t.bn / 2) : tl_ceil_div(N, t.bn); }

// us of a product in tiles of t and `shares`: whole rounds of work-groups over the 256 CUs, or W from memory, or what the CUs
// load, whichever is more, and of tiles that the same bound holds for those that keep the CUs least busy: where W from memory is
// the bound tiles of 256 rows are slower than those of 128 (us, 256 and 128 rows and the library: a head of 152,064 x 3,584 for
// 65 rows 283, 234, 244, for 128 289, 252, 252; of 151,936 x 1,536 for 65 128, 109, 124); then the result's bytes, and the shares'
// second reading (by whoever takes them, or by a kernel)
static double gt_time(const GtTile& t, int M, int N, int K, bool gated, int shares, bool takes_shares) {
    const int mtiles = tl_ceil_div(M, t.bm);
    const double groups = (double)mtiles * gt_ntiles(t, N, gated) * shares, slots = 256.0 * t.per_cu;
    const double steps = tl_ceil_div(K / GT_KT, shares), full = floor(groups / slots), rest = groups - full * slots;
    const double step1 = t.step1 * (1.0 + 0.243 / mtiles), step2 = t.per_cu == 1 ? step1 : t.step2 * (1.0 + 0.760 / mtiles);
    double busy = full * (steps * step2 + t.ends);
    if (rest > 0) busy += steps * (rest <= 256 ? step1 : step2) + t.ends;
    const double weights = 0.233e-6 * 2.0 * N * K, loads = 0.060e-6 * groups * steps * (t.bm + t.bn) * 128.0;
    const double plane = 4e-6 * (double)M * N;           // MB of float
    double us = 3.4 + fmax(busy, fmax(weights, loads)) + 1e-4 * busy + 0.211 * (gated ? 0.25 : shares) * plane;
    if (shares > 1) us += takes_shares ? 0.2 * (shares - 1) * plane : 2.7 + 0.13 * (shares + 1) * plane;
    return us;
}

// Whether the gated form of a product that the formula cuts into tiles of t runs in tiles of 128 x 256 with W straight into registers, two to a
// CU: where there are more of them than CUs and the formula has them ahead.  It is 8% under their times in the mean of 33 sizes (of 9,728
// x 896 to 37,888 x 3,584, 200 to 6,000 rows, weights from memory; 2 to 13%), 10% under those of the other tiles.  The ten of these sizes that take them are 1.05 to 1.17
// times as fast as in the other tile, 1.09 in the mean: us, 801 rows of 17,920 x 1,536 53 and 47, 2,048 121 and 106, 380 of 37,888 x 3,584
// 112 and 104, 1,600 of 11,008 x 2,048 83 and 78.  The others take 5% longer in them in the mean (1,300 rows of 17,920 x 1,536 73 and 82, 513
// 36 and 43, 1,521 of 9,728 x 896 31 and 32), but for three that would take 3 to 8% less (1,000 of 17,920 x 1,536 68 and 63).  Plain products
// of up to 3,000 rows with a choice of shares were level at best (256 tiles) or slower (384 tiles 28 and 36), and have no such form.
static bool gt_goes_direct(const GtTile& t, const GtTile& direct, int M, int N, int K) {
    return (double)tl_ceil_div(M, direct.bm) * gt_ntiles(direct, N, true) > 256 &&
           gt_time(direct, M, N, K, true, 1, false) < gt_time(t, M, N, K, true, 1, false);
}

// The tile and the number of shares for a product (shares * 256 + tile), or -1: not one this file takes.
// More than 512 rows of a matrix that is large both ways stay in the library (us, library and here in the best tile):
// - plain products are level in sum: 513, 801 and 2,048 rows of 4,608 x 3,584 31, 39, 62 and 36, 40, 66; of 3,584 x 3,584 28, 34, 55 and
//   29, 38, 54; of 3,584 x 18,944 89, 116, 224 and 77, 127, 224; of 4,096 x 12,288 91, 98, 185 and 66, 88, 167;
// - gated ones would be faster here (of 37,888 x 3,584 with SiLU 175, 286, 553 and 143, 226, 444; 2,048 rows of 24,576 x 4,096 325 and
//   313) and stay for their results, not for speed: with another order of summation, and gate and up not rounded to bfloat16 ahead of
//   the SiLU, 15 to 31% of 48 draws at top-p 0.9 behind prompts of 150 to 2,300 tokens of the 7B shape came out differently, with
//   logits as far from 64 bits as before.  No
//   limit of the kernel lies here.
extern "C" int tl_gemm_tiles_plan(int M, int N, int K, int gated, int takes_shares) {
    if (M <= 0 || N <= 0 || K <= 0 || K % GT_KT || N % (gated ? 32 : 4) || (double)N * K * 2.0 >= 4e9) return -1;
    if (M > 512 && N > 2048 && K > 2048) return -1;
    int best = -1;
    double least = 0.0;
    for (int i = 0; i < GT_TILE_COUNT; ++i) {
        const GtTile& t = gt_tiles[i];
        if (t.direct || (gated && !t.pairs)) continue;
        const double plane = (double)tl_ceil_div(M, t.bm) * gt_ntiles(t, N, gated);
        for (int shares = 1; shares <= (gated ? 1 : GT_MAX_SHARES); ++shares) {
            if (shares > 1 && (K / GT_KT / shares < 4 || plane * shares > 1.35 * 256 * t.per_cu)) break;
            if (plane * shares >= 2e9) break;
            const double us = gt_time(t, M, N, K, gated, shares, takes_shares);
            if (best < 0 || us < least) best = shares * 256 + i, least = us;
        }
    }
    if (gated && best >= 0 && gt_goes_direct(gt_tiles[best & 255], gt_tiles[GT_DIRECT], M, N, K)) best = 256 + GT_DIRECT;
    return best;
}

// A [M, K] (row stride lda), W the matrix-core ordered copy of [N, K].  gated 0: C [M, N] (float or bfloat16) = act(A W^T + bias);
// 1: C [M, N / 2] bfloat16 = act(gate) * up without bias.  shares > 1 (not gated): partial products into ws [shares, M, N] float,
// added into C unless C is null.
extern "C" int tl_gemm_tiles(const void* A, const void* W, const float* bias, void* C, int c_dtype, float* ws, int M, int N, int K, int lda, int ldc,
                             int tile, int shares, int gated, int act, hipStream_t stream) {
    TL_CHECK_ARG(M > 0 && N > 0 && K > 0 && K % GT_KT == 0 && N % (gated ? 32 : 4) == 0 && lda >= K && lda % 8 == 0 && (uintptr_t)A % 16 == 0 && (uintptr_t)W % 16 == 0,
                 "tl_gemm_tiles: not sizes or an alignment this product takes: M=%d N=%d K=%d lda=%d", M, N, K, lda);
    TL_CHECK_ARG(tile >= 0 && tile < GT_TILE_COUNT && shares >= 1 && shares <= GT_MAX_SHARES && shares <= K / GT_KT && (shares == 1 || (!gated && ws && (uintptr_t)ws % 16 == 0)) &&
                     (C || shares > 1),
                 "tl_gemm_tiles: tile %d in %d shares", tile, shares);
    TL_CHECK_ARG((double)N * K * 2.0 < 4e9 && (double)lda * 512.0 < 4e9, "tl_gemm_tiles: N=%d K=%d lda=%d are beyond 32-bit offsets", N, K, lda);
    TL_CHECK_ARG(gated || !gt_tiles[tile].direct, "tl_gemm_tiles: tile %d serves the gated form", tile);
    TL_CHECK_ARG(!gated || (c_dtype == TL_BF16 && !bias && gt_tiles[tile].pairs), "tl_gemm_tiles: the gated form stores bfloat16, without bias, in tiles of whole pairs");
    TL_CHECK_ARG((gated && (act == 0 || act == 2)) || (!gated && (act == 0 || act == 1)), "tl_gemm_tiles: activation %d is not one this product applies", act);
    TL_CHECK_ARG(!C || (ldc >= (gated ? N / 2 : N) && ldc % 4 == 0 && (uintptr_t)C % (c_dtype == TL_F32 ? 16 : 8) == 0 && (c_dtype == TL_F32 || c_dtype == TL_BF16)),
                 "tl_gemm_tiles: bad output");
    const GtTile& t = gt_tiles[tile];
    const int mtiles = tl_ceil_div(M, t.bm), ntiles = gt_ntiles(t, N, gated);
    TL_CHECK_ARG((double)mtiles * ntiles * shares < 2e9, "tl_gemm_tiles: too many tiles");
    const dim3 grid((unsigned)tl_ceil_div(mtiles * ntiles * shares, 8) * 8);
    const GtOut direct = {C, ldc, bias, act}, partial = {ws, N, nullptr, 0};
    const GtOut& o = shares > 1 ? partial : direct;
    const bool alone = t.alone_lds && K / GT_KT / shares >= t.alone_from && (long long)mtiles * ntiles * shares <= GT_CUS;
#define GO_OF(WM, WN, MB, NB, AST, BST, LDS, GLU, TO)                                                                                              \
    hipLaunchKernelGGL((gemm_tiles_kernel<WM, WN, MB, NB, AST, BST, GLU, TO>), grid, dim3(64 * WM * WN), (size_t)LDS, stream, (const bf16_t*)A, lda, \
                       (const bf16_t*)W, o, M, N, K, mtiles, ntiles, shares)
#define GO(WM, WN, MB, NB, AST, BST, DEEP, GLU, TO)                                                            \
    do {                                                                                                       \
        if constexpr (DEEP != 0) {                                                                             \
            if (alone) { GO_OF(WM, WN, MB, NB, DEEP, DEEP, t.alone_lds, GLU, TO); break; }                     \
        }                                                                                                      \
        GO_OF(WM, WN, MB, NB, AST, BST, t.lds, GLU, TO);                                                       \
    } while (0)
#define X(ID, WM, WN, MB, NB, AST, BST, DEEP, FROM, CU, T1, T2, ENDS)          \
    case ID:                                                                   \
        if (gated) GO(WM, WN, MB, (NB % 2 ? NB + 1 : NB), AST, BST, DEEP, true, bf16_t); \
        else if constexpr (BST != 0) {                                         \
            if (shares > 1 || c_dtype == TL_F32) GO(WM, WN, MB, NB, AST, BST, DEEP, false, float); \
            else GO(WM, WN, MB, NB, AST, BST, DEEP, false, bf16_t);            \
        }                                                                      \
        break;
    switch (tile) { GT_TILES(X) }
#undef X
#undef GO
#undef GO_OF
    TL_CHECK_LAUNCH("tl_gemm_tiles");
    if (shares > 1 && C) {
        const dim3 blocks((unsigned)(((size_t)M * N / 4 + 255) / 256));
        if (c_dtype == TL_F32) hipLaunchKernelGGL(gt_add_kernel<float>, blocks, dim3(256), 0, stream, ws, shares, direct, M, N);
        else hipLaunchKernelGGL(gt_add_kernel<bf16_t>, blocks, dim3(256), 0, stream, ws, shares, direct, M, N);
        TL_CHECK_LAUNCH("tl_gemm_tiles (shares)");
    }
    return 0;
}
