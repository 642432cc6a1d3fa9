// The walk over k of a product whose operands' tiles go from memory straight into LDS (gemm_tiles.hip, moe.hip): bfloat16,
// v_mfma_f32_16x16x32_bf16, k in steps of 64 in two halves of 32, for a work-group of waves that each hold MB x NB blocks of 16 x 16.
//
// AST and BST stages of LDS for the rows of A and of W (equal, or 2 and 3); a wave asks for LA and LB pieces of a step.  The
// fragments of a half are read while the other half is multiplied, a few in front of each row of products.  The barrier lies in the
// middle of a step, between the reads of its second half and those of the next step's first; the loads of a later step follow it
// into the buffers of this one, spread over the products too.  A barrier waits for the next step's pieces only, the newer ones
// stay on their way: a CU gets 100 to 130 bytes a ns from L2 or the last-level cache where loads never drain, and 36 where each
// step's loads are waited for one step after they were asked for.
//
// load_a(buffer, i), load_b(buffer, i): ask for the i-th piece; next_a(), next_b(): go on to the next step (where there are fewer
// steps than stages, the last step stays); read_a(buffer, half, i), read_b(buffer, half, j): a block's fragment.  W's fragment is the
// first operand, so that lane 16 g + c ends with row c and the columns 4 g .. 4 g + 3 of each block.
#pragma once
#include "common.h"

#include <type_traits>

typedef float tw_f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 tw_bf16x8 __attribute__((ext_vector_type(8)));

template <int MB, int NB, int AST, int BST, int LA, int LB, typename LoadA, typename LoadB, typename NextA, typename NextB, typename ReadA, typename ReadB>
__device__ __forceinline__ void tile_walk(int nsteps, tw_f32x4 (&acc)[MB][NB], LoadA load_a, LoadB load_b, NextA next_a, NextB next_b,
                                          ReadA read_a, ReadB read_b) {
    static_assert(AST == BST || (AST == 2 && BST == 3), "the waits know these stages");
    auto stage_a = [&](int buf) {
#pragma unroll
        for (int i = 0; i < LA; ++i) load_a(buf, i);
        next_a();
    };
    auto stage_b = [&](int buf) {
#pragma unroll
        for (int i = 0; i < LB; ++i) load_b(buf, i);
        next_b();
    };
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] = (tw_f32x4){0.f, 0.f, 0.f, 0.f};
    tw_bf16x8 a[2][MB], b[2][NB];
    if (AST == BST) {
#pragma unroll
        for (int i = 0; i < AST; ++i) { stage_b(i); stage_a(i); }
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((AST - 1) * (LA + LB)) : "memory");
    } else {
        stage_b(0), stage_b(1), stage_a(0), stage_a(1), stage_b(2);    // in the order the waits below count in
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LA + LB) : "memory");
    }
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int j = 0; j < NB; ++j) b[0][j] = read_b(0, 0, j);
#pragma unroll
    for (int i = 0; i < MB; ++i) a[0][i] = read_a(0, 0, i);
    constexpr int RP = (2 * MB + NB - 1) / MB, LP = (LA + LB + MB - 1) / MB;      // reads and loads in front of a row of products
    int bufa = 0, bufb = 0;
    auto step = [&](int s, auto loads) {
        constexpr bool LOADS = decltype(loads)::value;
#pragma unroll
        for (int i = 0; i < MB; ++i) {
#pragma unroll
            for (int x = i * RP; x < (i + 1) * RP; ++x) {
                if (x < NB) b[1][x] = read_b(bufb, 1, x);
                else if (x < MB + NB) a[1][x - NB] = read_a(bufa, 1, x - NB);
            }
#pragma unroll
            for (int j = 0; j < NB; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[0][j], a[0][i], acc[i][j], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
        const int nexta = bufa == AST - 1 ? 0 : bufa + 1, nextb = bufb == BST - 1 ? 0 : bufb + 1;
        // step s + 1 is here (on their way: W of step s + 2, or all of the steps after s + 1); this wave's reads of step s are done
        if (LOADS || s + BST <= nsteps) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(AST == BST ? (AST - 2) * (LA + LB) : LB) : "memory");
        else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (!LOADS && AST < BST && s + AST < nsteps) stage_a(bufa);    // the rows of the last step, where they have fewer stages
#pragma unroll
        for (int i = 0; i < MB; ++i) {
#pragma unroll
            for (int x = i * RP; x < (i + 1) * RP; ++x) {
                if (x < NB) b[0][x] = read_b(nextb, 0, x);
                else if (x < MB + NB) a[0][x - NB] = read_a(nexta, 0, x - NB);
            }
            if (LOADS) {
#pragma unroll
                for (int x = i * LP; x < (i + 1) * LP; ++x) {          // into the buffers of step s
                    if (x < LA) load_a(bufa, x);
                    else if (x < LA + LB) load_b(bufb, x - LA);
                }
            }
#pragma unroll
            for (int j = 0; j < NB; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[1][j], a[1][i], acc[i][j], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (LOADS) next_a(), next_b();
        bufa = nexta, bufb = nextb;
    };
    int s = 0;
    for (; s + BST < nsteps; ++s) step(s, std::integral_constant<bool, true>());
    for (; s < nsteps; ++s) step(s, std::integral_constant<bool, false>());       // all of W is on its way or here
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");     // nothing may land in LDS that is no longer this work-group's
}

// The same walk with W's fragments straight from memory into the registers they are multiplied from: only the rows go through LDS,
// which four waves of 128 x 64 side by side then read 64 KB of a step.  A's stages are four, W's are two steps of registers; a half's
// registers are asked for again, two steps ahead, behind the products that used them.
// load_b(piece, token): W's fragment j of half h of the step that next_b counts (piece = 4 h + j), asked for behind all loads of A that gave `token`.
// How a stage of A is waited for: loads return in order, and W's fragments of half 1 of step s are asked for behind A's pieces of
// step s + 1, which the token that goes from those loads into these addresses makes sure of.  To have the one is to have the other,
// so a wave that has its fragments in registers (the empty asm reads them) may go to the barrier.
template <int MB, int NB, int LA, typename LoadA, typename LoadB, typename NextA, typename NextB, typename ReadA>
__device__ __forceinline__ void tile_walk_direct(int nsteps, tw_f32x4 (&acc)[MB][NB], uint32_t token, LoadA load_a, LoadB load_b, NextA next_a, NextB next_b,
                                                 ReadA read_a) {
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] = (tw_f32x4){0.f, 0.f, 0.f, 0.f};
    constexpr int AHEAD = MB / 2;            // fragments of A read ahead
    tw_bf16x8 a[AHEAD], b[2][2][NB];
    auto ask_a = [&](int buf) {
#pragma unroll
        for (int i = 0; i < LA; ++i) load_a(buf, i, token);
        next_a();
    };
    auto ask_b = [&](auto set, auto half) {
#pragma unroll
        for (int j = 0; j < NB; ++j) b[decltype(set)::value][decltype(half)::value][j] = load_b(decltype(half)::value * NB + j, token);
    };
    auto here = [&](auto set, auto half) {
#pragma unroll
        for (int j = 0; j < NB; ++j) asm volatile("" ::"v"(b[decltype(set)::value][decltype(half)::value][j]) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    constexpr std::integral_constant<int, 0> _0;
    constexpr std::integral_constant<int, 1> _1;
    ask_a(0), ask_b(_0, _0), ask_a(1), ask_b(_0, _1), next_b(), ask_b(_1, _0), ask_a(2), ask_b(_1, _1), next_b();
    here(_0, _0);
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) a[i] = read_a(0, 0, i);
    int buf = 0;
    auto step = [&](auto set) {
        constexpr int S = decltype(set)::value;
        const int next = (buf + 1) & 3;
#pragma unroll
        for (int i = 0; i < MB; ++i) {
#pragma unroll
            for (int j = 0; j < NB; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[S][0][j], a[i % AHEAD], acc[i][j], 0, 0, 0);
            a[i % AHEAD] = i < MB - AHEAD ? read_a(buf, 0, i + AHEAD) : read_a(buf, 1, i + AHEAD - MB);
            __builtin_amdgcn_sched_barrier(0);
        }
        ask_b(set, _0);
        __builtin_amdgcn_sched_barrier(0);
        here(set, _1);                       // and so are the rows of the next step; nobody reads those of the step before this one
        ask_a((buf + 3) & 3);
#pragma unroll
        for (int i = 0; i < MB; ++i) {
#pragma unroll
            for (int j = 0; j < NB; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[S][1][j], a[i % AHEAD], acc[i][j], 0, 0, 0);
            a[i % AHEAD] = i < MB - AHEAD ? read_a(buf, 1, i + AHEAD) : read_a(next, 0, i + AHEAD - MB);
            __builtin_amdgcn_sched_barrier(0);
        }
        ask_b(set, _1);
        next_b();
        __builtin_amdgcn_sched_barrier(0);
        buf = next;
    };
    int s = 0;
    for (; s + 2 <= nsteps; s += 2) step(_0), step(_1);
    if (s < nsteps) step(_0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");     // nothing may land in LDS that is no longer this work-group's
}

// 16 bytes a lane from sbase + voff into LDS at lds_base + 16 * lane (lds_base is the same for the whole wave); tw_load_once: read
// once, leaving no trace in the caches
__device__ __forceinline__ void tw_load(uint32_t voff, const void* sbase, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_base), "v"(voff), "s"(sbase) : "memory", "m0");
}
// the same, with a token that goes through the load: what is computed from it comes behind
__device__ __forceinline__ void tw_load_token(uint32_t voff, const void* sbase, uint32_t lds_base, uint32_t& token) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %3" : "+v"(token) : "s"(lds_base), "v"(voff), "s"(sbase) : "memory", "m0");
}
__device__ __forceinline__ void tw_load_once(uint32_t voff, const void* sbase, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt" ::"s"(lds_base), "v"(voff), "s"(sbase) : "memory", "m0");
}
__device__ __forceinline__ void tw_store4(float* p, tw_f32x4 o) { *reinterpret_cast<tw_f32x4*>(p) = o; }
__device__ __forceinline__ void tw_store4(bf16_t* p, tw_f32x4 o) {
    *reinterpret_cast<uint2*>(p) = make_uint2(tl_pack_bf16(o[0], o[1]), tl_pack_bf16(o[2], o[3]));
}
