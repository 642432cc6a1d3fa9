// Float attention of steps that bring one token per sequence (the 32-bit path's decode steps): head sizes 64 and 128,
// pages of a power of two of at least four tokens, up to 8 (at 64) or 16 query heads to a key/value head, no cap and no
// bias.  Everything is float multiply-adds.
//
// What such a step has to do is read the cache: 75 MB a layer for 8 sequences of 2,300 keys and 4 key/value heads of 128.  The
// any-shape kernel, whose tiles of keys go through LDS to the matrix cores between two barriers with one chain of dependent
// products per wave, took 72 us for it with the merge, in runs of 256 keys.  Here a work-group of four waves takes a run of keys
// (a split) of one sequence and up to eight query heads of one key/value head; a wave takes 32 keys of every 128, straight
// into registers, 32 KB on their way at a time, and there is no barrier until the run is done.  33 us for the same in runs of 128
// keys (40 in runs of 256: fewer work-groups than the CUs hold; 45 in runs of 64: the waves have half as much to do).
// One sequence of 2,300 37 -> 21, 8 of 300 35 -> 19, 64 of 2,300 305 -> 157, 32 of 1,000 (2 x 64) 30 -> 19, 8 of 2,300 (8 x
// 128, a head each) 99 -> 41.  What bounds it is latency: the run's first key, page, keys and values are asked for one after the
// other, 2.6 TB/s over a layer.  Tried: 64 keys of a wave at a time 46; values asked for before the scores 41 (222 registers);
// values four lanes to a head dimension, coalesced, the lanes added at the end 46 (64 sums per lane).
//
// Scores: lane 4 k + part holds, of key k of a block of 16, the head dimensions 16 i + 4 part .. + 3; the queries come from LDS
// (the same four addresses for all keys) and the four parts are added across lanes.  Weighted sum: lane c has dimensions c (and
// c + 64), its keys 16 bytes at a time as the cache keeps them; the weights come from LDS, the same address for all lanes.
// Sums run over keys in ascending order within a wave's 32, over the blocks of 128, over the four waves in order: an
// order fixed by absolute positions and the length of a split.
#pragma once
#include "attention_generic_kernel.h"

#define AFD_HEADS 8
#define AFD_WAVES 4

// HC: the heads of a work-group, rounded up (numbers of heads that are not there are zero, and dropped at the end).
template <int D, int HC>
__global__ __launch_bounds__(AFD_WAVES * 64, 1) void attn_float_decode_kernel(
    const float* __restrict__ q, int q_stride, const float* __restrict__ k_cache, const float* __restrict__ v_cache,
    const int32_t* __restrict__ tables, int NB, const int32_t* __restrict__ q_start, const int32_t* __restrict__ pos,
    float* __restrict__ out, int out_stride, int nq, int nkv, int bs, int bs_shift, TlMask mask, float scale, int nsplit,
    int split_keys, float* __restrict__ ws_o, float* __restrict__ ws_ml, const float* __restrict__ sinks) {
    constexpr int PC = D / 16, DL = D / 64;              // 16-byte pieces of a key per lane, head dimensions per lane
    constexpr int KB = 2, WK = 16 * KB;                  // blocks of 16 keys, keys of a wave at a time
    __shared__ __attribute__((aligned(16))) float qs[HC][D];
    __shared__ __attribute__((aligned(16))) float ps[AFD_WAVES][HC][WK];
    __shared__ float os[AFD_WAVES][HC][D];
    __shared__ float mls[AFD_WAVES][HC][2];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int s = blockIdx.x, kvh = blockIdx.y, G = nq / nkv;
    const int chunk = blockIdx.z / nsplit, sp = blockIdx.z - chunk * nsplit;
    const int h0 = kvh * G + chunk * HC, heads = min(G - chunk * HC, HC);
    const int t = q_start[s];
    if (q_start[s + 1] <= t) return;
    const int p = pos[t], lo = tl_mask_lo(mask, p);
    const int32_t* table = tables + (size_t)s * NB;
    for (int i = tid; i < HC * D; i += AFD_WAVES * 64) qs[i / D][i % D] = i < heads * D ? q[(size_t)t * q_stride + (size_t)h0 * D + i] * scale : 0.f;
    __syncthreads();

    const int k_first = nsplit > 1 ? sp * split_keys : 0;
    const int k_end = nsplit > 1 ? min(p + 1, k_first + split_keys) : p + 1;
    float m[HC], l[HC], o[HC][DL];
#pragma unroll
    for (int h = 0; h < HC; ++h) {
        m[h] = -INFINITY;
        l[h] = 0.f;
#pragma unroll
        for (int x = 0; x < DL; ++x) o[h][x] = 0.f;
    }
    const int part = lane & 3, sub = lane >> 2;
    for (int k0 = k_first + wave * WK; k0 < k_end; k0 += AFD_WAVES * WK) {
        if (k0 + WK - 1 < lo && k0 >= mask.first) continue;    // the same for the whole wave: none of its keys is in sight
        // keys: block b, key sub; values: quad j of four keys.  A key past the last one is read from the last one's place.
        float4 kr[KB][PC], vr[WK / 4][DL];
        int kpage[KB];
#pragma unroll
        for (int b = 0; b < KB; ++b) kpage[b] = table[min(k0 + 16 * b + sub, k_end - 1) >> bs_shift];
#pragma unroll
        for (int b = 0; b < KB; ++b) {
            const int key = min(k0 + 16 * b + sub, k_end - 1);
            const float* kp = k_cache + (((size_t)kpage[b] * bs + (key & (bs - 1))) * nkv + kvh) * D + 4 * part;
#pragma unroll
            for (int i = 0; i < PC; ++i) kr[b][i] = *reinterpret_cast<const float4*>(kp + 16 * i);
        }
        float sc[KB][HC];
#pragma unroll
        for (int b = 0; b < KB; ++b)
#pragma unroll
            for (int h = 0; h < HC; ++h) sc[b][h] = 0.f;
#pragma unroll
        for (int h = 0; h < HC; ++h) {
            int at = 4 * part;
            asm volatile("" : "+v"(at));                   // opaque: no head's numbers are read ahead, eight heads' would take all registers
#pragma unroll
            for (int i = 0; i < PC; ++i) {
                const float4 qv = *reinterpret_cast<const float4*>(&qs[h][16 * i + at]);
#pragma unroll
                for (int b = 0; b < KB; ++b)
                    sc[b][h] = fmaf(qv.w, kr[b][i].w, fmaf(qv.z, kr[b][i].z, fmaf(qv.y, kr[b][i].y, fmaf(qv.x, kr[b][i].x, sc[b][h]))));
            }
            float mx = -INFINITY;
#pragma unroll
            for (int b = 0; b < KB; ++b) {
                float v = sc[b][h];
                v += __shfl_xor(v, 1, TL_WAVE);
                v += __shfl_xor(v, 2, TL_WAVE);
                const int key = k0 + 16 * b + sub;
                sc[b][h] = key < k_end && !tl_mask_hides(mask, key, lo) ? v : -INFINITY;
                mx = fmaxf(mx, sc[b][h]);
            }
#pragma unroll
            for (int off = 4; off < 64; off <<= 1) mx = fmaxf(mx, __shfl_xor(mx, off, TL_WAVE));
            const float m_new = fmaxf(m[h], mx);
            const float alpha = m_new > -INFINITY ? expf(m[h] - m_new) : 1.f;
            float sum = 0.f;
#pragma unroll
            for (int b = 0; b < KB; ++b) {
                sc[b][h] = sc[b][h] > -INFINITY ? expf(sc[b][h] - m_new) : 0.f;
                sum += sc[b][h];
            }
#pragma unroll
            for (int off = 4; off < 64; off <<= 1) sum += __shfl_xor(sum, off, TL_WAVE);
            l[h] = l[h] * alpha + sum;
            m[h] = m_new;
#pragma unroll
            for (int x = 0; x < DL; ++x) o[h][x] *= alpha;
            // lane part b hands on block b's weights
            static_assert(KB == 2, "two parts hand on two blocks");
            if (part < KB) ps[wave][h][16 * part + sub] = part == 1 ? sc[1][h] : sc[0][h];
        }
        // written and read by this wave only; LDS operations of a wave complete in order
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int j = 0; j < WK / 4; ++j) {
            const int key = min(k0 + 4 * j, (k_end - 1) & ~3);
            const float* vp = v_cache + ((size_t)table[key >> bs_shift] * nkv + kvh) * D * bs + (key & (bs - 1));   // one for the wave
#pragma unroll
            for (int x = 0; x < DL; ++x) vr[j][x] = *reinterpret_cast<const float4*>(vp + (unsigned)((lane + 64 * x) * bs));
        }
        // a value past the last key may be anything (a page's unused end): its weight is zero, and it must not make NaN of it
#pragma unroll
        for (int j = 0; j < WK / 4; ++j) {
            const int left = k_end - (k0 + 4 * j);
#pragma unroll
            for (int x = 0; x < DL; ++x) {
                vr[j][x].x = left > 0 ? vr[j][x].x : 0.f;
                vr[j][x].y = left > 1 ? vr[j][x].y : 0.f;
                vr[j][x].z = left > 2 ? vr[j][x].z : 0.f;
                vr[j][x].w = left > 3 ? vr[j][x].w : 0.f;
            }
        }
#pragma unroll
        for (int j = 0; j < WK / 4; ++j) {
            int at = 4 * j;
            asm volatile("" : "+v"(at));
#pragma unroll
            for (int h = 0; h < HC; ++h) {
                const float4 w = *reinterpret_cast<const float4*>(&ps[wave][h][at]);
#pragma unroll
                for (int x = 0; x < DL; ++x)
                    o[h][x] = fmaf(w.w, vr[j][x].w, fmaf(w.z, vr[j][x].z, fmaf(w.y, vr[j][x].y, fmaf(w.x, vr[j][x].x, o[h][x]))));
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
    // the four waves together, in their order
#pragma unroll
    for (int h = 0; h < HC; ++h) {
#pragma unroll
        for (int x = 0; x < DL; ++x) os[wave][h][lane + 64 * x] = o[h][x];
        if (lane == 0) {
            mls[wave][h][0] = m[h];
            mls[wave][h][1] = l[h];
        }
    }
    __syncthreads();
    for (int i = tid; i < heads * D; i += AFD_WAVES * 64) {
        const int h = i / D, c = i % D;
        float M = -INFINITY, den = 0.f, num = 0.f;
#pragma unroll
        for (int w = 0; w < AFD_WAVES; ++w) M = fmaxf(M, mls[w][h][0]);
#pragma unroll
        for (int w = 0; w < AFD_WAVES; ++w) {
            const float f = mls[w][h][0] > -INFINITY ? expf(mls[w][h][0] - M) : 0.f;      // a wave that saw no key: nothing
            den += f * mls[w][h][1];
            num += f * os[w][h][c];
        }
        if (nsplit > 1) {
            const size_t at = ((size_t)t * nq + h0 + h) * nsplit + sp;
            ws_o[at * D + c] = num;
            if (c == 0) {
                ws_ml[at * 2] = M;
                ws_ml[at * 2 + 1] = den;
            }
        } else {
            const float all = sinks ? den + expf(sinks[h0 + h] - M) : den;                // the head's sink: a key without a value
            out[(size_t)t * out_stride + (size_t)(h0 + h) * D + c] = den > 0.f ? num / all : 0.f;
        }
    }
}

// The heads and pages the kernel above is the faster one for.  More than eight query heads to a key/value head read the
// keys once per eight; us here and on the any-shape kernel, whose 16 rows take up to 16 heads of one read: 16 heads of 128
// 64 sequences of 1,000 40 and 42, of 16,000 526 and 567; 10 heads of 64 64 of 300 15 and 26, but 64 of 6,000 95 and 86, 8 of
// 16,000 50 and 40; 32 heads of 128 200 of 300 72 and 67, 8 of 16,000 122 and 81.
static bool afd_takes_heads(int nq, int nkv, int d, int bs) {
    return nkv > 0 && ((d == 64 && nq / nkv <= AFD_HEADS) || (d == 128 && nq / nkv <= 2 * AFD_HEADS)) && bs >= 4 && (bs & (bs - 1)) == 0;
}

// Whether a float launch runs on the kernel above.  (q rows need no alignment: they are read one number at a time.)
static bool afd_takes(const AgLaunch& a, int max_query_len, long long sequences) {
    const int chunks = tl_ceil_div(a.nq / a.nkv, AFD_HEADS);
    return max_query_len == 1 && afd_takes_heads(a.nq, a.nkv, a.d, a.bs) && a.softcap == 0.f && !a.bias.table &&
           (long long)chunks * a.nsplit <= 65535 && sequences <= 0x7fffffffLL && (uintptr_t)a.k_cache % 16 == 0 && (uintptr_t)a.v_cache % 16 == 0;
}

static void afd_launch(const AgLaunch& a, int S) {
    const int G = a.nq / a.nkv, chunks = tl_ceil_div(G, AFD_HEADS);
    const dim3 grid(S, a.nkv, chunks * a.nsplit), block(AFD_WAVES * 64);
#define AFD_GO(D, HC)                                                                                                         \
    hipLaunchKernelGGL((attn_float_decode_kernel<D, HC>), grid, block, 0, a.stream, (const float*)a.q, a.q_stride,             \
                       (const float*)a.k_cache, (const float*)a.v_cache, a.tables, a.NB, a.q_start, a.pos, (float*)a.out,      \
                       a.out_stride, a.nq, a.nkv, a.bs, a.bs_shift, a.mask, a.scale, a.nsplit, a.split_keys, a.ws_o, a.ws_ml, a.sinks)
#define AFD_HEADS_OF(D)                                                                                                       \
    if (G == 1) AFD_GO(D, 1);                                                                                                 \
    else if (G <= 4) AFD_GO(D, 4);                                                                                            \
    else AFD_GO(D, AFD_HEADS)
    if (a.d == 64) {
        AFD_HEADS_OF(64);
    } else {
        AFD_HEADS_OF(128);
    }
#undef AFD_HEADS_OF
#undef AFD_GO
    ag_merge<float>(a);
}
