// Windows with pooled blocks and sigmoid attention on the matrix cores (bfloat16 pages, float32 scores and weights).
//
// A workgroup of four waves takes one tile of up to 16 queries: 16 rows of one request and one head (prompt portions), or
// the heads of one key/value head of one row (steps of single rows).  The waves deal the tile's keys among themselves in
// pairs of blocks of 32 and meet in LDS at the end.  Nothing is staged: every operand is a 16-byte load straight from the pages, which
// hold 8 lanes of a key side by side and a value lane's tokens side by side.
//
//   S^T = K Q^T   v_mfma_f32_16x16x32_bf16, A = 16 keys x 32 lanes, B = Q^T: the result leaves lane l with its own query
//                 (l % 16) and four keys.  A's row c of tile j holds key (c / 4) * 8 + j * 4 + c % 4 of the block, so that
//                 the two tiles of a block leave lane group g = l / 16 with the keys g * 8 .. g * 8 + 7 in order,
//   O^T += V^T P^T  which is how the next product's B operand wants them (k = g * 8 + e) and how a value lane's tokens lie
//                 in a page (one 16-byte load).
// Weights stay float32: P goes into the product as the sum of two bfloat16 numbers (its rounding and what the rounding
// lost), two products a tile.  The means of blocks are float32 in memory and go in the same way, for keys and for values.
#include <algorithm>
#include <type_traits>

#include "api.h"
#include "common.h"

namespace {

constexpr int kThreads = 256;
constexpr int kWavesM = kThreads / kWave;

struct TileParams {
    const bf16_t *q;
    int q_stride;
    const bf16_t *k_pages, *v_pages;
    const float *pool_k, *pool_v;
    const int32_t *tables;
    int table_stride;
    const int32_t *row_pos, *row_seg, *seg_start;
    int num_segs;
    bf16_t *out;
    int rows, heads, kv_heads, page_size;
    float scale;
    int window, pool, slots;                  // pooled windows
    float softcap, temp_coef;                 // sigmoid weights
    int temp_every;
    const float *r1, *r2, *pb;
    int by_heads;                             // 1: a tile is the heads of one key/value head of one row
    int splits;                               // workgroups that share a tile's keys (blockIdx.z); more than one: partial results
    float *parts;                             // [tile][split][16 * DV sums, 16 maxima, 16 denominators] in the device workspace
    int *counters;                            // a tile's finished workgroups, zero between launches
};

// The hardware's exponential, logarithm and reciprocal (a unit or two in the last place of a float32): these kernels serve the
// bfloat16 path alone, whose operands are rounded to eight bits.
__device__ __forceinline__ float fast_exp(float x) { return __builtin_amdgcn_exp2f(x * 1.4426950408889634f); }
__device__ __forceinline__ float fast_log(float x) { return __builtin_amdgcn_logf(x) * 0.6931471805599453f; }
__device__ __forceinline__ float fast_rcp(float x) { return __builtin_amdgcn_rcpf(x); }

__device__ __forceinline__ void split_bf16(const float (&x)[8], bf16x8_t &hi, bf16x8_t &lo) {
#pragma unroll
    for (int e = 0; e < 8; e++) {
        hi[e] = (bf16_t)x[e];
        lo[e] = (bf16_t)(x[e] - (float)hi[e]);
    }
}

constexpr int kMostSplits = 32;

__device__ __forceinline__ void publish(float *at, float v) { __hip_atomic_store(at, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// VARIANT 0: window + pooled blocks, softmax.  VARIANT 1: every key up to the row, sigmoid weights.
// What bounds a step of single rows is its chain of trips to memory: the row's place with the arguments that are not in registers when a wave starts
// (the first 14 words are), its pages, its keys and values (of the pooled blocks as well: both are asked for before a score is known), and the
// hand-over of the shares: windows of 1,024 with pooled blocks, 2 rows of 12 heads on two of 128 13.9 -> 12.5 us, sigmoid weights 10.3 -> 9.9.
// Pages of a power of two have instances of their own: divisions by the page size, or the question at each address, cost more than they
// save (2,000 rows 57 us with divisions, 63 with the question, 55 like this).
// BY_HEADS: tiles of single rows.  Tiles of 16 rows have instances of their own, which ask for a pooled block's keys and values as they come: a prompt
// has enough workgroups to cover the trips, and what all of them at once hold in registers cost it a wave a SIMD (1,900 rows of 12 heads on two, windows of
// 1,024, keys and values of 64 and 96 lanes 47.5 us with one kernel that asks as they come, 48.6 with one that asks for all at once, 44.2 like this; 128 and 64
// 43.5, 45.3, 39.9, with pages of 48 tokens 44.0, 48.8, 44.2).
template <int KD, int VT, int VARIANT, bool POW2, bool BY_HEADS>
__global__ void __launch_bounds__(kThreads)
mixer_tile_kernel(const int32_t *__restrict__ row_seg, const int32_t *__restrict__ row_pos, const int32_t *__restrict__ tables,
                  const bf16_t *__restrict__ q, int table_stride, int heads, int kv_heads, int q_stride, int page_shift,
                  const TileParams p) {
    typedef const __attribute__((address_space(4))) int32_t *constant_t;      // the same for every lane: a scalar load
    constexpr int D = KD * 32, DV = VT * 16;
    __shared__ float sm_o[kWavesM][16][DV + 1];
    __shared__ float sm_m[kWavesM][16], sm_l[kWavesM][16];
    constexpr bool by_heads = BY_HEADS;
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const int qi = lane & 15, g = lane >> 4;
    // ---- which queries this tile holds
    int seg = -1, row0 = 0, count = 0, kvh = 0, head0 = 0, pos_here = 0;
    if (by_heads) {
        row0 = blockIdx.x;
        seg = ((constant_t)(uintptr_t)row_seg)[row0], pos_here = ((constant_t)(uintptr_t)row_pos)[row0];
        fetch_arguments(p.k_pages, p.v_pages, p.page_size, p.scale, p.window, p.pool, p.slots, p.splits, p.parts, p.counters, p.out, p.rows, pos_here);
    }
    const int G = heads / kv_heads;
    if (by_heads) {
        kvh = blockIdx.y;
        head0 = kvh * G;
        count = G;
        if (seg < 0) {      // padding row: zeros
            if (blockIdx.z == 0)
                for (int i = threadIdx.x; i < G * DV; i += kThreads) p.out[((size_t)row0 * heads + head0) * DV + i] = (bf16_t)0.f;
            return;
        }
    } else {
        int tile = blockIdx.x;
        for (int s = 0; s < p.num_segs; s++) {
            const int first = p.seg_start[s], n = p.seg_start[s + 1] - first;
            const int tiles = (n + 15) >> 4;
            if (tile < tiles) {
                row0 = first + tile * 16;
                count = n - tile * 16 < 16 ? n - tile * 16 : 16;
                seg = p.row_seg[row0];
                break;
            }
            tile -= tiles;
        }
        if (seg < 0) return;      // no such tile, or rows of padding (their outputs are never read in a step of portions)
        head0 = blockIdx.y;
        kvh = head0 / G;
    }
    const bool valid = qi < count;
    const int my_row = by_heads ? row0 : row0 + (valid ? qi : 0);
    const int my_head = by_heads ? head0 + (valid ? qi : 0) : head0;
    const int my_pos = by_heads ? pos_here : row_pos[my_row];
    const int pos_min = by_heads ? pos_here : row_pos[row0], pos_max = by_heads ? pos_here : row_pos[row0 + count - 1];
    const int32_t *tbl = tables + (size_t)seg * table_stride;
    const int ps = p.page_size;
    auto page_of = [&](int key) __attribute__((always_inline)) { return POW2 ? key >> page_shift : key / ps; };
    auto in_page = [&](int key) __attribute__((always_inline)) { return POW2 ? key & (ps - 1) : key % ps; };
    // ---- Q^T as the B operand: column = the lane's query, k = g * 8 + e of every 32 lanes of a head
    bf16x8_t qf[KD];
    {
        const bf16_t *qrow = q + (size_t)my_row * q_stride + (size_t)my_head * D;
#pragma unroll
        for (int kk = 0; kk < KD; kk++) {
            qf[kk] = *(const bf16x8_t *)(qrow + kk * 32 + g * 8);
            if (!valid)
#pragma unroll
                for (int e = 0; e < 8; e++) qf[kk][e] = (bf16_t)0.f;
        }
    }
    f32x4_t o[VT];
#pragma unroll
    for (int t = 0; t < VT; t++) o[t] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    float m_run = -INFINITY, l_run = 0.f;
    // what the lane's query sees
    int lo_q = 0, nb_q = 0;
    float temp = 1.f, a1 = 0.f, a2 = 0.f, bias = 0.f;
    if (VARIANT == 0) {
        lo_q = my_pos - p.window + 1 > 0 ? my_pos - p.window + 1 : 0;
        nb_q = lo_q / p.pool;
    } else {
        temp = 1.0f + p.temp_coef * logf((float)((my_pos + 1) / p.temp_every) + 1.0f);
        a1 = p.r1[my_head], a2 = p.r2[my_head], bias = p.pb[my_head];
    }
    const float sc = p.scale * temp;
    const float two_over_cap = VARIANT == 1 ? 2.0f / p.softcap : 0.f;
    int turn = 0;      // blocks are dealt to the waves in turn, over both kinds of keys

    // one block of 32 keys: scores in s[2], then weights, then the products with the values
    auto weigh_and_add = [&](f32x4_t (&s)[2], auto visible, auto distance, auto load_values) {
        float pvals[8];
        if (VARIANT == 0) {
            float m_blk = -INFINITY;
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    s[j][i] = visible(g * 8 + j * 4 + i) ? s[j][i] * sc : -INFINITY;
                    m_blk = fmaxf(m_blk, s[j][i]);
                }
            m_blk = max_16_apart(m_blk);
            m_blk = max_32_apart(m_blk);
            const float m_new = fmaxf(m_run, m_blk);
            const float alpha = m_run == -INFINITY ? 0.f : fast_exp(m_run - m_new);
            float sum = 0.f;
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float pv = s[j][i] == -INFINITY ? 0.f : fast_exp(s[j][i] - m_new);
                    pvals[j * 4 + i] = pv;
                    sum += pv;
                }
            l_run = l_run * alpha + sum;      // the lane's own keys; the lane groups are added at the end
            m_run = m_new;
#pragma unroll
            for (int t = 0; t < VT; t++) o[t] *= alpha;
        } else {
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const int slot = g * 8 + j * 4 + i;
                    // cap * tanh(x / cap) = cap - 2 cap / (exp(2 x / cap) + 1): an overflowing exponential gives cap, none -cap
                    float x = s[j][i] * sc;
                    x = p.softcap - 2.0f * p.softcap * fast_rcp(fast_exp(x * two_over_cap) + 1.0f);
                    x = x - a1 * fast_log(fmaf(a2, distance(slot), 1.0f)) + bias;
                    pvals[j * 4 + i] = visible(slot) ? fast_rcp(1.0f + fast_exp(-x)) : 0.f;
                }
        }
        bf16x8_t p_hi, p_lo;
        split_bf16(pvals, p_hi, p_lo);
        load_values(p_hi, p_lo);
    };

    // ---- the means of blocks behind the window (VARIANT 0)
    if constexpr (VARIANT == 0) {
        const int lo_max = pos_max - p.window + 1 > 0 ? pos_max - p.window + 1 : 0;
        const int nb_max = lo_max / p.pool;
        for (int base = 0; base < nb_max; base += 32, turn++) {
            if ((turn & (kWavesM - 1)) != wave || (turn / kWavesM) % p.splits != (int)blockIdx.z) continue;
            // where a block's mean lies: the page of its last token, and its place there
            auto mean_of = [&](int b) __attribute__((always_inline)) {
                const int end = min(b, nb_max - 1) * p.pool + p.pool - 1;
                return ((size_t)tbl[page_of(end)] * kv_heads + kvh) * p.slots + (p.slots > 1 ? in_page(end) / p.pool : 0);
            };
            // A = V^T: row = a value lane, k = the blocks base + g * 8 + e, each in a page and slot of its own
            size_t vat[8];
            f32x4_t kx[2][KD][2];
            float vx[VT][8];
            auto ask_keys = [&](int j) __attribute__((always_inline)) {
                const float *kr = p.pool_k + mean_of(base + (qi >> 2) * 8 + j * 4 + (qi & 3)) * D;
#pragma unroll
                for (int kk = 0; kk < KD; kk++)
#pragma unroll
                    for (int i = 0; i < 2; i++) kx[j][kk][i] = *(const f32x4_t *)(kr + kk * 32 + g * 8 + 4 * i);
            };
            auto places = [&]() __attribute__((always_inline)) {
#pragma unroll
                for (int e = 0; e < 8; e++) vat[e] = mean_of(base + g * 8 + e) * DV;
            };
            auto ask_values = [&](int t) __attribute__((always_inline)) {
#pragma unroll
                for (int e = 0; e < 8; e++) vx[t][e] = p.pool_v[vat[e] + t * 16 + qi];
            };
            if constexpr (by_heads) {
                places();
#pragma unroll
                for (int j = 0; j < 2; j++) ask_keys(j);
#pragma unroll
                for (int t = 0; t < VT; t++) ask_values(t);
                __builtin_amdgcn_sched_barrier(0);      // all of them before the first product
            }
            f32x4_t s[2];
#pragma unroll
            for (int j = 0; j < 2; j++) {
                if constexpr (!by_heads) ask_keys(j);
                s[j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int kk = 0; kk < KD; kk++) {
                    float x[8];
                    *(f32x4_t *)x = kx[j][kk][0];
                    *(f32x4_t *)(x + 4) = kx[j][kk][1];
                    bf16x8_t hi, lo;
                    split_bf16(x, hi, lo);
                    s[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(hi, qf[kk], s[j], 0, 0, 0);
                    s[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(lo, qf[kk], s[j], 0, 0, 0);
                }
            }
            weigh_and_add(
                s, [&](int slot) { return valid && base + slot < nb_q; }, [&](int) { return 0.f; },
                [&](const bf16x8_t &p_hi, const bf16x8_t &p_lo) {
                    if constexpr (!by_heads) places();
#pragma unroll
                    for (int t = 0; t < VT; t++) {
                        if constexpr (!by_heads) ask_values(t);
                        bf16x8_t hi, lo;
                        split_bf16(vx[t], hi, lo);
                        o[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(hi, p_hi, o[t], 0, 0, 0);
                        o[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(hi, p_lo, o[t], 0, 0, 0);
                        o[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(lo, p_hi, o[t], 0, 0, 0);
                    }
                });
        }
    }
    // ---- the tokens: from the first one that the tile's first row sees, two blocks of 32 positions a turn.  All operands of a
    // turn are asked for before the first product, so that the second block's loads and both blocks' values travel while the
    // first block's scores are weighed.  Keys behind the tile's last row are read from an address that exists and masked.
    {
        const int first = VARIANT == 0 ? (pos_min - p.window + 1 > 0 ? pos_min - p.window + 1 : 0) : 0;
        for (int base0 = first & ~63; base0 <= pos_max; base0 += 64, turn++) {
            if ((turn & (kWavesM - 1)) != wave || (turn / kWavesM) % p.splits != (int)blockIdx.z) continue;
            bf16x8_t ka[2][2][KD], va[2][VT];
#pragma unroll
            for (int half = 0; half < 2; half++) {
                const int base = base0 + half * 32;
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    int key = base + (qi >> 2) * 8 + j * 4 + (qi & 3);
                    key = key <= pos_max ? key : pos_max;
                    const bf16_t *kr = p.k_pages + key_offset(tbl[page_of(key)], kv_heads, kvh, ps, D, in_page(key), g * 8);
#pragma unroll
                    for (int kk = 0; kk < KD; kk++) ka[half][j][kk] = *(const bf16x8_t *)(kr + (size_t)kk * 4 * ps * 8);      // 32 lanes on: four chunks of 8
                }
                int key = base + g * 8;                  // eight tokens side by side in one page (pages hold multiples of 16)
                key = key <= pos_max ? key : pos_max & ~7;
                const bf16_t *vr = p.v_pages + (((size_t)tbl[page_of(key)] * kv_heads + kvh) * DV + qi) * ps + in_page(key);
#pragma unroll
                for (int t = 0; t < VT; t++) va[half][t] = *(const bf16x8_t *)(vr + (size_t)t * 16 * ps);
            }
#pragma unroll
            for (int half = 0; half < 2; half++) {
                const int base = base0 + half * 32;
                f32x4_t s[2];
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    s[j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int kk = 0; kk < KD; kk++) s[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka[half][j][kk], qf[kk], s[j], 0, 0, 0);
                }
                weigh_and_add(
                    s, [&](int slot) { const int key = base + slot; return valid && key <= my_pos && key >= lo_q; },
                    [&](int slot) { const int dist = my_pos - (base + slot); return (float)(dist > 0 ? dist : 0); },
                    [&](const bf16x8_t &p_hi, const bf16x8_t &p_lo) {
#pragma unroll
                        for (int t = 0; t < VT; t++) {
                            o[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(va[half][t], p_hi, o[t], 0, 0, 0);
                            o[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(va[half][t], p_lo, o[t], 0, 0, 0);
                        }
                    });
            }
        }
    }
    // ---- the waves meet
    if (VARIANT == 0) {
        l_run = sum_16_apart(l_run);
        l_run = sum_32_apart(l_run);
        if (g == 0) sm_m[wave][qi] = m_run, sm_l[wave][qi] = l_run;
    }
#pragma unroll
    for (int t = 0; t < VT; t++)
#pragma unroll
        for (int i = 0; i < 4; i++) sm_o[wave][qi][t * 16 + g * 4 + i] = o[t][i];
    __syncthreads();
    float *part = p.splits > 1 ? p.parts + ((size_t)(blockIdx.y * p.rows + blockIdx.x) * p.splits + blockIdx.z) * (16 * DV + 32) : nullptr;
    for (int idx = threadIdx.x; idx < count * DV; idx += kThreads) {
        const int q = idx / DV, d = idx - q * DV;
        float acc = 0.f, l = 0.f;
        if (VARIANT == 0) {
            float m = -INFINITY;
#pragma unroll
            for (int w = 0; w < kWavesM; w++) m = fmaxf(m, sm_m[w][q]);
#pragma unroll
            for (int w = 0; w < kWavesM; w++) {
                const float f = sm_m[w][q] == -INFINITY ? 0.f : expf(sm_m[w][q] - m);
                l += sm_l[w][q] * f;
                acc += sm_o[w][q][d] * f;
            }
            if (part != nullptr) {      // this workgroup's share of the keys: the sums as they are, against its own maximum
                publish(part + q * DV + d, acc);
                if (d == 0) publish(part + 16 * DV + q, m), publish(part + 16 * DV + 16 + q, l);
                continue;
            }
            acc = l > 0.f ? acc / l : 0.f;
        } else {
#pragma unroll
            for (int w = 0; w < kWavesM; w++) acc += sm_o[w][q][d];
            if (part != nullptr) {
                publish(part + q * DV + d, acc);
                continue;
            }
        }
        const int row = by_heads ? row0 : row0 + q, head = by_heads ? head0 + q : head0;
        p.out[((size_t)row * heads + head) * DV + d] = (bf16_t)acc;
    }
    if (part == nullptr) return;
    // ---- the shares meet (tiles by heads): the workgroup that counts last puts them together in the order of the shares, all of
    // its loads asked for before it waits.  A kernel of its own for this took 8.4 us (softmax) and 6.0 (sigmoid) at 2 rows and 6 shares
    // (prompts and answers of 2 requests, 72 such launches: 14.46 -> 14.10 ms).
    __shared__ int s_seen;
    __shared__ float s_factor[kMostSplits][16], s_sum[kMostSplits][16];
    const int tile = blockIdx.y * p.rows + blockIdx.x, splits = p.splits;
    parts_published();
    __syncthreads();
    if (threadIdx.x == 0) s_seen = __hip_atomic_fetch_add(p.counters + tile, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (s_seen != splits - 1) return;
    parts_visible();
    if (threadIdx.x == 0) __hip_atomic_store(p.counters + tile, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);      // for the next launch
    constexpr int kStride = 16 * DV + 32, NI = 4, NS = 8;
    const float *all = p.parts + (size_t)tile * splits * kStride;
    auto fetch = [](const float *at) __attribute__((always_inline)) { return __hip_atomic_load(at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
    if (VARIANT == 0) {
        for (int i = threadIdx.x; i < splits * 16; i += kThreads) {
            const int q = i & 15;
            const float *of = all + (size_t)(i >> 4) * kStride + 16 * DV + q;
            if (q < count) s_factor[i >> 4][q] = fetch(of), s_sum[i >> 4][q] = fetch(of + 16);
        }
    }
    for (int base = 0; base < count * DV; base += NI * kThreads) {      // every thread the same trips
        const int idx0 = base + threadIdx.x;
        float acc[NI], m[NI], l[NI];
#pragma unroll
        for (int i = 0; i < NI; i++) acc[i] = l[i] = 0.f, m[i] = -INFINITY;
        for (int s0 = 0; s0 < splits; s0 += NS) {
            float v[NI][NS];
#pragma unroll
            for (int i = 0; i < NI; i++)
#pragma unroll
                for (int s = 0; s < NS; s++) {
                    const int idx = min(idx0 + i * kThreads, count * DV - 1), at = min(s0 + s, splits - 1);
                    v[i][s] = fetch(all + (size_t)at * kStride + idx);      // idx = q * DV + d
                }
            if (VARIANT == 0 && s0 == 0) {
                if (base == 0) __syncthreads();                             // the maxima and sums are in LDS
#pragma unroll
                for (int i = 0; i < NI; i++) {
                    const int q = min(idx0 + i * kThreads, count * DV - 1) / DV;
                    for (int s = 0; s < splits; s++) m[i] = fmaxf(m[i], s_factor[s][q]);
                }
            }
#pragma unroll
            for (int i = 0; i < NI; i++) {
                const int q = min(idx0 + i * kThreads, count * DV - 1) / DV;
#pragma unroll
                for (int s = 0; s < NS; s++) {
                    if (s0 + s >= splits) break;
                    if (VARIANT == 0) {
                        const float ms = s_factor[s0 + s][q], f = ms == -INFINITY ? 0.f : expf(ms - m[i]);
                        l[i] += s_sum[s0 + s][q] * f;
                        acc[i] += v[i][s] * f;
                    } else {
                        acc[i] += v[i][s];
                    }
                }
            }
        }
#pragma unroll
        for (int i = 0; i < NI; i++) {
            const int idx = idx0 + i * kThreads;
            if (idx >= count * DV) break;
            const int q = idx / DV, d = idx - q * DV;
            if (VARIANT == 0) acc[i] = l[i] > 0.f ? acc[i] / l[i] : 0.f;
            p.out[((size_t)row0 * heads + head0 + q) * DV + d] = (bf16_t)acc[i];
        }
    }
}

template <int VARIANT, int KD>
int launch_vt(const TileParams &p, int vt, dim3 grid, hipStream_t stream) {
    int shift = -1;
    if ((p.page_size & (p.page_size - 1)) == 0) shift = __builtin_ctz((unsigned)p.page_size);
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, dim3(kThreads), 0, stream, p.row_seg, p.row_pos, p.tables, p.q, p.table_stride, p.heads, p.kv_heads,
                           p.q_stride, shift, p);
    };
    auto of = [&](auto pow2, auto by_heads) {
        constexpr bool P = decltype(pow2)::value, B = decltype(by_heads)::value;
        switch (vt) {
        case 2: go(mixer_tile_kernel<KD, 2, VARIANT, P, B>); return 0;
        case 4: go(mixer_tile_kernel<KD, 4, VARIANT, P, B>); return 0;
        case 6: go(mixer_tile_kernel<KD, 6, VARIANT, P, B>); return 0;
        case 8: go(mixer_tile_kernel<KD, 8, VARIANT, P, B>); return 0;
        }
        return 1;
    };
    if (p.by_heads) return shift >= 0 ? of(std::true_type{}, std::true_type{}) : of(std::false_type{}, std::true_type{});
    return shift >= 0 ? of(std::true_type{}, std::false_type{}) : of(std::false_type{}, std::false_type{});
}

template <int VARIANT>
int launch_tiles(TileParams &p, int head_dim, int v_dim, int keys_bound, hipStream_t stream) {
    // takes: bfloat16, keys in chunks of 8 (checked by the caller), heads of 32, 64, 96 or 128 lanes, values of 32, 64, 96 or
    // 128, pages of a multiple of 16 tokens, and for steps of single rows at most 16 heads a key/value head
    if (head_dim % 32 != 0 || head_dim > 128 || v_dim % 32 != 0 || v_dim > 128 || p.page_size % 16 != 0) return 1;
    const int G = p.heads / p.kv_heads;
    p.by_heads = p.rows == p.num_segs ? 1 : 0;
    if (p.by_heads && G > 16) return 1;
    dim3 grid = p.by_heads ? dim3(p.rows, p.kv_heads) : dim3((p.rows + 15) / 16 + p.num_segs, p.heads);
    if (grid.y > 65535) return 1;
    // Steps of single rows have a tile a row and key/value head: with few of them, several workgroups share a tile's keys
    // (at least 256 keys each, two workgroups a compute unit at most), and whichever is last puts their shares together.
    p.splits = 1;
    p.parts = nullptr;
    if (p.by_heads) {
        const long tiles = (long)p.rows * p.kv_heads;
        long splits = std::min<long>(std::min<long>(512 / std::max<long>(tiles, 1), (keys_bound + 255) / 256), kMostSplits);
        void *base = nullptr;
        size_t bytes = 0;
        if (splits > 1 && fllm_device_workspace(&base, &bytes) && bytes > kWorkspaceCounterBytes) {
            const size_t room = (bytes - kWorkspaceCounterBytes) / sizeof(float), each = (size_t)tiles * (16 * v_dim + 32);
            splits = std::min<long>(splits, (long)(room / each));
            if (splits > 1) {      // and so there are fewer tiles than 256: a counter each
                p.splits = (int)splits;
                p.counters = (int *)base;
                p.parts = (float *)((char *)base + kWorkspaceCounterBytes);
                grid.z = (unsigned)splits;
            }
        }
    }
    int declined = 1;
    switch (head_dim / 32) {
    case 1: declined = launch_vt<VARIANT, 1>(p, v_dim / 16, grid, stream); break;
    case 2: declined = launch_vt<VARIANT, 2>(p, v_dim / 16, grid, stream); break;
    case 3: declined = launch_vt<VARIANT, 3>(p, v_dim / 16, grid, stream); break;
    case 4: declined = launch_vt<VARIANT, 4>(p, v_dim / 16, grid, stream); break;
    }
    return declined;
}

}  // namespace

// 0: launched; 1: the shape is not one these kernels take (the caller runs the plain kernel).
int fllm_pooled_window_attention_bf16_fast(const void *q, int q_stride, const void *k_pages, const void *v_pages, const float *pool_k,
                                           const float *pool_v, const int32_t *tables, int table_stride, const int32_t *row_pos,
                                           const int32_t *row_seg, const int32_t *seg_start, int num_segs, void *out, int rows,
                                           int heads, int kv_heads, int head_dim, int v_dim, int page_size, float scale, int window,
                                           int pool, int max_context, hipStream_t stream) {
    if (!fllm_fast_kernels_enabled() || seg_start == nullptr || num_segs <= 0) return 1;
    TileParams p = {};
    p.q = (const bf16_t *)q, p.q_stride = q_stride, p.k_pages = (const bf16_t *)k_pages, p.v_pages = (const bf16_t *)v_pages;
    p.pool_k = pool_k, p.pool_v = pool_v, p.tables = tables, p.table_stride = table_stride, p.row_pos = row_pos, p.row_seg = row_seg;
    p.seg_start = seg_start, p.num_segs = num_segs, p.out = (bf16_t *)out, p.rows = rows, p.heads = heads, p.kv_heads = kv_heads;
    p.page_size = page_size, p.scale = scale, p.window = window, p.pool = pool, p.slots = (page_size + pool - 1) / pool;
    const int span = max_context > 0 ? std::min(max_context, window + (max_context + pool - 1) / pool) : window;
    if (launch_tiles<0>(p, head_dim, v_dim, span, stream)) return 1;
    return fllm_check_launch("pooled_window_attention (matrix cores)");
}

int fllm_sigmoid_attention_bf16_fast(const void *q, int q_stride, const void *k_pages, const void *v_pages, const int32_t *tables,
                                     int table_stride, const int32_t *row_pos, const int32_t *row_seg, const int32_t *seg_start,
                                     int num_segs, void *out, int rows, int heads, int kv_heads, int head_dim, int v_dim, int page_size,
                                     float scale, float softcap, const float *r1, const float *r2, const float *pb, float temp_coef,
                                     int temp_every, int max_context, hipStream_t stream) {
    if (!fllm_fast_kernels_enabled() || seg_start == nullptr || num_segs <= 0) return 1;
    TileParams p = {};
    p.q = (const bf16_t *)q, p.q_stride = q_stride, p.k_pages = (const bf16_t *)k_pages, p.v_pages = (const bf16_t *)v_pages;
    p.tables = tables, p.table_stride = table_stride, p.row_pos = row_pos, p.row_seg = row_seg, p.seg_start = seg_start;
    p.num_segs = num_segs, p.out = (bf16_t *)out, p.rows = rows, p.heads = heads, p.kv_heads = kv_heads, p.page_size = page_size;
    p.scale = scale, p.softcap = softcap, p.temp_coef = temp_coef, p.temp_every = temp_every, p.r1 = r1, p.r2 = r2, p.pb = pb;
    p.window = 1, p.pool = 1, p.slots = 1;
    if (launch_tiles<1>(p, head_dim, v_dim, max_context, stream)) return 1;
    return fllm_check_launch("sigmoid_attention (matrix cores)");
}
