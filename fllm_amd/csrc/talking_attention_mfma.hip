// Matrix-core form of the attention whose heads talk to each other (talking_attention.hip says what is computed),
// bfloat16 operands, float32 scores, statistics and sums.
//
// A workgroup of eight waves takes 16 consecutive rows of one request (a prompt portion's row tile) with ALL heads, because a
// mixed score needs every head's raw score of the same (row, key).  It walks the keys the tile sees in blocks of 128; the
// blocks of a tile are dealt out in runs of `share_blocks` to several workgroups where a launch has few tiles, which leave
// their running maxima, sums and unnormalised outputs in a workspace that a second kernel merges.  (Decode steps, one row a
// request, have a kernel of their own further down.)
//
// Keys and values go straight from the pages into operands: a wave's 16 keys and a wave's 16 value lanes serve that wave
// alone, so a pass through LDS would share nothing.  What the waves share lies in LDS: the tile's queries, a block's maxima and
// its weights.  The products are the transposed ones, v_mfma_f32_16x16x32_bf16 with D[m = 4 (l / 16) + i][n = l % 16], so that a
// lane keeps one row throughout:
//
//   1. wave w takes the block's keys 16 w .. 16 w + 15: for every head  raw_g^T[key][row] = K_{g / group} Q_g^T
//      (A = 16 keys x 32 lanes, B = the rows' queries from LDS).  A lane then holds, for its four (key, row) pairs, the raw
//      scores of all heads: the mix  s_h = sum_g talk[h, g] (raw_g * scale * temp[g])  is lane-local, its factors come
//      through the scalar cache.
//   2. the block's largest score a (head, row) goes through LDS (eight waves hold different keys); every wave computes
//      the same running maximum, weighs its scores, keeps its share of the running sum and leaves the weights in LDS
//      as bfloat16, [head][row][128 keys] with a row's 16-byte pieces XORed by the row (16 rows at one place of the row
//      would meet in the same banks).
//   3. the outputs  O_h^T[lane of v][row] += V_{h / group}^T P_h^T: wave w owns the value lanes 16 (w % n) .. of every
//      head, n = v_dim / 16 rounded up to a power of two; where n < 8 the heads are dealt out among the waves of one n.
// The keys of the next block and the values of the next key/value head are on their way while this one is multiplied, and
// page numbers a block earlier still; two barriers a block.
//
// What bounds it: vector instructions (the mix alone is H^2 multiply-adds a (row, key) pair) and LDS reads (queries and
// weights, one 16-byte read a product).  Before, four waves held both value halves and staged keys and values through LDS
// in two stages a block of 64 keys: 416 to 512 registers a lane, so one wave a SIMD waited out every latency by itself.
// 1,900 rows from a request's first token on, two key/value heads of 128 lanes: 8 heads 264 -> 48 us, 12 heads 338 -> 75, 16
// heads 546 -> 139 (20 and 68 registers spilled at 12 and 16); 2,048 rows behind 8,192 keys, 12 heads, 2,609 -> 442.  The general instance:
// 12 heads on 4 of 64 lanes, 1,000 rows, 143 -> 88 us; 16 on 16 of 32 lanes 324 -> 186.
//
// Rows of a tile see different key ranges when a chunk of positions ends inside the tile: the mask is per (row, key).
#include "api.h"
#include "common.h"

namespace {

constexpr int kThreads = 256;
constexpr int kTileRows = 16;
constexpr int kKeyBlock = 64;               // keys a step of the decode kernel
constexpr int kTileThreads = 512;
constexpr int kTileKeys = 128;              // keys a step of the tile kernel: 16 a wave

struct TalkArgs {
    const bf16_t *q, *gate;
    int gate_stride;
    const bf16_t *k_pages, *v_pages;
    const int32_t *tables;
    int table_stride;
    const int32_t *row_pos, *row_seg, *seg_start;
    int num_segs;
    const float *talk, *temp;
    bf16_t *out;
    int rows, heads, kv_heads, k_dim, v_dim, page_size;
    float scale;
    int chunk;
    int splits;
    float *ws;       // splits > 1: [tile][split] { m [heads][16], l [heads][16], o [16][heads][v_dim] }
    int page_shift;        // log2 of page_size, -1 where it is no power of two
    int share_blocks;      // tile kernel: blocks of keys a workgroup takes
};

__device__ __forceinline__ size_t part_floats(int heads, int v_dim) { return (size_t)kTileRows * heads * (2 + v_dim); }

// which rows: the workgroup's tile among the tiles of all segments.  The segments' first rows come through LDS in one
// load where they fit (`starts`, kMaxSegsLds + 1 ints): a scan over memory would wait for every segment in turn.
constexpr int kMaxSegsLds = 255;

__device__ __forceinline__ bool find_tile(const TalkArgs &p, int tile, int *starts, int &seg, int &first, int &nrows) {
    const bool in_lds = p.num_segs <= kMaxSegsLds;
    if (in_lds) {
        if ((int)threadIdx.x <= p.num_segs) starts[threadIdx.x] = p.seg_start[threadIdx.x];
        __syncthreads();
    }
    int before = 0;
    for (int s = 0; s < p.num_segs; s++) {
        const int r0 = in_lds ? starts[s] : p.seg_start[s], n = (in_lds ? starts[s + 1] : p.seg_start[s + 1]) - r0;
        const int tiles = (n + kTileRows - 1) / kTileRows;
        if (tile < before + tiles) {
            const int t = tile - before;
            seg = s;
            first = r0 + t * kTileRows;
            nrows = n - t * kTileRows < kTileRows ? n - t * kTileRows : kTileRows;
            return true;
        }
        before += tiles;
    }
    return false;
}

// Which blocks of 128 keys a tile sees, and how many workgroups share them.
struct TileKeys {
    int pos0, plast, kb_start, blocks, per_share, shares;
};
__device__ __forceinline__ TileKeys tile_keys(const TalkArgs &p, int first, int nrows) {
    TileKeys t;
    t.pos0 = p.row_pos[first];
    t.plast = t.pos0 + nrows - 1;
    t.kb_start = (p.chunk > 0 ? t.pos0 - t.pos0 % p.chunk : 0) & ~15;
    t.blocks = (t.plast - t.kb_start) / kTileKeys + 1;
    const int even = (t.blocks + p.splits - 1) / p.splits;      // more blocks than the caller's bound: dealt out evenly
    t.per_share = even > p.share_blocks ? even : p.share_blocks;
    t.shares = (t.blocks + t.per_share - 1) / t.per_share;
    return t;
}

typedef const __attribute__((address_space(4))) float *scalar_floats;      // read through the scalar cache

// GS > 0 (1, 2 or 4): an instance for exactly HMAX heads on GS key/value heads, keys of 128 lanes, values of 80 to 128 and pages of a power
// of two from 8 on, whose loops carry no conditions and whose key/value heads are unrolled.  GS 0: up to HMAX heads on any
// number of key/value heads, any widths and pages of multiples of 4.
template <int HMAX, int GS>
__global__ void __launch_bounds__(kTileThreads)
talking_tile_kernel(const TalkArgs p) {
    constexpr bool EXACT = GS > 0;
    constexpr int KSM = EXACT ? 4 : 8;         // k_dim <= 256
    constexpr int NS = kTileKeys / 32;         // products over a block's keys
    constexpr int UNROLL = EXACT ? GS : 1;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
    const int H = EXACT ? HMAX : p.heads, G = EXACT ? GS : p.kv_heads, D = EXACT ? 128 : p.k_dim, DV = p.v_dim, PS = p.page_size;
    const int group = H / G, ks_n = D / 32, shift = p.page_shift;
    const int QP = H * D + 8;
    bf16_t *qs = (bf16_t *)lds_raw;                         // [16 rows][H][D], + 8 a row
    bf16_t *ps = qs + kTileRows * QP;                       // [H][16 rows][128 keys]
    float *mx = (float *)(ps + H * kTileRows * kTileKeys);  // [H][16 rows][8 waves]
    __shared__ int starts[kMaxSegsLds + 1];
    int seg, first, nrows;
    // the last tiles of a prompt see the most keys: they start first, so that the short ones fill the gaps at the end
    const int tile = gridDim.x - 1 - blockIdx.x;
    if (!find_tile(p, tile, starts, seg, first, nrows)) return;
    const int share = blockIdx.y;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 15, g = lane >> 4;
    const size_t out_row = (size_t)H * DV;
    if (p.row_seg[first] < 0) {   // padding rows of a captured step
        if (share == 0)
            for (int i = tid; i < nrows * H * DV; i += kTileThreads) p.out[(size_t)first * out_row + i] = (bf16_t)0.f;
        return;
    }
    const TileKeys tk = tile_keys(p, first, nrows);
    if (share >= tk.shares) return;
    const int plast = tk.plast;
    const int block0 = share * tk.per_share;
    const int my_blocks = tk.blocks - block0 < tk.per_share ? tk.blocks - block0 : tk.per_share;
    const int kb0 = tk.kb_start + kTileKeys * block0;
    const int32_t *tbl = p.tables + (size_t)seg * p.table_stride;
    const int pos_c = c < nrows ? tk.pos0 + c : tk.pos0;        // rows beyond the tile's end: zero queries, never written
    const int lo_c = p.chunk > 0 ? pos_c - pos_c % p.chunk : 0;
    const int lo_last = p.chunk > 0 ? plast - plast % p.chunk : 0;
    // which value lanes this wave owns, and which heads of them (h % HG == hg)
    const int DVT = DV / 16;
    const int vt_n = EXACT || DVT > 4 ? 8 : DVT > 2 ? 4 : DVT;
    const int hg = wave / vt_n, HG = EXACT ? 1 : 8 / vt_n;
    const bool owns = (wave & (vt_n - 1)) < DVT;
    const int vt = owns ? wave & (vt_n - 1) : 0;      // a wave without lanes of its own loads the first ones and drops them
    const bool eights = EXACT || (PS & 7) == 0;       // eight tokens of a value lane lie together; other pages: four and four
    auto page_of = [&](int key) __attribute__((always_inline)) { return EXACT || shift >= 0 ? key >> shift : key / PS; };
    auto in_page = [&](int key) __attribute__((always_inline)) { return EXACT || shift >= 0 ? key & (PS - 1) : key % PS; };
    auto seen = [&](int key) __attribute__((always_inline)) { return key <= plast ? key : plast; };      // beyond it: masked later

    // the pages of a block's keys: this lane's key of step 1, the lanes' keys of step 3
    auto key_page = [&](int kb) __attribute__((always_inline)) { return tbl[page_of(seen(kb + 16 * wave + c))]; };
    int vpage[NS], vpage4[NS];
    auto value_pages = [&](int kb) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < NS; s++) {
            vpage[s] = tbl[page_of(seen(kb + 32 * s + 8 * g))];
            if (!eights) vpage4[s] = tbl[page_of(seen(kb + 32 * s + 8 * g + 4))];
        }
    };
    auto load_keys = [&](bf16x8_t *kf, int kb, int page, int kvh) __attribute__((always_inline)) {
        const bf16_t *at = p.k_pages + key_offset(page, G, kvh, PS, D, in_page(seen(kb + 16 * wave + c)), 8 * g);
#pragma unroll
        for (int ks = 0; ks < KSM; ks++)
            if (EXACT || ks < ks_n) kf[ks] = *(const bf16x8_t *)(at + 32 * ks * PS);
    };
    auto load_values = [&](bf16x8_t *vf, int kb, int kvh) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < NS; s++) {
            const int key = kb + 32 * s + 8 * g;
            const bf16_t *at = p.v_pages + (((size_t)vpage[s] * G + kvh) * DV + 16 * vt + c) * PS + (key <= plast ? in_page(key) : 0);
            if (eights) {
                vf[s] = *(const bf16x8_t *)at;
            } else {
                const bf16_t *at4 = p.v_pages + (((size_t)vpage4[s] * G + kvh) * DV + 16 * vt + c) * PS + (key + 4 <= plast ? in_page(key + 4) : 0);
                const bf16x4_t a4 = *(const bf16x4_t *)at, b4 = *(const bf16x4_t *)at4;
#pragma unroll
                for (int e = 0; e < 4; e++) { vf[s][e] = a4[e]; vf[s][4 + e] = b4[e]; }
            }
        }
    };

    // the first block's keys are on their way while the queries go into LDS
    bf16x8_t kf[KSM], kn[KSM], vf[NS], vn[NS];
    int page_now = key_page(kb0);
    load_keys(kf, kb0, page_now, 0);
    {
        const int per_row = H * D / 8;
        for (int i = tid; i < kTileRows * per_row; i += kTileThreads) {
            const int r = i / per_row, e = (i - r * per_row) * 8;
            bf16x8_t v = {0, 0, 0, 0, 0, 0, 0, 0};
            if (r < nrows) v = *(const bf16x8_t *)(p.q + (size_t)(first + r) * H * D + e);
            *(bf16x8_t *)(qs + r * QP + e) = v;
        }
    }
    __syncthreads();

    // laundered where they are read: the loads stay in the loop instead of filling (and spilling) the scalar registers
    auto fresh = [](const float *ptr) __attribute__((always_inline)) {
        uintptr_t v = (uintptr_t)ptr;
        asm volatile("" : "+s"(v));
        return (scalar_floats)v;
    };
    float m_run[HMAX], l_part[HMAX];
    f32x4_t o[HMAX];
#pragma unroll
    for (int h = 0; h < HMAX; h++) {
        m_run[h] = -INFINITY;
        l_part[h] = 0.f;
        o[h] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    }

    for (int b = 0; b < my_blocks; b++) {
        const int kb = kb0 + kTileKeys * b;
        const int kb_next = b + 1 < my_blocks ? kb + kTileKeys : kb;
        value_pages(kb);
        const int page_next = key_page(kb_next);
        // ---- 1. raw scores of this wave's 16 keys
        f32x4_t raw[HMAX];
#pragma unroll
        for (int h = 0; h < HMAX; h++) raw[h] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll UNROLL
        for (int kvh = 0; kvh < G; kvh++) {
            if (kvh + 1 < G) load_keys(kn, kb, page_now, kvh + 1);
#pragma unroll
            for (int h = 0; h < HMAX; h++) {
                if (h % 3 == 0) __builtin_amdgcn_sched_barrier(0);      // registers: LDS reads of three heads ahead, not of all
                if (h >= kvh * group && h < (kvh + 1) * group) {
#pragma unroll
                    for (int ks = 0; ks < KSM; ks++)
                        if (EXACT || ks < ks_n) {
                            const bf16x8_t qf = *(const bf16x8_t *)(qs + c * QP + h * D + 32 * ks + 8 * g);
                            raw[h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[ks], qf, raw[h], 0, 0, 0);
                        }
                }
            }
#pragma unroll
            for (int ks = 0; ks < KSM; ks++) kf[ks] = kn[ks];
        }
        // ---- the mix, lane-local
        __builtin_amdgcn_sched_barrier(0);
        f32x4_t s[HMAX];
        const scalar_floats temp = fresh(p.temp);
#pragma unroll
        for (int h = 0; h < HMAX; h++)
            if (h < H) {
                const float f = p.scale * temp[h];
#pragma unroll
                for (int i = 0; i < 4; i++) raw[h][i] *= f;
            }
#pragma unroll
        for (int h = 0; h < HMAX; h++) {
            s[h] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
            if (h < H) {
                const scalar_floats talk = fresh(p.talk);
#pragma unroll
                for (int gg = 0; gg < HMAX; gg++) {
                    const int at = h * H + gg;
                    const float t = EXACT ? talk[at] : gg < H ? talk[at < H * H ? at : H * H - 1] : 0.f;
#pragma unroll
                    for (int i = 0; i < 4; i++) s[h][i] = fmaf(t, raw[gg][i], s[h][i]);
                }
            }
        }
        if (kb + kTileKeys - 1 > tk.pos0 || kb < lo_last) {      // uniform: some row does not see all of the block
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int key = kb + 16 * wave + 4 * g + i;
                const bool see = key >= lo_c && key <= pos_c;
#pragma unroll
                for (int h = 0; h < HMAX; h++) s[h][i] = see ? s[h][i] : -INFINITY;
            }
        }
        __builtin_amdgcn_sched_barrier(0);      // registers: the raw scores' are free from here on
        load_values(vf, kb, 0);                 // the first values arrive during the softmax
        // ---- 2. the block's largest score a (head, row), through LDS
#pragma unroll
        for (int h = 0; h < HMAX; h++) {
            if (h < H) {
                float v = fmaxf(fmaxf(s[h][0], s[h][1]), fmaxf(s[h][2], s[h][3]));
                v = max_16_apart(v);
                v = max_32_apart(v);
                mx[(h * kTileRows + c) * 8 + wave] = v;      // the four lanes of a row hold the same
            }
        }
        __syncthreads();      // also: every wave has multiplied the weights of the block before
#pragma unroll
        for (int h = 0; h < HMAX; h++) {
            if (h % 3 == 0) __builtin_amdgcn_sched_barrier(0);
            if (h < H) {
                const f32x4_t ma = *(const f32x4_t *)(mx + (h * kTileRows + c) * 8), mb = *(const f32x4_t *)(mx + (h * kTileRows + c) * 8 + 4);
                const float blk = fmaxf(fmaxf(fmaxf(ma[0], ma[1]), fmaxf(ma[2], ma[3])), fmaxf(fmaxf(mb[0], mb[1]), fmaxf(mb[2], mb[3])));
                const float m_new = fmaxf(m_run[h], blk);
                const float m_safe = m_new == -INFINITY ? 0.f : m_new;      // a row that has seen no key yet
                const float alpha = __expf(m_run[h] - m_safe);
                m_run[h] = m_new;
                float sum = 0.f;
                bf16x4_t w4;
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float e = __expf(s[h][i] - m_safe);
                    sum += e;
                    w4[i] = (bf16_t)e;
                }
                l_part[h] = l_part[h] * alpha + sum;
#pragma unroll
                for (int i = 0; i < 4; i++) o[h][i] *= alpha;
                // keys 16 wave + 4 g ..: half of the 16-byte piece 2 wave + g / 2
                *(bf16x4_t *)(ps + (h * kTileRows + c) * kTileKeys + 8 * ((2 * wave + (g >> 1)) ^ c) + 4 * (g & 1)) = w4;
            }
        }
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
        page_now = page_next;
        load_keys(kf, kb_next, page_now, 0);    // the next block's first keys arrive during the products
        // ---- 3. outputs: this wave's value lanes, keys 32 s + 8 g + e in the products' slots
        if (owns) {
            const bool ragged = kb + kTileKeys - 1 > plast;      // uniform
#pragma unroll UNROLL
            for (int kvh = 0; kvh < G; kvh++) {
                if (kvh + 1 < G) load_values(vn, kb, kvh + 1);
                if (ragged) {      // slots past the last token hold anything
#pragma unroll
                    for (int s2 = 0; s2 < NS; s2++)
#pragma unroll
                        for (int e = 0; e < 8; e++) vf[s2][e] = kb + 32 * s2 + 8 * g + e <= plast ? vf[s2][e] : (bf16_t)0.f;
                }
#pragma unroll
                for (int h = 0; h < HMAX; h++) {
                    if (h % 3 == 0) __builtin_amdgcn_sched_barrier(0);
                    if (h >= kvh * group && h < (kvh + 1) * group && (HG == 1 || (h & (HG - 1)) == hg)) {
#pragma unroll
                        for (int s2 = 0; s2 < NS; s2++) {
                            const bf16x8_t pf = *(const bf16x8_t *)(ps + (h * kTileRows + c) * kTileKeys + 8 * ((4 * s2 + g) ^ c));
                            o[h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[s2], pf, o[h], 0, 0, 0);
                        }
                    }
                }
#pragma unroll
                for (int s2 = 0; s2 < NS; s2++) vf[s2] = vn[s2];
            }
        }
    }
    // the rows' sums: lanes of one row, then the eight waves (nobody reads mx after the last block's second barrier)
#pragma unroll
    for (int h = 0; h < HMAX; h++) {
        if (h < H) {
            float v = l_part[h];
            v = sum_16_apart(v);
            v = sum_32_apart(v);
            if (g == 0) mx[(h * kTileRows + c) * 8 + wave] = v;
        }
    }
    __syncthreads();
    auto row_sum = [&](int h) __attribute__((always_inline)) {
        const f32x4_t a = *(const f32x4_t *)(mx + (h * kTileRows + c) * 8), b = *(const f32x4_t *)(mx + (h * kTileRows + c) * 8 + 4);
        return ((a[0] + a[1]) + (a[2] + a[3])) + ((b[0] + b[1]) + (b[2] + b[3]));
    };
    if (tk.shares > 1) {
        // this workgroup's share of the tile: maxima and sums [heads][16], unnormalised outputs [16][heads][v_dim]
        float *part = p.ws + ((size_t)tile * p.splits + share) * part_floats(H, DV);
        float *part_o = part + 2 * kTileRows * H;
#pragma unroll
        for (int h = 0; h < HMAX; h++) {
            if (h < H) {
                if (wave == 0 && g == 0) {
                    part[h * kTileRows + c] = m_run[h];
                    part[(H + h) * kTileRows + c] = row_sum(h);
                }
                if (owns && (HG == 1 || (h & (HG - 1)) == hg)) *(f32x4_t *)(part_o + ((size_t)c * H + h) * DV + 16 * vt + 4 * g) = o[h];
            }
        }
        return;
    }
    if (c >= nrows || !owns) return;
#pragma unroll
    for (int h = 0; h < HMAX; h++) {
        if (h < H && (HG == 1 || (h & (HG - 1)) == hg)) {
            const float l = row_sum(h);
            float f = l > 0.f ? 1.0f / l : 0.f;
            if (p.gate != nullptr) f *= 1.0f / (1.0f + __expf(-(float)p.gate[(size_t)(first + c) * p.gate_stride + h]));
            bf16x4_t r4;
#pragma unroll
            for (int i = 0; i < 4; i++) r4[i] = (bf16_t)(o[h][i] * f);
            *(bf16x4_t *)(p.out + (size_t)(first + c) * out_row + (size_t)h * DV + 16 * vt + 4 * g) = r4;
        }
    }
}

// The shares of a tile's workgroups into the rows' outputs, a workgroup a (tile, head): out = sum_s o_s e^(m_s - m) / sum_s l_s e^(m_s - m) * gate.
__global__ void __launch_bounds__(kThreads) talking_merge_kernel(const TalkArgs p) {
    __shared__ int starts[kMaxSegsLds + 1];
    int seg, first, nrows;
    if (!find_tile(p, blockIdx.x, starts, seg, first, nrows)) return;
    if (p.row_seg[first] < 0) return;      // padding rows: the tile kernel has written zeros
    const int H = p.heads, DV = p.v_dim, h = blockIdx.y;
    const int S = tile_keys(p, first, nrows).shares;
    if (S <= 1) return;                    // one workgroup had the whole tile: it has written the outputs
    const size_t per = part_floats(H, DV);
    const float *parts = p.ws + (size_t)blockIdx.x * p.splits * per;
    const int quads = DV / 4;
    for (int i = threadIdx.x; i < nrows * quads; i += kThreads) {
        const int c = i / quads, d4 = (i - c * quads) * 4;
        float m = -INFINITY;
#pragma unroll 4
        for (int s = 0; s < S; s++) m = fmaxf(m, parts[s * per + h * kTileRows + c]);
        float l = 0.f;
        f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
        if (m > -INFINITY) {
#pragma unroll 4
            for (int s = 0; s < S; s++) {
                const float *part = parts + s * per;
                const float w = __expf(part[h * kTileRows + c] - m);
                l += part[(H + h) * kTileRows + c] * w;
                const f32x4_t o4 = *(const f32x4_t *)(part + 2 * kTileRows * H + ((size_t)c * H + h) * DV + d4);
#pragma unroll
                for (int e = 0; e < 4; e++) acc[e] = fmaf(o4[e], w, acc[e]);
            }
        }
        float f = l > 0.f ? 1.0f / l : 0.f;
        if (p.gate != nullptr) f *= 1.0f / (1.0f + __expf(-(float)p.gate[(size_t)(first + c) * p.gate_stride + h]));
        bf16x4_t r4;
#pragma unroll
        for (int e = 0; e < 4; e++) r4[e] = (bf16_t)(acc[e] * f);
        *(bf16x4_t *)(p.out + (size_t)(first + c) * H * DV + (size_t)h * DV + d4) = r4;
    }
}

// ---- decode steps: one row a request -----------------------------------------------------------------------------------
// With a single row the 16 columns of a product are the HEADS that share a key/value head (the same position's queries),
// not 16 positions: one chain of products gives a block's raw scores of a whole group, and a lane keeps a few numbers, so
// many waves fit a compute unit and hide one another's waits.  A workgroup takes one request's row and walks its key
// blocks of 64 (or its share of them, `splits` as above):
//   1. wave w, keys 16 w .. 16 w + 15 straight from the pages: raw^T[key][head of the group] = K Q^T a key/value head;
//      the raw scores go to LDS as [key][head].
//   2. lane = key, wave w owns the heads w, w + 4, ..: the mix over a key's raw scores, then maximum, weights and sums of
//      a head's 64 keys inside one wave; the weights go to LDS as bfloat16 [head column][key].
//   3. wave w, value lanes 16 w .. and 64 + 16 w ..: O^T[value lane][head of the group] += V^T P^T a key/value head.
constexpr int kDecGMax = 8;        // key/value heads
constexpr int kDecHeads = 4;       // heads a wave owns in step 2: 16 in all
constexpr int kDecPPitch = kKeyBlock + 8;

__device__ __forceinline__ size_t decode_part_floats(int heads, int v_dim) { return (size_t)heads * (2 + v_dim); }

// All of a block's first loads (two key/value heads' keys and values) are asked for before anything waits, and sit behind no
// condition; a later block's are asked for while the one before is weighed.  Before, every load sat behind a condition and was waited for
// by itself.  With the merge, 12 heads on two key/value heads of 128 lanes, in a graph: one row of 1,900 keys 15.6 -> 10.7 us, 64 rows of
// 1,000 41.5 -> 20.6, one of 8,000 24.9 -> 15.0 (the general instance, 16 heads on 4 of 64 lanes, 4 rows of 1,000, 16.3 -> 14.1).
// GX > 0: up to GX key/value heads, keys and values of 128 lanes in pages of a power of two.  General and GX = 4, 12 heads on four: one
// row of 1,900 keys 15.3 -> 12.4 us, 64 of 1,000 38.3 -> 30.3; GX = 8, 16 heads on eight: 20.9 -> 16.5 and 75.7 -> 55.3.
template <int GX>
__global__ void __launch_bounds__(kThreads, 2)
talking_decode_kernel(const bf16_t *__restrict__ q, const int32_t *__restrict__ row_seg, const int32_t *__restrict__ row_pos,
                      const int32_t *__restrict__ tables, const float *__restrict__ talk, const float *__restrict__ temp, int table_stride,
                      int all_heads /* heads | kv_heads << 16 */, const TalkArgs p) {
    constexpr bool EXACT = GX > 0;
    typedef const __attribute__((address_space(4))) int32_t *constant_t;      // the same for every lane: a scalar load
    constexpr int HW = kDecHeads, KSM = EXACT ? 4 : 8, TS = 2, GM = EXACT ? GX : kDecGMax;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
    const int H = all_heads & 0xffff, G = (int)((unsigned)all_heads >> 16), D = EXACT ? 128 : p.k_dim, DV = EXACT ? 128 : p.v_dim, PS = p.page_size;
    // One trip to memory for the row's place, the other arguments and the first pieces of the queries and of the mix; then the pages, then keys and values.
    // The first 14 words of the arguments are in registers when a wave starts.  (12 heads on two of 128, one row of 1,900 keys 7.05 -> 6.8 us)
    const int row_of = blockIdx.x;      // every segment has one row: its first row is its own number, no lookup to wait for
    const int placed = ((constant_t)(uintptr_t)row_seg)[row_of], pos = ((constant_t)(uintptr_t)row_pos)[row_of];
    const bf16x8_t q_first = *(const bf16x8_t *)(q + (size_t)row_of * H * D + 8 * min((int)threadIdx.x, H * D / 8 - 1));
    const float talk_first = talk[min((int)threadIdx.x, H * H - 1)], temp_first = temp[threadIdx.x % H];
    fetch_arguments(p.k_pages, p.v_pages, p.page_size, p.page_shift, p.chunk, p.splits, p.scale, p.ws);
    const int group = H / G, KS = D / 32, DVT = DV / 16, HP = H | 1, shift = p.page_shift;
    float *tk = (float *)lds_raw;                       // [H][H]
    float *rawl = tk + H * H;                           // [64 keys][HP]
    float *alv = rawl + kKeyBlock * HP;                 // [H] factors of this block
    float *mlv = alv + H;                               // [2][H] maxima and sums at the end
    bf16_t *qs = (bf16_t *)(mlv + 2 * H + ((4 - ((H * H + kKeyBlock * HP + 3 * H) & 3)) & 3));      // [H][D], on 16 bytes
    bf16_t *ps2 = qs + H * D;                           // [G * 16 head columns][64 keys + 8]
    const int seg = blockIdx.x, split = blockIdx.y, S = p.splits;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 15, g = lane >> 4;
    const int r = row_of;
    const size_t out_row = (size_t)H * DV;
    const bool padding = placed < 0;      // of a captured step: zeros out, no keys (a return here would be a wait ahead of the loads)
    if (padding && split == 0)
        for (int i = tid; i < H * DV; i += kThreads) p.out[(size_t)r * out_row + i] = (bf16_t)0.f;
    const int lo = p.chunk > 0 && pos >= p.chunk ? pos - pos % p.chunk : 0;
    const int kb_start = lo & ~15;
    const int32_t *tbl = tables + (size_t)seg * table_stride;
    const int nblk = (pos - kb_start) / kKeyBlock + 1;
    const int my_blocks = !padding && split < nblk ? (nblk - split + S - 1) / S : 0;
    auto page_of = [&](int key) __attribute__((always_inline)) { return EXACT || shift >= 0 ? key >> shift : key / PS; };
    auto in_page = [&](int key) __attribute__((always_inline)) { return EXACT || shift >= 0 ? key & (PS - 1) : key % PS; };
    auto seen = [&](int key) __attribute__((always_inline)) { return key <= pos ? key : pos; };      // beyond it: masked in step 2
    auto block_at = [&](int b) __attribute__((always_inline)) { return kb_start + kKeyBlock * (split + S * b); };

    // a lane's key of step 1, and the eight neighbouring keys of each half of a block whose values it takes in step 3
    auto load_keys = [&](bf16x8_t *kf, int kb, int page, int kvh) __attribute__((always_inline)) {
        const bf16_t *at = p.k_pages + key_offset(page, G, kvh, PS, D, in_page(seen(kb + 16 * wave + c)), 8 * g);
#pragma unroll
        for (int ks = 0; ks < KSM; ks++)
            if (EXACT || ks < KS) kf[ks] = *(const bf16x8_t *)(at + 32 * ks * PS);
    };
    auto load_values = [&](bf16x8_t (*vf)[2], int kb, const int *vpage, int kvh) __attribute__((always_inline)) {
#pragma unroll
        for (int s2 = 0; s2 < 2; s2++) {
            const int key8 = kb + 32 * s2 + 8 * g;
            const bf16_t *at = p.v_pages + (((size_t)vpage[s2] * G + kvh) * DV + c) * PS + (key8 <= pos ? in_page(key8) : 0);
#pragma unroll
            for (int ts = 0; ts < TS; ts++) {
                const int t = wave + 4 * ts;
                vf[ts][s2] = *(const bf16x8_t *)(at + (size_t)16 * (EXACT || t < DVT ? t : 0) * PS);
            }
        }
    };
    bf16x8_t kf[KSM], kn[KSM], vf[TS][2], vn[TS][2];
    int vpage[2] = {0, 0}, kpage = 0;
    auto pages = [&](int kb) __attribute__((always_inline)) {
        kpage = tbl[page_of(seen(kb + 16 * wave + c))];
#pragma unroll
        for (int s2 = 0; s2 < 2; s2++) vpage[s2] = tbl[page_of(seen(kb + 32 * s2 + 8 * g))];
    };
    const int second = G > 1 ? 1 : 0;
    if (my_blocks > 0) pages(block_at(0));
    if (my_blocks > 0) {
        load_keys(kf, block_at(0), kpage, 0);
        load_keys(kn, block_at(0), kpage, second);
        load_values(vf, block_at(0), vpage, 0);
    }
    if (tid < H * D / 8) *(bf16x8_t *)(qs + 8 * tid) = q_first;
    if (tid < H * H) tk[tid] = talk_first * (p.scale * temp_first);
    for (int i = tid + kThreads; i < H * D / 8; i += kThreads) *(bf16x8_t *)(qs + 8 * i) = *(const bf16x8_t *)(q + (size_t)r * H * D + 8 * i);
    for (int i = tid + kThreads; i < H * H; i += kThreads) tk[i] = talk[i] * (p.scale * temp[i % H]);
    __syncthreads();

    float m_run[HW], l_run[HW];
#pragma unroll
    for (int j = 0; j < HW; j++) { m_run[j] = -INFINITY; l_run[j] = 0.f; }
    f32x4_t o[GM][TS];
#pragma unroll
    for (int k = 0; k < GM; k++)
#pragma unroll
        for (int ts = 0; ts < TS; ts++) o[k][ts] = (f32x4_t){0.f, 0.f, 0.f, 0.f};

    for (int b = 0; b < my_blocks; b++) {
        const int kb = block_at(b);
        // ---- 1. raw scores of this wave's 16 keys, a key/value head at a time
        for (int kvh = 0; kvh < G; kvh++) {
            const int hq = kvh * group + c < H ? kvh * group + c : H - 1;      // columns beyond the group: any finite query
            f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < KSM; ks++)
                if (EXACT || ks < KS) {
                    const bf16x8_t qf = *(const bf16x8_t *)(qs + hq * D + 32 * ks + 8 * g);
                    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[ks], qf, acc, 0, 0, 0);
                }
#pragma unroll
            for (int ks = 0; ks < KSM; ks++) kf[ks] = kn[ks];
            if (kvh + 2 < G) load_keys(kn, kb, kpage, kvh + 2);
            if (c < group) {
#pragma unroll
                for (int i = 0; i < 4; i++) rawl[(16 * wave + 4 * g + i) * HP + kvh * group + c] = acc[i];
            }
        }
        load_values(vn, kb, vpage, second);
        const int vpage_now[2] = {vpage[0], vpage[1]};
        const int kb_next = b + 1 < my_blocks ? block_at(b + 1) : kb;
        pages(kb_next);
        __syncthreads();
        // ---- 2. lane = key: the mix of its raw scores for this wave's heads, then the heads' maxima, weights and sums
        {
            const int key = kb + lane;
            const bool see = key >= lo && key <= pos;
            float sc[HW], mx[HW], sum[HW];
            const float *row[HW];
#pragma unroll
            for (int j = 0; j < HW; j++) {
                sc[j] = 0.f;
                const int h = wave + 4 * j;
                row[j] = tk + (h < H ? h : H - 1) * H;      // a wave without a j-th head works on the last one's, for nobody
            }
#pragma unroll 4
            for (int gg = 0; gg < H; gg++) {
                const float x = rawl[lane * HP + gg];
#pragma unroll
                for (int j = 0; j < HW; j++) sc[j] = fmaf(row[j][gg], x, sc[j]);
            }
#pragma unroll
            for (int j = 0; j < HW; j++) {
                sc[j] = see ? sc[j] : -INFINITY;
                mx[j] = sc[j];
            }
#pragma unroll
            for (int j = 0; j < HW; j++) mx[j] = wave_max(mx[j]);
            float alpha[HW];
#pragma unroll
            for (int j = 0; j < HW; j++) {
                const int h = wave + 4 * j;
                const float m_new = fmaxf(m_run[j], mx[j]);
                const float m_safe = m_new == -INFINITY ? 0.f : m_new;
                alpha[j] = __expf(m_run[j] - m_safe);
                m_run[j] = m_new;
                sum[j] = __expf(sc[j] - m_safe);
                if (h < H) {
                    ps2[((h / group) * 16 + h % group) * kDecPPitch + lane] = (bf16_t)sum[j];
                    if (lane == 0) alv[h] = alpha[j];
                }
            }
#pragma unroll
            for (int j = 0; j < HW; j++) sum[j] = wave_sum(sum[j]);
#pragma unroll
            for (int j = 0; j < HW; j++) l_run[j] = l_run[j] * alpha[j] + sum[j];
        }
        if (b + 1 < my_blocks) {
            load_keys(kf, kb_next, kpage, 0);
            load_keys(kn, kb_next, kpage, second);
        }
        __syncthreads();
        // ---- 3. outputs: this wave's value lanes, the heads of a key/value head as the columns
        const bool ragged = kb + kKeyBlock - 1 > pos;      // uniform
#pragma unroll
        for (int kvh = 0; kvh < GM; kvh++) {
            if (kvh < G) {
                const int ha = kvh * group + c < H ? kvh * group + c : H - 1;
                const float alpha = alv[ha];
                if (ragged) {      // slots past the last token hold anything
#pragma unroll
                    for (int ts = 0; ts < TS; ts++)
#pragma unroll
                        for (int s2 = 0; s2 < 2; s2++)
#pragma unroll
                            for (int e = 0; e < 8; e++) vf[ts][s2][e] = kb + 32 * s2 + 8 * g + e <= pos ? vf[ts][s2][e] : (bf16_t)0.f;
                }
                bf16x8_t pf[2];
#pragma unroll
                for (int s2 = 0; s2 < 2; s2++) pf[s2] = *(const bf16x8_t *)(ps2 + (kvh * 16 + c) * kDecPPitch + 32 * s2 + 8 * g);
#pragma unroll
                for (int ts = 0; ts < TS; ts++) {
                    f32x4_t acc = o[kvh][ts];
#pragma unroll
                    for (int i = 0; i < 4; i++) acc[i] *= alpha;
#pragma unroll
                    for (int s2 = 0; s2 < 2; s2++) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[ts][s2], pf[s2], acc, 0, 0, 0);
                    o[kvh][ts] = acc;      // a wave without a second piece of lanes: the first one's again, never written
                }
#pragma unroll
                for (int ts = 0; ts < TS; ts++)
#pragma unroll
                    for (int s2 = 0; s2 < 2; s2++) vf[ts][s2] = vn[ts][s2];
                if (kvh + 2 < G) load_values(vn, kb, vpage_now, kvh + 2);
            }
        }
        if (b + 1 < my_blocks) load_values(vf, kb_next, vpage, 0);
        __syncthreads();   // rawl, ps2 and alv are rewritten by the next block
    }
#pragma unroll
    for (int j = 0; j < HW; j++) {
        const int h = wave + 4 * j;
        if (h < H && lane == 0) { mlv[h] = m_run[j]; mlv[H + h] = l_run[j]; }
    }
    __syncthreads();
    float *part = S > 1 ? p.ws + ((size_t)seg * S + split) * decode_part_floats(H, DV) : nullptr;
    if (S > 1 && tid < 2 * H) part[tid] = mlv[tid];
    if (c >= group || padding) return;
#pragma unroll
    for (int kvh = 0; kvh < GM; kvh++) {
        if (kvh < G) {
            const int h = kvh * group + c;
#pragma unroll
            for (int ts = 0; ts < TS; ts++) {
                const int t = wave + 4 * ts;
                if (t >= DVT) continue;
                if (S > 1) {
                    *(f32x4_t *)(part + 2 * H + (size_t)h * DV + 16 * t + 4 * g) = o[kvh][ts];
                } else {
                    const float l = mlv[H + h];
                    float f = l > 0.f ? 1.0f / l : 0.f;
                    if (p.gate != nullptr) f *= 1.0f / (1.0f + __expf(-(float)p.gate[(size_t)r * p.gate_stride + h]));
                    bf16x4_t r4;
#pragma unroll
                    for (int i = 0; i < 4; i++) r4[i] = (bf16_t)(o[kvh][ts][i] * f);
                    *(bf16x4_t *)(p.out + (size_t)r * out_row + (size_t)h * DV + 16 * t + 4 * g) = r4;
                }
            }
        }
    }
}

// The shares of a decode row's workgroups into its output, a workgroup a (request, head): eight groups of 32 threads take
// every eighth share each (a thread four value lanes), then the eight partial merges meet in LDS.  A group asks for four of its shares at a
// time, behind no condition: a share a trip to memory were four trips for 31 shares (3.6 -> 2.7 us at best).
__global__ void __launch_bounds__(kThreads)
talking_decode_merge_kernel(const float *__restrict__ ws, const int32_t *__restrict__ row_seg, const bf16_t *__restrict__ gate, bf16_t *__restrict__ out,
                            int H, int DV, int S, int gate_stride) {
    __shared__ float gm[8], gl[8];
    __shared__ __attribute__((aligned(16))) float go[8][128];
    const int seg = blockIdx.x, h = blockIdx.y;
    const int r = seg;
    const bool padding = ((const __attribute__((address_space(4))) int32_t *)(uintptr_t)row_seg)[r] < 0;
    const size_t per = decode_part_floats(H, DV);
    const float *parts = ws + (size_t)seg * S * per;
    const int sg = threadIdx.x >> 5, d4 = 4 * (threadIdx.x & 31);
    float m = -INFINITY, l = 0.f;
    f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
    constexpr int AT = 4;      // shares of a group on their way together
    for (int s0 = sg; s0 < S; s0 += 8 * AT) {
        float ms[AT], ls[AT];
        f32x4_t o4[AT];
#pragma unroll
        for (int i = 0; i < AT; i++) {
            const float *part = parts + min(s0 + 8 * i, S - 1) * per;
            ms[i] = part[h], ls[i] = part[H + h];
            o4[i] = *(const f32x4_t *)(part + 2 * H + (size_t)h * DV + min(d4, DV - 4));
        }
#pragma unroll
        for (int i = 0; i < AT; i++) {
            if (s0 + 8 * i >= S || ms[i] == -INFINITY) continue;      // no share, or one that saw no key
            const float m_new = fmaxf(m, ms[i]);
            const float a = __expf(m - m_new), w = __expf(ms[i] - m_new);      // m = -inf: a = 0
            l = l * a + ls[i] * w;
#pragma unroll
            for (int e = 0; e < 4; e++) acc[e] = acc[e] * a + o4[i][e] * w;
            m = m_new;
        }
    }
    if ((threadIdx.x & 31) == 0) { gm[sg] = m; gl[sg] = l; }
    if (d4 < DV) *(f32x4_t *)&go[sg][d4] = acc;
    __syncthreads();
    if (sg != 0 || d4 >= DV || padding) return;      // a padding row: the decode kernel has written zeros
    float mt = -INFINITY;
#pragma unroll
    for (int k = 0; k < 8; k++) mt = fmaxf(mt, gm[k]);
    float lt = 0.f;
    f32x4_t tot = {0.f, 0.f, 0.f, 0.f};
    if (mt > -INFINITY) {
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const float w = __expf(gm[k] - mt);      // a group without a share: e^-inf = 0
            lt += gl[k] * w;
            const f32x4_t o4 = *(const f32x4_t *)&go[k][d4];
#pragma unroll
            for (int e = 0; e < 4; e++) tot[e] = fmaf(o4[e], w, tot[e]);
        }
    }
    float f = lt > 0.f ? 1.0f / lt : 0.f;
    if (gate != nullptr) f *= 1.0f / (1.0f + __expf(-(float)gate[(size_t)r * gate_stride + h]));
    bf16x4_t r4;
#pragma unroll
    for (int e = 0; e < 4; e++) r4[e] = (bf16_t)(tot[e] * f);
    *(bf16x4_t *)(out + (size_t)r * H * DV + (size_t)h * DV + d4) = r4;
}

// 1: not taken
int launch_decode(const TalkArgs &a, hipStream_t stream) {
    const int H = a.heads, G = a.kv_heads;
    if (H > 4 * kDecHeads || G > kDecGMax || a.page_size % 8 != 0 || (H % 2 != 0 && a.splits > 1)) return 1;
    const int HP = H | 1;
    size_t floats = (size_t)H * H + (size_t)kKeyBlock * HP + 3 * H;
    floats = (floats + 3) & ~(size_t)3;
    const size_t lds = floats * sizeof(float) + ((size_t)H * a.k_dim + (size_t)G * 16 * kDecPPitch) * sizeof(bf16_t);
    if (lds > 60 * 1024) return 1;
    const dim3 grid(a.num_segs, a.splits), block(kThreads);
    const bool exact = a.k_dim == 128 && a.v_dim == 128 && a.page_shift >= 3;
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, block, lds, stream, a.q, a.row_seg, a.row_pos, a.tables, a.talk, a.temp, a.table_stride, H | G << 16, a);
    };
    if (exact && G <= 2) go(talking_decode_kernel<2>);
    else if (exact && G <= 4) go(talking_decode_kernel<4>);
    else if (exact) go(talking_decode_kernel<kDecGMax>);
    else go(talking_decode_kernel<0>);
    int rc = fllm_check_launch("talking_attention (decode rows)");
    if (rc == 0 && a.splits > 1) {
        hipLaunchKernelGGL(talking_decode_merge_kernel, dim3(a.num_segs, H), dim3(kThreads), 0, stream, a.ws, a.row_seg, a.gate, a.out, H,
                           a.v_dim, a.splits, a.gate_stride);
        rc = fllm_check_launch("talking_attention (decode merge)");
    }
    return rc;
}

size_t tile_lds(int heads, int k_dim) {
    return ((size_t)kTileRows * (heads * k_dim + 8) + (size_t)heads * kTileRows * kTileKeys) * sizeof(bf16_t) +
           (size_t)heads * kTileRows * 8 * sizeof(float);
}

template <int HMAX, int GS>
int launch_tiles(const TalkArgs &a, int tiles, hipStream_t stream) {
    auto kernel = talking_tile_kernel<HMAX, GS>;
    constexpr size_t own = sizeof(int) * (kMaxSegsLds + 1);
    const size_t lds = tile_lds(a.heads, a.k_dim);
    if (own + lds > 160 * 1024) return 1;
    if (own + lds > 60 * 1024) {      // beyond the default 64 KiB the larger amount has to be asked for
        FLLM_REQUIRE(hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024 - (int)own) ==
                         hipSuccess, "talking_attention: cannot have %zu bytes of LDS", own + lds);
    }
    hipLaunchKernelGGL(kernel, dim3(tiles, a.splits), dim3(kTileThreads), lds, stream, a);
    int rc = fllm_check_launch("talking_attention (matrix cores)");
    if (rc == 0 && a.splits > 1) {
        hipLaunchKernelGGL(talking_merge_kernel, dim3(tiles, a.heads), dim3(kThreads), 0, stream, a);
        rc = fllm_check_launch("talking_attention (merge)");
    }
    return rc;
}

// 2: no instance for exactly these heads
template <int GS>
int launch_exact(const TalkArgs &a, int tiles, hipStream_t stream) {
    switch (a.heads) {
    case 4: return launch_tiles<4, GS>(a, tiles, stream);
    case 8: return launch_tiles<8, GS>(a, tiles, stream);
    case 12: return launch_tiles<12, GS>(a, tiles, stream);
    case 16: return launch_tiles<16, GS>(a, tiles, stream);
    }
    if constexpr (GS <= 2) {
        switch (a.heads) {
        case 6: return launch_tiles<6, GS>(a, tiles, stream);
        case 10: return launch_tiles<10, GS>(a, tiles, stream);
        case 14: return launch_tiles<14, GS>(a, tiles, stream);
        }
    }
    return 2;
}

}  // namespace

// Floats of workspace that `splits` workgroups a tile need for `rows` rows in `num_segs` segments.
extern "C" size_t fllm_talking_attention_workspace(int rows, int num_segs, int heads, int v_dim, int splits) {
    if (splits <= 1) return 0;
    return (size_t)(rows / kTileRows + num_segs) * splits * kTileRows * heads * (2 + v_dim);
}

// 1: the shape is not taken, the caller runs the plain kernel
int fllm_talking_attention_bf16_fast(const void *q, const void *gate, int gate_stride, const void *k_pages, const void *v_pages,
                                     const int32_t *tables, int table_stride, const int32_t *row_pos, const int32_t *row_seg,
                                     const int32_t *seg_start, int num_segs, const float *talk, const float *temp, void *out,
                                     int rows, int heads, int kv_heads, int k_dim, int v_dim, int page_size, float scale, int chunk,
                                     int key_chunk, int max_context, int splits, float *ws, size_t ws_floats, int single_rows,
                                     hipStream_t stream) {
    if (key_chunk != 8 || k_dim % 32 != 0 || k_dim > 256 || v_dim % 16 != 0 || v_dim > 128 || heads > 16 || page_size % 4 != 0)
        return 1;
    if (((uintptr_t)q | (uintptr_t)out | (uintptr_t)k_pages | (uintptr_t)v_pages) & 15) return 1;
    if (splits < 1) splits = 1;
    if (splits > 1) {
        FLLM_REQUIRE(ws != nullptr && ((uintptr_t)ws & 15) == 0 &&
                         ws_floats >= fllm_talking_attention_workspace(rows, num_segs, heads, v_dim, splits),
                     "talking_attention: %d workgroups a tile need a workspace of %zu floats, aligned to 16 bytes (%zu given)", splits,
                     fllm_talking_attention_workspace(rows, num_segs, heads, v_dim, splits), ws_floats);
    }
    TalkArgs a;
    a.q = (const bf16_t *)q;
    a.gate = (const bf16_t *)gate;
    a.gate_stride = gate_stride;
    a.k_pages = (const bf16_t *)k_pages;
    a.v_pages = (const bf16_t *)v_pages;
    a.tables = tables;
    a.table_stride = table_stride;
    a.row_pos = row_pos;
    a.row_seg = row_seg;
    a.seg_start = seg_start;
    a.num_segs = num_segs;
    a.talk = talk;
    a.temp = temp;
    a.out = (bf16_t *)out;
    a.rows = rows;
    a.heads = heads;
    a.kv_heads = kv_heads;
    a.k_dim = k_dim;
    a.v_dim = v_dim;
    a.page_size = page_size;
    a.scale = scale;
    a.chunk = chunk;
    a.splits = splits;
    a.ws = ws;
    a.page_shift = (page_size & (page_size - 1)) == 0 ? __builtin_ctz(page_size) : -1;
    // the blocks of the longest row tile, dealt out evenly: shorter tiles take fewer workgroups
    const long span = chunk > 0 && chunk + 2 * kTileRows < max_context ? chunk + 2 * kTileRows : max_context;
    const long blocks = (span + kTileRows + kTileKeys - 1) / kTileKeys;
    a.share_blocks = blocks > splits ? (int)((blocks + splits - 1) / splits) : 1;
    if (single_rows && rows == num_segs) {      // a decode step: every request has one row
        const int rc = launch_decode(a, stream);
        if (rc <= 0) return rc;
    }
    // every segment's rows in tiles of 16: at most rows / 16 full tiles and one ragged tile a segment
    const int tiles = rows / kTileRows + num_segs;
    // The kernel holds every head's scores and outputs of its rows in registers: an instance a bracket of head counts, and
    // one each for an even number of heads on 1, 2 or 4 key/value heads of 128 lanes, the counts whose loops unroll without
    // conditions.  What that is worth, 1,900 rows from a request's first token on, general and exact instance: 4 / 8 / 12 / 16 heads on
    // one 58 -> 30, 84 -> 47, 187 -> 66, 329 -> 102 us (the last spills 44 registers), on four 78 -> 36, 102 -> 50, 211 -> 82 (35
    // spilled), 353 -> 161 (126), 6 / 10 / 14 on two 77 -> 40, 169 -> 58, 299 -> 93 (48); 300 rows between 1.5 and 2.3 times.
    if (k_dim == 128 && v_dim > 64 && a.page_shift >= 3) {
        const int rc = kv_heads == 1 ? launch_exact<1>(a, tiles, stream) : kv_heads == 2 ? launch_exact<2>(a, tiles, stream)
                     : kv_heads == 4 ? launch_exact<4>(a, tiles, stream) : 2;
        if (rc <= 1) return rc;
    }
    if (heads <= 8) return launch_tiles<8, 0>(a, tiles, stream);
    if (heads <= 12) return launch_tiles<12, 0>(a, tiles, stream);
    return launch_tiles<16, 0>(a, tiles, stream);
}
