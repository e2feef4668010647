// Attention over cached latents on the matrix cores (bfloat16 pages, float32 scores and weights).
//
// A token's key is its latent (rank lanes) and one rotated part (rot lanes) for all heads; its value is the latent itself.  Two ways:
//
//   latent rows   few rows a request: queries come in the latent's space (W_uk^T q beside the rotated lanes), and a workgroup takes
//                 16 heads of one row and a share of its keys.  A tile of 64 keys lies in LDS once, key after key, and serves both
//                 products: S^T = K Q^T reads its rows, O^T += C^T P^T reads it transposed (ds_read_b64_tr_b16).  The waves deal the
//                 tile's keys among themselves in the first product and the latent's lanes in the second, and hand the weights over
//                 in LDS (as two bfloat16 terms each: a weight's rounding and what the rounding lost).
//   expanded      portions of prompts: the keys and values of the tokens that the portion sees are made once (latent_expand), a head
//                 at a time and laid out as pages of 64 tokens, and the row tiles of masked_attention_mfma.hip run over them.
//
//   headwise      the products between the two spaces, a matrix a head.
#include <algorithm>
#include <type_traits>

#include "api.h"
#include "common.h"

namespace {

constexpr int kThreads = 256;
constexpr int kWavesL = kThreads / kWave;
constexpr int KT = 64;               // keys of a tile
constexpr int PP = KT + 8;           // pitch of a query's weights in LDS
constexpr float kLog2e = 1.4426950408889634f;

typedef __attribute__((ext_vector_type(4))) short s16x4_t;

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

__device__ __forceinline__ bf16x8_t zero8() {
    bf16x8_t z;
#pragma unroll
    for (int e = 0; e < 8; e++) z[e] = (bf16_t)0.f;
    return z;
}

// Columns col .. col + 15 of rows row .. row + 7 of a matrix in LDS: lane l of sixteen gets column col + l, rows in order.
__device__ __forceinline__ bf16x8_t read_columns(const bf16_t *base, int pitch, int row, int col) {
    const int i = threadIdx.x & 15;
    const bf16_t *at = base + (row + (i >> 2)) * pitch + col + (i & 3) * 4;
    const s16x4_t a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4_t *)at);
    const s16x4_t b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4_t *)(at + 4 * pitch));
    const auto both = __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
    return __builtin_bit_cast(bf16x8_t, both);
}

struct LatentParams {
    const bf16_t *q;
    int q_stride;              // elements of a row: heads * D
    const bf16_t *pages;
    const int32_t *tables;
    int table_stride;
    const int32_t *row_pos, *row_seg;
    bf16_t *out;               // [row][head][rank]
    int heads, rank, D, page_size, ps_shift;
    float scale_log2;
    int window, splits;
    float *parts;              // [row][head tile][split][16 * rank sums, 16 maxima, 16 denominators]
};

// grid (rows, head tiles of 16, splits).  VTW: latent tiles of 16 lanes a wave; KDM: 16-byte pieces of a tile's keys a thread, and steps of
// 32 lanes of a key.
template <int VTW, int KDM>
__global__ void __launch_bounds__(kThreads, 2)
latent_rows_kernel(const LatentParams p) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int row = blockIdx.x, seg = p.row_seg[row], head0 = blockIdx.y * 16, nh = min(16, p.heads - head0);
    const int D = p.D, rank = p.rank, KD = (D + 31) / 32, DP = KD * 32 + 8;
    bf16_t *Ks = (bf16_t *)smem, *Ph = Ks + KT * DP, *Pl = Ph + 16 * PP;
    float *sm_m = (float *)(Pl + 16 * PP), *sm_l = sm_m + kWavesL * 16;
    if (seg < 0) {      // padding row: zeros (with several splits the merge writes them)
        if (p.splits == 1)
            for (int i = threadIdx.x; i < nh * rank; i += kThreads) p.out[((size_t)row * p.heads + head0) * rank + i] = (bf16_t)0.f;
        return;
    }
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const int c = lane & 15, g = lane >> 4;
    const int pos = p.row_pos[row], lo = p.window > 0 && pos - p.window + 1 > 0 ? pos - p.window + 1 : 0;
    const int32_t *tbl = p.tables + (size_t)seg * p.table_stride;
    const int main0 = lo & ~(KT - 1), tiles = (pos - main0) / KT + 1;
    const int psh = p.ps_shift, pmask = p.page_size - 1;

    bf16x8_t rk[KDM];
    auto issue = [&](int t) {
        const int key = max(min(main0 + t * KT + lane, pos), lo);      // keys outside the row's range: an address that exists; masked
        const bf16_t *kr = p.pages + key_offset(tbl[key >> psh], 1, 0, p.page_size, D, key & pmask, wave * 8);
#pragma unroll
        for (int i = 0; i < KDM; i++)
            if (wave + i * kWavesL < D / 8) rk[i] = *(const bf16x8_t *)(kr + (size_t)i * kWavesL * p.page_size * 8);
    };
    int t = blockIdx.z;
    if (t < tiles) issue(t);
    bf16x8_t qf[KDM];      // a head's query, and zeros behind it
    const bf16_t *qr = p.q + (size_t)row * p.q_stride + (size_t)(head0 + min(c, nh - 1)) * D;
#pragma unroll
    for (int kk = 0; kk < KDM; kk++) qf[kk] = c < nh && kk * 32 + g * 8 < D ? *(const bf16x8_t *)(qr + kk * 32 + g * 8) : zero8();
    for (int ch = D / 8 + wave; ch < KD * 4; ch += kWavesL) *(bf16x8_t *)(Ks + lane * DP + ch * 8) = zero8();

    f32x4_t o[VTW];
#pragma unroll
    for (int i = 0; i < VTW; i++) o[i] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    float m_run = -INFINITY, l_run = 0.f;
    for (; t < tiles; t += p.splits) {
        __syncthreads();      // the tile before has been read
#pragma unroll
        for (int i = 0; i < KDM; i++)
            if (wave + i * kWavesL < D / 8) *(bf16x8_t *)(Ks + lane * DP + (wave + i * kWavesL) * 8) = rk[i];
        if (t + p.splits < tiles) issue(t + p.splits);
        __syncthreads();
        f32x4_t st[2];
        st[0] = st[1] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
        const bf16_t *ka = Ks + (wave * 16 + c) * DP + g * 8;
#pragma unroll
        for (int kk = 0; kk < KDM; kk++)
            if (kk < KD) st[kk & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const bf16x8_t *)(ka + kk * 32), qf[kk], st[kk & 1], 0, 0, 0);
        float s[4], m_blk = -INFINITY;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int key = main0 + t * KT + wave * 16 + g * 4 + i;
            s[i] = key >= lo && key <= pos ? (st[0][i] + st[1][i]) * p.scale_log2 : -INFINITY;
            m_blk = fmaxf(m_blk, s[i]);
        }
        m_blk = max_16_apart(m_blk);
        m_blk = max_32_apart(m_blk);
        if (g == 0) sm_m[wave * 16 + c] = m_blk;
        __syncthreads();
        float m_new = m_run;
#pragma unroll
        for (int w = 0; w < kWavesL; w++) m_new = fmaxf(m_new, sm_m[w * 16 + c]);      // a number: the row sees a key of every tile
        const float alpha = m_run == -INFINITY ? 0.f : fast_exp2(m_run - m_new);
        m_run = m_new;
        bf16x4_t hi, lo4;
        float sum = 0.f;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float w = fast_exp2(s[i] - m_new);
            sum += w;
            hi[i] = (bf16_t)w;
            lo4[i] = (bf16_t)(w - (float)hi[i]);
        }
        l_run = l_run * alpha + sum;
        *(bf16x4_t *)(Ph + c * PP + wave * 16 + g * 4) = hi;
        *(bf16x4_t *)(Pl + c * PP + wave * 16 + g * 4) = lo4;
        __syncthreads();
        bf16x8_t ph[2], pl[2];
#pragma unroll
        for (int ks = 0; ks < 2; ks++) {
            ph[ks] = *(const bf16x8_t *)(Ph + c * PP + ks * 32 + g * 8);
            pl[ks] = *(const bf16x8_t *)(Pl + c * PP + ks * 32 + g * 8);
        }
#pragma unroll
        for (int i = 0; i < VTW; i++) {
            const int d0 = (wave + i * kWavesL) * 16;
            if (d0 >= rank) break;
            o[i] *= alpha;
#pragma unroll
            for (int ks = 0; ks < 2; ks++) {
                const bf16x8_t a = read_columns(Ks, DP, ks * 32 + g * 8, d0);
                o[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, ph[ks], o[i], 0, 0, 0);
                o[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, pl[ks], o[i], 0, 0, 0);
            }
        }
    }
    l_run = sum_16_apart(l_run);
    l_run = sum_32_apart(l_run);
    if (g == 0) sm_l[wave * 16 + c] = l_run;
    __syncthreads();
    float l = 0.f;
#pragma unroll
    for (int w = 0; w < kWavesL; w++) l += sm_l[w * 16 + c];
    float *part = p.parts + (((size_t)row * gridDim.y + blockIdx.y) * p.splits + blockIdx.z) * (16 * rank + 32);
    if (p.splits > 1 && wave == 0 && g == 0) part[16 * rank + c] = m_run, part[16 * rank + 16 + c] = l;
    if (c >= nh) return;
    const float inv = 1.0f / l;
#pragma unroll
    for (int i = 0; i < VTW; i++) {
        const int d = (wave + i * kWavesL) * 16 + g * 4;
        if (d >= rank) break;
        if (p.splits > 1) {
            *(f32x4_t *)(part + c * rank + d) = o[i];
        } else {
            bf16x4_t b;
#pragma unroll
            for (int e = 0; e < 4; e++) b[e] = (bf16_t)(o[i][e] * inv);
            *(bf16x4_t *)(p.out + ((size_t)row * p.heads + head0 + c) * rank + d) = b;
        }
    }
}

// ---- a row's latent into the pages, its rotated lanes to the queries --------------------------------------------------------------
// Eight lanes a thread: heads, latents and rotated parts in whole pieces of eight, neighbours paired, keys in chunks of eight.
struct StoreParams {
    const bf16_t *joint;
    int ld, dkv_at, rank, rot;
    const float *c_weight;
    float eps;
    int heads, dim;
    bf16_t *q_out;
    int q_width, rot_at, plain_lanes;
    const int32_t *row_pos, *row_seg, *tables;
    int table_stride;
    const float *cos_table, *sin_table;
    bf16_t *k_pages;
    int page_size;
};

__device__ __forceinline__ void store_row(const StoreParams &p, size_t r, float *scratch) {
    const bf16_t *joint = p.joint;
    const int ld = p.ld, dkv_at = p.dkv_at, rank = p.rank, rot = p.rot, heads = p.heads, dim = p.dim, q_width = p.q_width, rot_at = p.rot_at;
    const int plain_lanes = p.plain_lanes, page_size = p.page_size;
    const float *cos_table = p.cos_table, *sin_table = p.sin_table, *c_weight = p.c_weight;
    const float eps = p.eps;
    bf16_t *q_out = p.q_out, *k_pages = p.k_pages;
    const int seg = p.row_seg[r];
    if (seg < 0) return;
    const int pos = p.row_pos[r];
    const float *cs = cos_table + (size_t)pos * (rot / 2), *sn = sin_table + (size_t)pos * (rot / 2);
    const bf16_t *row = joint + r * ld;
    auto turn8 = [&](bf16x8_t v, int c) {      // lanes c .. c + 7 of a rotated part
        const f32x4_t co = *(const f32x4_t *)(cs + c / 2), si = *(const f32x4_t *)(sn + c / 2);
        bf16x8_t out;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float a = (float)v[2 * i], b = (float)v[2 * i + 1];
            out[2 * i] = (bf16_t)(a * co[i] - b * si[i]);
            out[2 * i + 1] = (bf16_t)(a * si[i] + b * co[i]);
        }
        return out;
    };
    const int pieces = (plain_lanes ? q_width : rot) / 8, first = plain_lanes ? 0 : rot_at;
    for (int idx = threadIdx.x; idx < heads * pieces; idx += kThreads) {
        const int h = idx / pieces, c = first + (idx - h * pieces) * 8;
        const bf16_t *src = row + (size_t)h * (dim + rot);
        bf16x8_t v;
        if (c >= rot_at && c < rot_at + rot) v = turn8(*(const bf16x8_t *)(src + dim + c - rot_at), c - rot_at);
        else if (c < dim) v = *(const bf16x8_t *)(src + c);
        else
#pragma unroll
            for (int e = 0; e < 8; e++) v[e] = (bf16_t)0.f;
        *(bf16x8_t *)(q_out + (r * heads + h) * q_width + c) = v;
    }
    if (k_pages == nullptr) return;
    const int page = p.tables[(size_t)seg * p.table_stride + pos / page_size], off = pos % page_size;
    const bf16_t *c_row = row + dkv_at;
    const int mine = threadIdx.x * 8;      // at most kThreads pieces (checked where this is launched)
    bf16x8_t v;
    float ss = 0.f;
    if (mine < rank + rot) v = *(const bf16x8_t *)(c_row + mine);
    if (mine < rank)
#pragma unroll
        for (int e = 0; e < 8; e++) ss = fmaf((float)v[e], (float)v[e], ss);
    const float inv = 1.0f / sqrtf(block_sum<kWavesL>(ss, scratch) / (float)rank + eps);
    if (mine >= rank + rot) return;
    if (mine < rank) {
        const f32x4_t w0 = *(const f32x4_t *)(c_weight + mine), w1 = *(const f32x4_t *)(c_weight + mine + 4);
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = (bf16_t)((float)v[e] * inv * (e < 4 ? w0[e & 3] : w1[e & 3]));
    } else {
        v = turn8(v, mine - rank);
    }
    *(bf16x8_t *)(k_pages + key_offset(page, 1, 0, page_size, rank + rot, off, mine)) = v;
}

__global__ void __launch_bounds__(kThreads) latent_rope_store_vec_kernel(const StoreParams p) {
    __shared__ float scratch[kWavesL];
    store_row(p, blockIdx.x, scratch);
}

// ---- a matrix a head ------------------------------------------------------------------------------------------------------------
// A wave's 16 columns from n0 on of head h for the 16 rows from r0 on.  D^T = W X^T: a lane ends with four neighbouring columns of one row.
__device__ __forceinline__ void headwise_tile(const bf16_t *__restrict__ x, int x_row, int x_head, const bf16_t *__restrict__ w,
                                              bf16_t *__restrict__ out, int out_row, int out_head, const bf16_t *__restrict__ gate, int gate_row,
                                              int rows, int N, int K, int h, int n0, int r0) {
    const int lane = threadIdx.x & (kWave - 1), c = lane & 15, g = lane >> 4;
    const bf16_t *wr = w + ((size_t)h * N + min(n0 + c, N - 1)) * K;
    const int r = min(r0 + c, rows - 1);
    const bf16_t *xr = x + (size_t)r * x_row + (size_t)h * x_head;
    f32x4_t acc[2];
    acc[0] = acc[1] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    int k = g * 8;
    auto steps = [&](auto count) {      // so many steps of 32, their operands asked for at once
        constexpr int U = decltype(count)::value;
        bf16x8_t a[U], b[U];
#pragma unroll
        for (int u = 0; u < U; u++) a[u] = *(const bf16x8_t *)(wr + k + u * 32), b[u] = *(const bf16x8_t *)(xr + k + u * 32);
#pragma unroll
        for (int u = 0; u < U; u++) acc[u & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[u], b[u], acc[u & 1], 0, 0, 0);
        k += U * 32;
    };
    int left = K / 32;
    for (; left >= 8; left -= 8) steps(std::integral_constant<int, 8>{});
    if (left & 4) steps(std::integral_constant<int, 4>{});
    if (left & 2) steps(std::integral_constant<int, 2>{});
    if (left & 1) steps(std::integral_constant<int, 1>{});
    if (K % 32 != 0) {
        const bf16x8_t a = k < K ? *(const bf16x8_t *)(wr + k) : zero8(), b = k < K ? *(const bf16x8_t *)(xr + k) : zero8();
        acc[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc[0], 0, 0, 0);
    }
    if (r0 + c >= rows) return;
    float f = 1.0f;
    if (gate != nullptr) f = 1.0f / (1.0f + __expf(-(float)gate[(size_t)r * gate_row + h]));
    const int n = n0 + g * 4;
    bf16_t *dst = out + (size_t)r * out_row + (size_t)h * out_head + n;
    bf16x4_t v;
#pragma unroll
    for (int e = 0; e < 4; e++) v[e] = (bf16_t)((acc[0][e] + acc[1][e]) * f);
    if (n + 3 < N) *(bf16x4_t *)dst = v;
    else
        for (int e = 0; e < 4; e++)
            if (n + e < N) dst[e] = v[e];
}

// grid (heads, column blocks of 64, row tiles of 16)
__global__ void __launch_bounds__(kThreads)
headwise_linear_mfma_kernel(const bf16_t *__restrict__ x, int x_row, int x_head, const bf16_t *__restrict__ w, bf16_t *__restrict__ out,
                            int out_row, int out_head, const bf16_t *__restrict__ gate, int gate_row, int rows, int N, int K) {
    const int n0 = (blockIdx.y * kWavesL + threadIdx.x / kWave) * 16;
    if (n0 < N) headwise_tile(x, x_row, x_head, w, out, out_row, out_head, gate, gate_row, rows, N, K, blockIdx.x, n0, blockIdx.z * 16);
}

// The way into the latent's space in one launch: the first `rows` workgroups store their rows (store_row), the others take the plain query
// lanes through W_uk^T, a head, a column block of 64 and a row tile of 16 each.  Neither reads what the other writes.
__global__ void __launch_bounds__(kThreads) latent_enter_kernel(const StoreParams p, const bf16_t *__restrict__ w_uk_t, int rows, int blocks) {
    __shared__ float scratch[kWavesL];
    if ((int)blockIdx.x < rows) {
        store_row(p, blockIdx.x, scratch);
        return;
    }
    int b = blockIdx.x - rows;
    const int h = b % p.heads;
    b /= p.heads;
    const int n0 = (b % blocks * kWavesL + threadIdx.x / kWave) * 16, head_lanes = p.dim + p.rot, D = p.rank + p.rot;
    if (n0 < p.rank)
        headwise_tile(p.joint, p.ld, head_lanes, w_uk_t, p.q_out, p.heads * D, D, nullptr, 0, rows, p.rank, p.dim, h, n0, b / blocks * 16);
}

// The way out: the shares of a row's keys put together and taken through W_uv, times the gate.  Grid (rows in R, heads, column blocks of 64).
// The matrix is asked for before the shares are waited for; the product's columns repeat the R latents.
constexpr int kMostSplits = 20;
template <int KS, int R>
__global__ void __launch_bounds__(kThreads)
latent_leave_kernel(const float *__restrict__ parts, int splits, const int32_t *__restrict__ row_seg, const bf16_t *__restrict__ w_uv,
                    const bf16_t *__restrict__ gate, int gate_row, bf16_t *__restrict__ out, int rows, int heads, int rank, int vdim) {
    static_assert(R == 1 || R == kWavesL, "a wave finds the factors of one row");
    __shared__ float s_factor[R][kMostSplits];
    __shared__ __attribute__((aligned(16))) bf16_t s_latent[R][KS * 32 + 8];
    const int row0 = blockIdx.x * R, h = blockIdx.y, q = h & 15, n0 = (blockIdx.z * kWavesL + threadIdx.x / kWave) * 16;
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave, c = lane & 15, g = lane >> 4;
    const bf16_t *wr = w_uv + ((size_t)h * vdim + min(n0 + c, vdim - 1)) * rank;
    bf16x8_t w[KS];
#pragma unroll
    for (int kk = 0; kk < KS; kk++) w[kk] = kk * 32 + g * 8 < rank ? *(const bf16x8_t *)(wr + kk * 32 + g * 8) : zero8();
    const int stride = 16 * rank + 32, head_tiles = (heads + 15) / 16, d = threadIdx.x * 2;      // two lanes of a latent a thread
    auto shares_of = [&](int r) { return parts + ((size_t)min(row0 + r, rows - 1) * head_tiles + h / 16) * splits * stride; };
    auto there = [&](int r) { return row0 + r < rows && row_seg[row0 + r] >= 0; };              // padding rows have no shares
    float2 v[R == 1 ? kMostSplits : 1];
    if constexpr (R == 1) {
        const float *mine = shares_of(0);
#pragma unroll
        for (int s = 0; s < kMostSplits; s++)
            if (s < splits && d < rank) v[s] = *(const float2 *)(mine + (size_t)s * stride + q * rank + d);
    }
    if (wave < R) {
        const float *mine = shares_of(wave);
        const bool have = lane < splits && there(wave);
        const float m_s = have ? mine[(size_t)lane * stride + 16 * rank + q] : -INFINITY;
        const float l_s = have ? mine[(size_t)lane * stride + 16 * rank + 16 + q] : 0.f;
        const float m = wave_max(m_s);
        const float f = m_s == -INFINITY ? 0.f : fast_exp2(m_s - m);
        const float l = wave_sum(f * l_s);
        if (lane < splits) s_factor[wave][lane] = l > 0.f ? f / l : 0.f;
    }
    __syncthreads();
    if (d < KS * 32)
#pragma unroll
        for (int r = 0; r < R; r++) {
            float a = 0.f, b = 0.f;
            if (d < rank && there(r)) {
                if constexpr (R == 1) {
#pragma unroll
                    for (int s = 0; s < kMostSplits; s++)
                        if (s < splits) {
                            a = fmaf(v[s].x, s_factor[0][s], a);
                            b = fmaf(v[s].y, s_factor[0][s], b);
                        }
                } else {
                    const float *mine = shares_of(r) + q * rank + d;
#pragma unroll 4
                    for (int s = 0; s < splits; s++) {
                        const float2 x = *(const float2 *)(mine + (size_t)s * stride);
                        a = fmaf(x.x, s_factor[r][s], a);
                        b = fmaf(x.y, s_factor[r][s], b);
                    }
                }
            }
            bf16x2_t two;
            two[0] = (bf16_t)a, two[1] = (bf16_t)b;
            *(bf16x2_t *)(s_latent[r] + d) = two;
        }
    __syncthreads();
    if (n0 >= vdim) return;
    f32x4_t acc[2];
    acc[0] = acc[1] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < KS; kk++)
        acc[kk & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[kk], *(const bf16x8_t *)(s_latent[c % R] + kk * 32 + g * 8), acc[kk & 1], 0, 0, 0);
    const int row = row0 + c;
    if (c >= R || row >= rows) return;
    float f = 1.0f;
    if (gate != nullptr && there(c)) f = 1.0f / (1.0f + __expf(-(float)gate[(size_t)row * gate_row + h]));
    bf16_t *dst = out + ((size_t)row * heads + h) * vdim + n0 + g * 4;
#pragma unroll
    for (int e = 0; e < 4; e++)
        if (n0 + g * 4 + e < vdim) dst[e] = (bf16_t)((acc[0][e] + acc[1][e]) * f);
}

// ---- keys and values a head made of latents --------------------------------------------------------------------------------------
// grid (pages of 64 tokens, groups of heads).  pages_of [page][4]: the segment, the position of the page's first token, the first and
// one past the last position that anyone reads.  Out: keys [page][head][k_width / 8][64][8] (dim lanes made, rot lanes copied, zeros
// behind), values [page][head][v_width][64] (zeros behind vdim).  A wave makes two tiles of 16 lanes at a time for the page's tokens.
// Half of a job's weights (KS / 2 steps of 32 latent lanes) are asked for while the half before is multiplied, the first before the
// tokens are staged.
template <int KS>
__global__ void __launch_bounds__(kThreads, 2)
latent_expand_kernel(const bf16_t *__restrict__ pages, const int32_t *__restrict__ tables, int table_stride, const int32_t *__restrict__ pages_of,
                     const bf16_t *__restrict__ w_uk, const bf16_t *__restrict__ w_uv, bf16_t *__restrict__ k_out, bf16_t *__restrict__ v_out,
                     int heads, int heads_each, int rank, int rot, int dim, int vdim, int k_width, int v_width, int page_size, int ps_shift) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    bf16_t *Cs = (bf16_t *)smem;
    constexpr int CP = KS * 32 + 8;
    const int D = rank + rot;
    const size_t page = blockIdx.x;
    const int seg = pages_of[page * 4], pos0 = pages_of[page * 4 + 1], first = pages_of[page * 4 + 2], last = pages_of[page * 4 + 3] - 1;
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const int c = lane & 15, g = lane >> 4;
    const int h0 = blockIdx.y * heads_each, h1 = min(heads, h0 + heads_each);
    const int pos = max(min(pos0 + lane, last), first);      // tokens nobody reads repeat one that exists
    const bf16_t *token = pages + key_offset(tables[(size_t)seg * table_stride + (pos >> ps_shift)], 1, 0, page_size, D, pos & (page_size - 1), 0);
    const int kp = (dim + 31) / 32, vp = (vdim + 31) / 32, each = kp + vp, jobs = (h1 - h0) * each;      // pairs of tiles: keys' first
    constexpr int HS = KS / 2;
    bf16x8_t wa[2][HS], wb[2][HS];
    auto ask = [&](int job, auto half) {
        constexpr int B = decltype(half)::value;
        const int h = h0 + job / each, j = job % each;
        const bool keys = j < kp;
        const int n0 = (keys ? j : j - kp) * 32, N = keys ? dim : vdim;
        const bf16_t *wh = (keys ? w_uk : w_uv) + (size_t)h * N * rank;
        const bf16_t *w0 = wh + (size_t)min(n0 + c, N - 1) * rank, *w1 = wh + (size_t)min(n0 + 16 + c, N - 1) * rank;
#pragma unroll
        for (int kk = 0; kk < HS; kk++) {
            const int k = (B * HS + kk) * 32 + g * 8;
            wa[B][kk] = k < rank ? *(const bf16x8_t *)(w0 + k) : zero8();
            wb[B][kk] = k < rank ? *(const bf16x8_t *)(w1 + k) : zero8();
        }
    };
    const std::integral_constant<int, 0> first_half;
    const std::integral_constant<int, 1> second_half;
    if (wave < jobs) ask(wave, first_half);
    for (int ch = wave; ch < KS * 4; ch += kWavesL)
        *(bf16x8_t *)(Cs + lane * CP + ch * 8) = ch * 8 < rank ? *(const bf16x8_t *)(token + (size_t)ch * page_size * 8) : zero8();
    for (int ch = wave; ch < k_width / 8; ch += kWavesL) {      // the rotated part, and zeros
        if (ch * 8 < dim) continue;
        const int at = ch * 8 - dim;
        const bf16x8_t v = at < rot ? *(const bf16x8_t *)(token + (size_t)(rank + at) / 8 * page_size * 8) : zero8();
        for (int h = h0; h < h1; h++) *(bf16x8_t *)(k_out + (((page * heads + h) * (k_width / 8) + ch) * 64 + lane) * 8) = v;
    }
    for (int h = h0; h < h1; h++)
        for (int i = threadIdx.x; i < (v_width - vdim) * 8; i += kThreads)
            *(bf16x8_t *)(v_out + ((page * heads + h) * v_width + vdim) * 64 + (size_t)i * 8) = zero8();
    __syncthreads();
    for (int job = wave; job < jobs; job += kWavesL) {
        const int h = h0 + job / each, j = job % each;
        const bool keys = j < kp;
        const int n0 = (keys ? j : j - kp) * 32;
        f32x4_t acc[2][4];
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
            for (int t = 0; t < 4; t++) acc[a][t] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
        // keys: lanes as rows (four lanes of a token meet in a thread); values: tokens as rows (four tokens of a lane)
        auto multiply = [&](auto keys_form, auto half) {
            constexpr int B = decltype(half)::value;
#pragma unroll
            for (int kk = 0; kk < HS; kk++) {
#pragma unroll
                for (int t = 0; t < 4; t++) {
                    const bf16x8_t b = *(const bf16x8_t *)(Cs + (t * 16 + c) * CP + (B * HS + kk) * 32 + g * 8);
                    if constexpr (decltype(keys_form)::value) {
                        acc[0][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wa[B][kk], b, acc[0][t], 0, 0, 0);
                        acc[1][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wb[B][kk], b, acc[1][t], 0, 0, 0);
                    } else {
                        acc[0][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b, wa[B][kk], acc[0][t], 0, 0, 0);
                        acc[1][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b, wb[B][kk], acc[1][t], 0, 0, 0);
                    }
                }
                if (kk & 1) __builtin_amdgcn_sched_barrier(0);      // operands of two steps ahead of the products, no more: registers
            }
        };
        ask(job, second_half);
        if (keys) multiply(std::true_type{}, first_half);
        else multiply(std::false_type{}, first_half);
        if (job + kWavesL < jobs) ask(job + kWavesL, first_half);
        if (keys) multiply(std::true_type{}, second_half);
        else multiply(std::false_type{}, second_half);
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
            for (int t = 0; t < 4; t++) {
                bf16x4_t v;
#pragma unroll
                for (int e = 0; e < 4; e++) v[e] = (bf16_t)acc[a][t][e];
                if (keys) {      // four lanes of token t * 16 + c
                    const int d = n0 + a * 16 + g * 4;
                    if (d < dim) *(bf16x4_t *)(k_out + (((page * heads + h) * (k_width / 8) + d / 8) * 64 + t * 16 + c) * 8 + d % 8) = v;
                } else {         // lane n0 + a * 16 + c of four tokens
                    const int d = n0 + a * 16 + c;
                    if (d < vdim) *(bf16x4_t *)(v_out + ((page * heads + h) * v_width + d) * 64 + t * 16 + g * 4) = v;
                }
            }
    }
}

template <typename F> int allow_lds(F kernel, size_t bytes, bool &done) {
    if (done) return 0;
    const hipError_t e = hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    FLLM_REQUIRE(e == hipSuccess, "latent attention: %zu bytes of LDS: %s", bytes, hipGetErrorString(e));
    done = true;
    return 0;
}

template <int VTW, int KDM> int launch_rows(const LatentParams &p, dim3 grid, size_t smem, hipStream_t stream) {
    static bool done = false;
    if (allow_lds(latent_rows_kernel<VTW, KDM>, smem, done) != 0) return -1;
    hipLaunchKernelGGL((latent_rows_kernel<VTW, KDM>), grid, dim3(kThreads), smem, stream, p);
    return 0;
}

}  // namespace

extern "C" int fllm_latent_attention(const void *q, const void *k_pages, const int32_t *tables, int table_stride, const int32_t *row_pos,
                                     const int32_t *row_seg, const void *w_uv, const void *gate, int gate_row, void *latent, void *out, int rows,
                                     int heads, int rank, int rot, int vdim, int page_size, float scale, int window, int max_context,
                                     hipStream_t stream) {
    FLLM_REQUIRE(rows >= 0 && heads > 0 && rank > 0 && rot > 0 && vdim > 0 && page_size > 0 && table_stride > 0 && window >= 0, "latent_attention: bad sizes");
    FLLM_REQUIRE(q && k_pages && tables && row_pos && row_seg && w_uv && latent && out, "latent_attention: operands missing");
    const int head_dim = rank + rot, q_stride = heads * head_dim;
    if (!fllm_fast_kernels_enabled()) return 1;
    if (rot % 8 != 0 || rank % 8 != 0 || rank > 512 || rot > 64) return 1;
    if ((page_size & (page_size - 1)) != 0 || (((uintptr_t)q | (uintptr_t)w_uv) & 15) != 0 || heads > 16 * 65535) return 1;
    if (rows == 0) return 0;
    LatentParams p = {};
    p.q = (const bf16_t *)q, p.q_stride = q_stride, p.pages = (const bf16_t *)k_pages, p.tables = tables, p.table_stride = table_stride;
    p.row_pos = row_pos, p.row_seg = row_seg, p.out = (bf16_t *)latent, p.heads = heads, p.rank = rank, p.D = head_dim, p.page_size = page_size;
    while ((1 << p.ps_shift) < page_size) p.ps_shift++;
    p.scale_log2 = scale * kLog2e;
    p.window = window;
    const int head_tiles = (heads + 15) / 16;
    int span = max_context > 0 ? max_context : 1 << 20;
    if (window > 0) span = std::min(span, window + KT);
    const long groups = (long)rows * head_tiles;
    long splits = std::max(1L, std::min(std::min(512 / std::max(groups, 1L), (long)(span + KT - 1) / KT), (long)kMostSplits));
    if (splits > 1) {
        void *base = nullptr;
        size_t bytes = 0;
        if (!fllm_device_workspace(&base, &bytes) || bytes <= kWorkspaceCounterBytes) splits = 1;
        else {
            const size_t room = (bytes - kWorkspaceCounterBytes) / sizeof(float), each = (size_t)groups * (16 * rank + 32);
            splits = std::max(1L, std::min<long>(splits, (long)(room / each)));
            p.parts = (float *)((char *)base + kWorkspaceCounterBytes);
        }
    }
    p.splits = (int)splits;
    const int DP = (head_dim + 31) / 32 * 32 + 8;
    const size_t smem = (size_t)KT * DP * 2 + 2 * 16 * PP * 2 + 2 * kWavesL * 16 * sizeof(float);
    const dim3 grid(rows, head_tiles, p.splits);
    int rc;
    if (rank <= 64) rc = launch_rows<1, 4>(p, grid, smem, stream);
    else if (rank <= 128) rc = launch_rows<2, 6>(p, grid, smem, stream);
    else if (rank <= 256) rc = launch_rows<4, 10>(p, grid, smem, stream);
    else rc = launch_rows<8, 18>(p, grid, smem, stream);
    if (rc != 0) return rc;
    if (p.splits > 1) {      // the shares go through W_uv where they meet; many rows: four of them at a time, so that the matrix is read less
        const int R = rows <= 16 ? 1 : kWavesL;
        const dim3 leave((rows + R - 1) / R, heads, (vdim + 63) / 64);
        FLLM_REQUIRE(heads <= 65535 && leave.z <= 65535, "latent_attention: too many heads");
#define FLLM_LEAVE(KS, R)                                                                                                                   \
    hipLaunchKernelGGL((latent_leave_kernel<KS, R>), leave, dim3(kThreads), 0, stream, p.parts, p.splits, row_seg, (const bf16_t *)w_uv,     \
                       (const bf16_t *)gate, gate_row, (bf16_t *)out, rows, heads, rank, vdim)
        if (R == 1) {
            if (rank <= 128) FLLM_LEAVE(4, 1);
            else if (rank <= 256) FLLM_LEAVE(8, 1);
            else FLLM_LEAVE(16, 1);
        } else {
            if (rank <= 128) FLLM_LEAVE(4, kWavesL);
            else if (rank <= 256) FLLM_LEAVE(8, kWavesL);
            else FLLM_LEAVE(16, kWavesL);
        }
#undef FLLM_LEAVE
        return fllm_check_launch("latent_attention (matrix cores)");
    }
    rc = fllm_check_launch("latent_attention (matrix cores)");
    if (rc != 0) return rc;
    return fllm_headwise_linear(latent, heads * rank, rank, w_uv, out, heads * vdim, vdim, gate, gate_row, rows, heads, vdim, rank, FLLM_BF16, stream);
}

int fllm_headwise_linear_bf16_fast(const void *x, int x_row, int x_head, const void *w, void *out, int out_row, int out_head, const void *gate,
                                   int gate_row, int rows, int heads, int N, int K, hipStream_t stream) {
    if (!fllm_fast_kernels_enabled() || K % 8 != 0 || x_row % 8 != 0 || x_head % 8 != 0 || out_row % 4 != 0 || out_head % 4 != 0) return 1;
    if ((((uintptr_t)x | (uintptr_t)w) & 15) != 0 || ((uintptr_t)out & 7) != 0 || (N + 63) / 64 > 65535 || (rows + 15) / 16 > 65535) return 1;
    hipLaunchKernelGGL(headwise_linear_mfma_kernel, dim3(heads, (N + 63) / 64, (rows + 15) / 16), dim3(kThreads), 0, stream, (const bf16_t *)x, x_row,
                       x_head, (const bf16_t *)w, (bf16_t *)out, out_row, out_head, (const bf16_t *)gate, gate_row, rows, N, K);
    return fllm_check_launch("headwise_linear (matrix cores)");
}

static bool store_params(StoreParams &p, const void *joint, int ld, int dkv_at, int rank, int rot, const float *c_weight, float eps, int heads, int dim,
                         void *q_out, int q_width, int rot_at, int plain_lanes, const int32_t *row_pos, const int32_t *row_seg,
                         const int32_t *tables, int table_stride, const float *cos_table, const float *sin_table, int pairing, void *k_pages,
                         int page_size, int key_chunk) {
    if (ld % 8 != 0 || dkv_at % 8 != 0 || rank % 8 != 0 || rot % 8 != 0 || dim % 8 != 0 || q_width % 8 != 0 || rot_at % 8 != 0) return false;
    if (rank + rot > kThreads * 8 || key_chunk != 8 || pairing != 1 || (((uintptr_t)joint | (uintptr_t)q_out) & 15) != 0) return false;
    p.joint = (const bf16_t *)joint, p.ld = ld, p.dkv_at = dkv_at, p.rank = rank, p.rot = rot, p.c_weight = c_weight, p.eps = eps;
    p.heads = heads, p.dim = dim, p.q_out = (bf16_t *)q_out, p.q_width = q_width, p.rot_at = rot_at, p.plain_lanes = plain_lanes;
    p.row_pos = row_pos, p.row_seg = row_seg, p.tables = tables, p.table_stride = table_stride, p.cos_table = cos_table, p.sin_table = sin_table;
    p.k_pages = (bf16_t *)k_pages, p.page_size = page_size;
    return true;
}

int fllm_latent_rope_store_vec(const void *joint, int ld, int dkv_at, int rank, int rot, const float *c_weight, float eps, int heads, int dim,
                               void *q_out, int q_width, int rot_at, int plain_lanes, const int32_t *row_pos, const int32_t *row_seg,
                               const int32_t *tables, int table_stride, const float *cos_table, const float *sin_table, int pairing, void *k_pages,
                               int page_size, int key_chunk, int rows, hipStream_t stream) {
    StoreParams p = {};
    if (!store_params(p, joint, ld, dkv_at, rank, rot, c_weight, eps, heads, dim, q_out, q_width, rot_at, plain_lanes, row_pos, row_seg, tables,
                      table_stride, cos_table, sin_table, pairing, k_pages, page_size, key_chunk))
        return 1;
    hipLaunchKernelGGL(latent_rope_store_vec_kernel, dim3(rows), dim3(kThreads), 0, stream, p);
    return fllm_check_launch("latent_rope_store");
}

extern "C" int fllm_latent_enter(const void *joint, int ld, int dkv_at, int rank, int rot, const float *c_weight, float eps, int heads, int dim,
                                 const void *w_uk_t, void *q_out, const int32_t *row_pos, const int32_t *row_seg, const int32_t *tables,
                                 int table_stride, const float *cos_table, const float *sin_table, int table_positions, int pairing,
                                 void *k_pages, int page_size, int key_chunk, int rows, hipStream_t stream) {
    FLLM_REQUIRE(rows >= 0 && rank > 0 && rot > 0 && heads > 0 && dim > 0 && page_size > 0 && table_stride > 0 && table_positions > 0,
                 "latent_enter: bad sizes");
    FLLM_REQUIRE(dkv_at >= heads * (dim + rot) && ld >= dkv_at + rank + rot && eps > 0.f, "latent_enter: rows of %d values cannot hold queries and latent", ld);
    FLLM_REQUIRE(joint && c_weight && w_uk_t && q_out && row_pos && row_seg && tables && cos_table && sin_table && k_pages, "latent_enter: operands missing");
    StoreParams p = {};
    if (!fllm_fast_kernels_enabled() || ((uintptr_t)w_uk_t & 15) != 0 ||
        !store_params(p, joint, ld, dkv_at, rank, rot, c_weight, eps, heads, dim, q_out, rank + rot, rank, 0, row_pos, row_seg, tables, table_stride,
                      cos_table, sin_table, pairing, k_pages, page_size, key_chunk))
        return 1;
    if (rows == 0) return 0;
    const int blocks = (rank + 63) / 64;
    const long grid = rows + (long)heads * blocks * ((rows + 15) / 16);
    if (grid > 0x7fffffff) return 1;
    hipLaunchKernelGGL(latent_enter_kernel, dim3((unsigned)grid), dim3(kThreads), 0, stream, p, (const bf16_t *)w_uk_t, rows, blocks);
    return fllm_check_launch("latent_enter");
}

extern "C" int fllm_latent_expand(const void *pages, const int32_t *tables, int table_stride, const int32_t *pages_of, int num_pages,
                                  const void *w_uk, const void *w_uv, void *k_out, void *v_out, int heads, int rank, int rot, int dim, int vdim,
                                  int k_width, int v_width, int page_size, hipStream_t stream) {
    FLLM_REQUIRE(num_pages >= 0 && heads > 0 && rank > 0 && rot > 0 && dim > 0 && vdim > 0 && table_stride > 0, "latent_expand: bad sizes");
    FLLM_REQUIRE(rank % 8 == 0 && rot % 8 == 0 && dim % 8 == 0 && vdim % 8 == 0 && rank <= 512 && page_size > 0 && (page_size & (page_size - 1)) == 0,
                 "latent_expand: takes lanes in pieces of 8, latents of up to 512 and pages of a power of two (rank %d, rot %d, dim %d, vdim %d, "
                 "page %d)", rank, rot, dim, vdim, page_size);
    FLLM_REQUIRE(k_width % 8 == 0 && k_width >= dim + rot && v_width >= vdim, "latent_expand: widths %d and %d are too small", k_width, v_width);
    FLLM_REQUIRE(pages && tables && pages_of && w_uk && w_uv && k_out && v_out, "latent_expand: operands missing");
    if (num_pages == 0) return 0;
    int psh = 0;
    while ((1 << psh) < page_size) psh++;
    const int heads_each = (int)std::max(1L, std::min<long>(heads, (long)num_pages * heads / 512));
    const int groups = (heads + heads_each - 1) / heads_each;
    FLLM_REQUIRE(groups <= 65535, "latent_expand: too many heads");
    const dim3 grid(num_pages, groups);
    int rc;
    auto launch = [&](auto kernel, int ks, bool &done) {
        const size_t smem = (size_t)64 * (ks * 32 + 8) * 2;
        if (allow_lds(kernel, smem, done) != 0) return -1;
        hipLaunchKernelGGL(kernel, grid, dim3(kThreads), smem, stream, (const bf16_t *)pages, tables, table_stride, pages_of, (const bf16_t *)w_uk,
                           (const bf16_t *)w_uv, (bf16_t *)k_out, (bf16_t *)v_out, heads, heads_each, rank, rot, dim, vdim, k_width, v_width,
                           page_size, psh);
        return 0;
    };
    static bool done4 = false, done8 = false, done16 = false;
    if (rank <= 128) rc = launch(latent_expand_kernel<4>, 4, done4);
    else if (rank <= 256) rc = launch(latent_expand_kernel<8>, 8, done8);
    else rc = launch(latent_expand_kernel<16>, 16, done16);
    if (rc != 0) return rc;
    return fllm_check_launch("latent_expand");
}
