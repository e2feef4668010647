// Routed experts of decode steps (bfloat16, few (row, pick) pairs): the picked experts' matrices stream once from their
// tile-major copies straight into matrix-core operands.
//
// What bounds it is the bytes of the picked experts' weights, so everything else is kept out of their way: no list of
// pairs is made by a kernel of its own (every wave finds its expert's pairs in `ids` itself; one wave for all with a barrier
// behind it cost prompts and answers of 12 requests 12.40 ms where this takes 12.29), no scaled copies of the rows are
// made (an operand is scaled where it is loaded, rounded to bfloat16 as a stored copy would be), and the down product is not cut
// into planes that a further kernel adds.  A workgroup takes 16 output columns (of gate and of up) or 32 of one expert, its eight waves
// cut K between them with 4 to 12 KiB asked for at a time each, and they meet in LDS once.  A load of the tile-major copy is
// 1 KiB in a row, whole cache lines that carry the non-temporal hint; the same kernel reading the rows as the checkpoint has them
// (64 bytes of each of 16) runs at 4.4 instead of 5.9 TB/s, and through LDS in whole rows, a tile at a time, at 4.0.
// A load of an expert's weights serves up to 32 pairs from registers.
//
// MFMA operand layout (v_mfma_f32_16x16x32_bf16): A lane l holds A[m = l%16][k = 8*(l/16) .. +7]; B likewise with n = l%16;
// D lane l holds D[m = 4*(l/16) + i][n = l%16], i = 0..3.
#include <type_traits>

#include "api.h"
#include "common.h"

namespace {

constexpr int kThreads = 512, kWaves = kThreads / kWave;
constexpr int kMostPairs = 512;

// MODE 0: act[pair, c] = a(g) * (u + up_offset), x = h[pair / top] times the pick's weight (weights null: as it is), w [E][2 N][K]
// MODE 1: out[pair, c] = w[e][c] . x[pair], float32, w [E][N][K]
// MODE 2: act[pair, c] = relu(w[e][c] . h[pair / top])^2, w [E][N][K]
// w is tile-major: [16 rows][K / 32] blocks of 64 lanes x 8 values (fllm_tile_weights' order; rows and K whole tiles).
// G: groups of 16 pairs that share a load of the weights.
// SHARED (modes 1 and 2): one more expert, which every row uses, is the last row of workgroups: its matrix [shared_n][shared_k] is
// w_shared, its activations lie behind the pairs'.  A row's outputs are then top + 1 neighbouring rows of `out`, the picks' times
// out_weights[pair], so that one sum of a row's parts is all that follows: of one layer's launches (2 rows, 8 experts and a shared one of
// 4,480 lanes at a width of 1,536) two products of 6 to 8 us and a sum of 4 are gone
// (a prompt and eight decode steps of twelve such layers 15.6 -> 14.5 ms).
// U: products a wave asks for at a time (launch_groups).
template <int MODE, int G, bool SHARED, int U>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(4)))
expert_stream_kernel(const bf16_t *__restrict__ x, const int32_t *__restrict__ ids, const bf16_t *__restrict__ w, int ldx, int pairs, int top, int E,
                     int N, int K, int by_pair, const float *__restrict__ weights, bf16_t *__restrict__ act,
                     float *__restrict__ out, float limit, float alpha, float up_offset, const bf16_t *__restrict__ w_shared, int shared_n,
                     int shared_k, const float *__restrict__ out_weights, int out_top) {
    static_assert(!SHARED || MODE != 0, "a shared expert comes with experts without a gate");
    constexpr int RT = MODE == 1 ? 1 : 2;                  // 16-row weight tiles a workgroup
    constexpr int COLS = MODE == 2 ? 32 : 16;              // output columns a workgroup
    __shared__ __attribute__((aligned(16))) f32x4_t red[kWaves][RT][kWave];
    __shared__ short s_pairs[kWaves][kMostPairs];          // a wave's own list: no barrier before the first loads
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const int l16 = lane & 15, lg = lane >> 4;
    const int c0 = blockIdx.x * COLS;
    typedef const __attribute__((address_space(4))) int32_t *constant_t;      // the same for every lane: a scalar load
    auto in_stack = [&](int e) { return e < 0 ? 0 : (e >= E ? E - 1 : e); };      // never outside the stack of experts
    // blockIdx.y names an expert, or (by_pair) a pair: then the first pair of an expert stands for it
    const bool shared = SHARED && (int)blockIdx.y == (by_pair ? pairs : E);
    const int first_id = ids[min(lane, pairs - 1)];        // of the first 64 pairs, on its way with the workgroup's own
    const int own_id = ((constant_t)(uintptr_t)ids)[by_pair && !shared ? (int)blockIdx.y : 0];
    const int e = shared ? 0 : by_pair ? in_stack(own_id) : (int)blockIdx.y;
    if (shared) {                                          // every row: `pairs` and the pointers become the shared expert's own
        if (MODE == 1) x += (size_t)pairs * ldx;
        if (MODE == 2) act += (size_t)pairs * N;
        pairs = pairs / out_top;
        if (MODE == 1) ldx = shared_k;
        w = w_shared;
        N = shared_n;
        K = shared_k;
        top = 1;
    }
    if (SHARED && c0 >= N) return;                         // the grid covers the wider of the two kinds of experts
    const bf16_t *tiles[RT];
#pragma unroll
    for (int t = 0; t < RT; t++) {
        const int c = min(c0 + (MODE == 2 ? 16 * t : 0), N - 16);      // a tile beyond the matrix reads its last one again
        tiles[t] = w + ((size_t)e * (MODE == 0 ? 2 : 1) * N + (MODE == 0 && t == 1 ? N : 0) + c) * K + lane * 8;
    }
    const int k_per = ((K + kWaves - 1) / kWaves + 31) / 32 * 32;
    const int k_begin = wave * k_per, k_end = min(K, k_begin + k_per);
    // Ahead of the first weights lies one trip to memory, for the pairs' experts; the arguments that are not among the first 14 words (those arrive with
    // the wave) ride on it.  It was three, an argument line, the workgroup's own pair and the list: 4,480 lanes at a width of 1,536, 2 rows
    // with a shared expert 16.5 -> 15.2 and 14.2 -> 13.2 us, 8 rows 33.9 -> 32.3 and 19.5 -> 18.5.  Asking for the first weights ahead of the list as well spilled registers.
    fetch_arguments(weights, act, out, limit, alpha, up_offset, out_weights, out_top);
    short *s_pair = s_pairs[wave];
    int count = 0;
    if (shared) {
        if (lane < pairs) s_pair[lane] = (short)lane;      // 16 rows at most
        count = pairs;
    } else {
        for (int p0 = 0; p0 < pairs; p0 += kWave) {
            const int p = p0 + lane;
            const bool mine = p < pairs && in_stack(p0 == 0 ? first_id : ids[min(p, pairs - 1)]) == e;
            const unsigned long long mask = __ballot(mine);
            if (mine) s_pair[count + __popcll(mask & ((1ull << lane) - 1))] = (short)p;
            count += __popcll(mask);
        }
    }
    __builtin_amdgcn_wave_barrier();
    __threadfence_block();
    if (count == 0 || (by_pair && !shared && s_pair[0] != (int)blockIdx.y)) return;      // the same for all waves

    for (int g0 = 0; g0 < count; g0 += 16 * G) {
        const bf16_t *src[G];
        float scale[G];
        f32x4_t acc[G][RT];
#pragma unroll
        for (int g = 0; g < G; g++) {
            const int pair = s_pair[min(g0 + 16 * g + l16, count - 1)];
            src[g] = x + (size_t)(MODE == 1 ? pair : pair / top) * ldx + 8 * lg;
            scale[g] = MODE == 0 && weights != nullptr ? weights[pair] : 1.0f;
#pragma unroll
            for (int t = 0; t < RT; t++) acc[g][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        }
        // U products, all of their loads asked for before the first product; a wave's last ones masked where they are fewer
        auto block = [&](int k0, auto whole) {
            bf16x8_t a[RT][U], b[G][U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int k = decltype(whole)::value ? k0 + 32 * u : min(k0 + 32 * u, k_end - 32);
#pragma unroll
                for (int t = 0; t < RT; t++) a[t][u] = __builtin_nontemporal_load((const bf16x8_t *)(tiles[t] + (size_t)k * 16));
#pragma unroll
                for (int g = 0; g < G; g++) b[g][u] = *(const bf16x8_t *)(src[g] + k);
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                if (!decltype(whole)::value && k0 + 32 * u >= k_end) break;
#pragma unroll
                for (int g = 0; g < G; g++) {
                    if (MODE == 0 && weights != nullptr) {
#pragma unroll
                        for (int i = 0; i < 8; i++) b[g][u][i] = (bf16_t)((float)b[g][u][i] * scale[g]);
                    }
#pragma unroll
                    for (int t = 0; t < RT; t++) acc[g][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[t][u], b[g][u], acc[g][t], 0, 0, 0);
                }
            }
        };
        int k0 = k_begin;
        for (; k0 + 32 * U <= k_end; k0 += 32 * U) block(k0, std::true_type{});
        if (k0 < k_end) block(k0, std::false_type{});
#pragma unroll
        for (int g = 0; g < G; g++) {
            if (g0 + 16 * g >= count) break;
            if (g0 + g > 0) __syncthreads();               // the sums of the pairs before have been read
#pragma unroll
            for (int t = 0; t < RT; t++) red[wave][t][lane] = acc[g][t];
            __syncthreads();
            // a thread an output: neighbours are neighbouring columns of one pair; the waves' sums in wave order
            for (int o = threadIdx.x; o < 16 * COLS; o += kThreads) {
                const int m = o % COLS, n = o / COLS, tile = m / 16, mm = m % 16;
                if (g0 + 16 * g + n >= count || c0 + m >= N) continue;
                const int from = n + 16 * (mm / 4), at = mm % 4;
                float v = 0.f, u = 0.f;
#pragma unroll
                for (int s = 0; s < kWaves; s++) {
                    v += red[s][MODE == 2 ? tile : 0][from][at];
                    if (MODE == 0) u += red[s][RT - 1][from][at];
                }
                const int pair = s_pair[g0 + 16 * g + n];
                const size_t to = (size_t)pair * N + c0 + m;
                if (MODE == 0) {
                    if (limit > 0.f) {
                        v = fminf(v, limit);
                        u = fminf(fmaxf(u, -limit), limit);
                    }
                    act[to] = (bf16_t)(v / (1.0f + expf(-alpha * v)) * (u + up_offset));
                } else if (MODE == 2) {
                    v = fmaxf(v, 0.f);
                    act[to] = (bf16_t)(v * v);
                } else if (SHARED) {
                    const int row = shared ? pair : pair / out_top, part = shared ? out_top : pair - row * out_top;
                    out[((size_t)row * (out_top + 1) + part) * N + c0 + m] = shared ? v : v * out_weights[pair];
                } else {
                    out[to] = v;
                }
            }
        }
    }
}

struct Shared {
    const void *w = nullptr;
    int n = 0, k = 0;
    const float *out_weights = nullptr;
    int top = 1;
};

template <int MODE, int G, bool SHARED>
void launch_groups(const void *x, int ldx, const int32_t *ids, const float *weights, long pairs, int top, const void *w, int E, int N, int K,
                   void *act, float *out, float limit, float alpha, float up_offset, const Shared &sh, hipStream_t stream) {
    const int by_pair = pairs < E;
    const int cols = MODE == 2 ? 32 : 16, widest = sh.n > N ? sh.n : N;
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3((widest + cols - 1) / cols, (by_pair ? (unsigned)pairs : (unsigned)E) + (SHARED ? 1 : 0)), dim3(kThreads), 0, stream,
                           (const bf16_t *)x, ids, (const bf16_t *)w, ldx, (int)pairs, top, E, N, K, by_pair, weights, (bf16_t *)act, out, limit, alpha,
                           up_offset, (const bf16_t *)sh.w, sh.n, sh.k, sh.out_weights, sh.top);
    };
    // Products a wave asks for at a time.  Two tiles of one group: two or three, so that 64 to 75 registers hold three or four workgroups a compute
    // unit where six left two: how many workgroups are there to ask while others' sums meet counts for more than how much each asks for.  Which of the
    // two: three, unless a wave has few products and a third of them would be asked for twice.  Microseconds of both products with two, three, four, six:
    //   gated experts of 2,048 lanes    width 1,024 (4 products a wave), 1 row 11.7, 12.3, 11.6, 11.4;  8 rows 21.2, 23.2, 22.0, 22.4
    //                                   width 2,048 (8), 1 row 14.7, 14.8, 14.8, 15.5;  8 rows 38.6, 39.2, 38.8, 41.5
    //   gated experts of 4,480 lanes    width 1,024, 1 row 19.0, 20.1, 19.8, 19.9;  8 rows 37.8, 40.5, 41.4, 41.3
    //                                   width 1,536 (6), 1 row 23.4, 23.1, 24.9, 24.1;  8 rows 53.7, 53.3, 57.7, 55.4
    //                                   width 4,096 (16), 1 row 43.3, 43.2, 42.5, 42.9;  8 rows 134.0, 132.3, 134.0, 131.9
    //   4,480 lanes beside a shared expert, width 1,536, 2 rows 26.1, 26.2, 26.4, 28.8;  16 rows 49.2, 49.4, 49.7, 53.1
    // One tile: six (4,480 lanes at 1,536, the down product alone, four: 18.5 and 18.4, 20.2 and 20.4, with a shared expert 13.2 and 13.7; nine 21.4, 22.8,
    // 13.2).  Two groups: 128 registers.
    if constexpr (G == 1 && MODE != 1) {
        const int each = ((K + kWaves - 1) / kWaves + 31) / 32;
        if (each % 3 != 0 && each <= 8) go(expert_stream_kernel<MODE, G, SHARED, 2>);
        else go(expert_stream_kernel<MODE, G, SHARED, 3>);
    } else {
        go(expert_stream_kernel<MODE, G, SHARED, MODE == 0 ? 3 : 6>);
    }
}

template <int MODE, bool SHARED = false>
void launch(int groups, const void *x, int ldx, const int32_t *ids, const float *weights, long pairs, int top, const void *w, int E, int N,
            int K, void *act, float *out, float limit, float alpha, float up_offset, hipStream_t stream, const Shared &sh = Shared()) {
    if (groups == 1) launch_groups<MODE, 1, SHARED>(x, ldx, ids, weights, pairs, top, w, E, N, K, act, out, limit, alpha, up_offset, sh, stream);
    else if constexpr (!SHARED) launch_groups<MODE, 2, SHARED>(x, ldx, ids, weights, pairs, top, w, E, N, K, act, out, limit, alpha, up_offset, sh, stream);
}

}  // namespace

// 0: launched, negative: error, 1: shape declined.  h bfloat16 [rows, K] (row stride ldh); ids / weights [rows, top] (weights null: all
// 1); w_up the tile-major copy of [E * 2 inter, K] (gate rows, then up rows of an expert), or with gated 0 of [E * inter, K] and a
// relu(.)^2 activation (weights must be null); w_down that of [E * N, inter]; act bfloat16 [rows * top, inter] (scratch); out float32
// [rows * top, N].
extern "C" int fllm_experts_stream(const void *h, int ldh, const int32_t *ids, const float *weights, int rows, int top, const void *w_up,
                                   const void *w_down, int E, int inter, int K, int N, int gated, void *act, float *out, float limit,
                                   float alpha, float up_offset, hipStream_t stream) {
    FLLM_REQUIRE(rows >= 0 && top > 0 && E > 0 && inter > 0 && K > 0 && N > 0 && ldh >= K, "experts_stream: bad sizes");
    FLLM_REQUIRE(h && ids && w_up && w_down && act && out, "experts_stream: operands missing");
    FLLM_REQUIRE(gated || !weights, "experts_stream: experts without a gate carry their weights on the outputs");
    if (!fllm_fast_kernels_enabled()) return 1;
    // every wave has a product at least
    if (K % 32 != 0 || inter % 32 != 0 || K < 32 * kWaves || inter < 32 * kWaves || N % 16 != 0 || ldh % 8 != 0 || E > 4096) return 1;
    if ((((uintptr_t)h | (uintptr_t)w_up | (uintptr_t)w_down | (uintptr_t)act) & 15) != 0) return 1;
    const long pairs = (long)rows * top;
    if (pairs == 0) return 0;
    if (pairs > kMostPairs || pairs > 16L * E) return 1;      // more pairs an expert: tiles of 64 and 128 pairs are faster (below)
    // Measured, microseconds of both products (grouped_tiles_kernel with what it needs around it -> this kernel with one, with two groups),
    // weights from memory, 8 experts of 4,480 lanes at a width of 1,536, two picks a row:
    //   1 row (one pair at a time -> this) 25 -> 22;  4 rows 55 -> 39;  8 rows 70 -> 51, 54;  16 rows 75 -> 57, 59;
    //   32 rows 77 -> 61, 62;  48 rows 77 -> 80, 70;  64 rows 78 -> 92, 75;  96 rows 83 -> 123, 92
    // (165 of 330 MB at one row's share; 5.8 TB/s at 16 rows); 8 experts of 2,048 lanes at 1,024: 8 rows 37 -> 19, 64 rows 42 -> 38, 32.
    const int groups = pairs <= 8L * E ? 1 : 2;
    if (gated) launch<0>(groups, h, ldh, ids, weights, pairs, top, w_up, E, inter, K, act, nullptr, limit, alpha, up_offset, stream);
    else launch<2>(groups, h, ldh, ids, nullptr, pairs, top, w_up, E, inter, K, act, nullptr, 0.f, 0.f, 0.f, stream);
    launch<1>(groups, act, inter, ids, nullptr, pairs, 1, w_down, E, N, inter, nullptr, out, 0.f, 0.f, 0.f, stream);
    return fllm_check_launch("experts_stream");
}

// The same for experts without a gate beside a shared expert (w_shared_up [shared, K], w_shared_down [N, shared], both tile-major) whose
// output counts once for every row: out float32 [rows * (top + 1), N], row r's picks times their weights and then the shared expert's
// output; act bfloat16 [rows * top * inter + rows * shared] (scratch).  1..16 rows.
extern "C" int fllm_experts_stream_shared(const void *h, int ldh, const int32_t *ids, const float *weights, int rows, int top, const void *w_up,
                                          const void *w_down, int E, int inter, int K, int N, const void *w_shared_up,
                                          const void *w_shared_down, int shared, void *act, float *out, hipStream_t stream) {
    FLLM_REQUIRE(rows >= 0 && top > 0 && E > 0 && inter > 0 && K > 0 && N > 0 && shared > 0 && ldh >= K, "experts_stream_shared: bad sizes");
    FLLM_REQUIRE(h && ids && weights && w_up && w_down && w_shared_up && w_shared_down && act && out, "experts_stream_shared: operands missing");
    if (!fllm_fast_kernels_enabled()) return 1;
    // 16 rows meet the shared expert's weights in one pass, and a row's pairs fit into one group of 16 an expert
    if (rows > 16 || K % 32 != 0 || inter % 32 != 0 || shared % 32 != 0 || K < 32 * kWaves || inter < 32 * kWaves || shared < 32 * kWaves ||
        N % 16 != 0 || ldh % 8 != 0 || E > 4096)
        return 1;
    if ((((uintptr_t)h | (uintptr_t)w_up | (uintptr_t)w_down | (uintptr_t)w_shared_up | (uintptr_t)w_shared_down | (uintptr_t)act) & 15) != 0) return 1;
    const long pairs = (long)rows * top;
    if (pairs == 0) return 0;
    if (pairs > kMostPairs || pairs > 16L * E) return 1;
    Shared up, down;
    up.w = w_shared_up, up.n = shared, up.k = K, up.top = top;
    down.w = w_shared_down, down.n = N, down.k = shared, down.top = top, down.out_weights = weights;
    launch<2, true>(1, h, ldh, ids, nullptr, pairs, top, w_up, E, inter, K, act, nullptr, 0.f, 0.f, 0.f, stream, up);
    launch<1, true>(1, act, inter, ids, nullptr, pairs, 1, w_down, E, N, inter, nullptr, out, 0.f, 0.f, 0.f, stream, down);
    return fllm_check_launch("experts_stream_shared");
}
