// Products of many bfloat16 rows on the tiles of gemm_tiles.h: gate and up with the activation in the epilogue, the squared ReLU, and plain
// products (with a bias, or where their tiles fill the device).
#include "api.h"
#include "gemm_tiles.h"
#include "plans.h"

using namespace fllm_tiles;

namespace {

bool operands_fit(const void *x, int ldx, const void *w, const void *out, int ldo, int M, long w_rows, int N, int K) {
    return ((((uintptr_t)x | (uintptr_t)w | (uintptr_t)out) & 15) == 0) && ldx % 8 == 0 && ldo % 8 == 0 && N % 8 == 0 &&
           (uint64_t)M * ldx * 2 < (1ull << 32) && (uint64_t)w_rows * K * 2 < (1ull << 32);      // byte offsets of 32 bits
}

TileArgs tile_args(const void *x, int ldx, const void *w, void *out, int ldo, int M, int N, int K) {
    TileArgs a = {};
    a.x = (const bf16_t *)x, a.w = (const bf16_t *)w, a.out = out;
    a.ldx = ldx, a.ldo = ldo, a.M = M, a.N = N, a.K = K;
    return a;
}
fllm_plan::TilePlan plan_of(long M, int N, int cols, int K, int force) {
    const long columns = (N + cols - 1) / cols;
    return fllm_plan::tile_plan((M + 255) / 256 * columns, (M + 127) / 128 * columns, K, force, fllm_option_half_tiles());
}

}  // namespace

// 0: launched, negative: error, 1: declined (the shape, or with `force` 0 a shape that the general path is faster at; `force` 256 or 128
// asks for that row tile and is declined where K is too short for it or no whole steps, as is any value but 0, 1 and these).
//
// The fused product against the library's product and an activation kernel, inside a graph, weights from memory, microseconds at 512 /
// 1,024 / 2,048 rows: 2 x 14,336 x 4,096 116 -> 104 / 212 -> 185 / 398 -> 352; 2 x 8,192 x 2,048 43 -> 37 / 69 -> 57 / 123 -> 109; 2 x 8,960 x 1,536
// 45 -> 43 / 82 -> 63 / 137 -> 106; 2 x 4,096 x 1,024 20 -> 18 / 27 -> 21 / 42 -> 35.  Where few rows or half-empty rounds make it slower: activation_joins in plans.h.
extern "C" int fllm_gate_up_tiles(const void *x, int ldx, const void *w_gate_up, void *out, int M, int inter, int K, float limit, float alpha,
                                  float up_offset, int force, hipStream_t stream) {
    FLLM_REQUIRE(M >= 0 && inter > 0 && K > 0 && ldx >= K && x && w_gate_up && out, "gate_up_tiles: bad sizes or operands missing");
    if (!fllm_fast_kernels_enabled() || !operands_fit(x, ldx, w_gate_up, out, inter, M, 2L * inter, inter, K)) return 1;
    if (M == 0) return 0;
    const fllm_plan::TilePlan plan = plan_of(M, inter, 128, K, force);
    if (plan.bm == 0 || (!force && !fllm_plan::activation_joins(M, 2L * inter, K, plan))) return 1;
    TileArgs a = tile_args(x, ldx, w_gate_up, out, inter, M, inter, K);
    a.limit = limit, a.alpha = alpha, a.up_offset = up_offset;
    return launch_tiles<EPI_GLU, false>(a, plan.bm, plan.halves, plan.tiles, stream);
}

// mode 0: out = x w^T (+ bias); 2: out = relu(x w^T)^2; bfloat16.  1: float32, where K is cut into slices (tile_slices in plans.h).
//
// The squared ReLU against the library's product and a kernel of its own (13,312 x 1,536): 37 -> 28 us at 512 rows, 95 -> 79 at 2,048; fewer rows
// as above.  A bias (2,048 x 1,536; the general path is linear_tiled_mfma_kernel): 32 -> 23 us at 136 rows, 34 -> 24 at 2,048.  Without either
// the library has kernels for every tile of the device's time, and these tiles are ahead only where they fill whole rounds over the compute
// units: 4,096 x 14,336 at 2,048 rows (256 tiles) 207 -> 188 us, at 1,900 (240) 191 -> 182, at 1,536 (192) 167 -> 177; 4,096 x 4,096 at
// 2,048 rows 59 -> 55; 6,144 x 4,096 at 2,048 rows (192 of 256 rows) 80 -> 77, at 1,900 76 -> 78.  Hence nine
// tenths of the rounds, and what that means where a last round runs as halves: plain_takes_tiles in plans.h.
extern "C" int fllm_linear_tiles(const void *x, int ldx, const void *w, const float *bias, void *out, int ldo, int M, int N, int K, int mode,
                                 int force, hipStream_t stream) {
    FLLM_REQUIRE(M >= 0 && N >= 0 && K >= 0 && mode >= 0 && mode <= 2, "linear_tiles: bad sizes");
    // rows that share memory, products without columns or steps: the general path's
    if (N == 0 || K == 0 || ldx < K || ldo < N || !x || !w || !out) return 1;
    if (!fllm_fast_kernels_enabled() || (bias && mode != 0) || !operands_fit(x, ldx, w, out, ldo, M, N, N, K)) return 1;
    if (M == 0) return 0;
    TileArgs a = tile_args(x, ldx, w, out, ldo, M, N, K);
    a.bias = bias;
    if (!force && mode != 2 && !bias) {
        void *base = nullptr;
        size_t bytes = 0;
        const bool have_ws = fllm_device_workspace(&base, &bytes);
        const long tiles = (long)((M + 127) / 128) * ((N + 255) / 256);
        a.slices = fllm_plan::tile_slices(M, tiles, K, bytes, have_ws, fllm_option_tile_slices());
        if (a.slices > 1) {
            a.counters = (int *)base;
            a.parts = (float *)((unsigned char *)base + fllm_plan::kCounterBytes);
            return mode == 1 ? launch_sliced<EPI_F32>(a, tiles, stream) : launch_sliced<EPI_STORE>(a, tiles, stream);
        }
    }
    if (mode == 1) return 1;
    const fllm_plan::TilePlan plan = plan_of(M, N, 256, K, force);
    if (plan.bm == 0) return 1;
    if (!force && mode == 2 && !fllm_plan::activation_joins(M, N, K, plan)) return 1;
    if (!force && mode == 0 && !bias && !fllm_plan::plain_takes_tiles(M, N, K, plan)) return 1;
    if (mode == 0) return launch_tiles<EPI_STORE, false>(a, plan.bm, plan.halves, plan.tiles, stream);
    return launch_tiles<EPI_RELU2, false>(a, plan.bm, plan.halves, plan.tiles, stream);
}
