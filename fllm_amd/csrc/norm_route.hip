// A decode step's row on its way into routed experts in one kernel: a branch behind a norm joins the stream (or none does), the norm before
// the experts, and the router: what postnorm_add (stream_ops.hip) and the routers (routed_experts.hip) do one after the other.
//
// One workgroup a row.  What bounds it is its launch and its trips to memory, where the two kernels pay both twice: the row, its
// branch, the vectors and a wave's first two experts are asked for together, and the normed row stays in LDS for the
// router's products.  A wave has its SIMD to itself, so it takes two experts at a time (two chains of sums) and asks for the next two
// before; a chain is added in the order of row_score.  With one expert at a time, asked for when the one before was done, it was slower than
// the two kernels from 24 experts on.  Microseconds in a graph behind a branch, this and the two kernels, sigmoid scores, at 1 and 64 rows:
//   8 experts of 1,536 lanes   5.1 / 6.4,   5.5 / 7.1       64 experts of 512     9.6 / 10.0, 10.1 / 10.8
//   8 of 4,096                 6.7 / 8.2,   7.1 / 9.0       64 of 2,048          12.2 / 14.5, 12.7 / 15.4 (one at a time 18.7, 18.9)
//   32 of 1,024                7.2 / 8.4,   7.8 / 9.1       64 of 4,096          16.7 / 21.0, 17.8 / 22.2
// Prompts and answers of models with 12, 6 and 4 such layers a step, 8 experts of 1,536 lanes: 14.10 -> 13.87, 11.57 -> 11.42, 8.44 -> 8.31 ms with
// one expert at a time.
#include <type_traits>

#include "api.h"
#include "common.h"
#include "router_picks.h"

namespace {

constexpr int kBlock = 256;
constexpr int kWaves = kBlock / kWave;
constexpr int kMostExperts = 64;
constexpr int kStep = kWave * 8;      // lanes of a row that a wave takes at a time: widths are multiples of it

struct RouteArgs {
    const float *correction;          // GROUPED: [experts]
    int top, groups, kept, score_mode, renormalize;
    float scale;
    int32_t *ids;
    float *weights;
};

// NV pieces of four lanes a thread (width <= NV * 4 * kBlock); BRANCH: x[r] += branch * rsqrt(mean branch^2 + eps) * gain first
// (`normalize` 0: without the norm); GROUPED: the router with corrections and groups.
template <int NV, bool BRANCH, bool GROUPED>
__global__ void __launch_bounds__(kBlock)
norm_route_kernel(float *__restrict__ x, const float *__restrict__ branch, const float *__restrict__ gain, const float *__restrict__ norm_w,
                  const bf16_t *__restrict__ router /* [experts][width] */, int width, int experts, int normalize, float eps, float norm_eps,
                  bf16_t *__restrict__ out, const RouteArgs p) {
    constexpr int AHEAD = NV * 4 * kBlock / kStep;      // pieces of a router's row
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    __shared__ float scratch[2][kWaves];
    __shared__ float score[kMostExperts], choice[kMostExperts], gsum[kMostExperts], picks[kMostExperts];
    bf16_t *row = (bf16_t *)smem;                       // [width]
    const size_t r = blockIdx.x;
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const int pieces = width / kStep;
    f32x4_t v[NV], s[NV], w[NV], w2[NV];
#pragma unroll
    for (int i = 0; i < NV; i++) {
        const int c = min((i * kBlock + (int)threadIdx.x) * 4, width - 4);
        if (BRANCH) {
            v[i] = *(const f32x4_t *)(branch + r * width + c);
            w[i] = *(const f32x4_t *)(gain + c);
        }
        s[i] = *(const f32x4_t *)(x + r * width + c);
        w2[i] = *(const f32x4_t *)(norm_w + c);
    }
    // this wave's experts' rows of the router, two at work at a time, up to 2,048 lanes the next two on their way
    constexpr bool DEEP = NV <= 2;
    bf16x8_t b[2][AHEAD], ahead[2][DEEP ? AHEAD : 1];
    auto ask = [&](auto &to, int e0) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < 2; k++)
#pragma unroll
            for (int j = 0; j < AHEAD; j++)
                to[k][j] = *(const bf16x8_t *)(router + (size_t)min(e0 + k * kWaves, experts - 1) * width + lane * 8 + min(j, pieces - 1) * kStep);
    };
    ask(b, wave);
    fetch_arguments(norm_eps, out, p.correction, p.top, p.groups, p.kept, p.score_mode, p.renormalize, p.scale, p.ids, p.weights);
    float corrected[2] = {0.f, 0.f};      // of this wave's first two experts
#pragma unroll
    for (int k = 0; k < 2; k++)
        if (GROUPED) corrected[k] = p.correction[min(wave + k * kWaves, experts - 1)];
    auto mine = [&](int i) { return (i * kBlock + (int)threadIdx.x) * 4 < width; };
    if (BRANCH) {
        float inv = 1.0f;
        if (normalize) {
            float ss = 0.f;
#pragma unroll
            for (int i = 0; i < NV; i++)
                if (mine(i))
#pragma unroll
                    for (int e = 0; e < 4; e++) ss = fmaf(v[i][e], v[i][e], ss);
            inv = 1.0f / sqrtf(block_sum_once<kWaves>(ss, scratch[0]) / (float)width + eps);
        }
#pragma unroll
        for (int i = 0; i < NV; i++) {
            if (!mine(i)) break;
#pragma unroll
            for (int e = 0; e < 4; e++) s[i][e] += v[i][e] * inv * w[i][e];
            *(f32x4_t *)(x + r * width + (i * kBlock + threadIdx.x) * 4) = s[i];
        }
    }
    float ss2 = 0.f;
#pragma unroll
    for (int i = 0; i < NV; i++)
        if (mine(i))
#pragma unroll
            for (int e = 0; e < 4; e++) ss2 = fmaf(s[i][e], s[i][e], ss2);
    const float inv2 = 1.0f / sqrtf(block_sum_once<kWaves>(ss2, scratch[1]) / (float)width + norm_eps);
#pragma unroll
    for (int i = 0; i < NV; i++) {
        const int c = (i * kBlock + threadIdx.x) * 4;
        if (!mine(i)) break;
        bf16x4_t h;
#pragma unroll
        for (int e = 0; e < 4; e++) h[e] = (bf16_t)(s[i][e] * inv2 * w2[i][e]);
        *(bf16x4_t *)(out + r * width + c) = h;
        *(bf16x4_t *)(row + c) = h;
    }
    __syncthreads();
    // two experts of this wave: their sums, with the next two on their way where there may be any
    auto two = [&](int e0, auto last) __attribute__((always_inline)) {
        float c[2] = {0.f, 0.f}, z[2] = {0.f, 0.f};
#pragma unroll
        for (int k = 0; k < 2; k++)
            if (GROUPED) c[k] = decltype(last)::value ? corrected[k] : p.correction[min(e0 + k * kWaves, experts - 1)];
        if constexpr (DEEP && !decltype(last)::value) ask(ahead, e0 + 2 * kWaves);
#pragma unroll
        for (int j = 0; j < AHEAD; j++) {
            if (j >= pieces) break;
            const bf16x8_t a = *(const bf16x8_t *)(row + j * kStep + lane * 8);
#pragma unroll
            for (int i = 0; i < 8; i++)
#pragma unroll
                for (int k = 0; k < 2; k++) z[k] = fmaf((float)a[i], (float)b[k][j][i], z[k]);
        }
        if constexpr (decltype(last)::value) {
        } else if constexpr (DEEP) {
#pragma unroll
            for (int k = 0; k < 2; k++)
#pragma unroll
                for (int j = 0; j < AHEAD; j++) b[k][j] = ahead[k][j];
        } else {
            ask(b, e0 + 2 * kWaves);
        }
#pragma unroll
        for (int k = 0; k < 2; k++) z[k] = wave_sum(z[k]);
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const int e = e0 + k * kWaves;
            if (lane == 0 && e < experts) {
                const float sigmoid = 1.0f / (1.0f + expf(-z[k]));
                score[e] = GROUPED || p.score_mode == 0 ? sigmoid : z[k];
                if (GROUPED) choice[e] = sigmoid + c[k];
            }
        }
    };
    // up to eight experts are a pass of the four waves: nothing is asked for ahead, which the pass would wait for (with the picks in registers, 8 experts of
    // 1,536 lanes: grouped scores at 2 rows 6.6 -> 5.0 us, plain at 4 rows 4.8 -> 3.8)
    if (experts <= 2 * kWaves) two(wave, std::true_type{});
    else
        for (int e0 = wave; e0 < experts; e0 += 2 * kWaves) two(e0, std::false_type{});
    __syncthreads();
    if (wave != 0) return;
    if (GROUPED) pick_grouped(score, choice, gsum, picks, experts, p.top, p.groups, p.kept, p.ids + r * p.top, p.weights + r * p.top, p.scale, lane);
    else pick_plain(score, picks, experts, p.top, p.ids + r * p.top, p.weights + r * p.top, p.score_mode, p.renormalize, p.scale, lane);
}

template <bool BRANCH, bool GROUPED>
void launch(float *x, const float *branch, const float *gain, float eps, int normalize, const float *norm_w, float norm_eps, void *out, int rows,
            int width, const void *router, int experts, const RouteArgs &p, hipStream_t stream) {
    const size_t smem = (size_t)width * sizeof(bf16_t);
#define FLLM_NORM_ROUTE(NV)                                                                                                              \
    hipLaunchKernelGGL((norm_route_kernel<NV, BRANCH, GROUPED>), dim3(rows), dim3(kBlock), smem, stream, x, branch, gain, norm_w, \
                       (const bf16_t *)router, width, experts, normalize, eps, norm_eps, (bf16_t *)out, p)
    if (width <= 4 * kBlock) FLLM_NORM_ROUTE(1);
    else if (width <= 8 * kBlock) FLLM_NORM_ROUTE(2);
    else FLLM_NORM_ROUTE(4);
#undef FLLM_NORM_ROUTE
}

}  // namespace

// 0: launched; negative: error; 1: declined (a width that is no multiple of 512 or beyond 4,096, more than 64 experts or rows, the plain kernels
// asked for), nothing was written
extern "C" int fllm_norm_route(float *x, const float *branch, const float *gain, float eps, int normalize, const float *norm_w, float norm_eps,
                               void *out, int rows, int width, const void *w_router, const float *correction, int experts, int top, int groups,
                               int kept, int score_mode, int renormalize, float route_scale, int32_t *ids, float *weights, hipStream_t stream) {
    FLLM_REQUIRE(rows >= 0 && width > 0 && experts > 0 && top > 0 && top <= experts && norm_eps > 0.f, "norm_route: bad sizes");
    FLLM_REQUIRE(x && norm_w && out && w_router && ids && weights && ((branch == nullptr) == (gain == nullptr)), "norm_route: operands missing");
    FLLM_REQUIRE(branch == nullptr || !normalize || eps > 0.f, "norm_route: a norm needs an eps");
    FLLM_REQUIRE(score_mode == 0 || score_mode == 1, "norm_route: unknown score %d", score_mode);
    if (correction != nullptr)
        FLLM_REQUIRE(groups > 0 && experts % groups == 0 && kept > 0 && kept <= groups && top <= kept * (experts / groups),
                     "norm_route: %d experts in %d groups, %d kept, %d picked", experts, groups, kept, top);
    if (rows == 0) return 0;
    if (!fllm_fast_kernels_enabled() || width % kStep != 0 || width > 16 * kBlock || experts > kMostExperts || rows > 64) return 1;
    if (((uintptr_t)x | (uintptr_t)branch | (uintptr_t)gain | (uintptr_t)norm_w | (uintptr_t)out | (uintptr_t)w_router) & 15) return 1;
    const RouteArgs p = {correction, top, groups, kept, score_mode, renormalize, route_scale, ids, weights};
    if (branch != nullptr && correction != nullptr) launch<true, true>(x, branch, gain, eps, normalize, norm_w, norm_eps, out, rows, width, w_router, experts, p, stream);
    else if (branch != nullptr) launch<true, false>(x, branch, gain, eps, normalize, norm_w, norm_eps, out, rows, width, w_router, experts, p, stream);
    else if (correction != nullptr) launch<false, true>(x, branch, gain, eps, normalize, norm_w, norm_eps, out, rows, width, w_router, experts, p, stream);
    else launch<false, false>(x, branch, gain, eps, normalize, norm_w, norm_eps, out, rows, width, w_router, experts, p, stream);
    return fllm_check_launch("norm_route");
}
