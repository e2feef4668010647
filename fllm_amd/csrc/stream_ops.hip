// Small kernels on the residual stream and around the feed-forward that the dense decoder's own kernels do not
// cover: two RMSNorms of one row in one pass (blocks whose branches read the same stream), a gated activation with
// clamped operands, a vector and the embedding added to the stream between passes of looped layers, and logits times
// a constant.  All arithmetic is float32; the element type only says how operands are stored.
#include "api.h"
#include "common.h"

namespace {

constexpr int kBlock = 256;
constexpr int kWaves = kBlock / kWave;

// One workgroup a row.  The sum of squares is added in a fixed order (thread t its columns t, t + 256, ..., then
// lanes, then waves): a row gives the same bits whatever else is in the batch.  Both norms share the sum.
template <typename T>
__global__ void __launch_bounds__(kBlock)
rmsnorm_pair_kernel(const float *__restrict__ x, const float *__restrict__ w1, const float *__restrict__ w2,
                    T *__restrict__ out1, T *__restrict__ out2, int width, float eps1, float eps2) {
    __shared__ float scratch[kWaves];
    const size_t r = blockIdx.x;
    const float *src = x + r * width;
    float ss = 0.f;
    for (int c = threadIdx.x; c < width; c += kBlock) ss += src[c] * src[c];
    ss = block_sum<kWaves>(ss, scratch);
    const float mean = ss / (float)width;
    const float inv1 = 1.0f / sqrtf(mean + eps1), inv2 = 1.0f / sqrtf(mean + eps2);
    for (int c = threadIdx.x; c < width; c += kBlock) {
        const float v = src[c];
        out1[r * width + c] = from_f32<T>(v * inv1 * w1[c]);
        if (out2 != nullptr) out2[r * width + c] = from_f32<T>(v * inv2 * w2[c]);
    }
}

// out = a(g) * (u + up_offset) with g = min(gate, limit), u = clamp(up, -limit, limit) (limit <= 0: neither is
// clamped) and a(g) = g * sigmoid(alpha * g)
template <typename T>
__global__ void __launch_bounds__(kBlock)
glu_clamped_kernel(const T *__restrict__ gu, T *__restrict__ out, int inter, float limit, float alpha, float up_offset) {
    const size_t r = blockIdx.y;
    const T *g = gu + r * 2 * inter, *u = g + inter;
    T *o = out + r * inter;
    const int c = blockIdx.x * kBlock + threadIdx.x;
    if (c >= inter) return;
    float gf = to_f32<T>(g[c]), uf = to_f32<T>(u[c]);
    if (limit > 0.f) {
        gf = fminf(gf, limit);
        uf = fminf(fmaxf(uf, -limit), limit);
    }
    o[c] = from_f32<T>(gf / (1.0f + expf(-alpha * gf)) * (uf + up_offset));
}

// the same for bfloat16 rows whose width is a multiple of 8: a thread takes 8 neighbours, 16 bytes of gate and of up
__global__ void __launch_bounds__(kBlock)
glu_clamped_vec_kernel(const bf16_t *__restrict__ gu, bf16_t *__restrict__ out, int inter, float limit, float alpha, float up_offset) {
    const size_t r = blockIdx.y;
    const int c = (blockIdx.x * kBlock + threadIdx.x) * 8;
    if (c >= inter) return;
    const bf16x8_t g8 = *(const bf16x8_t *)(gu + r * 2 * inter + c), u8 = *(const bf16x8_t *)(gu + r * 2 * inter + inter + c);
    bf16x8_t o8;
#pragma unroll
    for (int e = 0; e < 8; e++) {
        float gf = (float)g8[e], uf = (float)u8[e];
        if (limit > 0.f) {
            gf = fminf(gf, limit);
            uf = fminf(fmaxf(uf, -limit), limit);
        }
        o8[e] = (bf16_t)(gf / (1.0f + expf(-alpha * gf)) * (uf + up_offset));
    }
    *(bf16x8_t *)(out + r * inter + c) = o8;
}

__global__ void __launch_bounds__(kBlock) scale_kernel(float *__restrict__ x, size_t total, float scale) {
    for (size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x; i < total; i += (size_t)gridDim.x * kBlock) x[i] *= scale;
}

// x[r, :] = (x[r, :] + scale * table[ids[r], :]) + vec[:]; either addend may be absent
template <typename T>
__global__ void __launch_bounds__(kBlock)
stream_add_kernel(float *__restrict__ x, const int32_t *__restrict__ ids, const T *__restrict__ table, int vocab, float scale,
                  const float *__restrict__ vec, int width) {
    const size_t r = blockIdx.x;
    const T *src = nullptr;
    if (table != nullptr) {
        int id = ids[r];
        id = id < 0 ? 0 : (id >= vocab ? vocab - 1 : id);   // ids are validated on the host; never read outside the table
        src = table + (size_t)id * width;
    }
    float *dst = x + r * width;
    for (int c = threadIdx.x; c < width; c += kBlock) {
        float v = dst[c];
        if (src != nullptr) v += to_f32<T>(src[c]) * scale;
        if (vec != nullptr) v += vec[c];
        dst[c] = v;
    }
}

// A branch that is normed on its way into the stream: v = sum of the row's `parts` partial branches (in index order),
// x[r] += v * rsqrt(mean(v^2) + eps) * gain (normalize 0: x[r] += v * gain).  `gain` is whatever multiplies the normed
// branch lane by lane: the norm's weight, a layer scale and the constant of the residual sum in one vector.  With
// `next_w`, the RMSNorm of the new row (its own eps) is written to `next_out` as well, the norm that reads the stream
// next; with `next_ssq` what the products behind a prepared norm take instead: the row times next_w, and its sum of squares there (a
// q/k/v product of 8 rows of 1,536 lanes that finds its norm prepared takes 6.6 us, one that norms the stream itself 8.6).
// One workgroup a row, sums in a fixed order: a row gives the same bits whatever else is in the batch.
template <typename B, typename T>
__global__ void __launch_bounds__(kBlock)
postnorm_add_kernel(float *__restrict__ x, const B *__restrict__ branch, int parts, const float *__restrict__ part_weights,
                    const float *__restrict__ gain, float eps, int normalize, const float *__restrict__ next_w, float next_eps, T *__restrict__ next_out,
                    float *__restrict__ next_ssq, int width) {
    __shared__ float scratch[kWaves];
    const size_t r = blockIdx.x;
    const B *src = branch + r * parts * width;
    float *dst = x + r * width;
    const float *pw = part_weights == nullptr ? nullptr : part_weights + r * parts;      // a weight a partial row
    auto value = [&](int c) {
        if (pw != nullptr) {
            float v = to_f32<B>(src[c]) * pw[0];
            for (int k = 1; k < parts; k++) v = fmaf(to_f32<B>(src[(size_t)k * width + c]), pw[k], v);
            return v;
        }
        float v = to_f32<B>(src[c]);
        for (int k = 1; k < parts; k++) v += to_f32<B>(src[(size_t)k * width + c]);
        return v;
    };
    float inv = 1.0f;
    if (normalize) {
        float ss = 0.f;
        for (int c = threadIdx.x; c < width; c += kBlock) {
            const float v = value(c);
            ss += v * v;
        }
        ss = block_sum<kWaves>(ss, scratch);
        inv = 1.0f / sqrtf(ss / (float)width + eps);
    }
    float ss2 = 0.f;
    for (int c = threadIdx.x; c < width; c += kBlock) {
        const float v = dst[c] + value(c) * inv * gain[c];
        dst[c] = v;
        ss2 += v * v;
    }
    if (next_w == nullptr) return;
    ss2 = block_sum<kWaves>(ss2, scratch);
    if (next_ssq != nullptr && threadIdx.x == 0) next_ssq[r] = ss2;
    const float inv2 = next_ssq != nullptr ? 1.0f : 1.0f / sqrtf(ss2 / (float)width + next_eps);
    for (int c = threadIdx.x; c < width; c += kBlock) next_out[r * width + c] = from_f32<T>(dst[c] * inv2 * next_w[c]);   // the thread's own stores
}

// The same for P float32 branches a row and widths in steps of 4: a thread holds NV pieces of four lanes of everything the row needs, asked
// for at once, so that a row costs one wait for memory and two sums over the workgroup (two branches of 1,536 lanes at 8 rows: 9.1 us
// lane by lane, 4.8 like this).  What addresses and sums need are the first 14 words of the arguments, which arrive with the wave, and no
// load sits behind a condition: a thread without lanes of its own reads the row's last ones again, an operand that is not there another one.  With conditions
// the compiler awaited a piece before it asked for the next (one branch of 1,536 lanes at 4 and 8 rows 2.8 -> 2.0 and 3.2 -> 2.4 us at best, two at 16 rows 3.4 -> 2.4).
template <int NV, int P, typename T>
__global__ void __launch_bounds__(kBlock)
postnorm_add_vec_kernel(float *__restrict__ x, const float *__restrict__ branch, const float *__restrict__ gain, const float *__restrict__ next_w,
                        const float *__restrict__ part_weights, int width, int normalize, float eps, float next_eps,
                        T *__restrict__ next_out, float *__restrict__ next_ssq) {
    __shared__ float scratch[2][kWaves];
    const size_t r = blockIdx.x;
    f32x4_t v[NV], s[NV], w[NV], w2[NV], more[NV][P];
    float pw[P];
    float ss = 0.f;
    auto mine = [&](int i) { return (i * kBlock + (int)threadIdx.x) * 4 < width; };
    const float *after = next_w != nullptr ? next_w : gain, *scales = part_weights != nullptr ? part_weights + r * P : gain;
#pragma unroll
    for (int i = 0; i < NV; i++) {
        const int c = min((i * kBlock + (int)threadIdx.x) * 4, width - 4);
        v[i] = *(const f32x4_t *)(branch + r * P * width + c);
#pragma unroll
        for (int k = 1; k < P; k++) more[i][k] = *(const f32x4_t *)(branch + (r * P + k) * width + c);
        s[i] = *(const f32x4_t *)(x + r * width + c);
        w[i] = *(const f32x4_t *)(gain + c);
        w2[i] = *(const f32x4_t *)(after + c);
    }
#pragma unroll
    for (int k = 0; k < P; k++) pw[k] = scales[k];      // (a row has four lanes at least)
    fetch_arguments(next_out, next_ssq);
#pragma unroll
    for (int k = 0; k < P; k++) pw[k] = part_weights == nullptr ? 1.0f : pw[k];
    // the row's branches in index order: x * 1 + y is x + y
#pragma unroll
    for (int i = 0; i < NV; i++) {
        v[i] *= pw[0];
#pragma unroll
        for (int k = 1; k < P; k++)
#pragma unroll
            for (int e = 0; e < 4; e++) v[i][e] = fmaf(more[i][k][e], pw[k], v[i][e]);
    }
    float inv = 1.0f;
    if (normalize) {
#pragma unroll
        for (int i = 0; i < NV; i++)
            if (mine(i))
#pragma unroll
                for (int e = 0; e < 4; e++) ss = fmaf(v[i][e], v[i][e], ss);
        inv = 1.0f / sqrtf(block_sum_once<kWaves>(ss, scratch[0]) / (float)width + eps);
    }
    float ss2 = 0.f;
#pragma unroll
    for (int i = 0; i < NV; i++) {
        if (!mine(i)) break;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            s[i][e] += v[i][e] * inv * w[i][e];
            ss2 = fmaf(s[i][e], s[i][e], ss2);
        }
        *(f32x4_t *)(x + r * width + (i * kBlock + threadIdx.x) * 4) = s[i];
    }
    if (next_w == nullptr) return;
    ss2 = block_sum_once<kWaves>(ss2, scratch[1]);
    if (next_ssq != nullptr && threadIdx.x == 0) next_ssq[r] = ss2;
    const float inv2 = next_ssq != nullptr ? 1.0f : 1.0f / sqrtf(ss2 / (float)width + next_eps);
#pragma unroll
    for (int i = 0; i < NV; i++) {
        const int c = (i * kBlock + threadIdx.x) * 4;
        if (!mine(i)) break;
        if constexpr (sizeof(T) == 2) {
            bf16x4_t b;
#pragma unroll
            for (int e = 0; e < 4; e++) b[e] = (bf16_t)(s[i][e] * inv2 * w2[i][e]);
            *(bf16x4_t *)((bf16_t *)next_out + r * width + c) = b;
        } else {
            *(f32x4_t *)((float *)next_out + r * width + c) = s[i] * inv2 * w2[i];
        }
    }
}

// A request's first step finds the state of its slot at zero in every tensor that keeps one: all tensors and all such requests of a step
// in one launch (12 requests of a model with 14 tensors were 168 fills of 2 us and their launches: prompts and answers of those 13.11 ->
// 12.76 ms).  table[i]: where tensor i begins and the bytes of a slot of it.
constexpr int kSlotsALaunch = 60;      // by value in the kernel's arguments
constexpr int kClearBytes = 32 * 1024; // of a slot a workgroup

struct ClearTable {
    const unsigned long long *table;
    int slots[kSlotsALaunch];
};

__global__ void __launch_bounds__(256) clear_slots_kernel(const ClearTable p) {
    const unsigned long long bytes = p.table[2 * blockIdx.y + 1];
    const unsigned long long from = (unsigned long long)blockIdx.x * kClearBytes;
    if (from >= bytes) return;
    unsigned char *at = (unsigned char *)p.table[2 * blockIdx.y] + (unsigned long long)p.slots[blockIdx.z] * bytes + from;
    const int n = (int)(bytes - from < kClearBytes ? bytes - from : kClearBytes);
    const int head = min(n, (int)((16 - ((uintptr_t)at & 15)) & 15)), whole = (n - head) / 16;
    if ((int)threadIdx.x < head) at[threadIdx.x] = 0;
    const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
    for (int i = threadIdx.x; i < whole; i += 256) *(f32x4_t *)(at + head + 16 * i) = zero;
    for (int i = head + 16 * whole + threadIdx.x; i < n; i += 256) at[i] = 0;
}

}  // namespace

extern "C" int fllm_postnorm_add(float *x, const void *branch, int branch_dtype, int parts, const float *part_weights, const float *gain,
                                 float eps, int normalize,
                                 const float *next_w, float next_eps, void *next_out, int next_dtype, float *next_ssq, int rows, int width,
                                 hipStream_t stream) {
    FLLM_REQUIRE(rows >= 0 && width > 0 && parts > 0, "postnorm_add: bad sizes");
    FLLM_REQUIRE(x && branch && gain && ((next_w == nullptr) == (next_out == nullptr)), "postnorm_add: operands missing");
    FLLM_REQUIRE(next_ssq == nullptr || next_w != nullptr, "postnorm_add: a sum of squares is of a prepared norm");
    if (rows == 0) return 0;
    const uintptr_t bases = (uintptr_t)x | (uintptr_t)branch | (uintptr_t)gain | (uintptr_t)next_w | (uintptr_t)next_out;
    // up to 4 branches in registers beside the rest, of rows of up to 8,192 lanes (one branch) or 4,096
    if (branch_dtype == FLLM_F32 && parts <= 4 && width % 4 == 0 && width <= (parts == 1 ? 8 : 4) * 4 * kBlock && (bases & 15) == 0 &&
        (next_dtype == FLLM_F32 || next_dtype == FLLM_BF16)) {
#define FLLM_POSTNORM_VEC(NV, P, T)                                                                                                       \
    hipLaunchKernelGGL((postnorm_add_vec_kernel<NV, P, T>), dim3(rows), dim3(kBlock), 0, stream, x, (const float *)branch, gain, next_w, part_weights, \
                       width, normalize, eps, next_eps, (T *)next_out, next_ssq)
#define FLLM_POSTNORM_PARTS(NV, T)                     \
    do {                                               \
        if (parts == 1) FLLM_POSTNORM_VEC(NV, 1, T);   \
        else if (parts == 2) FLLM_POSTNORM_VEC(NV, 2, T); \
        else if (parts == 3) FLLM_POSTNORM_VEC(NV, 3, T); \
        else FLLM_POSTNORM_VEC(NV, 4, T);              \
    } while (0)
#define FLLM_POSTNORM_ROW(T)                           \
    do {                                               \
        if (pieces <= 1) FLLM_POSTNORM_PARTS(1, T);    \
        else if (pieces <= 2) FLLM_POSTNORM_PARTS(2, T); \
        else if (pieces <= 4) FLLM_POSTNORM_PARTS(4, T); \
        else FLLM_POSTNORM_VEC(8, 1, T);               \
    } while (0)
        const int pieces = (width / 4 + kBlock - 1) / kBlock;
        if (next_dtype == FLLM_F32) FLLM_POSTNORM_ROW(float);
        else FLLM_POSTNORM_ROW(bf16_t);
#undef FLLM_POSTNORM_ROW
#undef FLLM_POSTNORM_PARTS
#undef FLLM_POSTNORM_VEC
        return fllm_check_launch("postnorm_add");
    }
#define FLLM_POSTNORM(B, T) hipLaunchKernelGGL((postnorm_add_kernel<B, T>), dim3(rows), dim3(kBlock), 0, stream, x, (const B *)branch, \
                                               parts, part_weights, gain, eps, normalize, next_w, next_eps, (T *)next_out, next_ssq, width)
    if (branch_dtype == FLLM_F32 && next_dtype == FLLM_F32) FLLM_POSTNORM(float, float);
    else if (branch_dtype == FLLM_F32 && next_dtype == FLLM_BF16) FLLM_POSTNORM(float, bf16_t);
    else if (branch_dtype == FLLM_BF16 && next_dtype == FLLM_F32) FLLM_POSTNORM(bf16_t, float);
    else if (branch_dtype == FLLM_BF16 && next_dtype == FLLM_BF16) FLLM_POSTNORM(bf16_t, bf16_t);
    else FLLM_REQUIRE(false, "postnorm_add: unknown dtypes %d, %d", branch_dtype, next_dtype);
#undef FLLM_POSTNORM
    return fllm_check_launch("postnorm_add");
}

extern "C" int fllm_rmsnorm_pair(const float *x, const float *w1, const float *w2, void *out1, void *out2, int rows, int width,
                                 float eps1, float eps2, int out_dtype, hipStream_t stream) {
    FLLM_REQUIRE(rows >= 0 && width > 0, "rmsnorm_pair: bad sizes");
    FLLM_REQUIRE(x && w1 && out1 && ((w2 == nullptr) == (out2 == nullptr)), "rmsnorm_pair: operands missing");
    if (rows == 0) return 0;
    if (out_dtype == FLLM_F32)
        hipLaunchKernelGGL(rmsnorm_pair_kernel<float>, dim3(rows), dim3(kBlock), 0, stream, x, w1, w2, (float *)out1, (float *)out2,
                           width, eps1, eps2);
    else if (out_dtype == FLLM_BF16)
        hipLaunchKernelGGL(rmsnorm_pair_kernel<bf16_t>, dim3(rows), dim3(kBlock), 0, stream, x, w1, w2, (bf16_t *)out1,
                           (bf16_t *)out2, width, eps1, eps2);
    else
        FLLM_REQUIRE(false, "rmsnorm_pair: unknown dtype %d", out_dtype);
    return fllm_check_launch("rmsnorm_pair");
}

extern "C" int fllm_glu_clamped(const void *gate_up, void *out, int rows, int inter, float limit, float alpha, float up_offset,
                                int dtype, hipStream_t stream) {
    FLLM_REQUIRE(rows >= 0 && inter > 0 && rows <= 65535, "glu_clamped: bad sizes");
    if (rows == 0) return 0;
    const dim3 grid((inter + kBlock - 1) / kBlock, rows);
    if (dtype == FLLM_F32)
        hipLaunchKernelGGL(glu_clamped_kernel<float>, grid, dim3(kBlock), 0, stream, (const float *)gate_up, (float *)out, inter,
                           limit, alpha, up_offset);
    else if (dtype == FLLM_BF16 && inter % 8 == 0 && (((uintptr_t)gate_up | (uintptr_t)out) & 15) == 0)
        hipLaunchKernelGGL(glu_clamped_vec_kernel, dim3((inter / 8 + kBlock - 1) / kBlock, rows), dim3(kBlock), 0, stream,
                           (const bf16_t *)gate_up, (bf16_t *)out, inter, limit, alpha, up_offset);
    else if (dtype == FLLM_BF16)
        hipLaunchKernelGGL(glu_clamped_kernel<bf16_t>, grid, dim3(kBlock), 0, stream, (const bf16_t *)gate_up, (bf16_t *)out, inter,
                           limit, alpha, up_offset);
    else
        FLLM_REQUIRE(false, "glu_clamped: unknown dtype %d", dtype);
    return fllm_check_launch("glu_clamped");
}

extern "C" int fllm_scale_f32(float *x, size_t total, float scale, hipStream_t stream) {
    if (total == 0) return 0;
    const size_t blocks = (total + kBlock - 1) / kBlock;
    hipLaunchKernelGGL(scale_kernel, dim3((unsigned)(blocks < 4096 ? blocks : 4096)), dim3(kBlock), 0, stream, x, total, scale);
    return fllm_check_launch("scale_f32");
}

extern "C" int fllm_stream_add(float *x, const int32_t *ids, const void *table, int table_dtype, int vocab, float scale,
                               const float *vec, int rows, int width, hipStream_t stream) {
    FLLM_REQUIRE(rows >= 0 && width > 0, "stream_add: bad sizes");
    FLLM_REQUIRE(table == nullptr || (ids != nullptr && vocab > 0), "stream_add: a table needs ids");
    if (rows == 0 || (table == nullptr && vec == nullptr)) return 0;
    if (table_dtype == FLLM_F32)
        hipLaunchKernelGGL(stream_add_kernel<float>, dim3(rows), dim3(kBlock), 0, stream, x, ids, (const float *)table, vocab, scale,
                           vec, width);
    else if (table_dtype == FLLM_BF16)
        hipLaunchKernelGGL(stream_add_kernel<bf16_t>, dim3(rows), dim3(kBlock), 0, stream, x, ids, (const bf16_t *)table, vocab,
                           scale, vec, width);
    else
        FLLM_REQUIRE(false, "stream_add: unknown dtype %d", table_dtype);
    return fllm_check_launch("stream_add");
}

// Zeroes slots `slots` (host memory, `count` of them) of `tensors` tensors: table (device memory) holds an address and the bytes of a
// slot for each, `largest` is the largest of those sizes.
extern "C" int fllm_clear_slots(const uint64_t *table, int tensors, size_t largest, const int32_t *slots, int count, hipStream_t stream) {
    FLLM_REQUIRE(tensors >= 0 && tensors <= 65535 && count >= 0, "clear_slots: bad sizes");
    if (tensors == 0 || count == 0 || largest == 0) return 0;
    FLLM_REQUIRE(table != nullptr && slots != nullptr, "clear_slots: operands missing");
    const size_t blocks = (largest + kClearBytes - 1) / kClearBytes;
    FLLM_REQUIRE(blocks <= 0x7fffffff, "clear_slots: slots of %zu bytes are too large", largest);
    for (int at = 0; at < count; at += kSlotsALaunch) {
        const int n = count - at < kSlotsALaunch ? count - at : kSlotsALaunch;
        ClearTable p = {};
        p.table = (const unsigned long long *)table;
        for (int i = 0; i < n; i++) {
            FLLM_REQUIRE(slots[at + i] >= 0, "clear_slots: slot %d", slots[at + i]);
            p.slots[i] = slots[at + i];
        }
        hipLaunchKernelGGL(clear_slots_kernel, dim3((unsigned)blocks, tensors, n), dim3(256), 0, stream, p);
        const int rc = fllm_check_launch("clear_slots");
        if (rc != 0) return rc;
    }
    return 0;
}
