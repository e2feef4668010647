// Shared helpers of the gfx950 kernels: element types, wave64 reductions, error reporting.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define FLLM_F32 0
#define FLLM_BF16 1

typedef __bf16 bf16_t;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4_t;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
typedef __attribute__((ext_vector_type(16))) float f32x16_t;

constexpr int kWave = 64;

// Records the first failure of a call; every entry point returns 0 or a negative code and the
// text is read back through fllm_last_error().
void fllm_set_error(const char *fmt, ...);
int fllm_check_launch(const char *what);
// 0 when the MFMA kernels are switched off (tests compare them with the plain kernels)
int fllm_fast_kernels_enabled(void);
// 1: prompt portions of heads of 64 and 128 use the 128-row attention kernel (default); 0: the 64-row kernel
int fllm_option_tile32(void);
// 0: the decode-shaped products choose their number of K slices themselves (default); n: n slices where that is possible
int fllm_option_linear_slices(void);
// 1: the parts of a split decode context are merged by the split that arrives last (default); 0: by a second kernel
int fllm_option_fused_merge(void);
// 1: prompt portions with long contexts and few rows share a row tile's keys among workgroups (default); 0: one workgroup a row tile
int fllm_option_prefill_parts(void);
// 1: decode-shaped products read bfloat16 activations straight from global memory (default); 0: they stage them in LDS
int fllm_option_x_direct(void);
// products of 17 to 64 rows: 1 (default) the kernel that suits the shape; 0 activations pass through LDS in chunks wherever
// that kernel can serve; 2 a K slice of the activations stays in LDS wherever that kernel can serve
int fllm_option_slab(void);
// products of many rows on 256-row tiles: 1 (default) a last round of at most 128 tiles runs as tiles of half the rows where that takes less
// time; 0 never; 2 wherever it can
int fllm_option_half_tiles(void);
int fllm_option_wide_waves(void);
int fllm_option_resident_tiles(void);
int fllm_option_tile32_rows(void);
// 1: decode-shaped products of up to 8 rows use 8-row weight tiles with two K halves a product (default); 0: 16-row tiles
int fllm_option_dual_k(void);
int fllm_option_tile_slices(void);

// The device workspace of the current device (fllm_set_device_workspace): its first kWorkspaceCounterBytes are
// counters that every kernel leaves at zero, the rest is for partial results of the kernel that is running.
constexpr size_t kWorkspaceCounterBytes = 64 * 1024;      // plans.h counts with the same number (checked where both are seen)
bool fllm_device_workspace(void **base, size_t *bytes);

// Workgroups of one launch that meet in the workspace: a workgroup leaves its partial results there (relaxed
// agent-scope atomic stores, or the sc0 sc1 buffer stores of linear_skinny.hip), calls parts_published() and then
// counts itself with a relaxed agent-scope add; the workgroup that counts last calls parts_visible() and reads the
// parts of all (relaxed agent-scope atomic loads, sc0 sc1 buffer loads).
//
// FLLM_HANDOVER_SCOPE "agent" makes the two calls the release and acquire fences at agent scope that the HIP memory
// model asks for.  On gfx950 such a release writes the die's whole L2 back and the acquire drops it, and a decode
// step of 8 rows at the Llama-3.1-8B sizes takes 4.76 ms instead of 3.73 (measured; its K-sliced products and split
// contexts hand over 200 times a step), 3.41 instead of 3.34 ms at one row.  The default is therefore the form that
// rests on what the hardware does with these particular accesses, which is all the hand-over needs:
//   1. every part is written by stores with the sc1 bit (what an agent-scope atomic store is on gfx950): they are
//      written through to the memory side, which all eight dies share, and do not stay in the writer's L2;
//   2. s_waitcnt vmcnt(0) returns when those stores have been acknowledged from there;
//   3. only then is the counter's add issued, an atomic performed at the same memory-side point;
//   4. the reader issues its loads after the add that told it it is last has returned, and they carry sc1 too: they
//      are served from the memory side, not from a line its own die's L2 may still hold.
// A compiler fence at workgroup scope keeps the compiler from moving the stores, the add and the loads across each other.
// What this depends on and a change of hardware or compiler could break: that sc1 stores are acknowledged only once
// visible to the other dies (2), and that agent-scope atomic loads never hit in a die's L2 (4).
#ifndef FLLM_HANDOVER_SCOPE
#define FLLM_HANDOVER_SCOPE "workgroup"
#endif
__device__ __forceinline__ void parts_published() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, FLLM_HANDOVER_SCOPE);
    __builtin_amdgcn_s_waitcnt(0);
}
__device__ __forceinline__ void parts_visible() { __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, FLLM_HANDOVER_SCOPE); }

#define FLLM_REQUIRE(cond, ...)            \
    do {                                   \
        if (!(cond)) {                     \
            fllm_set_error(__VA_ARGS__);   \
            return -1;                     \
        }                                  \
    } while (0)

// Partial sums that workgroups hand to each other go through the device workspace in 16-byte pieces that pass by the
// caches of the compute units and of their die on both ways (the sc0 sc1 forms of the buffer instructions: written
// through to memory, read from memory), as device-scope atomics do for single words.  The workspace is one buffer
// for these instructions; offsets are in bytes from its base.
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4_t;
constexpr int kThroughCaches = 17;        // cache policy bits sc0 (1) and sc1 (16)
__device__ __forceinline__ __amdgpu_buffer_rsrc_t workspace_buffer(float *base) {
    return __builtin_amdgcn_make_buffer_rsrc(base, 0, 0x7fffffff, 0x00020000);      // raw buffer, offsets up to 2 GiB
}
__device__ __forceinline__ void hand_over(__amdgpu_buffer_rsrc_t ws, unsigned int byte_offset, f32x4_t v) {
    u32x4_t bits = {__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]), __float_as_uint(v[3])};
    __builtin_amdgcn_raw_buffer_store_b128(bits, ws, byte_offset, 0, kThroughCaches);
}
__device__ __forceinline__ f32x4_t take_over(__amdgpu_buffer_rsrc_t ws, unsigned int byte_offset) {
    const u32x4_t bits = __builtin_amdgcn_raw_buffer_load_b128(ws, byte_offset, 0, kThroughCaches);
    return (f32x4_t){__uint_as_float(bits[0]), __uint_as_float(bits[1]), __uint_as_float(bits[2]), __uint_as_float(bits[3])};
}

// Where a key's value lies in the pages.  Inside a page the keys of a key/value head are stored chunk by chunk:
// [kv_head][head_dim / 8][token][8], so that the 8 neighbouring values (16 bytes in bfloat16) of all tokens of the page lie
// together.  A decode step's products take 16 keys x 8 values a lane group: from this order that is 256 bytes in a row
// (two cache lines), from [token][head_dim] it would be 16 bytes of each of 16 rows (sixteen lines), which is what the
// memory pipeline of a compute unit is short of, not bytes (decode attention 8 x 32,768 keys: 182 -> 148 us).
// head_dim must be a multiple of 8.  Values are stored [kv_head][head_dim][token].
__host__ __device__ __forceinline__ size_t key_offset(size_t page, int kv_heads, int kvh, int page_size, int head_dim, int token, int d) {
    return ((((size_t)page * kv_heads + kvh) * (head_dim >> 3) + (d >> 3)) * page_size + token) * 8 + (d & 7);
}

// The same for keys stored in chunks of `kc` values ([kv_head][head_dim / kc][token][kc]; kc divides head_dim): 8 is the
// order above, 1 stores a head's lanes one after the other over the tokens, for head sizes that are no multiple of 8.
__host__ __device__ __forceinline__ size_t key_offset_chunked(size_t page, int kv_heads, int kvh, int page_size, int head_dim, int token,
                                                              int d, int kc) {
    return ((((size_t)page * kv_heads + kvh) * (head_dim / kc) + (d / kc)) * page_size + token) * kc + (d % kc);
}

template <typename T> __device__ __forceinline__ float to_f32(T v);
template <> __device__ __forceinline__ float to_f32<float>(float v) { return v; }
template <> __device__ __forceinline__ float to_f32<bf16_t>(bf16_t v) { return (float)v; }

template <typename T> __device__ __forceinline__ T from_f32(float v);
template <> __device__ __forceinline__ float from_f32<float>(float v) { return v; }
template <> __device__ __forceinline__ bf16_t from_f32<bf16_t>(float v) { return (bf16_t)v; }

// Sums and maxima over lanes, without LDS: what two lanes hold meets by the swaps of half waves and of rows of 16 lanes and by rotations inside a row.
// Through LDS (a shuffle each) every step waits for the one before it, some 100 cycles six times over; these steps are a few cycles each.
// The lanes meet as in a butterfly over the bits 32, 16, 8, 4, 2, 1 of their numbers, so no bit differs from that: once lanes 8 (4, 2) apart
// hold the same, the lane 4 (2, 1) further along the row holds what the one across has.  All lanes of the wave take part.
// Microseconds with shuffles -> with these: q/k/v 3,072 x 2,048 behind a norm at 8 / 16 rows 8.7 -> 8.1 / 11.1 -> 10.1 (four rows' sums side by side
// either way), a token step of layers of twelve small kernels (Dumizen, 1.5B sizes, two requests) 1.5 % less.
struct LanePair {
    float a, b;      // what the two lanes hold, the same in both
};
__device__ __forceinline__ LanePair lanes_32_apart(float v) {
    const unsigned int bits = __float_as_uint(v);
    const auto r = __builtin_amdgcn_permlane32_swap(bits, bits, false, false);
    return {__uint_as_float(r[0]), __uint_as_float(r[1])};
}
__device__ __forceinline__ LanePair lanes_16_apart(float v) {
    const unsigned int bits = __float_as_uint(v);
    const auto r = __builtin_amdgcn_permlane16_swap(bits, bits, false, false);
    return {__uint_as_float(r[0]), __uint_as_float(r[1])};
}
// the lane N further along this lane's row of 16
template <int N> __device__ __forceinline__ float along_row(float v) {
    return __uint_as_float(__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(v), 0x120 + N, 0xf, 0xf, false));      // row_ror:N
}
__device__ __forceinline__ float sum_32_apart(float v) { const LanePair p = lanes_32_apart(v); return p.a + p.b; }
__device__ __forceinline__ float sum_16_apart(float v) { const LanePair p = lanes_16_apart(v); return p.a + p.b; }
__device__ __forceinline__ float max_32_apart(float v) { const LanePair p = lanes_32_apart(v); return fmaxf(p.a, p.b); }
__device__ __forceinline__ float max_16_apart(float v) { const LanePair p = lanes_16_apart(v); return fmaxf(p.a, p.b); }
__device__ __forceinline__ float wave_sum(float v) {
    v = sum_16_apart(sum_32_apart(v));
    v += along_row<8>(v);
    v += along_row<4>(v);
    v += along_row<2>(v);
    v += along_row<1>(v);
    return v;
}
__device__ __forceinline__ float wave_max(float v) {
    v = max_16_apart(max_32_apart(v));
    v = fmaxf(v, along_row<8>(v));
    v = fmaxf(v, along_row<4>(v));
    v = fmaxf(v, along_row<2>(v));
    v = fmaxf(v, along_row<1>(v));
    return v;
}

// Sum over a workgroup of NW waves, the same value in every thread; the waves' partial sums
// are added in wave order, so the result depends only on the data and the launch shape.
template <int NW> __device__ __forceinline__ float block_sum(float v, float *scratch /* NW floats */) {
    v = wave_sum(v);
    __syncthreads();
    if ((threadIdx.x & (kWave - 1)) == 0) scratch[threadIdx.x / kWave] = v;
    __syncthreads();
    float total = 0.f;
#pragma unroll
    for (int i = 0; i < NW; i++) total += scratch[i];
    return total;
}
// The same over a place that nothing has used yet: one meeting instead of two.
template <int NW> __device__ __forceinline__ float block_sum_once(float v, float *scratch /* NW floats, this sum's own */) {
    v = wave_sum(v);
    if ((threadIdx.x & (kWave - 1)) == 0) scratch[threadIdx.x / kWave] = v;
    __syncthreads();
    float total = 0.f;
#pragma unroll
    for (int i = 0; i < NW; i++) total += scratch[i];
    return total;
}
// Arguments that no register holds at the start of a wave, asked for here: behind the first loads, whose trip to memory theirs then shares.
// Left to itself the compiler fetches an argument just ahead of its use, which is a trip of its own (0.3 to 0.5 us, the line is cold).
template <typename... A> __device__ __forceinline__ void fetch_arguments(A... a) {
    __builtin_amdgcn_sched_barrier(0);      // no load of before moves behind the wait
    const int done[] = {([](auto one) { asm volatile("" ::"s"(one)); return 0; }(a))...};
    (void)done;
}
template <int NW> __device__ __forceinline__ float block_max(float v, float *scratch) {
    v = wave_max(v);
    __syncthreads();
    if ((threadIdx.x & (kWave - 1)) == 0) scratch[threadIdx.x / kWave] = v;
    __syncthreads();
    float total = -INFINITY;
#pragma unroll
    for (int i = 0; i < NW; i++) total = fmaxf(total, scratch[i]);
    return total;
}

// Philox-4x32 with ten rounds (Salmon et al., "Parallel random numbers: as easy as 1, 2, 3"): the counter words in,
// the output words in their place.  The sampler's draws and the random-weights generator use it.
struct Philox {
    uint32_t c0, c1, c2, c3;
    __device__ __forceinline__ void ten_rounds(uint32_t key_lo, uint32_t key_hi) {
#pragma unroll
        for (int round = 0; round < 10; round++) {
            const uint64_t left = (uint64_t)0xD2511F53u * c0;
            const uint64_t right = (uint64_t)0xCD9E8D57u * c2;
            const uint32_t next0 = (uint32_t)(right >> 32) ^ c1 ^ key_lo;
            const uint32_t next2 = (uint32_t)(left >> 32) ^ c3 ^ key_hi;
            c1 = (uint32_t)right;
            c3 = (uint32_t)left;
            c0 = next0;
            c2 = next2;
            key_lo += 0x9E3779B9u;
            key_hi += 0xBB67AE85u;
        }
    }
};
