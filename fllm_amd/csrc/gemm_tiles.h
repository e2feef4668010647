// Matrix products of many rows in bfloat16, y = x W^T, as tiles of 256 x 256 or 128 x 256 a workgroup (device code; launched by
// linear_tiles.hip and routed_experts_mfma.hip).
//
// What bounds such a product is how much of the time the matrix cores have operands.  A tile is 64 columns of K deep in LDS, filled by loads
// that go straight there (global_load_lds, 16 bytes a lane, seven half tiles ahead of their use) and waited for by count, never all.  Eight
// waves, two a SIMD, work in two groups that are half a step apart: while one group issues the 16 products of a quarter tile, the other
// reads its next operands from LDS and asks for a half tile of a later step; a barrier swaps them.  A half tile's place is filled again one
// step after it was read, behind a barrier that follows the read's own wait (a tile's first read of W, which lies ahead of the two
// groups' first step, has a barrier of its own).  16-byte chunk c of row r lies at place c ^ (r % 8) of the row:
// the lanes of an operand then meet every bank once.  Rows of W are dealt to LDS so that a lane ends up with 8 neighbouring columns (a
// 16-byte store); a workgroup asks for its next tile's first steps before it stores the last one.
//
// Measured (one MI355X, random operands, weights from memory, launches that follow one another, beside the GEMM library; boxes differ by
// 5 %): 8,192 x 8,192 x 8,192 720 us (1.53 PFLOP/s, library 703); 2,048 x 28,672 x 4,096 with the SwiGLU in the epilogue 346 to 356 us (1.39 to
// 1.35; library and a SwiGLU kernel 382 to 422), 368 where its last round runs as whole tiles; 2,048 x 4,096 x 14,336 as 128-row tiles 197 us
// (1.22; library 217), as 256-row tiles 257 (half of the compute units).
//
// MFMA operand layout (v_mfma_f32_16x16x32_bf16): A lane l holds A[m = l%16][k = 8*(l/16) .. +7]; B likewise with n = l%16; D lane l holds
// D[m = 4*(l/16) + i][n = l%16], i = 0..3.  A is W here, B the rows of x.
#pragma once
#include "common.h"

namespace fllm_tiles {

enum { EPI_STORE = 0, EPI_GLU = 1, EPI_RELU2 = 2, EPI_F32 = 3 };      // EPI_F32: grouped and sliced products alone

struct TileArgs {
    const bf16_t *x;        // rows, row stride ldx (a multiple of 8)
    const bf16_t *w;        // [N][K], EPI_GLU [2 N][K]: gate rows, then up rows; grouped: one such matrix an expert
    void *out;              // [rows][N], row stride ldo (a multiple of 8): bfloat16, EPI_F32 float32
    const float *bias;      // EPI_STORE: [N] or null
    int ldx, ldo, M, N, K;  // N a multiple of 8, K of 64 (128-row tiles, at least 192) or 128 (256-row tiles, at least 256)
    float limit, alpha, up_offset;
    // grouped by expert: see group_pairs_kernel
    const int32_t *work;    // null: the rows of x as they are
    int max_tiles;
    int top;                // the row of x a pair reads: > 0 pair / top, 0 its slot, -1 the pair
    // K cut into slices, a workgroup each (128-row tiles): the tiles' parts [tile][slice][128 x 256 floats] and a counter a tile, zero between launches
    int slices;
    float *parts;
    int *counters;
    int halves;             // the 256-row kernel: whether a last round of at most 128 tiles runs as tiles of half the rows
};

constexpr int kThreads = 512;
constexpr int BK = 64;
constexpr int kHalf = 128 * BK * 2;      // bytes of a half tile in LDS
constexpr int kLds256 = 8 * kHalf, kLds128 = 9 * kHalf;

// 16 bytes a lane from base + off (bytes) to LDS address l (the same in every lane) + 16 * lane
__device__ __forceinline__ void to_lds(const bf16_t *base, uint32_t off, uint32_t l) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(l), "v"(off), "s"(base) : "memory", "m0");
}
#define FLLM_VM(n) asm volatile("s_waitcnt vmcnt(" #n ")" ::: "memory")
#define FLLM_LGKM0 asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory")
#define FLLM_SWAP                             \
    do {                                      \
        __builtin_amdgcn_sched_barrier(0);    \
        __builtin_amdgcn_s_barrier();         \
        __builtin_amdgcn_sched_barrier(0);    \
    } while (0)
typedef const __attribute__((address_space(3))) bf16x8_t lds_piece;

// Row r (0 .. 127) of half h of W in LDS -> column of the tile
template <int EPI> __device__ __forceinline__ int tile_column(int r, int h) {
    const int c = ((r % 16) / 4) * 8 + ((r / 16) % 2) * 4 + r % 4;
    return EPI == EPI_GLU ? (r / 32) * 32 + c : (r / 32) * 64 + h * 32 + c;
}

// Which tile a workgroup works on.  The dies (workgroup number modulo 8) take runs of neighbouring tiles, in groups of 8 row tiles, so that
// what a die's workgroups read at a time fits its L2.
// HALVES: tiles of 128 rows, two for each of the 256-row tiles of a last round.
template <int EPI, bool GROUPED, int BM, bool HALVES = false>
struct Place {
    int total, mt, nt;
    int m0, n0;              // first row (grouped: slot) and column
    int rows;                // rows the tile has
    const bf16_t *w;
    static constexpr int kRows = HALVES ? 256 : BM;      // that a tile of the order below has
    __device__ __forceinline__ Place(const TileArgs &a) {
        mt = GROUPED ? __builtin_amdgcn_readfirstlane(a.work[0]) : (a.M + kRows - 1) / kRows;
        nt = (a.N + (EPI == EPI_GLU ? 127 : 255)) / (EPI == EPI_GLU ? 128 : 256);
        total = mt * nt;
        w = a.w;
    }
    // tiles of the last round that run as halves: their workgroups would take a whole tile's time and leave the others idle
    __device__ __forceinline__ int in_halves(const TileArgs &a) const { return a.halves && total % 256 <= 128 ? total % 256 : 0; }
    __device__ __forceinline__ void go(const TileArgs &a, int id) {
        int half = 0;
        if (HALVES) {                                        // both halves of a tile on the tile's die
            half = (id / 8) & 1;
            id = total - in_halves(a) + id / 16 * 8 + id % 8;
        }
        const int q = total / 8, r = total % 8, die = id % 8;
        id = (die < r ? die * (q + 1) : r * (q + 1) + (die - r) * q) + id / 8;
        const int per = 8 * nt, g = id / per, first = g * 8, tall = min(8, mt - first), in = id - g * per;
        const int t = first + in % tall;
        n0 = in / tall * (EPI == EPI_GLU ? 128 : 256);
        if (GROUPED) {
            const int32_t *tile = a.work + 1 + 3 * t;
            const int e = __builtin_amdgcn_readfirstlane(tile[0]);
            m0 = __builtin_amdgcn_readfirstlane(tile[1]) + half * BM;
            rows = __builtin_amdgcn_readfirstlane(tile[2]) - half * BM;
            w = a.w + (size_t)e * (EPI == EPI_GLU ? 2 : 1) * a.N * a.K;
        } else {
            m0 = t * kRows + half * BM;
            rows = a.M - m0;
        }
    }
    // the pair in row m of the tile (grouped), or the row itself
    __device__ __forceinline__ int row(const TileArgs &a, int m) const {
        return GROUPED ? a.work[1 + 3 * a.max_tiles + m0 + m] : m0 + m;
    }
    __device__ __forceinline__ uint32_t x_offset(const TileArgs &a, int m, int chunk) const {
        m = min(m, rows - 1);            // rows that the tile has not read its last one
        int from = row(a, m);
        if (GROUPED) from = a.top > 0 ? from / a.top : (a.top == 0 ? m0 + m : from);
        return ((uint32_t)from * (uint32_t)a.ldx + chunk * 8) * 2;
    }
    __device__ __forceinline__ uint32_t w_offset(const TileArgs &a, int r, int h, int chunk) const {
        const int n = min(n0 + tile_column<EPI>(r, h), a.N - 1) + (EPI == EPI_GLU ? h * a.N : 0);
        return ((uint32_t)n * (uint32_t)a.K + chunk * 8) * 2;
    }
};

// 8 neighbouring columns of one row: c0 from the first half of W, c1 from the second (EPI_GLU: gate and up)
template <int EPI>
__device__ __forceinline__ void store_columns(const TileArgs &a, int row, int n, const f32x4_t (&c)[2], const f32x4_t (&u)[2]) {
    const size_t at = (size_t)row * a.ldo + n;
    if (EPI == EPI_F32) {
        *(f32x4_t *)((float *)a.out + at) = c[0];
        *(f32x4_t *)((float *)a.out + at + 4) = c[1];
        return;
    }
    bf16x8_t o;
#pragma unroll
    for (int e = 0; e < 8; e++) {
        float v = c[e / 4][e % 4];
        if (EPI == EPI_GLU) {
            float up = u[e / 4][e % 4];
            if (a.limit > 0.f) {
                v = fminf(v, a.limit);
                up = fminf(fmaxf(up, -a.limit), a.limit);
            }
            v = v / (1.0f + expf(-a.alpha * v)) * (up + a.up_offset);
        } else if (EPI == EPI_RELU2) {
            v = fmaxf(v, 0.f);
            v = v * v;
        } else if (a.bias != nullptr) {
            v += a.bias[n + e];
        }
        o[e] = (bf16_t)v;
    }
    *(bf16x8_t *)((bf16_t *)a.out + at) = o;
}
template <int EPI>
__device__ __forceinline__ void store_row(const TileArgs &a, int row, int n0, int wn, int lg, const f32x4_t (&c0)[2], const f32x4_t (&c1)[2]) {
    if (EPI == EPI_GLU) {
        const int n = n0 + wn * 32 + lg * 8;
        if (n < a.N) store_columns<EPI>(a, row, n, c0, c1);
    } else {
        const int n = n0 + wn * 64 + lg * 8;
        if (n < a.N) store_columns<EPI>(a, row, n, c0, c0);
        if (n + 32 < a.N) store_columns<EPI>(a, row, n + 32, c1, c1);
    }
}

// One quarter of a tile: 64 rows x 32 columns a wave, 64 columns of K
__device__ __forceinline__ void multiply(f32x4_t (&c)[4][2], const bf16x8_t (&x)[4][2], const bf16x8_t (&w)[2][2]) {
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int s = 0; s < 2; s++)
#pragma unroll
        for (int t = 0; t < 4; t++)
#pragma unroll
            for (int u = 0; u < 2; u++) c[t][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[u][s], x[t][s], c[t][u], 0, 0, 0);
    __builtin_amdgcn_s_setprio(0);
}

// 256 x 256 (EPI_GLU: 256 x 128 gate and up columns).  LDS: two buffers of [x rows 0..127][x rows 128..255][W half 0][W half 1].
// K step k: quarter 0 reads x half 0 of k and asks for W half 0 of k + 2; quarter 1 reads W half 1, asks for x half 0 of k + 2; quarter 2
// reads x half 1, asks for W half 1; quarter 3 reads W half 0 of k + 1 and asks for x half 1 of k + 2.  Every quarter ends its reading side
// by waiting until at most 12 loads (six half tiles) are outstanding: then what the next quarter reads has arrived.
template <int EPI, bool GROUPED>
__device__ __forceinline__ void tiles256(const TileArgs &a) {
    extern __shared__ __attribute__((aligned(16))) bf16_t lds[];
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    const int wm = w >> 2, wn = w & 3, l16 = lane & 15, lg = lane >> 4;
    Place<EPI, GROUPED, 256> at(a);
    const int total = at.total - at.in_halves(a);
    int id = blockIdx.x;
    if (id >= total) return;
    const uint32_t base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) bf16_t *)lds;
    const uint32_t mine = __builtin_amdgcn_readfirstlane(base + w * 1024);
    uint32_t off_x[2][2], off_w[2][2];      // bytes from x and from the matrix to what this lane loads of a half tile, in two pieces
    auto offsets = [&]() {
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const int r = w * 8 + (lane >> 3) + j * 64, chunk = (lane & 7) ^ (r & 7);
                off_x[h][j] = at.x_offset(a, h * 128 + r, chunk);
                off_w[h][j] = at.w_offset(a, r, h, chunk);
                asm volatile("" : "+v"(off_x[h][j]));      // kept as they are: the compiler would hold many sums of them instead
                asm volatile("" : "+v"(off_w[h][j]));
            }
    };
    auto ask_x = [&](int buf, int h, int k) {
#pragma unroll
        for (int j = 0; j < 2; j++) to_lds(a.x + k * BK, off_x[h][j], mine + buf * 4 * kHalf + h * kHalf + j * 8192);
    };
    auto ask_w = [&](int buf, int h, int k) {
#pragma unroll
        for (int j = 0; j < 2; j++) to_lds(at.w + k * BK, off_w[h][j], mine + buf * 4 * kHalf + (2 + h) * kHalf + j * 8192);
    };
    uint32_t rx[2][2], rw[2][2];            // LDS addresses of a lane's pieces, by buffer and k-step of 32
#pragma unroll
    for (int buf = 0; buf < 2; buf++)
#pragma unroll
        for (int s = 0; s < 2; s++) {
            const uint32_t piece = ((s * 4 + lg) ^ (l16 & 7)) * 16;
            rx[buf][s] = base + buf * 4 * kHalf + (wm * 64 + l16) * BK * 2 + piece;
            rw[buf][s] = base + buf * 4 * kHalf + 2 * kHalf + (wn * 32 + l16) * BK * 2 + piece;
            asm volatile("" : "+v"(rx[buf][s]));
            asm volatile("" : "+v"(rw[buf][s]));
        }
    bf16x8_t xs[4][2], wx[2][2], wy[2][2];
    auto read_x = [&](int buf, int h) {
#pragma unroll
        for (int t = 0; t < 4; t++)
#pragma unroll
            for (int s = 0; s < 2; s++) xs[t][s] = *(lds_piece *)(uintptr_t)(rx[buf][s] + h * kHalf + t * 16 * BK * 2);
    };
    auto read_w = [&](int buf, int h, bf16x8_t (&to)[2][2]) {
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int s = 0; s < 2; s++) to[t][s] = *(lds_piece *)(uintptr_t)(rw[buf][s] + h * kHalf + t * 16 * BK * 2);
    };
    f32x4_t acc[2][2][4][2];
    auto first_steps = [&]() {
        ask_w(0, 0, 0); ask_x(0, 0, 0); ask_w(0, 1, 0); ask_x(0, 1, 0);
        ask_w(1, 0, 1); ask_x(1, 0, 1); ask_w(1, 1, 1); ask_x(1, 1, 1);
    };
    const int T = a.K / BK;                 // even, at least 4
#define FLLM_STEP(buf, w0, w1, k, ASK, V0, V1, V2, V3, NEXT)                              \
    do {                                                                                  \
        read_x(buf, 0);                                                                   \
        if (ASK) ask_w(buf, 0, (k) + 2);                                                  \
        FLLM_VM(V0); FLLM_LGKM0; FLLM_SWAP; multiply(acc[0][0], xs, w0); FLLM_SWAP;       \
        read_w(buf, 1, w1);                                                               \
        if (ASK) ask_x(buf, 0, (k) + 2);                                                  \
        FLLM_VM(V1); FLLM_LGKM0; FLLM_SWAP; multiply(acc[0][1], xs, w1); FLLM_SWAP;       \
        read_x(buf, 1);                                                                   \
        if (ASK) ask_w(buf, 1, (k) + 2);                                                  \
        FLLM_VM(V2); FLLM_LGKM0; FLLM_SWAP; multiply(acc[1][1], xs, w1); FLLM_SWAP;       \
        if (NEXT) read_w((buf) ^ 1, 0, w1);                                               \
        if (ASK) ask_x(buf, 1, (k) + 2);                                                  \
        FLLM_VM(V3); FLLM_LGKM0; FLLM_SWAP; multiply(acc[1][0], xs, w0); FLLM_SWAP;       \
    } while (0)
    at.go(a, id);
    offsets();
    first_steps();
    for (;;) {
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int t = 0; t < 4; t++)
#pragma unroll
                    for (int u = 0; u < 2; u++) acc[i][j][t][u] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        FLLM_VM(12);                        // (stores still on their way only make this wait longer: loads arrive in their order)
        FLLM_SWAP;
        read_w(0, 0, wx);
        FLLM_LGKM0;
        FLLM_SWAP;                          // step 0 asks for what takes that half tile's place: every wave has read it
        if (wm == 1) FLLM_SWAP;             // the second group runs half a quarter behind the first
        int k = 0;
        for (; k + 4 <= T; k += 2) {
            FLLM_STEP(0, wx, wy, k, true, 12, 12, 12, 12, true);
            FLLM_STEP(1, wy, wx, k + 1, true, 12, 12, 12, 12, true);
        }
        FLLM_STEP(0, wx, wy, k, false, 10, 8, 6, 4, true);
        FLLM_STEP(1, wy, wx, k + 1, false, 2, 0, 0, 0, false);
        if (wm == 0) FLLM_SWAP;
        // every wave has read what it needs: the next tile's first steps are on their way while this one is stored
        const Place<EPI, GROUPED, 256> done = at;
        int to[2][4];
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int t = 0; t < 4; t++) {
                to[i][t] = done.row(a, min(i * 128 + wm * 64 + t * 16 + l16, done.rows - 1));
                if (GROUPED) asm volatile("" : "+v"(to[i][t]));      // looked up before the next tile's loads are in the way
            }
        id += gridDim.x;
        const bool more = id < total;
        if (more) {
            at.go(a, id);
            offsets();
            first_steps();
        }
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int t = 0; t < 4; t++) {
                const int m = i * 128 + wm * 64 + t * 16 + l16;
                if (m < done.rows) store_row<EPI>(a, to[i][t], done.n0, wn, lg, acc[i][0][t], acc[i][1][t]);
            }
        if (!more) break;
    }
#undef FLLM_STEP
}

// The slices of a 128-row tile meet (below): whether this workgroup goes on with the sums of all.
__device__ __forceinline__ bool meet_slices(const TileArgs &a, int tile, int slice, f32x4_t (&acc)[2][4][2], int *seen);

// 128 x 256 (EPI_GLU: 128 x 128), for launches whose 256-row tiles would leave much of the device idle: an operand read from LDS serves half
// the products, so LDS and the matrix cores are busy alike.  LDS: three buffers of [x][W half 0][W half 1].  K step k: half 0 reads x of k
// and asks for W half 1 of k + 2 and W half 0 of k + 3; half 1 reads W half 1 of k and W half 0 of k + 1 and asks for x of k + 3.
// SLICED: workgroup number b takes slice b / tiles of tile b % tiles; see meet_slices.
template <int EPI, bool GROUPED, bool HALVES = false, bool SLICED = false>
__device__ __forceinline__ void tiles128(const TileArgs &a) {
    extern __shared__ __attribute__((aligned(16))) bf16_t lds[];
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    const int wm = w >> 2, wn = w & 3, l16 = lane & 15, lg = lane >> 4;
    Place<EPI, GROUPED, 128, HALVES> at(a);
    const int slice = SLICED ? blockIdx.x / at.total : 0;
    int id = SLICED ? blockIdx.x % at.total : blockIdx.x;
    const int tile = id;
    const int total = HALVES ? (at.in_halves(a) + 7) / 8 * 16 : at.total;      // HALVES: at most one a workgroup
    const int first_step = SLICED ? (int)((long)(a.K / BK) * slice / a.slices) : 0;
    if (id >= total || (HALVES && id / 16 * 8 + id % 8 >= at.in_halves(a))) return;
    constexpr uint32_t kSlot = 3 * kHalf;
    const uint32_t base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) bf16_t *)lds;
    const uint32_t mine = __builtin_amdgcn_readfirstlane(base + w * 1024);
    uint32_t off_x[2], off_w[2][2];
    auto offsets = [&]() {
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int r = w * 8 + (lane >> 3) + j * 64, chunk = (lane & 7) ^ (r & 7);
            off_x[j] = at.x_offset(a, r, chunk);
            asm volatile("" : "+v"(off_x[j]));
#pragma unroll
            for (int h = 0; h < 2; h++) {
                off_w[h][j] = at.w_offset(a, r, h, chunk);
                asm volatile("" : "+v"(off_w[h][j]));
            }
        }
    };
    auto ask_x = [&](uint32_t slot, int k) {
#pragma unroll
        for (int j = 0; j < 2; j++) to_lds(a.x + (first_step + k) * BK, off_x[j], mine + slot + j * 8192);
    };
    auto ask_w = [&](uint32_t slot, int h, int k) {
#pragma unroll
        for (int j = 0; j < 2; j++) to_lds(at.w + (first_step + k) * BK, off_w[h][j], mine + slot + (1 + h) * kHalf + j * 8192);
    };
    uint32_t rx[2], rw[2];
#pragma unroll
    for (int s = 0; s < 2; s++) {
        const uint32_t piece = ((s * 4 + lg) ^ (l16 & 7)) * 16;
        rx[s] = base + (wm * 64 + l16) * BK * 2 + piece;
        rw[s] = base + kHalf + (wn * 32 + l16) * BK * 2 + piece;
        asm volatile("" : "+v"(rx[s]));
        asm volatile("" : "+v"(rw[s]));
    }
    bf16x8_t xs[4][2], w0[2][2], w1[2][2];
    auto read_x = [&](uint32_t slot) {
#pragma unroll
        for (int t = 0; t < 4; t++)
#pragma unroll
            for (int s = 0; s < 2; s++) xs[t][s] = *(lds_piece *)(uintptr_t)(rx[s] + slot + t * 16 * BK * 2);
    };
    auto read_w = [&](uint32_t slot, int h, bf16x8_t (&to)[2][2]) {
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int s = 0; s < 2; s++) to[t][s] = *(lds_piece *)(uintptr_t)(rw[s] + slot + h * kHalf + t * 16 * BK * 2);
    };
    f32x4_t acc[2][4][2];
    auto first_steps = [&]() {
        ask_w(0, 0, 0); ask_x(0, 0); ask_w(0, 1, 0);
        ask_w(kSlot, 0, 1); ask_x(kSlot, 1); ask_w(kSlot, 1, 1);
        ask_w(2 * kSlot, 0, 2); ask_x(2 * kSlot, 2);
    };
    const int T = SLICED ? (int)((long)(a.K / BK) * (slice + 1) / a.slices) - first_step : a.K / BK;      // at least 3
    at.go(a, id);
    if (HALVES && at.rows <= 0) return;
    offsets();
    first_steps();
    for (;;) {
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int t = 0; t < 4; t++)
#pragma unroll
                for (int u = 0; u < 2; u++) acc[j][t][u] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        FLLM_VM(12);
        FLLM_SWAP;
        read_w(0, 0, w0);
        FLLM_LGKM0;
        FLLM_SWAP;                          // as above
        if (wm == 1) FLLM_SWAP;
        uint32_t s0 = 0, s1 = kSlot, s2 = 2 * kSlot;      // where steps k, k + 1 and k + 2 lie
        int k = 0;
        for (; k < T - 3; k++) {
            read_x(s0);
            ask_w(s2, 1, k + 2);
            ask_w(s0, 0, k + 3);
            FLLM_VM(12); FLLM_LGKM0; FLLM_SWAP; multiply(acc[0], xs, w0); FLLM_SWAP;
            read_w(s0, 1, w1);
            read_w(s1, 0, w0);
            ask_x(s0, k + 3);
            FLLM_VM(12); FLLM_LGKM0; FLLM_SWAP; multiply(acc[1], xs, w1); FLLM_SWAP;
            const uint32_t s = s0;
            s0 = s1, s1 = s2, s2 = s;
        }
        read_x(s0);
        ask_w(s2, 1, k + 2);
        FLLM_VM(10); FLLM_LGKM0; FLLM_SWAP; multiply(acc[0], xs, w0); FLLM_SWAP;
        read_w(s0, 1, w1);
        read_w(s1, 0, w0);
        FLLM_VM(8); FLLM_LGKM0; FLLM_SWAP; multiply(acc[1], xs, w1); FLLM_SWAP;
        read_x(s1);
        FLLM_VM(4); FLLM_LGKM0; FLLM_SWAP; multiply(acc[0], xs, w0); FLLM_SWAP;
        read_w(s1, 1, w1);
        read_w(s2, 0, w0);
        FLLM_VM(2); FLLM_LGKM0; FLLM_SWAP; multiply(acc[1], xs, w1); FLLM_SWAP;
        read_x(s2);
        FLLM_VM(0); FLLM_LGKM0; FLLM_SWAP; multiply(acc[0], xs, w0); FLLM_SWAP;
        read_w(s2, 1, w1);
        FLLM_LGKM0; FLLM_SWAP; multiply(acc[1], xs, w1); FLLM_SWAP;
        if (wm == 0) FLLM_SWAP;
        if constexpr (SLICED)
            if (!meet_slices(a, tile, slice, acc, (int *)lds)) return;
        const Place<EPI, GROUPED, 128, HALVES> done = at;
        int to[4];
#pragma unroll
        for (int t = 0; t < 4; t++) {
            to[t] = done.row(a, min(wm * 64 + t * 16 + l16, done.rows - 1));
            if (GROUPED) asm volatile("" : "+v"(to[t]));
        }
        id += gridDim.x;
        const bool more = !HALVES && !SLICED && id < total;
        if (more) {
            at.go(a, id);
            offsets();
            first_steps();
        }
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const int m = wm * 64 + t * 16 + l16;
            if (m < done.rows) store_row<EPI>(a, to[t], done.n0, wn, lg, acc[0][t], acc[1][t]);
        }
        if (!more) break;
    }
}

// The kernels, products of their own and grouped ones under names of their own in a trace; the modes of the grouped ones are those of
// the small grouped tiles: 0 gate and up with the activation, 1 float32 sums, 2 the squared ReLU.
// HALVES: a last round of at most 128 tiles of 256 rows runs as twice as many of 128 rows, which take 0.73 to 0.85 of its time.
template <int EPI, int ROWS, bool HALVES>
__global__ void __launch_bounds__(kThreads, 2) tiles_kernel(const TileArgs a) {
    if constexpr (ROWS == 256) tiles256<EPI, false>(a);
    if constexpr (ROWS == 128 || HALVES) tiles128<EPI, false, HALVES>(a);
}
template <int MODE, int ROWS, bool HALVES>
__global__ void __launch_bounds__(kThreads, 2) large_grouped_tiles_kernel(const TileArgs a) {
    constexpr int EPI = MODE == 0 ? EPI_GLU : MODE == 1 ? EPI_F32 : EPI_RELU2;
    if constexpr (ROWS == 256) tiles256<EPI, true>(a);
    if constexpr (ROWS == 128 || HALVES) tiles128<EPI, true, HALVES>(a);
}
template <int EPI, bool GROUPED, int ROWS, bool HALVES>
auto tiles_entry() -> void (*)(TileArgs) {
    if constexpr (GROUPED) return large_grouped_tiles_kernel<EPI == EPI_GLU ? 0 : EPI == EPI_F32 ? 1 : 2, ROWS, HALVES>;
    else return tiles_kernel<EPI, ROWS, HALVES>;
}

// The slices of a 128-row tile meet: every workgroup leaves its sums in the device workspace and counts the tile, the one that counts last goes on
// with the sum of all in slice order (so it does not matter which one that is), the others are done: false.  Nobody waits for another.
__device__ __forceinline__ bool meet_slices(const TileArgs &a, int tile, int slice, f32x4_t (&acc)[2][4][2], int *seen) {
    const __amdgpu_buffer_rsrc_t parts = workspace_buffer(a.parts);
    const unsigned int part = 128 * 256 * 4, mine = threadIdx.x * 16;      // bytes; 256 workgroups at most: 32 MiB
    const unsigned int first = (unsigned int)tile * a.slices * part + mine;
#pragma unroll
    for (int p = 0; p < 16; p++) hand_over(parts, first + slice * part + p * kThreads * 16, acc[p >> 3][(p >> 1) & 3][p & 1]);
    parts_published();
    __syncthreads();
    if (threadIdx.x == 0) *seen = __hip_atomic_fetch_add(a.counters + tile, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (*seen != a.slices - 1) return false;
    parts_visible();
    if (threadIdx.x == 0) __hip_atomic_store(a.counters + tile, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);      // for the next launch
    f32x4_t sum[16];
    for (int s = 0; s < a.slices; s++) {
        f32x4_t v[16];
#pragma unroll
        for (int p = 0; p < 16; p++) v[p] = take_over(parts, first + s * part + p * kThreads * 16);
#pragma unroll
        for (int p = 0; p < 16; p++) sum[p] = s == 0 ? v[p] : sum[p] + v[p];
    }
#pragma unroll
    for (int p = 0; p < 16; p++) acc[p >> 3][(p >> 1) & 3][p & 1] = sum[p];
    return true;
}

// What bounds it is what bounds the 128-row tiles, 0.88 us a step of K, and then the sums' way through memory: 2,048 x 2,048 x 8,192 in two slices of 128
// tiles 69 us (1.0 PFLOP/s; library 75), 13 of them before the first and behind the last step; 1,735 x 1,536 x 13,312 in three of 84 77 (89).
template <int EPI>
__global__ void __launch_bounds__(kThreads, 2) sliced_tiles_kernel(const TileArgs a) {
    tiles128<EPI, false, false, true>(a);
}
// `tiles` 128-row tiles in a.slices slices: tiles * slices workgroups, no more than compute units
template <int EPI>
int launch_sliced(const TileArgs &a, long tiles, hipStream_t stream) {
    static bool raised = false;
    if (!raised) {
        const hipError_t e = hipFuncSetAttribute((const void *)sliced_tiles_kernel<EPI>, hipFuncAttributeMaxDynamicSharedMemorySize, kLds128);
        FLLM_REQUIRE(e == hipSuccess, "gemm tiles: cannot raise the LDS limit: %s", hipGetErrorString(e));
        raised = true;
    }
    hipLaunchKernelGGL(sliced_tiles_kernel<EPI>, dim3((unsigned)(tiles * a.slices)), dim3(kThreads), kLds128, stream, a);
    return fllm_check_launch("sliced gemm tiles");
}

// Launches one of them on one workgroup a compute unit at most (grouped: as many tiles as there may be).
template <int EPI, bool GROUPED, int ROWS, bool HALVES>
int launch_entry(const TileArgs &a, unsigned blocks, hipStream_t stream) {
    constexpr int lds = ROWS == 256 && !HALVES ? kLds256 : kLds128;
    static_assert(kLds128 >= kLds256, "both kinds of tiles in one launch");
    static bool raised = false;      // more than 64 KiB of LDS has to be asked for once
    if (!raised) {
        const hipError_t e = hipFuncSetAttribute((const void *)tiles_entry<EPI, GROUPED, ROWS, HALVES>(), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        FLLM_REQUIRE(e == hipSuccess, "gemm tiles: cannot raise the LDS limit: %s", hipGetErrorString(e));
        raised = true;
    }
    hipLaunchKernelGGL((tiles_entry<EPI, GROUPED, ROWS, HALVES>()), dim3(blocks), dim3(kThreads), lds, stream, a);
    return fllm_check_launch("gemm tiles");
}
template <int EPI, bool GROUPED>
int launch_tiles(TileArgs a, int bm, bool halves, long tiles, hipStream_t stream) {
    a.halves = halves;
    if (halves) return launch_entry<EPI, GROUPED, 256, true>(a, 256, stream);
    const unsigned blocks = (unsigned)(tiles < 256 ? tiles : 256);
    return bm == 256 ? launch_entry<EPI, GROUPED, 256, false>(a, blocks, stream) : launch_entry<EPI, GROUPED, 128, false>(a, blocks, stream);
}

}  // namespace fllm_tiles
