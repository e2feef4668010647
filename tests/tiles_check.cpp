// The tile products of csrc/gemm_tiles.h as a host program (tests/test_tile_schedule.py puts the calls below in the place of the header's
// inline assembly).  One lane of each of the eight waves walks through the kernel, and every load into LDS, every wait and every read
// of LDS is noted with the number of barriers that its wave has passed.  All barriers are the workgroup's: events of two waves are in order where that number
// differs, and may fall in either order where it is the same.  Checked for every read of a half tile:
//   1. every wave had waited for the pieces that it loads, before an earlier barrier (the reading wave's own: before the read);
//   2. no wave asks for the half tile that comes to the same place next before a barrier behind the end of the read;
// and that steps come in their order, all that is asked for is read, and no load leaves the operands.
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <vector>

using std::max;
using std::min;

struct Index { unsigned int x; };
static Index threadIdx, blockIdx, gridDim;
constexpr int kWave = 64, kWaves = 8, kPlaces = 9, kPlaceBytes = 64 * 128 * 2;

struct bf16_t {
    uint16_t bits;
    bf16_t() = default;
    explicit bf16_t(float) : bits(0) {}
};
struct f32x4_t {
    float v[4];
    float operator[](int i) const { return v[i]; }
};
namespace fllm_tiles { alignas(16) bf16_t lds[kPlaces * kPlaceBytes / 2]; }

struct Fill { int step, asked, landed; long order, landed_order; bool of_x; };      // asked, landed: barriers passed
struct Read { int begin, end; long order; };
static std::vector<Fill> fills[kWaves][kPlaces];      // half a half tile each
static std::vector<Read> reads[kWaves][kPlaces];      // 16 bytes each
static std::vector<std::pair<int, size_t>> on_the_way, unread;      // place and index
static int wave, barriers;
static long order;
static const char *x_from, *x_to, *w_from, *w_to;

[[noreturn]] static void stop(const char *what, long n) { printf("%s (%ld)\n", what, n); exit(1); }

static long place_of(uintptr_t address) {             // the kernel holds LDS addresses in 32 bits
    const uint32_t off = (uint32_t)address - (uint32_t)(uintptr_t)fllm_tiles::lds;
    return off < kPlaces * kPlaceBytes ? (long)(off / kPlaceBytes) : -1;
}
struct bf16x8_t {
    bf16_t v[8];
    bf16_t &operator[](int i) { return v[i]; }
    bf16x8_t() = default;
    bf16x8_t &operator=(const bf16x8_t &o) {          // a copy from LDS is a read of it
        const long place = (uintptr_t)&o <= 0xffffffffu ? place_of((uintptr_t)&o) : -1;
        if (place < 0) { memcpy(v, o.v, sizeof(v)); return *this; }
        unread.push_back({(int)place, reads[wave][place].size()});
        reads[wave][place].push_back({barriers, -1, order++});
        return *this;
    }
};
static void sim_fill(const void *base, uint32_t off, uint32_t to) {
    const char *b = (const char *)base;
    const bool of_x = b >= x_from && b < x_to;
    if (!of_x && !(b >= w_from && b < w_to)) stop("a load from outside of the operands", off);
    if (b + off + 16 > (of_x ? x_to : w_to)) stop("a load past the end of an operand", off);
    const long place = place_of(to);
    if (place < 0) stop("a load to outside of LDS", to);
    on_the_way.push_back({(int)place, fills[wave][place].size()});
    fills[wave][place].push_back({(int)((b - (of_x ? x_from : w_from)) / 128), barriers, -1, order++, -1, of_x});
}
static void sim_vm(size_t left) {                     // loads arrive in the order they were asked for
    while (on_the_way.size() > left) {
        Fill &f = fills[wave][on_the_way[0].first][on_the_way[0].second];
        f.landed = barriers, f.landed_order = order++;
        on_the_way.erase(on_the_way.begin());
    }
}
static void sim_lgkm0() {
    for (auto &u : unread) reads[wave][u.first][u.second].end = barriers;
    unread.clear();
}
static void sim_barrier() { barriers++; }

#define __device__
#define __forceinline__ inline
#define __shared__
#define __attribute__(x)
#define __builtin_amdgcn_readfirstlane(x) (x)
#define __builtin_amdgcn_s_setprio(x)
#define __builtin_amdgcn_sched_barrier(x)
#define __builtin_amdgcn_s_barrier() sim_barrier()
#define __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, d, e, f) (c)
#include "tiles_host.h"
#undef __attribute__

using namespace fllm_tiles;

static int faults, M, N, K, rows;
static void fault(const char *what, int place, const Fill &f, int reader, int other) {
    if (++faults <= 12)
        printf("%d rows a tile, M %d N %d K %d: place %d, step %d: %s (wave %d reads, wave %d loads)\n", rows, M, N, K, place, f.step, what, reader, other);
}

template <int EPI, int ROWS>
static void check(int m, int n, int k, int workgroups) {
    M = m, N = n, K = k, rows = ROWS;
    std::vector<bf16_t> x((size_t)M * K), w((size_t)(EPI == EPI_GLU ? 2 : 1) * N * K);
    std::vector<float> out((size_t)M * N);
    TileArgs a = {};
    a.x = x.data(), a.w = w.data(), a.out = out.data();
    a.ldx = K, a.ldo = N, a.M = M, a.N = N, a.K = K;
    x_from = (const char *)a.x, x_to = x_from + x.size() * 2, w_from = (const char *)a.w, w_to = w_from + w.size() * 2;
    gridDim.x = workgroups;
    const int T = K / 64, ring = ROWS == 256 ? 2 : 3;
    for (blockIdx.x = 0; (int)blockIdx.x < workgroups; blockIdx.x++) {
        int first = -1;
        for (wave = 0; wave < kWaves; wave++) {
            threadIdx.x = wave * kWave;
            for (int p = 0; p < kPlaces; p++) fills[wave][p].clear(), reads[wave][p].clear();
            on_the_way.clear(), unread.clear();
            barriers = 0, order = 0;
            if (ROWS == 256) tiles256<EPI, false>(a);
            else tiles128<EPI, false>(a);
            if (first >= 0 && barriers != first) stop("waves that pass other numbers of barriers", barriers);
            first = barriers;
            if (!on_the_way.empty() || !unread.empty()) stop("loads or reads never waited for", (long)on_the_way.size());
        }
        for (int p = 0; p < kPlaces; p++) {
            const size_t loads = fills[0][p].size();
            if (loads == 0) continue;
            const size_t pieces = fills[0][p][0].of_x ? 8 : 4;      // reads of a half tile by a wave
            for (size_t i = 0; i + 2 < loads; i += 2) {             // steps of a place: every second (third) one, then the next tile's first
                const int now = fills[0][p][i].step, next = fills[0][p][i + 2].step;
                if (next != (now + ring < T ? now + ring : now % ring)) fault("steps out of their order", p, fills[0][p][i], 0, 0);
            }
            for (int r = 0; r < kWaves; r++) {
                if (reads[r][p].size() != loads / 2 * pieces) stop("half tiles that are not read once", (long)reads[r][p].size());
                for (size_t i = 0; i < reads[r][p].size(); i++) {
                    const Read &read = reads[r][p][i];
                    const size_t at = i / pieces * 2;               // the two loads of this half tile by every wave
                    for (int o = 0; o < kWaves; o++) {
                        if (fills[o][p].size() != loads) stop("waves that load other numbers of pieces", (long)fills[o][p].size());
                        for (int j = 0; j < 2; j++) {
                            const Fill &f = fills[o][p][at + j];
                            if (f.step != fills[0][p][at].step) fault("waves that load other steps", p, f, r, o);
                            if (o == r ? f.landed_order > read.order : f.landed >= read.begin) fault("read before it has arrived", p, f, r, o);
                            if (at + 2 + j >= loads) continue;
                            const Fill &next = fills[o][p][at + 2 + j];
                            if (o == r ? next.order < read.order || next.asked < read.end : next.asked <= read.end) fault("asked for again before it is read", p, next, r, o);
                        }
                    }
                }
            }
        }
    }
}

int main() {
    for (int k : {256, 384, 512, 640, 1024}) {      // the shortest (no trip through the loop), one trip, more
        check<EPI_STORE, 256>(300, 264, k, 1);      // several tiles a workgroup
        check<EPI_STORE, 256>(200, 264, k, 2);      // one tile
        check<EPI_GLU, 256>(300, 264, k, 1);
        check<EPI_F32, 256>(300, 264, k, 1);
    }
    for (int k : {192, 256, 320, 384, 448, 512, 1024}) {
        check<EPI_STORE, 128>(300, 264, k, 1);
        check<EPI_STORE, 128>(100, 264, k, 2);
        check<EPI_GLU, 128>(300, 264, k, 1);
        check<EPI_F32, 128>(300, 264, k, 1);
    }
    if (faults) { printf("%d faults\n", faults); return 1; }
    printf("tiles ok\n");
    return 0;
}
