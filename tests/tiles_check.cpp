// The tile products of csrc/gemm_tiles.h as a host program (tests/test_tile_schedule.py puts the calls below in the place of the header's
// inline assembly).  One lane of each of the eight waves walks through the kernel, and every load into LDS, every wait and every read
// of LDS is noted with the number of barriers that its wave has passed.  All barriers are the workgroup's: events of two waves are in order where that number
// differs, and may fall in either order where it is the same.  Checked for every read of a half tile:
//   1. every wave had waited for the pieces that it loads, before an earlier barrier (the reading wave's own: before the read);
//   2. no wave asks for the half tile that comes to the same place next before a barrier behind the end of the read;
// and that steps come in their order, all that is asked for is read, and no load leaves the operands.
// A workgroup that goes on from tiles of 256 rows to one of 128 (the halves of a last round) is one walk: its places are the same, and what the
// second part asks for first lies behind the first part's last reads.  Slices of K walk their own steps; where they meet, LDS is written only when
// every wave has read its last half tile, and parts lie inside what the plan says they need.
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
    f32x4_t operator+(const f32x4_t &) const { return *this; }
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

// ---- what slices meet through: only what touches LDS or has an address is looked at
typedef int __amdgpu_buffer_rsrc_t;
static unsigned int parts_bytes;
static int counted_at;                                // barriers that the first thread had passed when it wrote the count to LDS
static bool comes_last;
static __amdgpu_buffer_rsrc_t workspace_buffer(float *) { return 0; }
static void sim_part(unsigned int at) { if (at % 16 != 0 || at + 16 > parts_bytes) stop("a part outside of the workspace", at); }
static void hand_over(__amdgpu_buffer_rsrc_t, unsigned int at, f32x4_t) { sim_part(at); }
static f32x4_t take_over(__amdgpu_buffer_rsrc_t, unsigned int at) { sim_part(at); return f32x4_t(); }
static int published_at;                              // the most barriers that a wave had passed when its parts were on their way to memory
static void parts_published() { sim_vm(0), published_at = max(published_at, barriers); }
static void parts_visible() {}
static int sim_count(int slices) {
    counted_at = barriers;
    return comes_last ? slices - 1 : 0;
}
#define __hip_atomic_fetch_add(p, v, order, scope) sim_count(a.slices)
#define __hip_atomic_store(p, v, order, scope) (*(p) = (v))
#define __HIP_MEMORY_SCOPE_AGENT 0
#define __syncthreads() sim_barrier()

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

enum Form { WHOLE256, WHOLE128, THEN_HALVES, SLICED };

// one part of a walk: its fills and reads of a place are those from `fill` and `read` on, up to the next part's
struct Part {
    int ring, from, to;                               // steps [from, to)
    size_t fill[kPlaces], read[kPlaces];
    void begins(int w) {
        for (int p = 0; p < kPlaces; p++) fill[p] = fills[w][p].size(), read[p] = reads[w][p].size();
    }
};

static void check_part(const Part &part, const Part *next_part) {
    for (int p = 0; p < kPlaces; p++) {
        const size_t f0 = part.fill[p], r0 = part.read[p], f1 = next_part ? next_part->fill[p] : fills[0][p].size();
        const size_t loads = f1 - f0;
        if (loads == 0) continue;
        const size_t pieces = fills[0][p][f0].of_x ? 8 : 4;         // reads of a half tile by a wave
        for (size_t i = f0; i + 2 < f1; i += 2) {                   // steps of a place: every second (third) one, then the next tile's first
            const int now = fills[0][p][i].step - part.from, next = fills[0][p][i + 2].step - part.from;
            if (next != (now + part.ring < part.to - part.from ? now + part.ring : now % part.ring)) fault("steps out of their order", p, fills[0][p][i], 0, 0);
        }
        for (int r = 0; r < kWaves; r++) {
            const size_t r1 = next_part ? next_part->read[p] : reads[r][p].size();
            if (r1 - r0 != loads / 2 * pieces) stop("half tiles that are not read once", (long)(r1 - r0));
            for (size_t i = r0; i < r1; i++) {
                const Read &read = reads[r][p][i];
                const size_t at = f0 + (i - r0) / pieces * 2;       // the two loads of this half tile by every wave
                for (int o = 0; o < kWaves; o++) {
                    if (fills[o][p].size() != fills[0][p].size()) stop("waves that load other numbers of pieces", (long)fills[o][p].size());
                    for (int j = 0; j < 2; j++) {
                        const Fill &f = fills[o][p][at + j];
                        if (f.step != fills[0][p][at].step) fault("waves that load other steps", p, f, r, o);
                        if (o == r ? f.landed_order > read.order : f.landed >= read.begin) fault("read before it has arrived", p, f, r, o);
                        if (at + 2 + j >= fills[o][p].size()) continue;
                        const Fill &next = fills[o][p][at + 2 + j];         // the next part's first among them
                        if (o == r ? next.order < read.order || next.asked < read.end : next.asked <= read.end) fault("asked for again before it is read", p, next, r, o);
                    }
                }
            }
        }
    }
}

template <int EPI, int FORM>
static void check(int m, int n, int k, int workgroups, int slices = 1, int walked = 0) {
    M = m, N = n, K = k, rows = FORM == WHOLE256 || FORM == THEN_HALVES ? 256 : 128;
    std::vector<bf16_t> x((size_t)M * K), w((size_t)(EPI == EPI_GLU ? 2 : 1) * N * K);
    std::vector<float> out((size_t)M * N);
    const int tiles = (M + rows - 1) / rows * ((N + (EPI == EPI_GLU ? 127 : 255)) / (EPI == EPI_GLU ? 128 : 256));
    std::vector<int> counters(tiles);
    TileArgs a = {};
    a.x = x.data(), a.w = w.data(), a.out = out.data();
    a.ldx = K, a.ldo = N, a.M = M, a.N = N, a.K = K;
    a.halves = FORM == THEN_HALVES, a.slices = slices, a.counters = counters.data();
    parts_bytes = (unsigned int)tiles * slices * 128 * 256 * 4;
    x_from = (const char *)a.x, x_to = x_from + x.size() * 2, w_from = (const char *)a.w, w_to = w_from + w.size() * 2;
    gridDim.x = workgroups;
    const int T = K / 64;
    int both = 0;
    for (blockIdx.x = 0; (int)blockIdx.x < (walked ? walked : workgroups); blockIdx.x++) {
        const int slice = blockIdx.x / tiles;
        Part parts[2];
        parts[0].ring = rows == 256 ? 2 : 3, parts[1].ring = 3;
        parts[0].from = parts[1].from = FORM == SLICED ? T * slice / slices : 0;
        parts[0].to = parts[1].to = FORM == SLICED ? T * (slice + 1) / slices : T;
        comes_last = slice == slices / 2, published_at = 0;
        int first = -1;
        for (wave = 0; wave < kWaves; wave++) {
            threadIdx.x = wave * kWave;
            for (int p = 0; p < kPlaces; p++) fills[wave][p].clear(), reads[wave][p].clear();
            on_the_way.clear(), unread.clear();
            barriers = 0, order = 0;
            parts[0].begins(wave);
            if constexpr (FORM == WHOLE256 || FORM == THEN_HALVES) tiles256<EPI, false>(a);
            if constexpr (FORM == WHOLE128) tiles128<EPI, false>(a);
            if constexpr (FORM == SLICED) tiles128<EPI, false, false, true>(a);
            if (!on_the_way.empty() || !unread.empty()) stop("loads or reads never waited for", (long)on_the_way.size());
            const Part before = parts[1];
            parts[1].begins(wave);
            for (int p = 0; wave > 0 && FORM == THEN_HALVES && p < kPlaces; p++)
                if (parts[1].fill[p] != before.fill[p] || parts[1].read[p] != before.read[p]) stop("waves whose parts end elsewhere", p);
            if constexpr (FORM == THEN_HALVES) tiles128<EPI, false, true>(a);
            if (first >= 0 && barriers != first) stop("waves that pass other numbers of barriers", barriers);
            first = barriers;
            if (!on_the_way.empty() || !unread.empty()) stop("loads or reads never waited for", (long)on_the_way.size());
        }
        check_part(parts[0], FORM == THEN_HALVES ? &parts[1] : nullptr);
        if (FORM == THEN_HALVES) {
            check_part(parts[1], nullptr);
            both += parts[1].fill[0] > 0 && fills[0][0].size() > parts[1].fill[0];
        }
        if (FORM == SLICED && published_at >= counted_at) stop("a tile counted before all waves' parts are there", counted_at);
        if (FORM == SLICED)                           // the count is written over the first place
            for (int r = 0; r < kWaves; r++)
                for (const Read &read : reads[r][0])
                    if (read.end >= counted_at) fault("the count is written before it is read", 0, fills[r][0].back(), r, 0);
    }
    if (FORM == THEN_HALVES && walked && both == 0) stop("no workgroup that takes a whole tile and a half one", both);
}

int main() {
    for (int k : {256, 384, 512, 640, 1024}) {      // the shortest (no trip through the loop), one trip, more
        check<EPI_STORE, WHOLE256>(300, 264, k, 1);      // several tiles a workgroup
        check<EPI_STORE, WHOLE256>(200, 264, k, 2);      // one tile
        check<EPI_GLU, WHOLE256>(300, 264, k, 1);
        check<EPI_F32, WHOLE256>(300, 264, k, 1);
    }
    for (int k : {192, 256, 320, 384, 448, 512, 1024}) {
        check<EPI_STORE, WHOLE128>(300, 264, k, 1);
        check<EPI_STORE, WHOLE128>(100, 264, k, 2);
        check<EPI_GLU, WHOLE128>(300, 264, k, 1);
        check<EPI_F32, WHOLE128>(300, 264, k, 1);
    }
    for (int k : {256, 384, 512, 640}) {             // two row tiles (the last one's second half has no rows), 260 tiles: four of them in halves
        check<EPI_STORE, THEN_HALVES>(300, 130 * 256, k, 256, 1, 18);
        check<EPI_GLU, THEN_HALVES>(400, 130 * 128, k, 256, 1, 18);
        check<EPI_F32, THEN_HALVES>(1000, 129 * 256 / 2, k, 256, 1, 18);
        check<EPI_RELU2, THEN_HALVES>(300, 264, k, 256, 1, 0);      // halves alone
    }
    for (int slices : {2, 3, 5, 8})
        for (int k : {3 * 64, 4 * 64, 5 * 64 + 32, 7 * 64}) {       // steps a slice at least, some with one more
            const int steps = k * slices / 64;
            check<EPI_STORE, SLICED>(300, 264, steps * 64, 6 * slices, slices);
            check<EPI_F32, SLICED>(100, 264, steps * 64, 2 * slices, slices);
        }
    if (faults) { printf("%d faults\n", faults); return 1; }
    printf("tiles ok\n");
    return 0;
}
