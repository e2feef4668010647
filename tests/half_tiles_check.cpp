// The order of tiles in a launch of 256-row tiles whose last round runs as halves (csrc/gemm_tiles.h: Place), on the host: every output is
// made once, whichever workgroup makes it, on its own rows or in rows grouped by expert, and no workgroup takes two halves.
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>

#include <algorithm>
#include <vector>

#include "plans.h"

using std::min;
struct bf16_t { uint16_t bits; };
#define __device__
#define __forceinline__ inline
#define __builtin_amdgcn_readfirstlane(x) (x)
enum { EPI_STORE = 0, EPI_GLU = 1 };
struct TileArgs {
    const bf16_t *w;
    int ldx, M, N, K, halves, max_tiles, top;
    const int32_t *work;
};
static int tile_column_unused;
template <int EPI> int tile_column(int, int) { return tile_column_unused; }
#include "place_host.h"

#define REQUIRE(c, ...) do { if (!(c)) { printf(__VA_ARGS__); printf(" (%s)\n", #c); exit(1); } } while (0)

template <int EPI, bool GROUPED> static void check(const std::vector<int> &experts, int N) {
    const int cols = EPI == EPI_GLU ? 128 : 256;
    std::vector<int32_t> work(1);
    int M = 0;
    for (size_t e = 0; e < experts.size(); M += experts[e], e++)
        for (int r = 0; GROUPED && r < experts[e]; r += 256) work.insert(work.end(), {(int)e, M + r, min(256, experts[e] - r)}), work[0]++;
    TileArgs a = {};
    a.M = M, a.N = N, a.K = 256, a.halves = 1, a.work = work.data(), a.max_tiles = work[0];
    const int columns = (N + cols - 1) / cols;
    std::vector<int> made((size_t)M * columns);
    auto take = [&](int m0, int n0, int rows, int most) {
        REQUIRE(n0 % cols == 0 && n0 < N && m0 >= 0 && rows > 0, "tile at %d, %d of %d rows", m0, n0, rows);
        for (int m = m0; m < m0 + min(rows, most) && (GROUPED || m < M); m++) {
            REQUIRE(m < M, "row %d of %d", m, M);
            made[(size_t)m * columns + n0 / cols]++;
        }
    };
    Place<EPI, GROUPED, 256> whole(a);
    const int halves = whole.in_halves(a);
    REQUIRE(halves <= 128 && (whole.total - halves) % 256 == 0 || halves == 0, "%d of %d tiles in halves", halves, whole.total);
    REQUIRE((halves != 0) == fllm_plan::last_round_in_halves(whole.total), "the plan takes %d tiles otherwise", whole.total);
    for (int block = 0; block < 256; block++) {
        for (int id = block; id < whole.total - halves; id += 256) {
            whole.go(a, id);
            take(whole.m0, whole.n0, whole.rows, 256);
        }
        if (block >= (halves + 7) / 8 * 16 || block / 16 * 8 + block % 8 >= halves) continue;
        Place<EPI, GROUPED, 128, true> half(a);
        half.go(a, block);
        if (half.rows > 0) take(half.m0, half.n0, half.rows, 128);
    }
    for (size_t i = 0; i < made.size(); i++) REQUIRE(made[i] == 1, "M %d N %d: row %zu, columns %zu made %d times", M, N, i / columns, i % columns, made[i]);
}

int main() {
    for (int M : {1, 128, 129, 256, 257, 300, 385, 1900, 2048, 2049, 2305})
        for (int N : {8, 264, 1536, 4096, 6144, 8960, 14336}) check<EPI_STORE, false>({M}, N), check<EPI_GLU, false>({M}, N);
    for (int N : {128, 1536, 4480, 8960})
        for (auto &e : std::vector<std::vector<int>>{{0, 1, 700, 128}, {500, 480, 470, 512, 475, 460, 490, 413}, {2000}, {129, 127, 256, 257, 0, 3}})
            check<EPI_STORE, true>(e, N), check<EPI_GLU, true>(e, N);
    // the plan: halves only where they take less time, or wherever they can be where that is asked for
    for (long t256 = 1; t256 < 1500; t256++)
        for (long t128 : {2 * t256, 2 * t256 - 1, t256})
            for (int K : {64, 192, 256, 1536})
                for (int asked : {0, 1, 128, 256, 192})
                    for (int halves : {0, 1, 2}) {
                        const auto p = fllm_plan::tile_plan(t256, t128, K, asked, halves);
                        const int bm = fllm_plan::row_tile(t256, t128, K, asked);
                        REQUIRE((p.bm == 0) == (bm == 0), "%ld tiles", t256);
                        REQUIRE(p.halves || p.bm == bm, "%ld tiles", t256);
                        if (!p.halves) continue;
                        REQUIRE(halves && p.bm == 256 && p.tiles == t256 && K % 128 == 0 && asked != 128, "%ld tiles", t256);
                        const double without = bm == 256 ? (t256 + 255) / 256 : fllm_plan::kShortRound * ((t128 + 255) / 256);
                        REQUIRE(halves == 2 || p.rounds < without, "%ld tiles: %f rounds, %f without", t256, p.rounds, without);
                    }
    printf("half tiles ok\n");
    return 0;
}
