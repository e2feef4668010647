// Sweeps the launch plans of csrc/plans.h over shapes, on the host: every plan keeps LDS within a compute unit's, its
// counters within the counters' part of the workspace, cuts K into slices none of which is empty, and addresses
// partial results inside the bytes it said it needs (the buffers here have exactly that size, so that the address
// sanitizer sees a step outside them).  Built and run by tests/test_plans.py.
#include "plans.h"

#include <stdio.h>
#include <stdlib.h>
#include <vector>

using namespace fllm_plan;

static long checks = 0;
#define REQUIRE(cond, ...)                                   \
    do {                                                     \
        checks++;                                            \
        if (!(cond)) {                                       \
            fprintf(stderr, "FAILED %s: ", #cond);           \
            fprintf(stderr, __VA_ARGS__);                    \
            fprintf(stderr, "\n");                           \
            exit(1);                                         \
        }                                                    \
    } while (0)

static void slices_cover(int K, int S, int slice, const char *what) {
    REQUIRE(S >= 1 && slice > 0, "%s K=%d S=%d slice=%d", what, K, S, slice);
    REQUIRE((long)S * slice >= K, "%s: slices do not cover K=%d (S=%d slice=%d)", what, K, S, slice);
    REQUIRE((long)(S - 1) * slice < K, "%s: an empty slice at K=%d (S=%d slice=%d)", what, K, S, slice);
}

// A stretch of the workspace of exactly the floats a plan said it needs.  Small ones are real memory, so that the
// address sanitizer sees a step outside them; large ones (up to the 192 MiB of a workspace) are checked by arithmetic.
struct Stretch {
    size_t floats;
    std::vector<float> real;
    explicit Stretch(size_t n) : floats(n), real(n <= (1u << 18) ? n : 0) {}
};
// touches the first and last float that a (tile, slice) part of `floats` floats would use
static void touch(Stretch &buf, size_t offset, size_t floats) {
    REQUIRE(floats > 0 && offset + floats <= buf.floats, "a part at %zu + %zu lies outside the %zu floats planned", offset, floats, buf.floats);
    if (!buf.real.empty()) {
        buf.real[offset] = 1.f;
        buf.real[offset + floats - 1] = 1.f;
    }
}

int main() {
    const int Ks[] = {8, 72, 264, 1000, 1024, 2072, 4096, 8192, 14336, 30008, 65536};
    const int Ns[] = {16, 30, 1000, 4096, 5001, 28672, 128256, 262144};
    const size_t workspaces[] = {0, (size_t)1 << 20, (size_t)192 << 20};
    const int cus_list[] = {1, 256, 304};
    for (size_t ws_bytes : workspaces)
        for (int cus : cus_list)
            for (int K : Ks)
                for (int N : Ns) {
                    const bool have_ws = ws_bytes > 0;
                    // ---- up to 16 rows ----
                    for (int M : {1, 3, 8, 9, 16})
                        for (int rt = 1; rt <= 2; rt++)
                            for (int forced : {0, 1, 2, 4, 8})
                                for (int xd = 0; xd < 2; xd++) {
                                    const int nt = rt == 2 ? 8 : 16;
                                    const int ntiles = (int)ceil_div(rt == 2 ? N / 2 : N, nt);
                                    if (ntiles == 0) continue;
                                    ResidentPlan p = plan_resident(M, K, ntiles, rt, ws_bytes, have_ws, xd != 0, forced);
                                    if (p.S == 0) continue;      // declined: the caller says so
                                    if (xd) {
                                        slice_direct(p, M, K, ntiles, rt, ws_bytes, have_ws, cus, forced);
                                        REQUIRE(p.S == 1 || (p.S == 2 && forced != 1 && M > 8 && 2 * ntiles <= cus && p.stage == 0), "direct slices %d", p.S);
                                    }
                                    slices_cover(K, p.S, p.slice, "resident");
                                    REQUIRE(p.slice % 128 == 0, "resident slice %d", p.slice);
                                    REQUIRE(p.smem * p.per_cu <= kLdsBytes, "resident LDS %zu x %d", p.smem, p.per_cu);
                                    REQUIRE(p.stage + p.red + (size_t)p.waves * 16 * 4 <= p.smem, "resident LDS layout");
                                    REQUIRE(xd || p.stage >= (size_t)M * (p.slice + 8) * 2, "resident staging");
                                    const int groups = resident_groups(p, ntiles, cus);
                                    REQUIRE(groups >= 1 && groups <= ntiles, "resident groups %d of %d tiles", groups, ntiles);
                                    if (p.S > 1) {
                                        REQUIRE(have_ws && (size_t)ntiles * 4 <= kCounterBytes, "resident counters");
                                        const size_t need = resident_workspace_need(ntiles, p.S, rt);
                                        REQUIRE(need <= ws_bytes, "resident workspace %zu of %zu", need, ws_bytes);
                                        Stretch buf((need - kCounterBytes) / 4);
                                        const size_t ssq = resident_ssq_offset_floats(ntiles, p.S, rt);
                                        for (int tile : {0, ntiles - 1})
                                            for (int sl : {0, p.S - 1}) {
                                                touch(buf, ((size_t)(tile * p.S + sl) * rt * kWaveLanes) * 4, (size_t)rt * kWaveLanes * 4);
                                                touch(buf, ssq + (size_t)(tile * p.S + sl) * 16, 16);
                                            }
                                    }
                                }
                    // ---- 17 to 64 rows ----
                    for (int mt = 2; mt <= 4; mt++)
                        for (int rt = 1; rt <= 2; rt++)
                            for (int forced : {0, 1, 2, 4, 8, 14}) {
                                const int nt = rt == 2 ? 8 : 16;
                                const int ntiles = (int)ceil_div(rt == 2 ? N / 2 : N, nt);
                                if (ntiles == 0) continue;
                              for (int waves : {-1, 0, 4, 6, 7, 8}) {      // -1: without a copy
                                const ChunkPlan c = waves < 0 ? plan_chunks(K, ntiles, mt, rt, ws_bytes, have_ws, cus, forced, 4)
                                                              : plan_chunks_even(K, ntiles, mt, rt, ws_bytes, have_ws, cus, forced, waves);
                                REQUIRE(c.waves == 4 || (waves >= 0 && c.waves >= 6 && c.waves <= 8), "chunks waves %d", c.waves);
                                REQUIRE(waves <= 0 || c.waves == waves, "chunks waves %d forced %d", c.waves, waves);
                                if (waves == 0)
                                    REQUIRE(chunk_plan_cost(c, ntiles, cus) <=
                                                chunk_plan_cost(plan_chunks_balanced(K, ntiles, mt, rt, ws_bytes, have_ws, cus, forced, 0), ntiles, cus),
                                            "chunks: %d waves leave more than four, seven or eight", c.waves);
                                REQUIRE(c.grid / c.S <= (int)ceil_div(ntiles, c.waves), "chunks grid %d beyond the row groups", c.grid);
                                slices_cover(K, c.S, c.slice, "chunks");
                                REQUIRE(c.grid >= 1 && c.grid % c.S == 0, "chunks grid %d S %d", c.grid, c.S);
                                if (c.S > 1) {
                                    REQUIRE(have_ws && (size_t)ntiles * 4 <= kCounterBytes, "chunks counters");
                                    const size_t need = chunk_workspace_need(ntiles, c.S, mt, rt);
                                    REQUIRE(need <= ws_bytes, "chunks workspace");
                                    Stretch buf((need - kCounterBytes) / 4);
                                    for (int tile : {0, ntiles - 1})
                                        for (int sl : {0, c.S - 1})
                                            touch(buf, (((size_t)tile * c.S + sl) * mt) * rt * kWaveLanes * 4, (size_t)mt * rt * kWaveLanes * 4);
                                    REQUIRE(need - kCounterBytes <= 0x7fffffffu, "chunks workspace offsets");
                                }
                              }
                                for (int norm = 0; norm < 2; norm++) {
                                    const int M = mt * 16 - 3;
                                    const SlabPlan s = plan_slab(M, ntiles, K, mt, rt, norm != 0, nt, ws_bytes, have_ws, cus, forced);
                                    if (s.S == 0) continue;
                                    slices_cover(K, s.S, s.slice, "slab");
                                    REQUIRE(s.slice % 256 == 0 && (!norm || s.slice % 512 == 0) && s.slice <= 1024 + 0 * K, "slab slice %d", s.slice);
                                    REQUIRE(s.smem <= kLdsBytes, "slab LDS %zu", s.smem);
                                    REQUIRE(s.cells_off >= (size_t)mt * 16 * (s.slice + 8) * 2 && s.cells_off % 16 == 0, "slab staging");
                                    REQUIRE(!norm || s.smem >= s.cells_off + (size_t)mt * 16 * ((s.slice + 511) / 512) * 4, "slab cells");
                                    REQUIRE(s.grid >= 1 && s.grid % s.S == 0 && s.grid <= (cus > s.S ? cus : s.S), "slab grid %d S %d", s.grid, s.S);
                                    if (s.S > 1) {
                                        REQUIRE(have_ws && (size_t)ntiles * 4 <= kCounterBytes, "slab counters");
                                        const size_t need = slab_workspace_need(ntiles, s.S, mt, rt);
                                        REQUIRE(need <= ws_bytes && need - kCounterBytes <= 0x7fffffffu, "slab workspace");
                                        Stretch buf((need - kCounterBytes) / 4);
                                        const size_t ssq = slab_ssq_offset_floats(ntiles, s.S, mt, rt);
                                        for (int tile : {0, ntiles - 1})
                                            for (int sl : {0, s.S - 1}) {
                                                touch(buf, ((size_t)tile * s.S + sl) * mt * rt * kWaveLanes * 4, (size_t)mt * rt * kWaveLanes * 4);
                                                touch(buf, ssq + ((size_t)tile * s.S + sl) * mt * 16, (size_t)mt * 16);
                                            }
                                    }
                                }
                            }
                }
    // six waves where they leave the least: q/k/v of 6,144 x 4,096 in four slices; and not where seven do
    const ChunkPlan six = plan_chunks_even(4096, 384, 3, 1, (size_t)192 << 20, true, 256, 0, 0);
    REQUIRE(six.waves == 6 && six.S == 4 && six.grid == 256, "%d waves, %d slices, %d workgroups", six.waves, six.S, six.grid);
    REQUIRE(plan_chunks_even(4096, 1792, 3, 1, (size_t)192 << 20, true, 256, 0, 0).waves == 7, "1,792 tiles");
    // two slices of products of 9 to 16 rows: K beyond 4,096, tiles for half of the compute units at most
    for (auto &t : {std::vector<int>{9, 4104, 128, 2}, {16, 8192, 1, 2}, {16, 4096, 128, 1}, {8, 8192, 128, 1}, {16, 8192, 129, 1}}) {
        ResidentPlan p = plan_resident(t[0], t[1], t[2], 1, (size_t)192 << 20, true, true, 0);
        slice_direct(p, t[0], t[1], t[2], 1, (size_t)192 << 20, true, 256, 0);
        REQUIRE(p.S == t[3], "%d rows, %d tiles of %d: %d slices", t[0], t[2], t[1], p.S);
    }
    // 49 to 64 rows, tiles of 16: slices for one workgroup a compute unit where that is four of them, but for one tile over
    struct { int tiles, K, mt, rt; bool copy; int slices; } sums[] = {
        {256, 4096, 4, 1, false, 4}, {256, 4096, 4, 1, true, 4}, {256, 14336, 4, 1, true, 4}, {256, 16384, 4, 1, true, 8}, {256, 16384, 4, 1, false, 4},
        {130, 8192, 4, 1, false, 4}, {129, 8192, 4, 1, false, 8}, {129, 8192, 4, 1, true, 8}, {128, 8192, 4, 1, false, 8}, {257, 4096, 4, 1, false, 4},
        {257, 2048, 4, 1, false, 4}, {256, 4096, 4, 2, false, 8}, {256, 4096, 3, 1, false, 4}, {129, 8192, 3, 1, false, 4}};
    for (auto &t : sums) {
        const ChunkPlan c = plan_chunks(t.K, t.tiles, t.mt, t.rt, (size_t)192 << 20, true, 256, 0, 4, t.copy);
        REQUIRE(c.S == t.slices, "%d tiles of %d, %d row tiles, copy %d: %d slices", t.tiles, t.K, t.mt, t.copy, c.S);
    }
    // ---- products of many rows on tiles ----
    // What a tile walks: 256 rows steps 0 1 .. in pairs, the last four apart, 128 rows the last three apart; a K that is not taken
    // would be cut short or read past its end, also where a caller asks for the tile.
    for (int K = 1; K <= 1024; K++)
        for (int asked : {0, 1, 2, 64, 128, 192, 256, 512, -1})
            for (long rows : {1, 129, 300, 4096}) {
                const int bm = row_tile((rows + 255) / 256 * 40, (rows + 127) / 128 * 40, K, asked);
                REQUIRE(bm == 0 || bm == 128 || bm == 256, "row tile %d", bm);
                REQUIRE(bm != 256 || (K % 128 == 0 && K / 64 >= 4), "256 rows at K %d (asked %d)", K, asked);
                REQUIRE(bm != 128 || (K % 64 == 0 && K / 64 >= 3), "128 rows at K %d (asked %d)", K, asked);
                REQUIRE(asked == 0 || asked == 1 || bm == 0 || bm == asked, "asked for %d, got %d", asked, bm);
                if (asked == 0 || asked == 1) REQUIRE((bm != 0) == (K % 64 == 0 && K >= 192), "K %d declined", K);
            }
    // An activation joins its product where both were measured and the tiles were ahead, and stays apart where they were behind
    // (16,384 columns, 1,030 rows: library 82 us, tiles 89 whole and 80 with the last round in halves, as they are planned).
    struct { int columns, K; long rows; bool joins; } measured[] = {
        {28672, 4096, 65, false}, {28672, 4096, 128, false}, {28672, 4096, 160, false}, {28672, 4096, 320, false},
        {28672, 4096, 513, false}, {28672, 4096, 420, true}, {28672, 4096, 512, true}, {28672, 4096, 900, true},
        {28672, 4096, 2048, true}, {16384, 2048, 65, false}, {16384, 2048, 192, false}, {16384, 2048, 256, false},
        {16384, 2048, 513, false}, {16384, 2048, 1030, true}, {16384, 2048, 1280, true}, {16384, 2048, 420, true}, {16384, 2048, 512, true},
        {16384, 2048, 2048, true}, {17920, 1536, 65, false}, {17920, 1536, 128, false}, {17920, 1536, 192, true},
        {17920, 1536, 320, true}, {17920, 1536, 2048, true}, {13312, 1536, 65, false}, {13312, 1536, 128, false},
        {13312, 1536, 320, true}, {13312, 1536, 2048, true}, {4480, 1536, 128, false}, {4480, 1536, 512, false},
        {4480, 1536, 900, true}, {8192, 1024, 65, true}, {8192, 1024, 2048, true}, {57344, 8192, 128, true},
        {28672, 4096, 640, false}, {28672, 4096, 645, true}, {28672, 4096, 700, true}, {16384, 4096, 1085, false}, {16384, 4096, 1120, false},
        {16384, 4096, 2304, true}, {24576, 4096, 768, true}, {12288, 4096, 1536, true}, {57344, 8192, 800, true}};
    for (auto &m : measured) {
        const long cols = (m.columns + 255) / 256;
        const TilePlan p = tile_plan((m.rows + 255) / 256 * cols, (m.rows + 127) / 128 * cols, m.K, 0, 1);
        REQUIRE(activation_joins(m.rows, m.columns, m.K, p) == m.joins, "%d columns of %d, %ld rows", m.columns, m.K, m.rows);
    }
    // A plain product leaves the library where the tiles were measured ahead, and stays where they were behind.
    struct { int columns, K; long rows; bool tiles; } plain[] = {
        {16384, 2048, 1536, true}, {16384, 2048, 1500, true}, {24576, 4096, 1024, true}, {8192, 8192, 3072, true}, {57344, 8192, 1280, true},
        {6144, 4096, 4096, true}, {6144, 4096, 2560, true}, {4096, 14336, 2048, true}, {6144, 4096, 2048, false}, {16384, 2048, 1100, false}, {16384, 2048, 1280, false},
        {16384, 2048, 2304, false}, {16384, 4096, 2304, false}, {28672, 4096, 513, false}, {24576, 4096, 513, true} /* 128-row tiles */, {24576, 4096, 768, false},
        {10240, 8192, 1537, false}, {10240, 8192, 2048, false}, {13824, 5120, 2560, false}, {28672, 1536, 2304, false}};
    for (auto &m : plain) {
        const long cols = (m.columns + 255) / 256;
        const TilePlan p = tile_plan((m.rows + 255) / 256 * cols, (m.rows + 127) / 128 * cols, m.K, 0, 1);
        REQUIRE(plain_takes_tiles(m.rows, m.columns, m.K, p) == m.tiles, "%d columns of %d, %ld rows", m.columns, m.K, m.rows);
    }
    // experts' row tiles where both were measured: experts x inner width x width, tokens that pick two
    struct { int experts, inter, width, tokens, rows; } grouped[] = {
        {4, 1024, 1024, 512, 128}, {4, 1024, 1024, 1024, 128}, {4, 1024, 1024, 1500, 128}, {8, 2048, 1024, 512, 128}, {4, 1024, 1024, 2048, 256},
        {8, 2048, 1024, 1024, 256}, {8, 4480, 1536, 1900, 256}, {16, 1408, 2048, 1024, 256}, {16, 1408, 2048, 512, 128}, {8, 7168, 2048, 1900, 256}};
    for (auto &m : grouped) {
        const int got = grouped_row_tile(2L * m.tokens, m.experts, (m.inter + 127) / 128, (m.width + 255) / 256, m.width, m.inter, 1);
        REQUIRE(got == m.rows, "%d experts of %d x %d, %d tokens: tiles of %d rows", m.experts, m.inter, m.width, m.tokens, got);
    }
    // ---- decode attention ----
    for (int head_dim : {32, 64, 128}) {      // a wave's 64 keys; one row of one head group, and the part that tips the choice
        const int unit = decode_unit(head_dim), last = 16 * unit - 31;
        REQUIRE(unit == decode_waves(head_dim) * 64, "unit %d", unit);
        int splits = 0, per = 0;
        decode_split_plan(1, 1, 1, last, unit, true, &splits, &per);
        REQUIRE(splits == 16 && per == unit, "%d parts of %d", splits, per);
        decode_split_plan(1, 1, 1, last + 1, unit, true, &splits, &per);
        REQUIRE(splits == 9 && per == 2 * unit, "%d parts of %d", splits, per);
    }
    for (int rows : {1, 2, 8, 24, 64, 256})
        for (int kv_heads : {1, 2, 8, 64})
            for (int group : {1, 4, 7, 16, 40})
                for (int head_dim : {32, 64, 128})
                    // around sixteen and thirty-two parts of one round (256 and 512 keys)
                    for (int context : {1, 31, 256, 1000, 4065, 4066, 4096, 8161, 8162, 16353, 16354, 40000, 131072})
                        for (int fused = 0; fused < 2; fused++) {
                            const int qtiles = (group + 15) / 16, unit = decode_unit(head_dim);
                            int splits = 0, per = 0;
                            decode_split_plan(rows, kv_heads, qtiles, context, unit, fused != 0, &splits, &per);
                            const long span = (long)context + 31;
                            REQUIRE(splits >= 1 && splits <= 64 && per % unit == 0, "decode splits %d per %d", splits, per);
                            REQUIRE((long)splits * per >= span && (long)(splits - 1) * per < span, "decode: %d splits of %d keys for %d", splits, per, context);
                            REQUIRE(!fused || per > unit || splits <= 16, "decode: %d parts of one round, the merge reads sixteen a trip", splits);
                            REQUIRE(decode_lds_bytes(head_dim, group) + 1024 <= kLdsBytes, "decode LDS");
                            const size_t need = decode_workspace_need(rows, kv_heads * group, head_dim, splits);
                            if (splits > 1) {
                                Stretch buf(need / 4);
                                const size_t heads = (size_t)kv_heads * group, ml = (size_t)rows * heads * splits * 2;
                                touch(buf, 0, 2);
                                touch(buf, (((size_t)rows - 1) * heads + heads - 1) * splits * 2 + (splits - 1) * 2, 2);
                                touch(buf, ml + ((((size_t)rows - 1) * heads + heads - 1) * splits + splits - 1) * head_dim, head_dim);
                            } else {
                                REQUIRE(need == 0, "decode workspace of an unsplit step");
                            }
                        }
    // ---- prompt attention ----
    for (int tiles : {1, 3, 17, 64, 513, 20000})
        for (int kv_heads : {1, 8})
            for (int context : {64, 1000, 2048, 30000, 131072})
                for (int window : {0, 512})
                    for (size_t room : {(size_t)0, (size_t)40, (size_t)4096, (size_t)1 << 20})
                        for (int slots : {2, 512})
                            for (int by_hand : {0, 1, 3, 40})
                            for (int rows : {1, context / 2, context, 4 * context}) {
                                int max_parts = -1;
                                const int per_part = prefill_part_plan(tiles, kv_heads, rows, context, window, room, slots, by_hand, &max_parts);
                                REQUIRE(max_parts >= 1 && max_parts <= 16, "parts %d", max_parts);
                                if (per_part == 0) {
                                    REQUIRE(max_parts == 1, "an unshared row tile has one part");
                                    continue;
                                }
                                const long most_tiles = ((long)context + 63) / 64, groups = (long)tiles * kv_heads;
                                REQUIRE(window == 0 && groups * 4 <= (long)kCounterBytes, "shared row tiles need counters");
                                REQUIRE((long)max_parts * per_part >= most_tiles && (long)(max_parts - 1) * per_part < most_tiles,
                                        "parts %d of %d key tiles for %ld", max_parts, per_part, most_tiles);
                                REQUIRE((size_t)groups * max_parts <= room, "parts %ld x %d in room %zu", groups, max_parts, room);
                            }
    // which steps are one prompt's: heads 32 on 8 (row tiles of 32 rows) and 12 on 2 (of 21), 512 slots
    struct { int longest, more, singles, group, kv_heads; bool one; } steps[] = {
        {1900, 0, 0, 4, 8, true},     {1900, 40, 0, 4, 8, true},    {1900, 0, 4, 4, 8, true},      {1500, 500, 0, 4, 8, true},
        {1450, 550, 0, 4, 8, false},  {1024, 1024, 0, 4, 8, false}, {1900, 0, 32, 4, 8, true},     {1900, 0, 40, 4, 8, false},
        {1900, 0, 100, 4, 8, false},  {1900, 0, 64, 6, 2, true},    {1900, 0, 160, 6, 2, true},    {300, 0, 100, 4, 8, true},
        {131072, 0, 0, 4, 8, true},   {1 << 30, 1 << 30, 0, 4, 8, false}};
    for (const auto &t : steps) {
        const int segs = 1 + (t.more > 0) + t.singles, rows = (int)((unsigned)t.longest + t.more - (t.more == 1 << 30 ? 1 : 0)) + t.singles;
        const int tiles = rows / (128 / t.group) + 1 + segs;
        const int got = rows_of_one_prompt(tiles, rows, segs, t.kv_heads, t.longest, 512);
        REQUIRE(got == (t.one ? rows : 0), "%d + %d rows and %d single ones: %d", t.longest, t.more, t.singles, got);
        // a step that is not one prompt's is planned by its slots alone
        int parts = 0, plain = 0;
        const int a = prefill_part_plan(tiles, t.kv_heads, got, t.longest, 0, (size_t)1 << 20, 512, 0, &parts);
        const int b = prefill_part_plan(tiles, t.kv_heads, t.one ? rows : 1, t.longest, 0, (size_t)1 << 20, 512, 0, &plain);
        REQUIRE(a == b && parts == plain, "parts of %d + %d rows and %d single ones", t.longest, t.more, t.singles);
    }
    printf("plans ok: %ld checks\n", checks);
    return 0;
}
