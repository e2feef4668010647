// How the kernels that meet across workgroups are launched: K slices, grid sizes, LDS bytes, where partial results
// lie in the device workspace.  Plain C++ without a device type in it, so that the same code that the launchers run
// is also compiled for the host alone and swept over shapes under the address and undefined-behaviour sanitizers
// (a mistake here is an access outside LDS or outside the workspace on the device).
#pragma once
#include <stddef.h>
#include <stdint.h>

namespace fllm_plan {

constexpr size_t kLdsBytes = 160 * 1024;            // LDS of a compute unit
constexpr size_t kCounterBytes = 64 * 1024;         // the counters at the start of the device workspace
constexpr int kWaveLanes = 64;
constexpr size_t kBf16 = 2, kF32 = 4, kF32x4 = 16;

inline long ceil_div(long a, long b) { return (a + b - 1) / b; }

// ---- products of up to 16 rows: activations of a K slice resident in LDS, waves split the slice ----
struct ResidentPlan {
    int S = 0, slice = 0, waves = 8, per_cu = 0;      // S == 0: no plan
    size_t stage = 0, red = 0, smem = 0;
};
constexpr int kMaxSlices = 32;

// bytes of the workspace that S slices of `ntiles` tiles need, counters included: partial sums [tile][slice][rt][64][4]
// and sums of squares [tile][slice][16]
inline size_t resident_workspace_need(int ntiles, int S, int rt) {
    return kCounterBytes + (size_t)ntiles * S * ((size_t)rt * kWaveLanes * 4 + 16) * kF32;
}
inline size_t resident_ssq_offset_floats(int ntiles, int S, int rt) { return (size_t)ntiles * S * rt * kWaveLanes * 4; }

// The fewest K slices whose activations fit into LDS (slicing costs more than it gains wherever it is not needed):
// twice into a compute unit's as two workgroups of 8 waves, else once as one workgroup of 16 waves, so that as
// many loads are in flight.  `forced`: 0, or the number of slices asked for by hand.
inline ResidentPlan plan_resident(int M, int K, int ntiles, int rt, size_t ws_bytes, bool have_ws, bool x_direct, int forced) {
    ResidentPlan best;
    if (x_direct) {   // nothing is staged: one slice, two workgroups of 8 waves a compute unit
        best.S = 1;
        best.slice = (K + 127) / 128 * 128;
        best.waves = 8;
        best.per_cu = 2;
        best.stage = 0;
        best.red = 8 * kWaveLanes * kF32x4;
        best.smem = best.red + 8 * 16 * kF32;
        return best;
    }
    for (int S = 1; S <= kMaxSlices; S *= 2) {
        const int slice = ((K + S - 1) / S + 127) / 128 * 128;
        if (S > 1 && (slice < 1024 || (long)(S - 1) * slice >= K)) break;
        if (S > 1) {
            if (!have_ws || resident_workspace_need(ntiles, S, rt) > ws_bytes || (size_t)ntiles * sizeof(int) > kCounterBytes) break;
        }
        ResidentPlan p;
        p.S = S;
        p.slice = slice;
        p.stage = ((size_t)M * (slice + 8) * kBf16 + 15) / 16 * 16;
        const size_t small = p.stage + 8 * (kWaveLanes * kF32x4 + 16 * kF32);
        const size_t large = p.stage + 16 * (kWaveLanes * kF32x4 + 16 * kF32);
        if (small <= 76 * 1024) p.waves = 8, p.per_cu = 2, p.smem = small;
        else if (large <= kLdsBytes) p.waves = 16, p.per_cu = 1, p.smem = large;
        else continue;
        p.red = (size_t)p.waves * kWaveLanes * kF32x4;
        if (forced == 0 || S == forced || best.S == 0) best = p;
        if (forced == 0 || S == forced) break;
    }
    return best;
}

// Nine to sixteen rows read where they lie, tiles for no more than half of the compute units and long K (up to eight rows there are 8-row tiles): K in
// two slices, whose workgroups fill the device.  What it costs is the tile's way through memory, about 1 us.  Microseconds at 9 / 16 rows whole ->
// sliced: 2,048 x 8,192 11.8 -> 10.2 / 14.7 -> 11.3, 1,536 x 13,312 17.6 -> 12.8 / 21.7 -> 14.8, 1,536 x 4,480 8.0 -> 7.6 / 9.8 -> 8.4, 2,048 x 4,224 7.9 -> 7.7 /
// 9.5 -> 8.5, 768 x 8,192 11.1 -> 8.6 / 13.6 -> 10.0; not so 1,024 x 4,096 6.9 -> 7.4 / 8.6 -> 8.1 and 2,048 x 2,048 5.5 -> 6.8 / 6.1 -> 7.1.  Four slices were
// slower than two (2,048 x 8,192 at 16 rows 12.5 where two took 11.4).  Over 16 to 2,048 columns of K 4,104 to 28,672, with a copy and without, stored
// and added, at 9 and 16 rows: 0.56 to 0.96 of the time whole (220 products; 16 x 28,672 the most).  `forced`: 1 keeps K whole, others leave the choice here.
inline void slice_direct(ResidentPlan &p, int M, int K, int ntiles, int rt, size_t ws_bytes, bool have_ws, int cus, int forced) {
    if (forced == 1 || M <= 8 || K <= 4096 || 2 * ntiles > cus) return;
    if (!have_ws || resident_workspace_need(ntiles, 2, rt) > ws_bytes || (size_t)ntiles * sizeof(int) > kCounterBytes) return;
    p.S = 2;
    p.slice = (K + 255) / 256 * 128;
}
// The most tiles that one compute unit has where `groups` workgroups take `ntiles` in turn and workgroups i and i + cus meet on one unit:
// the first unit's, since a workgroup has no more tiles than the ones before it
inline int busiest_unit(int ntiles, int groups, int cus) {
    return (ntiles + groups - 1) / groups + (groups > cus ? (ntiles - cus + groups - 1) / groups : 0);
}
// workgroups of a resident launch: one per slot of the device and slice, no more than there are tiles
inline int resident_groups(const ResidentPlan &p, int ntiles, int cus) {
    int groups = cus * p.per_cu / p.S;
    if (groups < 1) groups = 1;
    if (groups > ntiles) groups = ntiles;
    const int most = groups;
    // no more workgroups than give every one the same number of tiles: 1,792 tiles on 512 slots are 448 workgroups of 4
    // tiles, not 256 of 4 beside 256 of 3 that wait for them (gate/up of the 8B sizes at 8 rows: 40.2 -> 39.6 us)
    const int rounds = (ntiles + groups - 1) / groups;
    groups = (ntiles + rounds - 1) / rounds;
    // Two workgroups a compute unit: where that gives some units two such workgroups and others one, as many more as take more than an eighth
    // off what the busiest unit streams (to three tiles from four, to five from six).  1,120 tiles are 432 workgroups of 3 and 2 tiles,
    // where 374 of 3 left 138 units half of what the others had; all 512 slots were slower than the fewest that do.  Microseconds at one and
    // eight rows, by gate/up tiles and K: 1,120 of 1,536 14.7 -> 13.3 and 17.3 -> 15.9, of 4,096 29.0 -> 27.3 and 32.0 -> 29.5; 600 of 2,048
    // 11.9 -> 10.8 and 14.9 -> 13.3; 1,280 of 1,024 12.5 -> 11.9 and 15.8 -> 15.1.  An eighth and less is even: seven tiles from eight 42.4 -> 42.0
    // (1,700 of 4,096) and 40.3 -> 41.9 (1,792 of 4,096), nine from ten 30.7 -> 31.7 (2,300 of 2,048).
    // What the busiest unit has falls as workgroups are added, so the least is that of all slots, and the fewest that reach it are found by halving
    // (trying each of up to 256 took 0.3 to 0.9 us of host time a launch, this 0.05).
    if (p.S == 1 && p.per_cu == 2 && groups > cus) {
        const int old = busiest_unit(ntiles, groups, cus), least = busiest_unit(ntiles, most, cus);
        if (8 * (old - least) > old) {
            int enough = most;
            while (groups < enough) {
                const int middle = groups + (enough - groups) / 2;
                if (busiest_unit(ntiles, middle, cus) == least) enough = middle;
                else groups = middle + 1;
            }
        }
    }
    return groups;       // the grid is groups * S
}

// ---- products of 17 to 64 rows, activations in chunks through LDS ----
struct ChunkPlan {
    int S = 1, slice = 0, grid = 0, waves = 4;
};
inline size_t chunk_workspace_need(int ntiles, int S, int mt, int rt) {
    return kCounterBytes + (size_t)ntiles * S * mt * rt * kWaveLanes * 4 * kF32;
}
// `waves`: row tiles (waves) of a workgroup; a compute unit holds eight waves of this kernel, two workgroups of four or
// one of five to eight.  `copy`: whether the weights come from their tile-major copy
inline ChunkPlan plan_chunks(int K, int ntiles, int mt, int rt, size_t ws_bytes, bool have_ws, int cus, int forced, int waves = 4,
                             bool copy = false) {
    const int ngroups = (ntiles + waves - 1) / waves;
    const int slots = 8 / waves * cus;
    // K slices: as many as fill the chip with the row groups there are, each at least two chunks long.  Up to 48 rows a
    // workgroup has enough on its way for a compute unit of its own, and more slices only cost their sums' way through
    // memory (40 rows, with one workgroup a unit and with two: 4,096 x 4,096 13.3 and 16.2 us, 4,096 x 14,336 28.0 and
    // 29.6).  49 to 64 rows keep two, but where one still leaves four slices and a tile is 16 rows: from a tile-major copy up to K of 16,384, where
    // the loads of one workgroup begin to be too few; and where eight slices of one a unit would hold all tiles but one, they keep eight.
    // Microseconds at 49 and 64 rows, eight slices / four of workgroups of four waves: stored with a bias 4,096 x 4,096 18.9 / 15.7 and 18.8 / 15.5,
    // float32 results 16.5 / 14.0 and 16.7 / 14.1; sums that prepare a norm 4,096 x 8,192 25.3 / 25.0 and 25.8 / 25.1, x 14,336 38.1 / 34.3 and 37.9 / 33.3, 2,560 x
    // 8,192 24.2 / 21.7 and 24.9 / 21.8, 3,600 x 24,576 54.3 / 54.9 and 54.2 / 52.6; with a copy 4,096 x 8,192 23.4 / 22.0 and 24.1 / 22.0, x 14,336 31.7 / 30.3
    // and 32.1 / 29.6, but x 16,384 32.9 / 36.0 and 33.2 / 36.7, x 28,672 47.9 / 49.4 and 48.5 / 49.1; of 129 tiles (2,064 columns) x 8,192 19.8 / 20.8 and
    // 19.9 / 21.1, x 24,576 41.1 / 45.1 and 41.5 / 45.3.  Two slices instead of four (64 rows): 8,192 x 8,192 35.5 and 34.3, 8,192 x 28,672 91.5 and 90.3.
    const bool four = mt == 4 && rt == 1 && (K < 16384 || !copy) && 4 * ngroups <= cus && ntiles > cus / 8 * waves + 1;
    const int fill = mt <= 3 || four ? cus : slots;
    int S = 1;
    while (S < 8 && ngroups * S * 2 <= fill && (K + 2 * S - 1) / (2 * S) >= 512) S *= 2;
    if (forced > 0) S = forced;
    while (S > 1) {
        const size_t need = chunk_workspace_need(ntiles, S, mt, rt);      // the kernel's offsets into it are 32 bits
        if (have_ws && need <= ws_bytes && need - kCounterBytes <= 0x7fffffffu && (size_t)ntiles * sizeof(int) <= kCounterBytes &&
            (K + S - 1) / S >= 256)
            break;
        S /= 2;
    }
    ChunkPlan p;
    p.waves = waves;
    p.S = S;
    p.slice = ((K + S - 1) / S + 255) / 256 * 256;
    if (S > 1 && (long)(S - 1) * p.slice >= K) p.S = S = (K + p.slice - 1) / p.slice;   // no empty slice
    int per_slice = slots / S;
    if (per_slice < 1) per_slice = 1;
    if (per_slice > ngroups) per_slice = ngroups;
    p.grid = per_slice * S;
    return p;
}
// What the busiest compute unit streams under a plan, in weight rows x columns: its workgroups' row tiles over their
// slices, as often as the row groups of a slice come round.  Workgroups that are no more than the compute units have one
// each, also where two of four waves would fit: their tiles then spread over more units than those of seven waves would
// (microseconds of seven waves and of four, with the same slices, weights from memory, at 49 / 64 rows: 2,048 x 8,192
// 19.1 -> 16.5 / 19.6 -> 17.3, 2,048 x 14,336 26.2 -> 21.3 / 26.5 -> 21.7, 4,096 x 2,048 14.3 -> 12.9 / 14.7 -> 13.5, 6,144 x 1,024 13.2 ->
// 11.9 / 13.6 -> 12.3; gate/up of 2 x 4,096 x 1,024 14.7 -> 12.6 / 14.8 -> 12.8, of 2 x 2,048 x 2,048 15.3 -> 13.2 / 15.4 -> 13.7).
inline long chunk_plan_cost(const ChunkPlan &p, int ntiles, int cus) {
    const int ngroups = (ntiles + p.waves - 1) / p.waves;
    const int per_slice = p.grid / p.S;
    const long rounds = (ngroups + per_slice - 1) / per_slice;
    const long together = p.grid <= cus ? 1 : 8 / p.waves;       // workgroups of a compute unit
    return rounds * together * p.waves * (long)p.slice;
}
// From a copy: the number of waves (four, seven or eight) whose plan leaves the least to the busiest compute unit; on a tie four,
// but see below.
// 1,792 tiles over 256 compute units are seven a unit: workgroups of seven waves take a tile each in one round, where
// four or eight waves leave an eighth of the device idle in the last round.
inline ChunkPlan plan_chunks_balanced(int K, int ntiles, int mt, int rt, size_t ws_bytes, bool have_ws, int cus, int forced,
                                      int forced_waves) {
    if (forced_waves == 4 || forced_waves == 7 || forced_waves == 8)
        return plan_chunks(K, ntiles, mt, rt, ws_bytes, have_ws, cus, forced, forced_waves, true);
    ChunkPlan best = plan_chunks(K, ntiles, mt, rt, ws_bytes, have_ws, cus, forced, 4, true);
    long best_cost = chunk_plan_cost(best, ntiles, cus);
    for (int waves = 7; waves <= 8; waves++) {
        const ChunkPlan p = plan_chunks(K, ntiles, mt, rt, ws_bytes, have_ws, cus, forced, waves, true);
        const long cost = chunk_plan_cost(p, ntiles, cus);
        // a tie between four and eight waves, no slices either way, three or four row tiles of activations: eight waves
        // share one copy of a chunk in LDS where two workgroups of four hold one each (the vocabulary projection at
        // 64 rows: 207 -> 194 us)
        const bool shares = waves == 8 && cost == best_cost && mt >= 3 && p.S == 1 && best.S == 1 && best.waves == 4;
        if (cost < best_cost || shares) best = p, best_cost = cost;
    }
    return best;
}

// Six waves where they leave less still: 384 tiles in four slices are 256 workgroups of six, where seven waves make 220 and leave 36 units idle
// (q/k/v of 6,144 x 4,096 at 17 / 40 rows 18.2 -> 17.3 / 21.2 -> 20.3 us, of 10,240 x 8,192 37.4 -> 37.2 / 42.8 -> 41.3).
inline ChunkPlan plan_chunks_even(int K, int ntiles, int mt, int rt, size_t ws_bytes, bool have_ws, int cus, int forced, int forced_waves) {
    if (forced_waves == 6) return plan_chunks(K, ntiles, mt, rt, ws_bytes, have_ws, cus, forced, 6, true);
    const ChunkPlan best = plan_chunks_balanced(K, ntiles, mt, rt, ws_bytes, have_ws, cus, forced, forced_waves);
    if (forced_waves == 4 || forced_waves == 7 || forced_waves == 8) return best;
    const ChunkPlan six = plan_chunks(K, ntiles, mt, rt, ws_bytes, have_ws, cus, forced, 6, true);
    return chunk_plan_cost(six, ntiles, cus) < chunk_plan_cost(best, ntiles, cus) ? six : best;
}

// ---- products of 17 to 64 rows, a K slice of the activations resident in LDS ----
struct SlabPlan {
    int S = 0, slice = 0, grid = 0;       // S == 0: no plan
    size_t smem = 0, cells_off = 0;
};
inline size_t slab_workspace_need(int ntiles, int S, int mt, int rt) {
    return kCounterBytes + (size_t)ntiles * S * ((size_t)mt * rt * kWaveLanes * 4 + (size_t)mt * 16) * kF32;
}
inline size_t slab_ssq_offset_floats(int ntiles, int S, int mt, int rt) { return (size_t)ntiles * S * mt * rt * kWaveLanes * 4; }

// The slice length (256 to 1,024 columns; multiples of 512 for the norm prologue, whose sums of squares are kept per
// 512 columns) that costs a workgroup the fewest bytes: its items' weights, its staged slice, and its share of the
// partial sums that slices cost.
inline SlabPlan plan_slab(int M, int n_tiles, int K, int mt, int rt, bool norm, int nt, size_t ws_bytes, bool have_ws, int cus,
                          int forced) {
    SlabPlan best;
    double best_cost = 0.0;
    const int rows = mt * 16;
    const int ngroups = (n_tiles + 7) / 8;
    for (int slice = 1024; slice >= 256; slice -= 256) {
        if (norm && slice % 512 != 0) continue;
        int S = (K + slice - 1) / slice;
        int len = slice;
        const int step = norm ? 512 : 256;
        if (S == 1) len = (K + step - 1) / step * step;   // one slice: no longer than K needs
        if (forced > 0 && S != forced) continue;
        SlabPlan p;
        p.S = S;
        p.slice = len;
        p.cells_off = ((size_t)rows * (len + 8) * kBf16 + 15) / 16 * 16;
        p.smem = p.cells_off + (norm ? (size_t)rows * ((len + 511) / 512) * kF32 : 0);
        if (p.smem > kLdsBytes) continue;
        if (S > 1) {
            if (!have_ws || slab_workspace_need(n_tiles, S, mt, rt) > ws_bytes || (size_t)n_tiles * sizeof(int) > kCounterBytes) continue;
            if ((slab_workspace_need(n_tiles, S, mt, rt) - kCounterBytes) > 0x7fffffffu) continue;   // offsets of the 16-byte pieces are 32 bits
        }
        int per_slice = cus / S;
        if (per_slice < 1) per_slice = 1;
        if (per_slice > ngroups) per_slice = ngroups;
        p.grid = per_slice * S;
        const int items = (ngroups + per_slice - 1) / per_slice;
        const double weights = (double)items * 8 * (rt * nt) * len * 2.0;
        const double staged = (double)rows * len * (norm ? 4.0 : 2.0);
        const double parts = S > 1 ? (double)items * 8 * (double)M * rt * nt * 4.0 * 2.0 : 0.0;   // written, and read again by somebody
        const double cost = weights + staged + parts;
        if (best.S == 0 || cost < best_cost) best = p, best_cost = cost;
        if (S == 1) break;      // shorter slices of a K that fits in one gain nothing
    }
    return best;
}

// ---- products of many rows on tiles of 256 or 128 rows (gemm_tiles.h) ----
// K that the tiles can walk: in steps of 64, two steps a trip and four at least (256 rows), three at least (128 rows).
inline bool row_tile_takes(int bm, int K) { return bm == 256 ? K % 128 == 0 && K >= 256 : bm == 128 && K % 64 == 0 && K >= 192; }
// 256 or 128: the row tile whose rounds over the 256 compute units take less; 0: shapes they do not take.  A round of 128-row tiles takes
// kShortRound of one of 256-row tiles (measured 0.54 to 0.64: 28,672 columns of 4,096 57 against 89 us, 16,384 of 2,048 30 against 53; over
// several rounds 0.63 to 0.67).
// `asked`: 256 or 128 where a caller wants that one, 0 or 1 where it leaves the choice here.
constexpr double kShortRound = 0.62;
inline int row_tile(long tiles256, long tiles128, int K, int asked = 0) {
    if (asked != 0 && asked != 1) return row_tile_takes(asked, K) ? asked : 0;
    if (!row_tile_takes(256, K)) return row_tile_takes(128, K) ? 128 : 0;
    const double a = (double)((tiles256 + 255) / 256), b = kShortRound * (double)((tiles128 + 255) / 256);
    return a <= b ? 256 : 128;
}

// The row tile and whether a last round of at most 128 tiles of 256 rows runs as halves (twice as many tiles of 128 rows), which leaves no more
// than half of the compute units idle, for 0.73 to 0.85 of a round instead of a whole one (28,672 columns of 4,096 at 768 rows 0.74, 16,384 of 2,048 at
// 1,280 0.73, 57,344 of 8,192 at 1,024 0.85); a fuller round would take two of them.  `rounds`: the time in rounds of whole 256-row tiles over the
// compute units, a round of halves counted as kShortRound like one of 128-row tiles alone: where halves are planned by that they were ahead of whole
// rounds and of 128-row tiles at all 38 shapes measured.  Without -> with, microseconds: 28,672 columns of 4,096 at 700 / 1,200 / 2,048 rows (2, 3, 4
// rounds before) 167 -> 150 / 259 -> 238 / 368 -> 352; 17,920 of 1,536 at 1,024 / 2,048 75 -> 63 / 116 -> 106; both products of eight experts of 4,480
// of 1,536, 1,900 tokens that pick two 228 -> 209.
struct TilePlan {
    int bm = 0;                 // 0: a shape the tiles do not take
    bool halves = false;
    long tiles = 0;             // of bm rows
    double rounds = 0;
};
// The time of `tiles` 256-row tiles with the last round in halves where it can be
inline bool last_round_in_halves(long tiles) { return tiles % 256 != 0 && tiles % 256 <= 128; }
inline double rounds_with_halves(long tiles) { return (double)(tiles / 256) + (tiles % 256 == 0 ? 0.0 : last_round_in_halves(tiles) ? kShortRound : 1.0); }
// halves: 0 never, 1 where they take less time, 2 wherever they can be
inline TilePlan tile_plan(long tiles256, long tiles128, int K, int asked, int halves) {
    TilePlan p;
    p.bm = row_tile(tiles256, tiles128, K, asked);
    if (p.bm == 0) return p;
    p.tiles = p.bm == 256 ? tiles256 : tiles128;
    p.rounds = (double)((p.tiles + 255) / 256) * (p.bm == 256 ? 1.0 : kShortRound);
    const bool asked_other = asked != 0 && asked != 1 && asked != 256;
    if (halves == 0 || asked_other || !row_tile_takes(256, K) || !last_round_in_halves(tiles256)) return p;
    if (halves == 2 || (tiles256 > 256 && rounds_with_halves(tiles256) < p.rounds))
        p.bm = 256, p.halves = true, p.tiles = tiles256, p.rounds = rounds_with_halves(tiles256);
    return p;
}

// The row tile of both products of `pairs` (row, pick) pairs grouped by expert, `up` and `down` column tiles wide, with K_up and K_down steps: of 256
// and 128 the one whose two products take fewer rounds over the compute units, weighted with their K; how many row tiles the experts fill is known on
// the device alone, so half a tile an expert is assumed on top of the pairs.  On a tie (a round that could be halves) 128: tiles of 256 cost their
// halves' order and more rows that are not there (microseconds of 256 / 128, both products, tokens that pick two: 4 x 1,024 x 1,024 at 512 and 1,024
// 43.5 / 42.1 and 46.2 / 45.1, 8 x 2,048 x 1,024 at 512 67.2 / 65.6).
inline int grouped_row_tile(long pairs, long experts, long up, long down, int K_up, int K_down, int halves) {
    auto cost = [&](int bm) {
        const long rows = (pairs + experts * bm / 2 + bm - 1) / bm;
        if (bm == 256 && halves) return rounds_with_halves(rows * up) * K_up + rounds_with_halves(rows * down) * K_down;
        return (bm == 256 ? 1.0 : kShortRound) * ((double)((rows * up + 255) / 256) * K_up + (double)((rows * down + 255) / 256) * K_down);
    };
    return cost(256) < cost(128) ? 256 : 128;
}

// Whether a plain product (neither bias nor activation) goes to the tiles, or to the GEMM library: K of 2,048 at least and nine tenths of the rounds
// filled, in tiles (whole rounds) or, where a last round runs as halves, in outputs: such a round is short because half of the device is enough for it,
// and what its tiles do for rows that are not there counts all the more.  Microseconds library / halves by share, one MI355X, weights from memory:
// 0.90 and more 16,384 x 2,048 at 1,500 rows 86.7 / 84.6, x 3,072 at 1,536 124.8 / 122.7, 24,576 x 4,096 at 1,024 166.8 / 154.7, 8,192 x 8,192 at
// 3,072 293 / 283, 57,344 x 8,192 at 1,280 907 / 827; 0.80 to 0.87 16,384 x 2,048 at 2,304 128 / 138, x 4,096 at 2,304 234 / 239, 13,824 x 5,120 at 2,560
// 279 / 286, but 6,144 x 4,096 at 3,840 149 / 144; below 28,672 x 4,096 at 513 125 / 139, 10,240 x 8,192 at 1,537 and 2,048 238 / 247 and 269 / 269,
// 16,384 x 2,048 at 1,100 69 / 77.  (Where the library takes one of its slow kernels the tiles are up to 1.9 times as fast at any share.)
inline bool plain_takes_tiles(long M, long N, int K, const TilePlan &p) {
    if (p.bm == 0 || K < 2048) return false;
    if (p.halves) return (double)M * (double)N >= 0.9 * p.rounds * 256.0 * 65536.0;
    return 10 * p.tiles >= 9 * ((p.tiles + 255) / 256 * 256);
}

// K slices of a product whose 128-row tiles leave half of the compute units or more without one, a workgroup a slice; 1: whole.  What it costs is a
// tile's sums on their way through memory, some 10 us for two to four slices; what it is measured against is the GEMM library, which has smaller
// tiles.  Hence 32 steps of 64 columns a slice at least, K of 8,192 at least (4,096 x 4,096 at 1,024 rows 42.5 -> 43.7 us), and four fifths of the device
// taken (2,048 x 8,192 at 1,500 rows, two slices of 96 tiles 61.3 -> 61.8, at 405 rows, 128 workgroups 31.3 -> 37.2).  Microseconds library -> slices:
// 2,048 x 8,192 at 1,024 / 1,735 / 2,048 rows 51 -> 45 / 72 -> 66 / 75 -> 69; 1,536 x 13,312 at 700 / 1,500 / 1,735 65 -> 50 / 99 -> 73 / 89 -> 77 (float32 results
// 98 -> 79); 1,536 x 8,960 at 1,500 / 1,735 66 -> 55 / 62 -> 57; 4,096 x 14,336 at 257 / 405 / 1,024 75 -> 58 / 86 -> 69 / 139 -> 117.
// Over 512 to 8,192 columns of K 8,192 to 16,384 at 225 to 2,048 rows 0.45 to 1.0 (1,280 x 12,288 at 1,700 92 -> 62; float32 results of K 8,192 up to 1.07,
// 1,280 columns at 1,300 rows 42 -> 45), of K 28,672 0.27 to 0.7.
// Few rows: the tiles' own time is then the weights' way from memory, and the library's kernels for such rows are as good up to longer K.  Up to 128 rows
// K of 18,432 at least (65 rows: 16,384 x 8,192 64.5 -> 81.0, 8,192 x 16,384 64.7 -> 85.3, 28,672 x 12,288 154 -> 169, but 16,384 x 10,240 81 -> 75; from
// there on 8,192 x 18,432 135 -> 74, x 28,672 187 -> 102, 20,480 x 20,480 204 -> 157, 16,384 x 24,576 186 -> 192), up to 200 rows 10,240 (8,192 x 8,192 at
// 140 / 180 / 200 rows 49.8 -> 53.9 / 48.6 -> 52.7 / 53.7 -> 52.7, x 8,960 at 140 52 -> 55; 4,096 x 14,336 at 150 58 -> 51, 8,192 x 12,288 at 140 71 -> 63,
// 6,144 x 10,240 at 150 89 -> 52, 5,120 x 12,288 at 129 49 -> 53).
// `asked`: 0 never, 1 planned, more: as many as that and K allow.
inline size_t tile_slices_need(long tiles128, int slices) { return kCounterBytes + (size_t)tiles128 * slices * 128 * 256 * kF32; }
inline int tile_slices_from(long rows) { return rows > 200 ? 8192 : rows > 128 ? 10240 : 18432; }
inline int tile_slices(long rows, long tiles128, int K, size_t ws_bytes, bool have_ws, int asked) {
    if (asked == 0 || !have_ws || K % 64 != 0 || tiles128 < 1 || tiles128 > 128 || (asked == 1 && K < tile_slices_from(rows))) return 1;
    const int least = asked > 1 ? 3 : 32;      // steps a slice; the kernel needs three
    long s = asked > 1 ? asked : 256 / tiles128;
    if (s > 256 / tiles128) s = 256 / tiles128;
    if (s > K / 64 / least) s = K / 64 / least;
    if (s > 8) s = 8;
    if (s < 2 || tile_slices_need(tiles128, (int)s) > ws_bytes) return 1;
    return asked > 1 || 10 * s * tiles128 >= 8 * 256 ? (int)s : 1;
}

// Whether a product with its activation in the epilogue (gate and up: `columns` counts both; the squared ReLU) goes to the tiles, or to the GEMM
// library and a kernel for the activation.  A tile costs the same however few of its rows and columns are there and however few of the
// compute units have one, where the library has smaller tiles and cuts K; against that stands one pass over the product, which
// weighs less the longer K is.  share: what the rounds of the tiles do for this product, 1 where every compute unit has whole 256-row
// tiles all the time.  Measured inside a graph, weights from memory, microseconds library and kernel -> tiles at rows: 28,672 columns of
// 4,096 65 60 -> 67, 160 65 -> 68, 320 85 -> 97, 640 0.92x, then 420 1.08x, 512 114 -> 100, 900 1.10x (line at 0.65); 16,384 of 2,048 128 24 -> 34, 256 33 -> 34,
// 513 0.92x, then 420 1.18x, 512 43 -> 38, 768 1.08x (line at 0.57); 17,920 of 1,536 128 25.5 -> 29.6, then 192 29.3 -> 27.5, 320 34 -> 28;
// the squared ReLU of 4,480 of 1,536 128 19 -> 26, 512 22.9 -> 24.8, then 900 1.21x, of 13,312 of 1,536 128 22 -> 28, then 320 31 -> 26, 512 35 -> 28 (line at
// 0.29).  Up to K 1,024 the two sides are a few microseconds apart on the device (8,192 of 1,024 128 15.8 -> 20.3, 320 19.5 -> 19.2, 512 21.5 -> 19.9) and a
// prompt step of such a model waits for the host's launches, of which the tiles save one: 24 -> 18 to 20 at 65 to 512 rows launched one by one.
// Where a last round runs as halves the line is no lower than 0.68: 28,672 of 4,096 620 148 -> 150 (0.65), 640 144 -> 149 (0.67), then 645 159 -> 147
// (0.68), 700 162 -> 150; 16,384 of 4,096 1,085 140 -> 145 (0.65), 1,120 142 -> 146, then 1,280 150 -> 152, 2,304 257 -> 243; 24,576 of 4,096 768 155 -> 150;
// 16,384 of 2,048 1,030 82 -> 80 and 1,280 88 -> 86 (above its line of 0.57).
inline bool activation_joins(long M, long columns, int K, const TilePlan &p) {
    if (K <= 1024) return true;
    const double share = (double)M * (double)columns / (p.rounds * 256.0 * 65536.0), line = (K - 1024) / 1792.0, most = p.halves ? 0.68 : 0.65;
    return share >= (line < most ? line : most);
}

// ---- decode attention: contexts split over workgroups ----
// How a decode step of `rows` rows is split over the context.  A workgroup takes `unit` keys per round (64 a
// wave).  Contexts are split when the rows alone do not fill the machine: down to one round per workgroup when
// the parts are merged by the split that arrives last (`fused`), and only for long contexts when merging costs
// a second kernel.
inline void decode_split_plan(int rows, int kv_heads, int qtiles, int max_context, int unit, bool fused, int *splits,
                              int *keys_per_split) {
    const long base = (long)rows * kv_heads * qtiles;
    const long span = (long)max_context + 31;   // the first split starts at a multiple of 32 at or below the first key
    long want = 1;
    if (fused) {
        if (base < 512) want = (512 + base - 1) / base;
        const long most = (span + unit - 1) / unit;
        if (want > most) want = most;
        // Heads of 128 lanes, contexts of two rounds at most: whole.  The second round's keys are on their way before the first's are multiplied, where a
        // second part has to be handed over (us split / whole at 300 and 500 keys: 12 heads on 2, eight rows 8.3 / 7.0 and 8.7 / 8.1, one row
        // 7.1 / 6.2 and 7.4 / 6.8; 32 on 8, eight rows 8.0 / 7.2 and 8.4 / 8.6, forty 13.6 / 13.2 and 19.5 / 18.6).  Of 64 lanes a round is 512 keys,
        // and the two are even (700 and 1,000 keys, eight rows 7.8 / 7.1 and 8.1 / 8.6; 16 rows of 48 to 798 8.1 / 8.2).
        if (unit == 256 && max_context <= 2 * unit) want = 1;
    } else if (max_context > 2048 && base < 256) {
        want = (256 + base - 1) / base;
        const long most = (span + 2047) / 2048;
        if (want > most) want = most;
    }
    if (want > 64) want = 64;
    long per = (span + want - 1) / want;
    per = (per + unit - 1) / unit * unit;
    // more than sixteen parts of one round: half as many of two (the merge reads sixteen parts a trip; one row of 8,192
    // keys at the 8B sizes in pages of 64: 15.7 us in 32 parts, 13.8 in 16)
    if (fused && per == unit && (span + per - 1) / per > 16) per = 2 * (long)unit;
    *splits = (int)((span + per - 1) / per);
    *keys_per_split = (int)per;
}
inline int decode_waves(int head_dim) { return head_dim >= 128 ? 4 : 8; }
inline int decode_unit(int head_dim) { return decode_waves(head_dim) * 64; }      // keys that a workgroup takes per round
inline size_t decode_workspace_need(int rows, int heads, int head_dim, int splits) {
    return splits > 1 ? (size_t)rows * heads * splits * (head_dim + 2) * kF32 : 0;
}
inline size_t decode_lds_bytes(int head_dim, int group) {
    const int waves = decode_waves(head_dim), gq = group < 16 ? group : 16;
    return (size_t)(2 * waves * 16 + waves * gq * (head_dim + 2)) * kF32;
}
inline bool decode_counters_fit(int rows, int kv_heads, int qtiles) { return (size_t)rows * kv_heads * qtiles * sizeof(int) <= kCounterBytes; }

// ---- prompt attention: the key tiles of a row tile shared among workgroups ----
// what a part of a row tile leaves behind, in floats: every thread of the workgroup its outputs (head_dim / 2), a maximum and a sum
constexpr size_t part_floats(int head_dim, int threads = 256) { return (size_t)threads * (head_dim / 2 + 2); }
// The rows of a step as the plan below counts them against its longest context: all of them where they are mostly one prompt's, 0 where
// others keep the slots busy while the long row tiles run, which are then better whole (shared, their second halves wait behind
// all other row tiles).  All segments but one may be single rows.  Others are enough
//   - with a third of the longest prompt's rows, or where there are several a quarter (32 heads on 8 of 128 lanes, us shared / whole: 1,900
//     and 100 rows 67.9 / 72.5, 1,500 and 500 54.0 / 57.3, 1,450 and 550 59.1 / 55.6, 1,300 and 700 56.5 / 50.9, 500, 650 and 800
//     42.6 / 39.1, 1,200, 200, 100 and 50 45.4 / 40.1; of 64 lanes 44.2 / 45.4, 35.0 / 36.8, 38.4 / 35.6, 36.6 / 32.6, 27.9 / 25.1, 30.1 / 26.0);
//   - being single rows, where they take half of the slots and the prompt's row tiles fill the other half by themselves (1,900 rows and
//     40 / 64 / 100 single ones 85.7 / 74.2, 89.0 / 76.1 and 104 / 87.6; 12 heads on 2, whose row tiles do not, 50.1 / 61.1, 48.2 /
//     52.4 and 46.8 / 53.2).
inline int rows_of_one_prompt(int tiles, int rows, int num_segs, int kv_heads, int max_context, int slots) {
    const long others = num_segs - 1;
    const bool prompts = (num_segs > 2 ? 4 : 3) * (rows - others - max_context) > max_context;
    const bool singles = 2 * others * kv_heads > slots && 2 * (tiles - others) * kv_heads >= slots;
    return prompts || singles ? 0 : rows;
}
// The most key tiles one workgroup takes (0: row tiles are not shared) and the most parts a row tile can have.  Row
// tiles are shared when, one workgroup each, they would leave workgroup slots of the device empty: a part then has
// about the key tiles that a slot sees in all when every slot is taken, and at least 8, since every part pays for
// leaving its results and the last one for adding them up.  A step whose rows are as many as its longest context (a
// prompt from its first token on) has row tiles of every length up to the longest, half of it on average: up to 2,048
// tokens the long ones are shared in halves (8 to 16 key tiles a part), or the slots of the short ones would idle
// through the second half of the launch (longer prompts have row tiles enough to keep every slot busy).  `rows`: see
// rows_of_one_prompt.  `room`: parts that the workspace holds; `by_hand`: key tiles a part when set by hand (> 1).
inline int prefill_part_plan(int tiles, int kv_heads, int rows, int max_context, int window, size_t room, int slots, int by_hand,
                             int *max_parts) {
    *max_parts = 1;
    if (window > 0) return 0;     // a window keeps every context short
    const long groups = (long)tiles * kv_heads;
    if (groups <= 0 || groups * (long)sizeof(int) > (long)kCounterBytes) return 0;
    const long most_tiles = ((long)max_context + 63) / 64;        // key tiles of the longest context
    const long per_slot = (groups * most_tiles + slots - 1) / slots;
    long per_part = per_slot > 8 ? per_slot : 8;
    if (rows + 63 >= max_context && most_tiles <= 32) {       // contexts of every length; measured a gain up to 2,048 tokens only
        long half = most_tiles / 2;
        half = half < 8 ? 8 : (half > 16 ? 16 : half);
        if (half < per_part) per_part = half;
    }
    if (by_hand > 1) per_part = by_hand;
    long cap = (long)(room / (size_t)groups);   // parts a row tile may have
    if (cap > 16) cap = 16;
    if (cap < 2) return 0;
    const long least = (most_tiles + cap - 1) / cap;
    if (per_part < least) per_part = least;
    if (per_part >= most_tiles) return 0;
    *max_parts = (int)((most_tiles + per_part - 1) / per_part);
    return (int)per_part;
}

}  // namespace fllm_plan
