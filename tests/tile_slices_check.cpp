// K slices of products of many rows (csrc/plans.h), swept: no more workgroups than compute units, every slice long enough for the kernel (and for the
// plan where it chose), parts inside the workspace, counters inside theirs.  Built and run by tests/test_tile_slices.py.
#include "plans.h"

#include <initializer_list>
#include <stdio.h>

using namespace fllm_plan;

int main() {
    long cut = 0;
    for (size_t ws : {(size_t)0, (size_t)8 << 20, (size_t)192 << 20})
        for (long tiles = 0; tiles <= 300; tiles++)
            for (int K = 8; K <= 32768; K += K < 1024 ? 8 : 64)
                for (int asked : {0, 1, 2, 3, 8, 100}) {
                    const long rows = tiles % 3 == 0 ? 128 : tiles % 3 == 1 ? 200 : 2048;
                    const int s = tile_slices(rows, tiles, K, ws, ws > 0, asked);
                    bool ok = s >= 1 && s <= 8;
                    if (s > 1) {
                        cut++;
                        ok = ok && asked != 0 && ws > 0 && K % 64 == 0 && s * tiles <= 256 && tile_slices_need(tiles, s) <= ws &&
                             tiles * (long)sizeof(int) <= (long)kCounterBytes;
                        for (int i = 0; i < s; i++) {      // as the kernel deals the steps out
                            const long from = (long)(K / 64) * i / s, to = (long)(K / 64) * (i + 1) / s;
                            ok = ok && to - from >= (asked == 1 ? 32 : 3) && (i + 1 < s || to == K / 64);
                        }
                        if (asked == 1) ok = ok && K >= tile_slices_from(rows) && K >= 8192 && 10 * s * tiles >= 8 * 256;
                    }
                    if (!ok) {
                        fprintf(stderr, "FAILED tiles %ld K %d asked %d: %d slices\n", tiles, K, asked, s);
                        return 1;
                    }
                }
    // where both were measured: columns, K, rows, and whether slices were ahead of the library
    const struct { int columns, K, rows; bool slices; } measured[] = {
        {16384, 8192, 65, false}, {28672, 8192, 100, false}, {8192, 16384, 65, false}, {28672, 12288, 128, false}, {8192, 18432, 65, true}, {8192, 28672, 96, true},
        {20480, 20480, 100, true}, {8192, 8192, 140, false}, {8192, 8192, 180, false}, {8192, 8960, 140, false}, {8192, 12288, 140, true}, {4096, 14336, 150, true},
        {6144, 10240, 150, true}, {8192, 8192, 225, true}, {8192, 8192, 256, true}, {4096, 14336, 405, true}, {2048, 8192, 2048, true}, {1536, 13312, 1735, true},
        {1536, 8960, 2003, false}, {4096, 4096, 1024, false}};
    for (const auto &m : measured) {
        const long tiles = (long)(m.rows + 127) / 128 * ((m.columns + 255) / 256);
        if ((tile_slices(m.rows, tiles, m.K, (size_t)192 << 20, true, 1) > 1) != m.slices) {
            fprintf(stderr, "FAILED %d columns of %d, %d rows\n", m.columns, m.K, m.rows);
            return 1;
        }
    }
    printf("slices ok %ld\n", cut);
    return cut > 0 ? 0 : 1;
}
