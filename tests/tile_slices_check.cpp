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
                    const int s = tile_slices(tiles, K, ws, ws > 0, asked);
                    bool ok = s >= 1 && s <= 8;
                    if (s > 1) {
                        cut++;
                        ok = ok && asked != 0 && ws > 0 && K % 64 == 0 && s * tiles <= 256 && tile_slices_need(tiles, s) <= ws &&
                             tiles * (long)sizeof(int) <= (long)kCounterBytes;
                        for (int i = 0; i < s; i++) {      // as the kernel deals the steps out
                            const long from = (long)(K / 64) * i / s, to = (long)(K / 64) * (i + 1) / s;
                            ok = ok && to - from >= (asked == 1 ? 32 : 3) && (i + 1 < s || to == K / 64);
                        }
                        if (asked == 1) ok = ok && K >= 8192 && 10 * s * tiles >= 8 * 256;
                    }
                    if (!ok) {
                        fprintf(stderr, "FAILED tiles %ld K %d asked %d: %d slices\n", tiles, K, asked, s);
                        return 1;
                    }
                }
    printf("slices ok %ld\n", cut);
    return cut > 0 ? 0 : 1;
}
