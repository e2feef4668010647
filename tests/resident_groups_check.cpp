// The workgroups of a resident product (csrc/plans.h), over all tile counts of its range: no more than slots and tiles, no compute unit with more
// tiles than under the even split, and the busiest unit's count is the one that dealing the tiles out gives.  Built and run by
// tests/test_resident_groups.py.
#include "plans.h"

#include <initializer_list>
#include <stdio.h>
#include <stdlib.h>
#include <vector>

using namespace fllm_plan;

int main() {
    for (int cus : {1, 3, 256, 304})
        for (int per_cu : {1, 2})
            for (int S : {1, 2, 4})
                for (int tiles = 1; tiles <= 9 * cus + 5 && tiles <= 2600; tiles++) {
                    ResidentPlan p;
                    p.S = S, p.per_cu = per_cu;
                    const int groups = resident_groups(p, tiles, cus);
                    int slots = cus * per_cu / S;
                    if (slots < 1) slots = 1;
                    if (slots > tiles) slots = tiles;
                    const int rounds = (tiles + slots - 1) / slots, even = (tiles + rounds - 1) / rounds;
                    std::vector<int> unit(cus, 0);
                    for (int t = 0; t < tiles; t++) unit[t % groups % cus]++;
                    int most = 0;
                    for (int n : unit) most = n > most ? n : most;
                    const bool shared = S == 1 && per_cu == 2;
                    // the fewest workgroups, each number tried, that leave the busiest unit the least, where that is an eighth and more
                    int few = even, least = busiest_unit(tiles, even, cus);
                    for (int g = even + 1; g <= slots; g++)
                        if (busiest_unit(tiles, g, cus) < least) few = g, least = busiest_unit(tiles, g, cus);
                    const int before = busiest_unit(tiles, even, cus);
                    const int wanted = shared && even > cus && 8 * (before - least) > before ? few : even;
                    if (groups != wanted) {
                        fprintf(stderr, "FAILED cus %d per %d S %d tiles %d: %d groups, not %d\n", cus, per_cu, S, tiles, groups, wanted);
                        return 1;
                    }
                    if (groups < 1 || groups > slots || busiest_unit(tiles, groups, cus) > busiest_unit(tiles, even, cus) || (!shared && groups != even) ||
                        (shared && most != busiest_unit(tiles, groups, cus))) {
                        fprintf(stderr, "FAILED cus %d per %d S %d tiles %d: %d groups, busiest %d\n", cus, per_cu, S, tiles, groups, most);
                        return 1;
                    }
                }
    ResidentPlan p;
    p.S = 1, p.per_cu = 2;
    const int want[][2] = {{512, 512}, {513, 257}, {600, 344}, {768, 512}, {769, 385}, {1024, 512}, {1120, 432}, {1280, 512}, {1536, 512}, {1792, 448}};
    for (const auto &w : want)
        if (resident_groups(p, w[0], 256) != w[1]) {
            fprintf(stderr, "FAILED %d tiles: %d groups, not %d\n", w[0], resident_groups(p, w[0], 256), w[1]);
            return 1;
        }
    printf("groups ok\n");
    return 0;
}
