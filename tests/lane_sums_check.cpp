// Sums and maxima over a wave's lanes (csrc/common.h) as a host program: a value is what all 64 lanes hold, the swaps and rotations are written out
// as the instruction set describes them.  Against a butterfly over the bits 32, 16, .. 1 of the lanes' numbers, bit for bit (a NaN for a NaN, a zero for a zero), on
// finite values, infinities of both signs, NaN, zeros of both signs and subnormal values.  Built and run by tests/test_lane_sums.py.
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

#include <random>

struct Lanes {
    float l[64];
    Lanes operator+(const Lanes &o) const {
        Lanes r;
        for (int i = 0; i < 64; i++) r.l[i] = l[i] + o.l[i];
        return r;
    }
    Lanes &operator+=(const Lanes &o) { return *this = *this + o; }
};
struct Two {
    Lanes r[2];
    Lanes operator[](int i) const { return r[i]; }
};
static Lanes fmaxf(const Lanes &a, const Lanes &b) {
    Lanes r;
    for (int i = 0; i < 64; i++) r.l[i] = ::fmaxf(a.l[i], b.l[i]);
    return r;
}
#define __device__
#define __forceinline__ inline
#define __float_as_uint(v) (v)
#define __uint_as_float(v) (v)
// the first operand's upper half (odd rows of 16) and the second one's lower half (even rows) change places
static Two swapped(Lanes a, Lanes b, int span) {
    Two t = {{a, b}};
    for (int i = 0; i < 64; i++)
        if (i & span) t.r[0].l[i] = b.l[i - span], t.r[1].l[i - span] = a.l[i];
    return t;
}
#define __builtin_amdgcn_permlane32_swap(a, b, fi, bc) swapped(a, b, 32)
#define __builtin_amdgcn_permlane16_swap(a, b, fi, bc) swapped(a, b, 16)
// row_ror:N: lane i takes lane i - N of its row of 16
static Lanes rotated(const Lanes &v, int control) {
    Lanes r;
    for (int i = 0; i < 64; i++) r.l[i] = v.l[(i & ~15) | ((i - (control - 0x120)) & 15)];
    return r;
}
#define __builtin_amdgcn_update_dpp(old, v, control, rows, banks, bound) rotated(v, control)
#include "lane_sums_host.h"

static Lanes butterfly(Lanes v, bool sum, int from, int to) {
    for (int o = from; o >= to; o >>= 1) {
        Lanes across;
        for (int i = 0; i < 64; i++) across.l[i] = v.l[i ^ o];
        v = sum ? v + across : fmaxf(v, across);
    }
    return v;
}
static bool same(const Lanes &a, const Lanes &b, const char *what, int trial) {
    for (int i = 0; i < 64; i++)
        if (memcmp(&a.l[i], &b.l[i], 4) != 0 && !(isnan(a.l[i]) && isnan(b.l[i])) && !(a.l[i] == 0 && b.l[i] == 0)) {
            printf("%s, trial %d, lane %d: %a, not %a\n", what, trial, i, a.l[i], b.l[i]);
            return false;
        }
    return true;
}

int main() {
    std::mt19937 g(5);
    std::normal_distribution<float> normal;
    const float odd[] = {INFINITY, -INFINITY, NAN, 0.f, -0.f, 1e-42f, -3e38f, 3e38f};
    bool ok = true;
    for (int trial = 0; trial < 4000; trial++) {
        Lanes v;
        for (float &x : v.l) x = trial % 4 == 3 ? -INFINITY : normal(g) * (trial % 4 == 2 ? 1e30f : 1.f);
        for (int n = trial % 5; n > 0; n--) v.l[g() % 64] = odd[g() % 8];
        ok = ok && same(wave_sum(v), butterfly(v, true, 32, 1), "sum", trial) && same(wave_max(v), butterfly(v, false, 32, 1), "maximum", trial) &&
             same(sum_32_apart(v), butterfly(v, true, 32, 32), "sum 32 apart", trial) && same(max_32_apart(v), butterfly(v, false, 32, 32), "maximum 32 apart", trial) &&
             same(sum_16_apart(v), butterfly(v, true, 16, 16), "sum 16 apart", trial) && same(max_16_apart(v), butterfly(v, false, 16, 16), "maximum 16 apart", trial);
    }
    if (ok) printf("lanes ok\n");
    return ok ? 0 : 1;
}
