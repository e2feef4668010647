// How a router's one wave picks a row's experts from their scores in LDS: for the routers of routed_experts.hip and for the kernel that
// norms a row and routes it (norm_route.hip).
#pragma once
#include "common.h"

// shuffles that meet among `lanes` (a power of two) neighbouring lanes: the largest value, the lower index among equals
__device__ __forceinline__ void best_of_lanes(float &best, int &at, int lanes) {
    for (int o = lanes >> 1; o > 0; o >>= 1) {
        const float other = __shfl_xor(best, o, kWave);
        const int other_at = __shfl_xor(at, o, kWave);
        if (other > best || (other == best && other_at < at)) best = other, at = other_at;
    }
}
__device__ __forceinline__ int lanes_for(int n) {      // the lanes that hold something when lane l holds items l, l + 64, ..
    int lanes = 1;
    while (lanes < n && lanes < kWave) lanes *= 2;
    return lanes;
}

// Up to 64 experts the picks are made in registers, an expert a lane: a round is the wave's largest score by lane swaps and the first lane that
// holds it, some 100 cycles, where shuffles and a pass through LDS were 500 (two of 8 experts in four groups, two kept: 1 us of a launch).
__device__ __forceinline__ int first_lane_with(bool yes) {      // -1: none
    const unsigned long long lanes = __ballot(yes);
    return lanes ? __builtin_ctzll(lanes) : -1;
}
__device__ __forceinline__ float value_of_lane(float v, int lane) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane)); }

// `top` rounds over what the lanes hold: the largest `choice`, the lower lane among equals, taken out; the lanes' picks (of lane k the k-th), the
// sum of their scores in order.  A round whose choices compare with nothing picks expert k: still one of the stack.
struct LanePicks {
    int id;
    float score, sum;
};
__device__ __forceinline__ LanePicks pick_lanes(float choice, float score, int top, int lane, bool score_is_choice) {
    LanePicks out = {0, 0.f, 0.f};
    float left = choice > -INFINITY ? choice : -INFINITY;      // NaN: compares with nothing
    for (int k = 0; k < top; k++) {
        const float best = wave_max(left);
        int at = first_lane_with(left == best && left > -INFINITY);
        const float s = at < 0 && score_is_choice ? -INFINITY : value_of_lane(score, at < 0 ? k : at);
        if (at < 0) at = k;
        out.sum += s;
        if (lane == k) out.id = at, out.score = s;
        if (lane == at) left = -INFINITY;
    }
    return out;
}

// score[E]: sigmoid scores (score_mode 0) or logits whose softmax over all experts is the score (1).  ids[top] and weights[top]: the
// `top` largest, the lower index among equals; weights with `renormalize` divided by the sum of the picks' scores (+ 1e-20), times
// route_scale.  picks[top] is scratch.
__device__ __forceinline__ void pick_plain(float *score, float *picks, int E, int top, int32_t *ids, float *weights, int score_mode,
                                           int renormalize, float route_scale, int lane) {
    if (E <= kWave) {
        float s = lane < E ? score[lane] : -INFINITY;
        if (score_mode == 1) {
            const float top_z = wave_max(s);
            const float sum = wave_sum(lane < E ? expf(s - top_z) : 0.f);
            s = lane < E ? expf(s - top_z) / sum : -INFINITY;
        }
        const LanePicks got = pick_lanes(s, s, top, lane, true);
        const float factor = renormalize ? route_scale / (got.sum + 1e-20f) : route_scale;
        if (lane < top) {
            ids[lane] = got.id;
            weights[lane] = (renormalize || route_scale != 1.0f) ? got.score * factor : got.score;
        }
        return;
    }
    const int lanes = lanes_for(E);
    if (score_mode == 1) {   // softmax over all experts: the largest logit, the sum in index order a lane, then across lanes
        float top_z = -INFINITY;
        for (int e = lane; e < E; e += kWave) top_z = fmaxf(top_z, score[e]);
        top_z = wave_max(top_z);
        float sum = 0.f;
        for (int e = lane; e < E; e += kWave) sum += expf(score[e] - top_z);
        sum = wave_sum(sum);
        for (int e = lane; e < E; e += kWave) score[e] = expf(score[e] - top_z) / sum;
        __builtin_amdgcn_wave_barrier();
        __threadfence_block();
    }
    float picked = 0.f;
    // one wave picks: every round the largest score not yet taken, the lowest index among equals
    for (int k = 0; k < top; k++) {
        float best = -INFINITY;
        int at = 0x7fffffff;
        for (int e = lane; e < E; e += kWave) {
            const float s = score[e];
            if (s > best) best = s, at = e;      // ascending e: the first of equals stays
        }
        best_of_lanes(best, at, lanes);
        if (at < 0 || at >= E) at = k;           // scores that compare with nothing (NaN rows): still an expert of the stack
        picked += best;
        if (lane == 0) {
            ids[k] = at;
            picks[k] = best;
            score[at] = -INFINITY;               // scores lie in [0, 1]: nothing real is that small
        }
        __builtin_amdgcn_wave_barrier();
        __threadfence_block();
    }
    const float factor = renormalize ? route_scale / (picked + 1e-20f) : route_scale;
    for (int k = lane; k < top; k += kWave)
        weights[k] = (renormalize || route_scale != 1.0f) ? picks[k] * factor : picks[k];
}

// score[E] sigmoid scores, choice[E] scores + corrections: picks by choice among the experts of the `kept` groups (of `groups` equal
// groups of neighbours) whose two largest choices sum highest, the lower group among equals; weights the plain scores of the
// picks divided by their sum (+ 1e-20), times route_scale.  gsum[groups] and picks[top] are scratch.
__device__ __forceinline__ void pick_grouped(const float *score, float *choice, float *gsum, float *picks, int E, int top, int groups,
                                             int kept, int32_t *ids, float *weights, float route_scale, int lane) {
    const int per = E / groups;
    if (E <= kWave) {
        const int g = lane / per;      // this lane's expert's group, and this lane's group below
        float c = lane < E ? choice[lane] : -INFINITY;
        const float s = lane < E ? score[lane] : 0.f;
        if (groups > 1) {
            float a = -INFINITY, b = -INFINITY;
            for (int i = 0; i < per; i++) {
                const float v = lane < groups ? choice[lane * per + i] : -INFINITY;
                if (v > a) b = a, a = v;
                else if (v > b) b = v;
            }
            float sum = per > 1 ? a + b : a;
            for (int k = 0; k < kept; k++) {      // the best group not yet kept: marked with +inf
                const float left = lane < groups && sum != INFINITY && sum > -INFINITY ? sum : -INFINITY;
                const float best = wave_max(left);
                int at = first_lane_with(left == best && left > -INFINITY);
                if (at < 0) {                     // sums that compare with nothing: the first group not yet kept
                    at = first_lane_with(lane < groups && sum != INFINITY);
                    if (at < 0) at = groups - 1;
                }
                if (lane == at) sum = INFINITY;
            }
            const unsigned long long keeps = __ballot(lane < groups && sum == INFINITY);
            if (((keeps >> (g & 63)) & 1) == 0) c = -INFINITY;
        }
        const LanePicks got = pick_lanes(c, s, top, lane, false);
        const float factor = route_scale / (got.sum + 1e-20f);
        if (lane < top) {
            ids[lane] = got.id;
            weights[lane] = got.score * factor;
        }
        return;
    }
    const int lanes = lanes_for(E), group_lanes = lanes_for(groups);
    if (groups > 1) {
        for (int g = lane; g < groups; g += kWave) {      // a group counts the sum of its two largest choices (of its one, if it has one)
            float a = -INFINITY, b = -INFINITY;
            for (int e = g * per; e < (g + 1) * per; e++) {
                const float c = choice[e];
                if (c > a) b = a, a = c;
                else if (c > b) b = c;
            }
            gsum[g] = per > 1 ? a + b : a;
        }
        __builtin_amdgcn_wave_barrier();
        __threadfence_block();
        for (int k = 0; k < kept; k++) {                  // the best group not yet kept: marked with +inf
            float best = -INFINITY;
            int at = 0x7fffffff;
            for (int g = lane; g < groups; g += kWave) {
                const float s = gsum[g];
                if (s != INFINITY && s > best) best = s, at = g;
            }
            best_of_lanes(best, at, group_lanes);
            at = __shfl(at, 0, kWave);
            if (at < 0 || at >= groups) {                 // sums that compare with nothing: the first group not yet kept
                at = 0;
                while (at < groups - 1 && gsum[at] == INFINITY) at++;
            }
            __builtin_amdgcn_wave_barrier();
            if (lane == 0) gsum[at] = INFINITY;
            __builtin_amdgcn_wave_barrier();
            __threadfence_block();
        }
        for (int e = lane; e < E; e += kWave)
            if (gsum[e / per] != INFINITY) choice[e] = -INFINITY;
        __builtin_amdgcn_wave_barrier();
        __threadfence_block();
    }
    float picked = 0.f;
    for (int k = 0; k < top; k++) {
        float best = -INFINITY;
        int at = 0x7fffffff;
        for (int e = lane; e < E; e += kWave) {
            const float s = choice[e];
            if (s > best) best = s, at = e;
        }
        best_of_lanes(best, at, lanes);
        if (at < 0 || at >= E) at = k;
        const float s = score[at];
        picked += s;
        __builtin_amdgcn_wave_barrier();
        if (lane == 0) {
            ids[k] = at;
            picks[k] = s;
            choice[at] = -INFINITY;
        }
        __builtin_amdgcn_wave_barrier();
        __threadfence_block();
    }
    const float factor = route_scale / (picked + 1e-20f);
    for (int k = lane; k < top; k += kWave) weights[k] = picks[k] * factor;
}
