// maya_route.hpp - the softmax router on one wave (up to 512 experts), exactly and by the order of the logits alone: what the kernels
// that route for themselves share (the routing kernels, the decode layers whose head rides in their gate/up launch).
#pragma once

#include "maya_dev.hpp"

namespace maya {

// The largest of a wave's values, in every lane's scalar copy: exchanges inside the rows of 16 lanes (lane ^ 1, lane ^ 2,
// the half-row and row mirrors), then lane 15 of a row to the next row and lane 31 to the upper half; lane 63 has it.
__device__ __forceinline__ int wave_max_i32(int v) {
    v = max(v, dpp_i<0xB1>(v));
    v = max(v, dpp_i<0x4E>(v));
    v = max(v, dpp_i<0x141>(v));
    v = max(v, dpp_i<0x140>(v));
    v = max(v, __builtin_amdgcn_update_dpp(v, v, 0x142, 0xa, 0xf, false));
    v = max(v, __builtin_amdgcn_update_dpp(v, v, 0x143, 0xc, 0xf, false));
    return __builtin_amdgcn_readlane(v, 63);
}

// Up to 64 R experts, ONE wave, sm.ex filled: lane L keeps experts L, L + 64, L + 128, ... in registers from the sum
// to the weights, so nothing but the result touches LDS and no workgroup barrier sits on the path.
//  * the sum: ascending, one add after the other (the reference's order).  The chain of dependent double adds is the
//    critical path, so every add takes its operand from a lane by v_readlane, eight fetched ahead; all lanes carry the sum.
//  * the k largest: k rounds of the reference's strict-> arg-max with the lower index on ties
//    (src/kernels/cuda/router_top10.cu:140-176).  Probabilities are non-negative, so their bit patterns order like the
//    values as signed integers and -1 marks "taken" or "no such expert"; a round is an R-way maximum a lane, the wave
//    maximum, and the first lane (lowest expert: lower register first, then lower lane) that holds it.
//  * renormalisation: the k weights summed in slot order in double, one division a lane.
// (the token's exponentials already R a lane in ex; the wave's lane i < k returns slot i: its expert and weight.  `tab`:
// the residency table's entries of the lane's experts (R = 4), NULL when no plan is wanted; the slot's blob address then
// comes back in my_ptr - read from the chosen expert's lane, no second trip to memory.)
template <int R>
__device__ __forceinline__ void route_narrow_regs(int n_expert, int k, const double (&ex)[R], const uint64_t* tab, int& my_id,
                                                  float& my_weight, uint64_t& my_ptr) {
    const int lane = threadIdx.x & 63;
    int lo[R], hi[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        lo[r] = __double2loint(ex[r]);
        hi[r] = __double2hiint(ex[r]);
    }
    double sum = 0.0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        if (64 * r < n_expert) {
#pragma unroll
            for (int j0 = 0; j0 < 64; j0 += 8) {
                int sl[8], sh[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    sl[j] = __builtin_amdgcn_readlane(lo[r], j0 + j);
                    sh[j] = __builtin_amdgcn_readlane(hi[r], j0 + j);
                }
#pragma unroll
                for (int j = 0; j < 8; ++j) sum += __hiloint2double(sh[j], sl[j]);
            }
        }
    }
    const float inv = (float) (1.0 / sum);
    int key[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        key[r] = 64 * r + lane < n_expert ? __float_as_int((float) (ex[r] * (double) inv)) : -1;
        // (a row with an infinity or a NaN is all NaN, of the sign the division gave it; beyond 256 experts such rows come out with
        // their lowest experts, as from route_token, whose keys are unsigned)
        if (R > 4 && 64 * r + lane < n_expert && key[r] < 0) key[r] = 0x7fffffff;
    }
    int id = 0, my_w = 0;
    uint64_t ptr = 0ull;
    for (int i = 0; i < k; ++i) {
        int best = max(key[0], key[1]);
#pragma unroll
        for (int q = 2; q < R; ++q) best = max(best, key[q]);
        const int top = wave_max_i32(best);
        unsigned long long b = __ballot(key[0] == top);
        int r = 0;
#pragma unroll
        for (int q = 1; q < R; ++q)
            if (b == 0ull) b = __ballot(key[q] == top), r = q;
        const int at = __builtin_amdgcn_readfirstlane(__builtin_ctzll(b));
#pragma unroll
        for (int q = 0; q < R; ++q) key[q] = (q == r && lane == at) ? -1 : key[q];
        if (lane == i) id = 64 * r + at, my_w = R > 4 && top == 0x7fffffff ? (int) 0xffc00000 : top;
        if (R == 4 && tab) {
            // (written out: as a loop over tab the select becomes an index, the table goes to memory, and the kernels whose launch holds
            // this router take 11 us longer)
            const uint64_t tq = r == 0 ? tab[0] : r == 1 ? tab[1] : r == 2 ? tab[2] : tab[3];
            const uint32_t plo = (uint32_t) __builtin_amdgcn_readlane((int) (uint32_t) tq, at);
            const uint32_t phi = (uint32_t) __builtin_amdgcn_readlane((int) (uint32_t) (tq >> 32), at);
            if (lane == i) ptr = ((uint64_t) phi << 32) | plo;
        }
    }
    double s = 0.0;
    for (int i = 0; i < k; ++i) s += (double) __int_as_float(__builtin_amdgcn_readlane(my_w, i));
    const double sc = fmax(s, 6.103515625e-05);
    my_id = id;
    my_weight = (float) ((double) __int_as_float(my_w) / sc);
    my_ptr = ptr;
}
// a float's bits as a signed integer that orders like the float (no -0.0 arises: p > 0 and p + bias = 0 rounds to +0.0)
__device__ __forceinline__ int float_order_key(float v) {
    const int b = __float_as_int(v);
    return b >= 0 ? b : b ^ 0x7fffffff;
}
// The softmax router on ONE wave, nothing but registers (up to 64 R experts, R a lane: lane L holds experts L, L + 64, ...;
// lv = -inf and tab = 0 past the end): the maximum, the exponentials, then route_narrow_regs.  Lane i < k returns slot i (its blob's
// address for R = 4 only).
template <int R>
__device__ __forceinline__ void route_wave_softmax(const float (&lv)[R], const uint64_t (&tab)[R], int n_expert, int k, int& id,
                                                   float& w, uint64_t& ptr) {
    const int lane = threadIdx.x & 63;
    float mx = fmaxf(lv[0], lv[1]);
#pragma unroll
    for (int r = 2; r < R; ++r) mx = fmaxf(mx, lv[r]);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, kWave));
    double ex[R];
#pragma unroll
    for (int r = 0; r < R; ++r) ex[r] = 64 * r + lane < n_expert ? exp((double) lv[r] - (double) mx) : 0.0;
    route_narrow_regs(n_expert, k, ex, tab, id, w, ptr);
}

// Which k experts the softmax router picks, and in which order, WITHOUT the probabilities: p = exp(l - max) / sum grows
// with the logit, so the k largest logits in descending order are the k largest probabilities in descending order as long
// as rounding cannot merge or reorder two of them.  Two logits more than 1e-6 apart give probabilities whose ratio
// exceeds 1 + 1e-6, far beyond the 2^-24 relative rounding of a float, and a probability within e^-60 of the largest
// is a normal float.  So: every logit finite, each pick more than 1e-6 above the next, the k-th more than 1e-6 above
// everything not picked, and all of that within 60 of the first - then the picks and their order are the exact router's.
// Anything else (ties, near ties, the sub-normal range, NaN / Inf) returns false and the caller runs the exact router.
//
// A round must be short (k + 1 of them run one after the other on one wave while its workgroup waits), so a key is one
// word that names its expert: the logit's ordered bits with the low byte (R = 8: nine bits) replaced by 255 - index.  The largest key
// of the wave IS the pick, with no search for the lane that holds it.  The bits given up make picks inside one
// 256-ulp bucket come out in index order: the check below therefore compares the picks' TRUE logits (a wrong order
// shows as a negative gap), and holds the k-th pick against the upper end of the (k + 1)-th pick's bucket, above which
// nothing unpicked can lie.  One wave, k < n_expert <= 64 R, k + 1 <= 64; s_lv [64 R] floats of LDS scratch; lane i < k
// gets slot i's expert.
// (The sigmoid router picks by the score p + bias itself, so its keys ARE the exact router's: margin 0 - any strictly
// descending order is the router's - and no range to keep; `fin` then says that no logit and no score is non-finite.)
template <int R>
__device__ __forceinline__ bool route_wave_order_only(const float (&lv)[R], bool fin, int n_expert, int k, float* s_lv, float margin,
                                                      float range, int& my_id) {
    const int lane = threadIdx.x & 63;
    constexpr int kNone = (int) 0x80000000, kIndex = 64 * R - 1;
    int key[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int e = 64 * r + lane;
        const bool have = e < n_expert;
        key[r] = have ? (int) (((uint32_t) float_order_key(lv[r]) & ~(uint32_t) kIndex) | (uint32_t) (kIndex - e)) : kNone;
        fin = fin && (!have || isfinite(lv[r]));
        s_lv[e] = lv[r];
    }
    int my_key = kNone;
    for (int i = 0; i <= k; ++i) {
        int best = max(max(key[0], key[1]), max(key[2], key[3]));
#pragma unroll
        for (int r = 4; r < R; ++r) best = max(best, key[r]);
        const int top = wave_max_i32(best);
#pragma unroll
        for (int r = 0; r < R; ++r) key[r] = key[r] == top ? kNone : key[r];
        my_key = lane == i ? top : my_key;
    }
    const int id = kIndex - (my_key & kIndex);
    const float val = lane <= k ? s_lv[id] : 0.0f;
    const int ub_key = my_key | kIndex;
    const float ub = __int_as_float(ub_key >= 0 ? ub_key : ub_key ^ 0x7fffffff);   // the bucket's upper end
    const float nxt = __shfl_down(lane == k ? ub : val, 1, kWave);
    const float first = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(val), 0));
    const bool apart = lane >= k || (val - nxt > margin && first - nxt <= range);
    my_id = id;
    return __all(fin && apart) != 0;
}

}  // namespace maya
