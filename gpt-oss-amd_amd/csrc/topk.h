// Top-k and softmax of one token by one wave, shared by the router kernels and the gate/up kernels that do it themselves.
#pragma once
#include "common.h"

namespace moe {
namespace {

// These kernels run their code once per wave, so their time is instruction fetch as much as
// anything: loops stay rolled (the round and segment counts are wave-uniform anyway).
//
// Sort key of a score: larger key = better candidate.  The score's bits mapped to an unsigned integer in score order (-0
// counts as +0, as in the reference's float comparison); key 0 is "nothing".
MOE_DEVICE uint32_t rank_key(float v) {
    const uint32_t u = __float_as_uint(v + 0.f);
    return max(u ^ ((uint32_t)((int32_t)u >> 31) | 0x80000000u), 1u);
}
MOE_DEVICE float rank_key_value(uint32_t m) { return __uint_as_float((m & 0x80000000u) ? m ^ 0x80000000u : ~m); }

// K rounds of wave-wide argmax over vals[0..E), E <= 64 C, ordered by (value desc, index asc).  Lane r < K ends up holding the
// winner of round r in (my_v, my_i).  The keys stay in registers (read anew in every round, for more than 128 experts : so, 64
// tokens, us: 256 experts, K = 8 10.2 : 5.2; 512, K = 4 10.8 : 5.5; 1000, K = 8 29 : 9.0).
// A round is a chain of dependent instructions and little else: the maximum of the 32-bit keys is one instruction per DPP
// step, and the lowest index that has it comes from a ballot.  (A 64-bit key with the index in it took five instructions a
// step: 850 cycles a round, 200 now.)
template <int C>
MOE_DEVICE void select_topk_of(const float* vals, int E, int K, int lane, float& my_v, int& my_i) {
    uint32_t key[C];
#pragma unroll
    for (int c = 0; c < C; ++c) key[c] = lane + 64 * c < E ? rank_key(vals[lane + 64 * c]) : 0u;
    my_v = -INFINITY;
    my_i = 0;
#pragma nounroll
    for (int r = 0; r < K; ++r) {
        uint32_t best = 0;
#pragma unroll
        for (int c = 0; c < C; ++c) best = max(best, key[c]);
#define MOE_STEP(CTRL, M) best = max(best, dpp_move<CTRL, M>(0u, best));
        MOE_DPP_STEPS(MOE_STEP)
#undef MOE_STEP
        best = __builtin_amdgcn_readlane(best, 63);
        int bi = 0;
        if constexpr (C <= 2) {
#pragma unroll
            for (int c = C - 1; c >= 0; --c) {
                const unsigned long long has = __ballot(key[c] == best);
                if (has) bi = 64 * c + (int)__builtin_ctzll(has);
            }
        } else {  // as many ballots would fill the scalar registers
            uint32_t miss = 0;  // ~index, or 0
#pragma unroll
            for (int c = C - 1; c >= 0; --c) miss = key[c] == best ? ~(uint32_t)(64 * c + lane) : miss;
#define MOE_STEP(CTRL, M) miss = max(miss, dpp_move<CTRL, M>(0u, miss));
            MOE_DPP_STEPS(MOE_STEP)
#undef MOE_STEP
            bi = (int)~(uint32_t)__builtin_amdgcn_readlane(miss, 63);
        }
#pragma unroll
        for (int c = 0; c < C; ++c) key[c] = bi == lane + 64 * c ? 0u : key[c];
        if (lane == r) {
            my_v = rank_key_value(best);
            my_i = bi;
        }
    }
}

// E <= 1024
MOE_DEVICE void select_topk(const float* vals, int E, int K, int lane, float& my_v, int& my_i) {
    if (E <= 64) select_topk_of<1>(vals, E, K, lane, my_v, my_i);  // wave-uniform
    else if (E <= 128) select_topk_of<2>(vals, E, K, lane, my_v, my_i);
    else if (E <= 256) select_topk_of<4>(vals, E, K, lane, my_v, my_i);
    else if (E <= 512) select_topk_of<8>(vals, E, K, lane, my_v, my_i);
    else select_topk_of<16>(vals, E, K, lane, my_v, my_i);
}

MOE_DEVICE float lane_value(float v, int src_lane) {
    return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), src_lane));
}

// Softmax of src/run.cpp:321-339 over the K selected values in its own order of operations (max,
// then exponentials, then their fp64 sum in index order), or the values themselves; lane r < K
// stores entry r.
MOE_DEVICE void write_topk(float my_v, int my_i, int K, int lane, int do_softmax, float* __restrict__ out_v,
                           int* __restrict__ out_i) {
    float o = my_v;
    if (do_softmax) {
        // the first of the selected values is the largest (or not a number, which no other compares greater than)
        const double max_val = lane_value(my_v, 0);
        const float ex = expf((float)((double)my_v - max_val));
        double sum = 0.0;
#pragma nounroll
        for (int r = 0; r < K; ++r) sum += (double)lane_value(ex, r);
        o = (float)((double)ex / sum);
    }
    if (lane < K) {
        out_v[lane] = o;
        out_i[lane] = my_i;
    }
}

}  // namespace
}  // namespace moe
