// Device code of the router top-k shared by the stand-alone route kernel, the router's scoring kernel and the fused route + pack kernel.
#pragma once
#include "common.h"

namespace dmoe {

// Monotone u32 key of an f32 for "ascending stable argsort, NaN last, -0 == +0".
// Never returns 0, so 0 can mark an entry that was already taken.
__device__ __forceinline__ uint32_t f32_sort_key(float c) {
    const uint32_t b = __float_as_uint(c);
    uint32_t k = (b & 0x80000000u) ? ~b : (b | 0x80000000u); // selects: a branch per register would be on the rounds' path
    k = c == 0.0f ? 0x80000000u : k;
    return c != c ? 0xffffffffu : k;
}

// v <- the larger of this lane's v and that of the lane the DPP control selects (one v_max_u32)
template <int CTRL>
__device__ __forceinline__ uint32_t route_max_step(uint32_t v) {
    const uint32_t o = (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, CTRL, 0xf, 0xf, false);
    return o > v ? o : v;
}

// The selection bias and the Smelt mask of a lane's experts l, l + 64, ...: every entry is requested before the first is used
// (one after the other they are eight round trips to memory), and by callers ahead of their own work.
template <int EPL>
struct RouteBias {
    float b[EPL];
    uint32_t on[EPL];
    bool has_bias, has_mask;
    __device__ __forceinline__ void load(const float *__restrict__ bias, const uint8_t *__restrict__ resident, int E, int lane) {
        has_bias = bias != nullptr, has_mask = resident != nullptr;
        if (has_bias) {
#pragma unroll
            for (int i = 0; i < EPL; ++i) b[i] = bias[lane + 64 * i < E ? lane + 64 * i : 0]; // loads stay in bounds and unconditional
        }
        if (has_mask) {
#pragma unroll
            for (int i = 0; i < EPL; ++i) on[i] = resident[lane + 64 * i < E ? lane + 64 * i : 0];
        }
    }
};

// One wavefront routes one token. Lane l holds the scores of experts l, l + 64, ... (EPL of them, E <= 64 * EPL; `sc`) and their
// keys. K rounds of a wave-wide maximum over the keys; round r fills column K-1-r, so the columns come out in ascending score
// order. Of experts with the same key the HIGHEST index wins - what "take the last K columns of a stable ascending argsort"
// selects: a ballot per register finds the winner behind the maximum. Lane j < K returns column j. Straight-line code.
// (A launch of a few tokens is as long as its one chain of memory round trips and dependent instructions. With bias and mask
// entries fetched one after the other, (key, index) pairs as 64-bit numbers, three instructions per comparison, and the winners'
// scores read back from memory, us per step or block, with the combine's rows one by one too: one token 34.8, block 44.1; now
// 33.4 and 41.9.)
template <int EPL>
__device__ __forceinline__ void route_from_registers(const float (&sc)[EPL], const RouteBias<EPL> &sel, int E, int K, int normalize,
                                                     int apply_scale, float route_scale, int lane, uint32_t &my_idx,
                                                     float &w) {
    uint32_t key[EPL];
#pragma unroll
    for (int i = 0; i < EPL; ++i) {
        float c = sc[i];
        c = sel.has_bias ? c + sel.b[i] : c;
        c = sel.has_mask ? c + (sel.on[i] ? 0.0f : -1e9f) : c;
        key[i] = lane + 64 * i < E ? f32_sort_key(c) : 0u; // 0 never wins: real keys are never 0
    }
    my_idx = 0;
    for (int it = 0; it < K; ++it) {
        uint32_t best = key[0];
#pragma unroll
        for (int i = 1; i < EPL; ++i) best = key[i] > best ? key[i] : best;
        // four cross-lane steps inside each row of 16 lanes (after them every lane holds its row's maximum), then the four
        // rows through scalar registers
        best = route_max_step<0xB1>(best);  // lane ^ 1 (quad_perm 1,0,3,2)
        best = route_max_step<0x4E>(best);  // lane ^ 2 (quad_perm 2,3,0,1)
        best = route_max_step<0x141>(best); // the other quad of each eight lanes (row_half_mirror)
        best = route_max_step<0x140>(best); // the other half of the row (row_mirror)
        uint32_t top = 0;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const uint32_t v = (uint32_t)__builtin_amdgcn_readlane((int)best, 16 * r);
            top = v > top ? v : top;
        }
        uint32_t bi = 0; // the winner's expert index, uniform
#pragma unroll
        for (int i = 0; i < EPL; ++i) {
            const uint64_t at = __ballot(key[i] == top);
            bi = at ? (uint32_t)(64 * i + 63 - __clzll((long long)at)) : bi;
        }
#pragma unroll
        for (int i = 0; i < EPL; ++i) key[i] = (bi == (uint32_t)(lane + 64 * i)) ? 0u : key[i]; // taken
        my_idx = (lane == K - 1 - it) ? bi : my_idx;
    }
    // the winners' unbiased scores: expert bi sits in register bi / 64 of lane bi % 64
    float my_w = 0.0f;
#pragma unroll
    for (int i = 0; i < EPL; ++i) {
        const float got = __shfl(sc[i], (int)(my_idx & 63u), 64);
        my_w = (my_idx >> 6) == (uint32_t)i ? got : my_w;
    }
    my_w = lane < K ? my_w : 0.0f;
    float sum = 0.0f;
    for (int c = 0; c < K; ++c) sum += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(my_w), c)); // left to right, like a row reduction
    float v = my_w;
    if (normalize) v = v / (sum + 1e-20f);
    if (apply_scale) v = v * route_scale;
    w = v;
}

// the same from the E scores of a token in memory
template <int EPL>
__device__ __forceinline__ void route_token(const float *__restrict__ s, const float *__restrict__ bias,
                                            const uint8_t *__restrict__ resident, int E, int K, int normalize, int apply_scale,
                                            float route_scale, int lane, uint32_t &my_idx, float &w) {
    float sc[EPL];
#pragma unroll
    for (int i = 0; i < EPL; ++i) sc[i] = s[lane + 64 * i < E ? lane + 64 * i : 0];
    RouteBias<EPL> sel;
    sel.load(bias, resident, E, lane);
    route_from_registers<EPL>(sc, sel, E, K, normalize, apply_scale, route_scale, lane, my_idx, w);
}

} // namespace dmoe
