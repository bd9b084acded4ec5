// The gated short convolution of one channel at batch 1, as the epilogue of the GEMVs that compute its b, c and x
// (gemv.hip, gemv_w4.hip): conv_step's arithmetic and roundings (step.hip), so the same bits.
#pragma once
#include "common.hpp"

namespace lfm2q {

struct ConvArgs {
    uint16_t *ring;        // [L, H]: b x of the last L positions, position p in row p mod L
    const uint16_t *wt;    // [L, H]
    const uint16_t *bias;  // [H] or null
    const int64_t *ctr;    // the position
};

constexpr int CONV_L = 3;  // taps of the fused form (LFM2's conv_L_cache)

// One channel's operands, loaded ahead of the GEMV's weights
struct ConvChannel {
    uint32_t ring[CONV_L], w[CONV_L], bias;
    int r;
    __device__ __forceinline__ void load(const ConvArgs &a, int n, int H) {
#pragma unroll
        for (int s = 0; s < CONV_L; ++s) {
            ring[s] = a.ring[(size_t)s * H + n];
            w[s] = a.wt[(size_t)s * H + n];
        }
        bias = a.bias ? a.bias[n] : 0u;
        r = (int)((a.ctr[0] % CONV_L + CONV_L) % CONV_L);
    }
    // b, c, x: the projection's bf16 values; stores the ring's new row and returns the gated output
    __device__ __forceinline__ uint16_t finish(const ConvArgs &a, int n, int H, float b, float c, float x) const {
#pragma clang fp contract(off)
        const uint32_t u = f2bf(b * x);
        a.ring[(size_t)r * H + n] = (uint16_t)u;
        float y = 0.f;
#pragma unroll
        for (int s = 0; s < CONV_L; ++s) {
            const uint32_t v = s == r ? u : ring[s];
            const int tap = s <= r ? CONV_L - 1 - (r - s) : s - r - 1;
            uint32_t wv = w[0];
#pragma unroll
            for (int k = 1; k < CONV_L; ++k)
                if (k == tap) wv = w[k];
            y += rbf(bf2f(v) * bf2f(wv));
        }
        y = rbf(y);
        if (a.bias) y = rbf(y + bf2f(bias));
        return (uint16_t)f2bf(c * y);
    }
};

}  // namespace lfm2q
