// The gated products of a feed-forward's two halves (SKYRL_ACT_*).
#pragma once
#include "elem.h"

namespace skyrl {

struct Gate {
    int act;
    float alpha, limit;  // of the clamped form
};

// The gated product of one pair.
__device__ __forceinline__ float gated(float g, float u, const Gate& f) {
    if (f.act == SKYRL_ACT_SILU) return siluf_(g) * u;
    if (f.act == SKYRL_ACT_CLAMPED) {
        g = fminf(g, f.limit);
        u = fminf(fmaxf(u, -f.limit), f.limit);
        return g / (1.f + expf(-f.alpha * g)) * (u + 1.f);
    }
    return 0.5f * g * (1.f + tanhf(0.7978845608028654f * (g + 0.044715f * g * g * g))) * u;
}

}  // namespace skyrl
