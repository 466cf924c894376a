// The gated product of a feed-forward's two halves for many rows (skyrl_gated_product): both products and the activation in
// one launch (wide.h).
#include "wide.h"

using namespace skyrl;

// Where it is the faster one: from three quarters of a round of workgroups on. Against the library's product and gate_mul, us,
// n x K rows and N: 8192 x 2048, 6144: 321 against 366; 6000: 255, 345; 4096: 166, 189; 1024: 51, 59; 512 (96 items): 49, 39.
// 3000 x 4096, 12288: 469, 614; 512: 87, 96; 384: 83, 81. 4096 x 1536, 8960: 204, 231; 512: 37, 45.
extern "C" int32_t skyrl_gated_product_fits(int32_t n, int32_t K, int32_t N) {
    return n >= 512 && N > 0 && wide_fits(K, N, true) && (int64_t)((n + 255) / 256) * (N / 128) >= kCUs * 3 / 4;
}

extern "C" int skyrl_gated_product(const void* x, int64_t ldx, int32_t n, int32_t K, const void* w, int64_t ldw, int32_t N,
                                   int32_t act, float alpha, float limit, void* out, void* stream) {
    SKYRL_REQUIRE(n > 0 && N > 0 && wide_fits(K, N, true), "gated_product: K must be a multiple of 64, N of 128");
    SKYRL_REQUIRE(x && w && out, "gated_product: null pointer");
    SKYRL_REQUIRE(act == SKYRL_ACT_SILU || act == SKYRL_ACT_GELU_TANH || act == SKYRL_ACT_CLAMPED, "gated_product: act");
    SKYRL_REQUIRE(aligned16(x) && aligned16(w) && aligned16(out) && ldx % 8 == 0 && ldw % 8 == 0 && ldw >= K && (n == 1 || ldx >= K),
                  "gated_product: rows must be 16-byte aligned");
    const Wide p{reinterpret_cast<const uint16_t*>(x), reinterpret_cast<const uint16_t*>(w), reinterpret_cast<uint16_t*>(out), K, N,
                 ldx, ldw, (n + 255) / 256, nullptr, nullptr, 1, 0, 0, nullptr, n, 256, Gate{act, alpha, limit}};
    if (act == SKYRL_ACT_SILU) return launch_wide<kGated, SKYRL_ACT_SILU>(p, as_stream(stream));
    if (act == SKYRL_ACT_CLAMPED) return launch_wide<kGated, SKYRL_ACT_CLAMPED>(p, as_stream(stream));
    return launch_wide<kGated, SKYRL_ACT_GELU_TANH>(p, as_stream(stream));
}
