// The gated product of a feed-forward's two halves for many rows (skyrl_gated_product): both products and the activation in
// one launch (wide.h).
#include "wide.h"

using namespace skyrl;

// Where it is the faster one. From 512 rows, by tiles of 256, from three quarters of a round of workgroups on. Against the library's
// product and gate_mul, us, n x K rows and N: 8192 x 2048, 6144: 297 against 366; 1024: 51, 59; 512 (96 items): 49, 39. 3000 x 4096, 12288:
// 469, 614; 512: 87, 96; 384: 83, 81. 4096 x 1536, 8960: 204, 231; 512: 37, 45.
// Below, by tiles of 64, against the library's and gate_mul, weights from HBM. In one round: 65 / 128 x 2048, 6144 21.3 / 22.1 against 21.5 /
// 23.1; 128, 256, 400 x 1536, 4608 12.2, 16.5, 19.3 against 17.4, 23.0, 28.8. An eighth more only of shallow products: 450 / 511 x 768, 4608
// 16.6 / 16.8 against 19.9 / 24.6, 256 x 768, 9216 16.9 against 22.2; but 289 x 1024, 7168 23.2 against 20.4, 450 x 1536, 4608 25.7
// against 24.8. Not 192 x 2048, 6144: 28.7, 27.9; 256 x 2048, 2048: 14.6, 13.6; 128 x 4096, 12288: 65, 61.
static bool few_rows(int32_t n, int32_t K, int32_t N) {
    return n > 64 && n < 512 && K <= (n <= 128 ? 2048 : 1536) && N >= 4096
           && (int64_t)((n + 63) / 64) * (N / 128) <= (K <= 768 ? kCUs * 9 / 8 : kCUs);
}
extern "C" int32_t skyrl_gated_product_fits(int32_t n, int32_t K, int32_t N) {
    if (N <= 0 || !wide_fits(K, N, true)) return 0;
    return few_rows(n, K, N) || (n >= 512 && (int64_t)((n + 255) / 256) * (N / 128) >= kCUs * 3 / 4);
}

extern "C" int skyrl_gated_product(const void* x, int64_t ldx, int32_t n, int32_t K, const void* w, int64_t ldw, int32_t N,
                                   int32_t act, float alpha, float limit, void* out, void* stream) {
    SKYRL_REQUIRE(n > 0 && N > 0 && wide_fits(K, N, true), "gated_product: K must be a multiple of 64, N of 128");
    SKYRL_REQUIRE(x && w && out, "gated_product: null pointer");
    SKYRL_REQUIRE(act == SKYRL_ACT_SILU || act == SKYRL_ACT_GELU_TANH || act == SKYRL_ACT_CLAMPED, "gated_product: act");
    SKYRL_REQUIRE(aligned16(x) && aligned16(w) && aligned16(out) && ldx % 8 == 0 && ldw % 8 == 0 && ldw >= K && (n == 1 || ldx >= K),
                  "gated_product: rows must be 16-byte aligned");
    const int rows = few_rows(n, K, N) ? 64 : 256;
    const Wide p{reinterpret_cast<const uint16_t*>(x), reinterpret_cast<const uint16_t*>(w), reinterpret_cast<uint16_t*>(out), K, N,
                 ldx, ldw, (n + rows - 1) / rows, nullptr, nullptr, 1, 0, 0, nullptr, n, rows, Gate{act, alpha, limit}};
    auto launch = [&](auto a) {
        if (rows == 64) return launch_wide<kGated, a, false, 64>(p, as_stream(stream));
        return launch_wide<kGated, a>(p, as_stream(stream));
    };
    if (act == SKYRL_ACT_SILU) return launch(std::integral_constant<int, SKYRL_ACT_SILU>{});
    if (act == SKYRL_ACT_CLAMPED) return launch(std::integral_constant<int, SKYRL_ACT_CLAMPED>{});
    return launch(std::integral_constant<int, SKYRL_ACT_GELU_TANH>{});
}
