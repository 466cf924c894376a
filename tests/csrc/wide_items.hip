// Test hook (never in the product libraries): which items of a launch of wide_kernel (csrc/wide.h) its workgroups take, for
// tests/test_wide_items.py.
#include "../../skyrl_amd/csrc/wide.h"

// Of a launch for up to `launched` items, of which there are `items`. seen[2 items]: how often the first and the second half of an
// item's columns is taken. Returns the most halves that a workgroup takes.
extern "C" int skyrl_test_wide_items(int64_t launched, int64_t items, int32_t* seen) {
    const int grid = skyrl::wide_grid(launched);
    int most = 0;
    for (int b = 0; b < grid; ++b) {
        const skyrl::Share share(items, grid, b);
        int halves = 0;
        for (int i = 0; i < share.mine; ++i) {
            const int it = share.nth(i), half = share.half_of(i);
            if (it < 0 || it >= items) return -1;
            for (int k = 0; k < 2; ++k)
                if (half != 2 - k) ++seen[2 * it + k], ++halves;
        }
        most = halves > most ? halves : most;
    }
    return grid % 8 == 0 && grid <= skyrl::kCUs ? most : -1;
}
