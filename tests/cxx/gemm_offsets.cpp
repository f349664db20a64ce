// Walks the Q8 GEMM's range-checked loads over tiles with partial rows, tokens and steps (the offset functions of
// kernels.hpp) and counts loads that pass the resource's check although they lie past its end, that are refused
// although they belong to the operand, or that address another element than meant. Exit status 1 after any.
#include <algorithm>
#include <cstdio>

#include "kernels.hpp"

int main() {
    int loads = 0, faults = 0;
    auto check = [&](unsigned off, int bytes, unsigned records, bool belongs, unsigned long long want) {
        loads++;
        const bool passes = off < records;  // what the range check lets through
        if (passes != belongs || (passes && (off + bytes > records || off != want))) faults++;
    };
    for (int cols : {32, 64, 96, 160, 2048, 2080, 1 << 22})
        for (int pad : {0, 4, 1000})
            for (int nr : {1, 100, 127, 128, 129, 214, 255, 256})
                for (int nt : {1, 6, 31, 32, 33, 96, 127, 128}) {
                    const int stride = std::min(cols, 3000000) + pad, nkb = cols / 32;
                    if (stride < cols) continue;  // strides that the other kernels take
                    if (!qw::gemm_offsets_fit(cols, stride)) faults++;
                    const unsigned wr = nr * cols, sr = nr * nkb * 4, xr = ((nt - 1) * stride + cols) * 4;
                    for (int k : {0, 1, (nkb + 1) / 2 - 1}) {  // the last step: half of one where nkb is odd
                        if (2 * k >= nkb) continue;
                        for (int row : {0, 1, nr - 1, nr, nr + 1, 255})
                            if (row >= 0 && row < 256) {
                                for (int q = 0; q < 4; q++)
                                    check(qw::gemm_w_off(row, q, k, cols, nkb), 16, wr, row < nr && 64 * k + 16 * q < cols,
                                          (unsigned long long)row * cols + 64 * k + 16 * q);
                                for (int j = 0; j < 2; j++)
                                    check(qw::gemm_s_off(row, j, k, nkb), 4, sr, row < nr && 2 * k + j < nkb,
                                          4ull * (row * nkb + 2 * k + j));
                            }
                        for (int tok : {0, 1, nt - 1, nt, nt + 1, 127})
                            if (tok >= 0 && tok < 128)
                                for (int q = 0; q < 16; q++)
                                    check(qw::gemm_x_off(tok, q, k, stride, nkb), 16, xr, tok < nt && 64 * k + 4 * q < cols,
                                          4ull * ((unsigned long long)tok * stride + 64 * k + 4 * q));
                    }
                }
    std::printf("loads %d faults %d\n", loads, faults);
    return faults || !loads;
}
