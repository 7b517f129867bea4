// The addresses of the TRSM items that keep X in LDS (ttad_types.hpp), against 64-bit arithmetic: every wave and column
// of a block, whole and ragged, up to the largest leading dimension that takes this form. Prints the number of
// addresses compared and exits with 1 at the first wrong one.
#include <cstdio>

#include <hip/hip_runtime.h>

#include "ttad_types.hpp"

using namespace ttad;

int main() {
    long cases = 0;
    for (int es : {4, 8})
        for (long ldx : {1L, 64L, 513L, (1L << 22) + 1, 1L << 23, 8521761L, TRSM_LDS_MAX_LD - 1})
            for (int cw : {1, 15, 16, 17, 33, 48, 63, 64})
                for (int w = 0; w < 4; w++)
                    for (int c = 0; c < 16; c++)
                        for (int row : {0, 15, 31}) {
                            const int col = 16 * w + c < cw ? 16 * w + c : cw - 1;
                            const long want = (row + (long)col * ldx) * es;
                            const long got = (long)trsm_wave_col(w, cw) * ldx * es + trsm_lane_offset(row, c, w, cw, ldx, es);
                            if (got != want) {
                                printf("es %d ldx %ld cw %d wave %d c %d row %d: %ld, not %ld\n", es, ldx, cw, w, c, row, got, want);
                                return 1;
                            }
                            cases++;
                        }
    printf("%ld\n", cases);
    return 0;
}
