// Which raw GEMM / SYRK calls take 64x64 items (ttad_types.hpp): a line "prec m n k syrk small" per five arguments.
#include <cstdio>
#include <cstdlib>

#include <hip/hip_runtime.h>

#include "ttad_types.hpp"

int main(int argc, char** argv) {
    for (int a = 1; a + 4 < argc; a += 5) {
        int v[5];
        for (int q = 0; q < 5; q++) v[q] = atoi(argv[a + q]);
        printf("%d %d %d %d %d %d\n", v[0], v[1], v[2], v[3], v[4], (int)ttad::raw_gemm_small(v[0], v[1], v[2], v[3], v[4] != 0));
    }
    return 0;
}
