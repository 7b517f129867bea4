// Which raw TRSM calls take the strips in LDS (ttad_types.hpp): a line "elem_bytes m n form" per triple of arguments.
#include <cstdio>
#include <cstdlib>

#include <hip/hip_runtime.h>

#include "ttad_types.hpp"

int main(int argc, char** argv) {
    for (int a = 1; a + 2 < argc; a += 3) {
        const int es = atoi(argv[a]), m = atoi(argv[a + 1]), n = atoi(argv[a + 2]);
        printf("%d %d %d %d\n", es, m, n, (int)ttad::trsm_in_lds(es, m, n));
    }
    return 0;
}
