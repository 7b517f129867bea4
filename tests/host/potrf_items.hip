// The numbering of a POTRF tile's items and flags (ttad_types.hpp): for each tile size given, a line "n items flags fin"
// and a line "r q tail flag(r, r) flag(r, q)" per item (the last one -1 in row 0).
#include <cstdio>
#include <cstdlib>

#include <hip/hip_runtime.h>

#include "ttad_types.hpp"

using namespace ttad;

int main(int argc, char** argv) {
    for (int a = 1; a < argc; a++) {
        const int n = atoi(argv[a]);
        printf("%d %d %d %d\n", n, potrf_items(n), potrf_flags(n), potrf_fin(n));
        for (int it = 0; it < potrf_items(n); it++) {
            const PotrfItem p = potrf_item(it);
            printf("%d %d %d %d %d\n", p.r, p.q, (int)p.tail, potrf_flag(p.r, p.r), p.q < 0 ? -1 : potrf_flag(p.r, p.q));
        }
    }
    return 0;
}
