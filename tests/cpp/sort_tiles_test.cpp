// The tiles that a sort's workspace is sized for are those of the kernel that is
// launched for it: for every number of keys, digits of 9 bits run on tiles of 1024
// threads, and those of 8 bits on 256, 512 or 1024.
#include "dgx_common.h"

#include <cstdio>

int main() {
    int bad = 0;
    for (int lg = 13; lg <= 28; ++lg)
        for (long long d = -1; d <= 1; ++d) {
            const size_t n = (size_t)((1ll << lg) + d);
            const int t8 = sort_threads(n, 8);
            bad += sort_threads(n, 9) != 1024;
            bad += t8 != 256 && t8 != 512 && t8 != 1024;
        }
    printf("%d failures\n", bad);
    return bad != 0;
}
