// Host build of the kernels' index arithmetic (bulbit_amd/csrc/bb_index.h):
// reads lines of a name and numbers, prints the results.
#include <cstdio>
#include <cstring>

#include "../bulbit_amd/csrc/bb_index.h"

int main()
{
    char what[16];
    while (std::scanf("%15s", what) == 1) {
        if (!std::strcmp(what, "pixel")) { // width height q -> px py
            int w, h, q, px = 0, py = 0;
            if (std::scanf("%d %d %d", &w, &h, &q) != 3) return 1;
            bb::order_pixel(w, h, q, px, py);
            std::printf("%d %d\n", px, py);
        }
    }
    return 0;
}
