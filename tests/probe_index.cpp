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
        } else if (!std::strcmp(what, "ray") || !std::strcmp(what, "film")) { // number -> place
            int i;
            if (std::scanf("%d", &i) != 1) return 1;
            std::printf("%zu\n", what[0] == 'r' ? bb::ray_at(i) : bb::film_at(i));
        } else if (!std::strcmp(what, "claim")) { // rb re n -> the n-th lane's query, the first one left
            int rb, re, n;
            if (std::scanf("%d %d %d", &rb, &re, &n) != 3) return 1;
            std::printf("%d %d\n", bb::claim(rb, re, n), bb::claims_left(rb, re, n));
        }
    }
    return 0;
}
