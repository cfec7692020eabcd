// bb_index.h — index arithmetic of the kernels that has to hold up to the
// largest images and batches a call accepts; shared by the kernels
// (kernels.hip) and a host-side test (compiled with g++).
#pragma once

#include <stddef.h>

#if defined(__HIPCC__)
#define BB_INDEX __host__ __device__ inline
#else
#define BB_INDEX inline
#endif

namespace bb
{

// Pixel number q (below width * height, at most 2^30) of the path order: down
// strips 8 pixels wide, row by row within a strip, so that 64 pixels in a row
// are an 8 x 8 square.  With the samples of a pixel next to each other too,
// the rays in flight at one time come from one small part of the image, and so
// do their first bounces: the traversal kernels read a quarter less from
// memory, and shading's lanes meet the same material more often (24 of 64
// active instead of 21).  The 1080p frame of 64 spp takes 66.3 instead of
// 68.4 ms, the textured 801 x 451 frame of 8 spp 6.6 instead of 7.2, the batch
// of 8 scenes 64.8 instead of 66.4.
BB_INDEX void order_pixel(int width, int height, int q, int& px, int& py)
{
    // (a narrower image is one strip of its own width: 8 * height would not
    // fit in 32 bits for the tallest of them, and no path order needs it)
    const int per_strip = (width < 8 ? width : 8) * height;
    const int strip = q / per_strip, r = q - strip * per_strip;
    const int left = width - 8 * strip;
    const int w = left < 8 ? left : 8;
    py = w == 8 ? r >> 3 : r / w;
    px = 8 * strip + r - py * w;
}

// where ray i of a batch starts in an array of 16-byte vectors, two to a ray
BB_INDEX size_t ray_at(int i) { return 2 * size_t(i); }

// where pixel p starts in a film's sums, three floats to a pixel
BB_INDEX size_t film_at(int p) { return 3 * size_t(p); }

// the query that an idle lane takes from its wave's claimed ones, [rb, re), as
// the rank-th of the idle lanes (0 to 63); -1 when there are not that many
BB_INDEX int claim(int rb, int re, int rank) { return rank < re - rb ? rb + rank : -1; }

// the first claimed query left over once n_idle lanes (up to 64) have taken theirs
BB_INDEX int claims_left(int rb, int re, int n_idle) { return n_idle < re - rb ? rb + n_idle : re; }

} // namespace bb
