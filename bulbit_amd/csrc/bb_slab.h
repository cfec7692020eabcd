// bb_slab.h — box tests of the traversal: RayCast's own, and those of the
// two-level records, whose boxes are rounded outwards and tested with a margin;
// shared by the kernels (kernels.hip), the scene set-up (host.cpp) and a
// host-side test (compiled with g++).  V is a vector of three floats x, y, z.
//
// The records are compressed wide nodes in the manner of Ylitie, Karras and
// Laine, "Efficient Incoherent Ray Traversal on GPUs Through Compressed Wide
// BVHs" (HPG 2017): an origin and a power of two per axis, a byte per plane.
#pragma once

#include <float.h>
#include <math.h>
#include <stdint.h>
#include <string.h>

#if defined(__HIPCC__)
#define BB_SLAB __host__ __device__ __forceinline__
#else
#define BB_SLAB inline
#endif

namespace bb
{

// ------------------------------------------------------------ the exact test

// AABB3::TestRay with precomputed inverse direction (bounding_box.h:443-484),
// split into the part that does not depend on t_max and the box's entry
// distance.
//
// The reference tests x, then y against the x-tightened interval, then z
// against the x,y-tightened interval, and ignores any NaN slab distance
// (every comparison with NaN is false).  Unrolled, it fails exactly when one
// of these pairs is out of order:
//   t_min  > t_max_i  (i = x, y, z)      t_min_i > t_max          (i = x, y, z)
//   t_min_i > t_max_j (i != j)
// (t_min is never compared with t_max, and t_min_i <= t_max_i always holds
// for one axis because both are computed with the same sign of inv.)  With
// NaN-ignoring max/min over the three axes, lo = max_i t_min_i and
// hi = min_i t_max_i, that is
//   fail = t_min > hi  or  lo > hi  or  lo > t_max.
// The first two do not involve t_max.  The last is monotone in t_max: a box
// that fails it fails again for any smaller t_max, and whether it passes
// later needs only lo, which does not change.
struct BoxHit
{
    bool ok;  // the t_max-independent part passed
    float lo; // entry distance: the box passes iff ok and !(lo > t_max)
};

template <class V>
BB_SLAB BoxHit box_part(V bmin, V bmax, V o, float t_min, V inv, bool n0, bool n1, bool n2)
{
    const float lx = ((n0 ? bmax.x : bmin.x) - o.x) * inv.x;
    const float hx = ((n0 ? bmin.x : bmax.x) - o.x) * inv.x;
    const float ly = ((n1 ? bmax.y : bmin.y) - o.y) * inv.y;
    const float hy = ((n1 ? bmin.y : bmax.y) - o.y) * inv.y;
    const float lz = ((n2 ? bmax.z : bmin.z) - o.z) * inv.z;
    const float hz = ((n2 ? bmin.z : bmax.z) - o.z) * inv.z;
    BoxHit h;
    h.lo = fmaxf(fmaxf(lx, ly), lz);
    const float hi = fminf(fminf(hx, hy), hz);
    h.ok = !((t_min > hi) | (h.lo > hi));
    return h;
}

BB_SLAB bool box_pass(BoxHit h, float t_max) { return h.ok && !(h.lo > t_max); }

// ------------------------------------------------------- tests with a margin

// The constants of a ray for box tests that need no division.  Planes are taken
// relative to the scene's centre c; with o' = o - c the slab distance of one at
// B' = B - c is
//   near = fma(B', inv, near0),  near0 = -o' inv - M
//   far  = fma(B', inv, far0),   far0  = -o' inv + M
// per axis, so that a box test passes whenever the exact one of a box inside
// does.
// half: every box lies within c +- half; rcp: 1 / d to one unit in the last
// place.
//
// With S = |o'| + half on an axis and u = 2^-24 the errors are, in units of
// u S |inv|: the record's planes three (quad_grid), o' one, the reciprocal two,
// near0 one, the two fused operations (quad_slabs, quad_entry) one each, the
// exact test's reciprocal, subtraction and product one each; M is 15.  It grows with the distance
// from the scene, not with the coordinates: a batch of 1 M rays on 328 K
// triangles takes 260 us wherever the scene lies (with planes as they are and
// M from |o|: 260 us around the origin, 1,540 moved by 10^4 on each axis, 22,600
// by 10^5).
//
// An axis the direction hardly moves along has an inverse so large that the
// distances overflow or, at the origin's own plane, are not a number; there
// |inv| is cut to 2^40 times the smallest of the three.  With t the distance at
// which the ray has left the scene, M is 4 t more on such an axis: a slab that
// holds the origin spans more than [-t, t] and decides nothing, as in the exact
// test, and one that the origin lies outside of by more than M's share still
// fails.
//
// False where this does not hold: for rays that
// are not finite, and for those whose distances or inverses come near the ends
// of the type's range.  Such a ray is tested exactly, on one-level records.  So
// is one that starts further than `far_away` from the scene (the sum over the
// axes), where M, 9e-7 of that distance, would pass too many boxes.
template <class V>
BB_SLAB bool slab_ray(V o, V rcp, V centre, V half, float far_away, V& inv, V& near0, V& far0)
{
    const float ox = o.x - centre.x, oy = o.y - centre.y, oz = o.z - centre.z;
    const float ax = fabsf(rcp.x), ay = fabsf(rcp.y), az = fabsf(rcp.z);
    const float sx = fabsf(ox) + half.x, sy = fabsf(oy) + half.y, sz = fabsf(oz) + half.z;
    const float least = fminf(fminf(ax, ay), az), most = least * 0x1p40f;
    const float s = sx + sy + sz, t = s * least;
    const float tiny = fmaf(most, 0x1p-125f, 1e-36f); // a grid's smallest step, and what underflows
    const float add = fmaf(4.0f, t, tiny);
    const bool cx = ax > most, cy = ay > most, cz = az > most;
    const float bx = cx ? most : ax, by = cy ? most : ay, bz = cz ? most : az;
    inv.x = copysignf(bx, rcp.x);
    inv.y = copysignf(by, rcp.y);
    inv.z = copysignf(bz, rcp.z);
    const float mx = fmaf(sx * bx, 9e-7f, cx ? add : tiny);
    const float my = fmaf(sy * by, 9e-7f, cy ? add : tiny);
    const float mz = fmaf(sz * bz, 9e-7f, cz ? add : tiny);
    near0.x = fmaf(-ox, inv.x, -mx);
    near0.y = fmaf(-oy, inv.y, -my);
    near0.z = fmaf(-oz, inv.z, -mz);
    far0.x = fmaf(-ox, inv.x, mx);
    far0.y = fmaf(-oy, inv.y, my);
    far0.z = fmaf(-oz, inv.z, mz);
    return (s < far_away) & (t < 1e20f) & (least > 1e-30f) & (least < 1e25f);
}

// The test of the scene's own box with the margin
template <class V>
BB_SLAB bool slab_root(V half, V inv, V near0, V far0, float t_min, float t_max)
{
    const float lo = fmaxf(fmaxf(fmaf(-half.x, fabsf(inv.x), near0.x), fmaf(-half.y, fabsf(inv.y), near0.y)),
                           fmaf(-half.z, fabsf(inv.z), near0.z));
    const float hi = fminf(fminf(fmaf(half.x, fabsf(inv.x), far0.x), fmaf(half.y, fabsf(inv.y), far0.y)),
                           fmaf(half.z, fabsf(inv.z), far0.z));
    return !((t_min > hi) | (lo > hi) | (lo > t_max));
}

// ---------------------------------------------------------- two-level records

// v 2^e
BB_SLAB float slab_scale(float v, int e)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_ldexpf(v, e);
#else
    return ldexpf(v, e);
#endif
}

// What the four entries of a record (SceneView::quads) share for one ray: the
// near and far distance of the grid's origin, the distance between its planes, and the packed rows of the planes that the ray meets first and last
template <class V>
struct QuadSlabs
{
    V n, f, s;
    uint32_t nx, ny, nz, fx, fy, fz;
};

// p: the grid's origin, e: its exponents, min and max: the entries' planes
template <class V>
BB_SLAB QuadSlabs<V> quad_slabs(V p, uint32_t e, uint32_t min_x, uint32_t min_y, uint32_t min_z, uint32_t max_x,
                                uint32_t max_y, uint32_t max_z, V inv, V near0, V far0, bool n0, bool n1, bool n2)
{
    QuadSlabs<V> q;
    q.n.x = fmaf(p.x, inv.x, near0.x);
    q.n.y = fmaf(p.y, inv.y, near0.y);
    q.n.z = fmaf(p.z, inv.z, near0.z);
    q.f.x = fmaf(p.x, inv.x, far0.x);
    q.f.y = fmaf(p.y, inv.y, far0.y);
    q.f.z = fmaf(p.z, inv.z, far0.z);
    q.s.x = slab_scale(inv.x, int8_t(e));
    q.s.y = slab_scale(inv.y, int8_t(e >> 8));
    q.s.z = slab_scale(inv.z, int8_t(e >> 16));
    q.nx = n0 ? max_x : min_x;
    q.fx = n0 ? min_x : max_x;
    q.ny = n1 ? max_y : min_y;
    q.fy = n1 ? min_y : max_y;
    q.nz = n2 ? max_z : min_z;
    q.fz = n2 ? min_z : max_z;
    return q;
}

// byte E of a packed row as a float
template <int E>
BB_SLAB float quad_byte(uint32_t row)
{
    return float((row >> (8 * E)) & 0xffu);
}

// entry E: false when the exact test of every box inside its own fails, else
// lo is at most the entry distance of each of them
template <int E, class V>
BB_SLAB bool quad_entry(const QuadSlabs<V>& q, float t_min, float t_max, float& lo)
{
    lo = fmaxf(fmaxf(fmaf(quad_byte<E>(q.nx), q.s.x, q.n.x), fmaf(quad_byte<E>(q.ny), q.s.y, q.n.y)),
               fmaf(quad_byte<E>(q.nz), q.s.z, q.n.z));
    const float hi = fminf(fminf(fmaf(quad_byte<E>(q.fx), q.s.x, q.f.x), fmaf(quad_byte<E>(q.fy), q.s.y, q.f.y)),
                           fmaf(quad_byte<E>(q.fz), q.s.z, q.f.z));
    return !((t_min > hi) | (lo > hi) | (lo > t_max));
}

// A record's grid, p + q 2^e on each axis relative to the scene's centre, and
// the entries' planes rounded outwards to it, a byte per entry (a missing entry
// gets an empty range); three axes, the fourth elements are of no use
struct QuadGrid
{
    float p[4];
    int32_t e[4];
    uint32_t lo[4], hi[4];
};

// box: the entries' boxes, bmin and bmax one after the other and one more float
// to be read (a missing entry repeats another); has: which entries there are.
// In floats, four at a time (three axes): the boxes' planes relative to the
// centre and to the grid's origin are rounded, by 3 u of what slab_ray's S is,
// which its margin holds.  In doubles, one axis after the other, the records of
// 5,200 triangles took 240 us of the host's time, and take 95.
inline QuadGrid quad_grid(const float* const box[4], const bool has[4], const float centre[3])
{
    typedef float f4 __attribute__((vector_size(16)));
    typedef int32_t i4 __attribute__((vector_size(16)));
    const f4 c = { centre[0], centre[1], centre[2], 0.0f };
    f4 bmin[4], bmax[4];
    for (int k = 0; k < 4; ++k) {
        memcpy(&bmin[k], box[k], 16);
        memcpy(&bmax[k], box[k] + 3, 16);
        bmin[k] -= c;
        bmax[k] -= c;
    }
    f4 p = bmin[0], top = bmax[0];
    for (int k = 1; k < 4; ++k) {
        p = bmin[k] < p ? bmin[k] : p;
        top = bmax[k] > top ? bmax[k] : top;
    }
    // 2^e > (top - p) / 254, from the exponent bits; the planes then end at 255
    const f4 step = (top - p) * (1.0f / 254.0f), zero = { 0.0f, 0.0f, 0.0f, 0.0f };
    i4 e = ((i4)step >> 23) - 126;
    e = step > zero ? e : (i4)zero;
    e = e < -126 ? (i4)zero - 126 : e;
    e = e > 126 ? (i4)zero + 126 : e;
    const f4 inv = (f4)((127 - e) << 23); // 2^-e
    i4 lo = { 0, 0, 0, 0 }, hi = { 0, 0, 0, 0 };
    const f4 last = { 255.0f, 255.0f, 255.0f, 255.0f };
    for (int k = 0; k < 4; ++k) {
        // (outside [0, 255] only for a box that is inverted, which no ray meets,
        // or not finite, as then the scene's is and no ray walks its records)
        f4 x = (bmin[k] - p) * inv, y = (bmax[k] - p) * inv;
        x = x > zero ? x : zero;
        x = x < last ? x : last;
        y = y > zero ? y : zero;
        y = y < last ? y : last;
        const i4 a = __builtin_convertvector(x, i4);
        i4 b = __builtin_convertvector(y, i4);
        b -= __builtin_convertvector(b, f4) < y; // (true is -1)
        lo |= (has[k] ? a : (i4)zero + 255) << (8 * k);
        hi |= (has[k] ? b : (i4)zero) << (8 * k);
    }
    QuadGrid g;
    memcpy(g.p, &p, 16);
    memcpy(g.e, &e, 16);
    memcpy(g.lo, &lo, 16);
    memcpy(g.hi, &hi, 16);
    return g;
}

// The largest distance from `centre` of a plane of [bmin, bmax], rounded up
inline float slab_half(float bmin, float bmax, float centre)
{
    const double a = double(centre) - bmin, b = double(bmax) - centre;
    const double d = a > b ? a : b;
    const float f = float(d);
    return double(f) < d ? nextafterf(f, INFINITY) : f;
}

} // namespace bb
