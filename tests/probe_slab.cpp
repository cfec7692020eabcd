// Host build of the traversal's box tests (bulbit_amd/csrc/bb_slab.h): random
// boxes, the records that hold them and rays of one kind, the tests with a
// margin against the exact one.  Arguments: scene kind, ray kind, seed.
// Prints, over all rays: the box tests, those that the exact test passes, those
// of rays with margins, then what may not happen, an entry (or the scene's box)
// that fails though the exact test passes or whose entry distance is larger, and
// the boxes that pass with the margin only.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <vector>

#include "../bulbit_amd/csrc/bb_slab.h"

struct V
{
    float x, y, z;
    float& operator[](int i) { return i == 0 ? x : (i == 1 ? y : z); }
    float operator[](int i) const { return i == 0 ? x : (i == 1 ? y : z); }
};

static std::mt19937_64 g;
static double uni(double a, double b) { return std::uniform_real_distribution<double>(a, b)(g); }
static int pick(int n) { return int(uni(0, n)); }

// 1 / d as the hardware gives it: one unit in the last place off, results and
// inputs below the normal range flushed
static float rcp(float d)
{
    if (std::isnan(d)) return d;
    if (std::fabs(d) < FLT_MIN) return std::copysign(INFINITY, d);
    float r = 1.0f / d;
    if (std::fabs(r) < FLT_MIN) return std::copysign(0.0f, d);
    const int k = pick(3);
    return k == 0 ? r : std::nextafter(r, k == 1 ? 0.0f : std::copysign(INFINITY, r));
}

template <int E>
static bool entry(const bb::QuadSlabs<V>& q, float t_min, float t_max, float& lo)
{
    return bb::quad_entry<E>(q, t_min, t_max, lo);
}

// A record's grid on one axis from eight numbers, the entries' planes (bmin
// bmax), and the centre: prints the grid and the packed rows
static int grid(char** argv)
{
    float box[4][7] = {};
    const float* at[4];
    for (int k = 0; k < 4; ++k) {
        box[k][0] = std::strtof(argv[2 + 2 * k], nullptr);
        box[k][3] = std::strtof(argv[3 + 2 * k], nullptr);
        at[k] = box[k];
    }
    const bool has[4] = { true, true, true, true };
    const float centre[3] = { std::strtof(argv[10], nullptr), 0.0f, 0.0f };
    const bb::QuadGrid q = bb::quad_grid(at, has, centre);
    std::printf("%.9g %d %u %u\n", q.p[0], q.e[0], q.lo[0], q.hi[0]);
    return 0;
}

int main(int argc, char** argv)
{
    if (argc == 11) return grid(argv);
    const char* scene = argv[1];
    const char* kind = argv[2];
    g.seed(std::strtoul(argv[3], nullptr, 10));
    // boxes 0.01 to 0.2 wide in [-1, 1], scaled and moved
    double scale = 1.0, move[3] = { 0, 0, 0 };
    if (!std::strcmp(scene, "moved")) {
        move[0] = 1e5;
        move[1] = -3e4;
        move[2] = 7e5;
    } else if (!std::strcmp(scene, "large")) {
        scale = 1e18;
    } else if (!std::strcmp(scene, "huge")) {
        scale = 1e37;
    } else if (!std::strcmp(scene, "small")) {
        scale = 1e-12;
    }
    std::vector<V> mn(64), mx(64);
    V wmin{ INFINITY, INFINITY, INFINITY }, wmax{ -INFINITY, -INFINITY, -INFINITY };
    for (int b = 0; b < 64; ++b)
        for (int a = 0; a < 3; ++a) {
            double c = uni(-1, 1), w = 0.5 * std::pow(10.0, uni(-2, -0.7));
            if (!std::strcmp(scene, "mixed")) w *= std::pow(10.0, -uni(0, 6)), c *= std::pow(10.0, -uni(0, 3));
            if (!std::strcmp(scene, "flat") && a == 1) c = 0.25, w = b % 2 ? 0.0 : 1e-38;
            mn[b][a] = float(scale * (c - w) + move[a]);
            mx[b][a] = float(scale * (c + w) + move[a]);
            wmin[a] = std::min(wmin[a], mn[b][a]);
            wmax[a] = std::max(wmax[a], mx[b][a]);
        }
    V centre, half;
    for (int a = 0; a < 3; ++a) {
        centre[a] = float(0.5 * (double(wmin[a]) + wmax[a]));
        half[a] = bb::slab_half(wmin[a], wmax[a], centre[a]);
    }
    const double size = std::max({ double(wmax.x) - wmin.x, double(wmax.y) - wmin.y, double(wmax.z) - wmin.z });
    long tests = 0, exact_passes = 0, with_margin = 0, lost = 0, loose = 0;
    for (int r = 0; r < 4000; ++r) {
        V o, d;
        for (int a = 0; a < 3; ++a) {
            o[a] = float(uni(wmin[a], wmax[a]));
            d[a] = float(uni(-1, 1));
        }
        if (pick(4) == 0) o[pick(3)] = pick(2) ? mn[pick(64)][pick(3)] : mx[pick(64)][pick(3)]; // on a plane
        double len = 1.0, away = 0.0, t0 = 1e-4, t1 = INFINITY;
        const bool any = !std::strcmp(kind, "any");
        if (!std::strcmp(kind, "axis") || (any && pick(4) == 0)) {
            const int a = pick(3);
            for (int k = 0; k < 3; ++k) {
                const double least = pick(3) == 0 ? 0.0 : std::pow(10.0, -uni(2, 44));
                if (k != a) d[k] = float(pick(2) ? least : -least);
            }
        }
        if (!std::strcmp(kind, "far") || (any && pick(3) == 0)) away = size * std::pow(10.0, any ? uni(0, 30) : uni(0, 4));
        if (!std::strcmp(kind, "length") || (any && pick(3) == 0)) len = std::pow(10.0, uni(-40, 38));
        if (pick(4)) { // at a corner of a box, or a point in it
            const int b = pick(64), corner = pick(2);
            for (int a = 0; a < 3; ++a) {
                const double at = corner ? (pick(2) ? mn[b][a] : mx[b][a]) : uni(mn[b][a], mx[b][a]);
                if (d[a] * d[a] < 1e-9 || !std::strcmp(kind, "axis")) o[a] = float(at);
                else d[a] = float((at - o[a]) / size);
            }
        }
        for (int a = 0; a < 3; ++a) {
            o[a] = float(o[a] - away * d[a]);
            d[a] = float(len * d[a]);
        }
        if (any && pick(50) == 0) d[pick(3)] = pick(2) ? INFINITY : NAN;
        if (any && pick(50) == 0) o[pick(3)] = pick(2) ? -INFINITY : NAN;
        if (any && pick(100) == 0) d = V{ 0.0f, -0.0f, 0.0f };
        if (pick(3) == 0) {
            t0 = (size * uni(-1, 1) + away) / len;
            t1 = t0 + size * uni(0, 1) / len;
        }
        const float t_min = float(t0), t_max = float(t1);
        const V ei{ 1.0f / d.x, 1.0f / d.y, 1.0f / d.z };
        const bool e0 = ei.x < 0.0f, e1 = ei.y < 0.0f, e2 = ei.z < 0.0f;
        const V ri{ rcp(d.x), rcp(d.y), rcp(d.z) };
        V inv, near0, far0;
        const bool ok = bb::slab_ray(o, ri, centre, half, FLT_MAX, inv, near0, far0);
        const bool n0 = ri.x < 0.0f, n1 = ri.y < 0.0f, n2 = ri.z < 0.0f;
        for (int b = 0; b < 64; b += 4) {
            const bool has[4] = { true, b % 8 == 0, true, true };
            float box[4][7];
            const float* at[4];
            for (int k = 0; k < 4; ++k) {
                const int from = has[k] ? b + k : b; // (a missing entry repeats another)
                for (int a = 0; a < 3; ++a) {
                    box[k][a] = mn[from][a];
                    box[k][3 + a] = mx[from][a];
                }
                box[k][6] = NAN;
                at[k] = box[k];
            }
            const float at_centre[3] = { centre.x, centre.y, centre.z };
            const bb::QuadGrid q = bb::quad_grid(at, has, at_centre);
            const uint32_t e = uint32_t(uint8_t(q.e[0])) | uint32_t(uint8_t(q.e[1])) << 8 | uint32_t(uint8_t(q.e[2])) << 16;
            const bb::QuadSlabs<V> s = bb::quad_slabs(V{ q.p[0], q.p[1], q.p[2] }, e, q.lo[0], q.lo[1], q.lo[2], q.hi[0],
                                                      q.hi[1], q.hi[2], inv, near0, far0, n0, n1, n2);
            for (int k = 0; k < 4; ++k) {
                if (!has[k]) continue;
                const bb::BoxHit h = bb::box_part(mn[b + k], mx[b + k], o, t_min, ei, e0, e1, e2);
                const bool exact = bb::box_pass(h, t_max);
                ++tests;
                exact_passes += exact;
                if (exact && ok) lost += !bb::slab_root(half, inv, near0, far0, t_min, t_max);
                if (!ok) continue;
                ++with_margin;
                float lo;
                const bool pass = k == 0 ? entry<0>(s, t_min, t_max, lo) : k == 1 ? entry<1>(s, t_min, t_max, lo)
                                : k == 2 ? entry<2>(s, t_min, t_max, lo) : entry<3>(s, t_min, t_max, lo);
                lost += exact && (!pass || lo > h.lo);
                // (its own box with the margin)
                V box_centre, box_half;
                for (int a = 0; a < 3; ++a) {
                    box_centre[a] = float(0.5 * (double(mn[b + k][a]) + mx[b + k][a]));
                    box_half[a] = bb::slab_half(mn[b + k][a], mx[b + k][a], box_centre[a]);
                }
                V n = near0, f = far0;
                for (int a = 0; a < 3; ++a) {
                    n[a] = std::fma(box_centre[a] - centre[a], inv[a], n[a]);
                    f[a] = std::fma(box_centre[a] - centre[a], inv[a], f[a]);
                }
                loose += !exact && bb::slab_root(box_half, inv, n, f, t_min, t_max);
            }
        }
    }
    std::printf("%ld %ld %ld %ld %ld\n", tests, exact_passes, with_margin, lost, loose);
    return 0;
}
