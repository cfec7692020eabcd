// Host build of the kernels' sine, cosine and fifth power
// (bulbit_amd/csrc/bb_trig.h) against the C library's long double ones over
// every `step`-th float of a range: prints how many values there were, how
// many results are not the correctly rounded float, and the largest error in
// units of the last place.
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "../bulbit_amd/csrc/bb_trig.h"

static float from_bits(uint32_t b)
{
    float f;
    std::memcpy(&f, &b, 4);
    return f;
}

static uint32_t to_bits(float f)
{
    uint32_t b;
    std::memcpy(&b, &f, 4);
    return b;
}

int main(int argc, char** argv)
{
    const char* what = argv[1];
    const uint32_t lo = to_bits(std::strtof(argv[2], nullptr)), hi = to_bits(std::strtof(argv[3], nullptr));
    const uint32_t step = uint32_t(std::atoi(argv[4]));
    const float sign = argc > 5 ? -1.0f : 1.0f;
    long n = 0, off = 0;
    double worst = 0.0;
    auto check = [&](float got, long double want) {
        ++n;
        const float w = float(want);
        if (to_bits(got) == to_bits(w)) return;
        ++off;
        const double ulp = std::abs(double(got) - double(w)) / (nextafterf(fabsf(w), INFINITY) - fabsf(w));
        if (!(ulp <= worst)) worst = ulp;
    };
    for (uint64_t b = lo; b <= hi; b += step) {
        const float x = sign * from_bits(uint32_t(b));
        if (what[0] == 'p') {
            const long double t = x;
            check(bb::pow5(x), t * t * t * t * t);
        } else {
            float s, c;
            bb::sincos_small(x, s, c);
            check(s, sinl((long double)x));
            check(c, cosl((long double)x));
        }
    }
    std::printf("%ld %ld %g\n", n, off, worst);
    return 0;
}
