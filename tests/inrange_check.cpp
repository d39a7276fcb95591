// Host check of by_const (fenice_amd/csrc/fvg_device.hpp, compiled for the host from the same source): x / c through
// the correctly rounded reciprocal of c must give the bits of the IEEE division for every x in its range, and
// value_in_range must have the bounds the kernels' comments derive their operand ranges from.
// usage: inrange_check <samples> <seed>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "../fenice_amd/csrc/fvg_device.hpp"

static uint64_t g_state;
static uint64_t next_u64() {   // splitmix64
    uint64_t z = (g_state += 0x9e3779b97f4a7c15ull);
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
    return z ^ (z >> 31);
}
static double make(uint64_t sig, int e, int neg) {
    const uint64_t b = ((uint64_t)(e + 1023) << 52) | (sig & ((1ull << 52) - 1)) | ((uint64_t)neg << 63);
    double d;
    std::memcpy(&d, &b, 8);
    return d;
}
static bool same(double a, double b) { return std::memcmp(&a, &b, 8) == 0; }

int main(int argc, char** argv) {
    const long long n = argc > 1 ? std::atoll(argv[1]) : 1000000;
    g_state = argc > 2 ? std::strtoull(argv[2], nullptr, 10) : 1;
    long long bad = 0;
    for (long long s = 0; s < n; ++s) {
        // divisors: random, near both ends of a binade (reciprocals next to midpoints), and gamma - 1 or a mesh width
        uint64_t sig = next_u64();
        const uint64_t kind = next_u64() % 4;
        if (kind == 1) sig = ((1ull << 52) - 1) - next_u64() % 4096;
        else if (kind == 2) sig = next_u64() % 4096;
        volatile double c = make(sig, (int)(next_u64() % 200) - 100, 0);
        if (kind == 3) c = (next_u64() & 1) ? 1.4 - 1.0 : 6.283185307179586 / (double)(1 + next_u64() % 1024);
        const double inv = 1.0 / c;
        for (int k = 0; k < 8; ++k) {
            volatile double x = make(next_u64(), (int)(next_u64() % 1600) - 850, (int)(next_u64() & 1));
            if (k == 1) x = make(next_u64(), 0, 0) * c;                       // exact or nearly exact quotients
            else if (k == 2) x = std::nextafter((double)x, 0.0) * c;
            else if (k == 3) {   // quotients next to a midpoint of two doubles
                const double q = make(next_u64(), (int)(next_u64() % 60) - 30, 0);
                x = q * c + 0.5 * (std::nextafter(q, 2.0 * q) - q) * c;
            } else if (k == 4) x = (next_u64() & 1) ? 0.0 : -0.0;
            const double want = x / c, got = fvg::by_const<true>(x, c, inv);
            if (!same(want, got)) {
                if (bad < 5) std::printf("differs: %a / %a = %a, by_const %a\n", (double)x, (double)c, want, got);
                ++bad;
            }
        }
    }
    const bool range = fvg::value_in_range(0.0) && fvg::value_in_range(-0.0) && fvg::value_in_range(0x1p-400) && fvg::value_in_range(-0x1p100) &&
                       !fvg::value_in_range(0x1.fffffffffffffp-401) && !fvg::value_in_range(0x1.0000000000001p100) &&
                       !fvg::value_in_range(INFINITY) && !fvg::value_in_range(-INFINITY) && !fvg::value_in_range(NAN) &&
                       !fvg::value_in_range(4.9e-324);
    std::printf("differing: %lld, bounds %s\n", bad, range ? "ok" : "WRONG");
    return bad == 0 && range ? 0 : 1;
}
