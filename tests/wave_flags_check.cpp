// wave_flags_check.cpp -- CPU check of the one-wave kernel's track flags
// (supertrack_amd/csrc/layout.{hpp,cpp}) against a brute-force count of what a
// flush would keep, built with g++ by tests/test_wave_flags.py.  Prints one
// line per track kind and "ALL OK".
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <set>
#include <vector>

#include "../supertrack_amd/csrc/layout.hpp"

using namespace st;

static st_geometry geometry(double half_length, double diameter)
{
    // SphericalGeometry (SphericalGeometry.cu:34-58)
    st_geometry g{};
    g.n_linear = (int)std::floor(half_length * 2 / diameter);
    g.length = g.n_linear * diameter;
    g.half_length = g.length / 2;
    g.diameter = diameter;
    g.radius = diameter / 2;
    g.gso = -g.half_length + g.radius;
    return g;
}

int main()
{
    std::mt19937_64 rng(7);
    auto uni = [&](double a, double b) { return std::uniform_real_distribution<double>(a, b)(rng); };
    int waves = 0, hots = 0, rest = 0;
    for (int trial = 0; trial < 240; ++trial) {
        const int kind = trial % 6;
        const double D = kind < 2 ? 2.0 : kind < 4 ? 10.0 : 100.0;
        const st_geometry g = geometry(kind == 5 ? 400.0 : 2500.0, D);
        const int n = (int)uni(1, 6000);
        const double spread = kind == 1 ? 40.0 : kind == 3 ? 120.0 : kind == 5 ? 390.0 : 15.0;
        const double length = uni(1, 4000);
        std::vector<double> z(n), x(n), y(n);
        for (double &v : z) v = uni(0, length);
        std::sort(z.begin(), z.end());
        const double x0 = uni(-300, 300);
        for (int i = 0; i < n; ++i) {
            x[i] = x0 + uni(-spread, spread);
            y[i] = uni(-spread, spread);
        }
        const auto mx = std::minmax_element(x.begin(), x.end());
        const auto my = std::minmax_element(y.begin(), y.end());
        const uint32_t f = wave_flags(x.data(), y.data(), z.data(), n, g, *mx.first, *mx.second, *my.first, *my.second);
        if (f == 0) {
            ++rest;
            continue;
        }
        (f & kFlagHot) ? ++hots : ++waves;
        size_t most = 0;
        for (int s = 0; s < 6; ++s) {
            const double sx = uni(-D, D), sy = uni(-D, D), sz = uni(-D, D);
            std::set<std::pair<long, long>> kept;   // spheres of the layer the point before lies in
            long layer = -(1l << 40);
            for (int i = 0; i < n; ++i) {
                const long k = std::lrint((z[i] + sz) / D);
                if (k != layer) kept.clear();
                layer = k;
                kept.insert({std::lrint((x[i] + sx) / D), std::lrint((y[i] + sy) / D)});
                most = std::max(most, kept.size());
            }
        }
        if (most > (size_t)((f & kFlagHot) ? kHotWindow : kWaveWindow)) {
            std::printf("FAIL trial %d: %zu spheres kept, flags %u\n", trial, most, f);
            return 1;
        }
        double bits = (f & kFlagHot) ? 2 : 0;
        for (double range : {*mx.second - *mx.first, *my.second - *my.first, z[n - 1] - z[0]})
            bits += std::floor(std::log2(std::min((double)g.n_linear, std::floor(range / D) + 6.0))) + 1;
        if (bits > kWaveKeyBits) {
            std::printf("FAIL trial %d: %g key bits\n", trial, bits);
            return 1;
        }
    }
    std::printf("%d wave, %d hot, %d other tracks\n", waves, hots, rest);
    if (waves < 20 || hots < 10 || rest < 10) return 1;
    std::printf("ALL OK\n");
    return 0;
}
