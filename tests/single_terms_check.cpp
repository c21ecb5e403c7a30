// Checks the FP32 terms of block records (single_terms) on the CPU: points laid
// out by fill_chunk are brought to lattice units in FP32 as wave_kernel does,
// for random shifts and key boxes, and every decision that the thresholds call
// certain is compared with long double arithmetic on the FP64 points.
#include <algorithm>
#include <cstdio>
#include <cstring>
#include <random>
#include <vector>

#include "../supertrack_amd/csrc/layout.hpp"

using namespace st;

static st_geometry make(double half, double d)
{
    st_geometry g{};
    const double r = d / 2;
    const int n = (int)std::floor(half * 2 / d);
    g.length = n * d;
    g.half_length = g.length / 2;
    g.diameter = d;
    g.radius = r;
    g.gso = -g.half_length + r;
    g.n_linear = n;
    return g;
}

int main()
{
    std::mt19937_64 rng(12345);
    auto uni = [&](double a, double b) { return a + (b - a) * std::uniform_real_distribution<double>(0, 1)(rng); };
    const double geos[][2] = {{2.5e3, 10.0}, {2.5e3, 2.0}, {1e3, 1.0}, {5e3, 100.0}, {2.5e3, 7.3}, {300.0, 0.37}};
    long long sure = 0, outside = 0, near = 0;
    for (const auto &gd : geos) {
        const st_geometry g = make(gd[0], gd[1]);
        for (double spread : {0.4, 30.0, 900.0, 20000.0}) {
            const int n = 5 * kBlk + 17;
            std::vector<double> x(n), y(n), z(n), e(n, 1.0);
            for (int i = 0; i < n; ++i) {
                x[i] = uni(-spread, spread);
                y[i] = uni(-spread, spread) + 0.3 * g.half_length;
                z[i] = uni(-g.half_length, g.half_length);
                if (i % 3 == 0) {   // close to a face of a sphere's cell, or to its sphere
                    const double c = std::round((x[i] - g.gso) / g.diameter) * g.diameter + g.gso;
                    x[i] = c + (i % 2 ? 0.5 : 0.4999) * g.diameter * (1.0 + uni(-1e-6, 1e-6));
                }
            }
            const int64_t off[2] = {0, n};
            const int32_t geom = 0;
            TrackDesc td{};
            const int64_t nb = plan_chunk(off, 1, &geom, 0, 0, &td);
            ChunkLayout lay;
            fill_chunk(x.data(), y.data(), z.data(), e.data(), off, 1, &g, ST_F32, 0, 0, nb, &td, lay);
            for (int trial = 0; trial < 20; ++trial) {
                const double s[3] = {uni(-g.half_length, g.half_length), uni(-g.half_length, g.half_length),
                                     uni(-g.half_length, g.half_length)};
                const double k0[3] = {std::floor(uni(0, g.n_linear)), std::floor(uni(0, g.n_linear)),
                                      std::floor(uni(0, g.n_linear))};
                const double invD = 1.0 / g.diameter;
                const float inv = (float)invD;
                for (int p = 0; p < n; ++p) {
                    const BlockF32 &bk = lay.blocks[p / kBlk];
                    const float f[3] = {bk.fx, bk.fy, bk.fz};
                    const int32_t k[3] = {bk.kx, bk.ky, bk.kz};
                    const float pt[3] = {lay.p32[p].x, lay.p32[p].y, lay.p32[p].z};
                    const double c64[3] = {lay.x[p], lay.y[p], lay.z[p] + g.half_length};
                    float u[3];
                    long double d2 = 0, low = 0, high = 0;
                    bool same = true;
                    for (int a = 0; a < 3; ++a) {
                        const double o = s[a] * invD - k0[a], ok = std::rint(o);
                        const float b = f[a] + (float)(o - ok);
                        const float q = std::fmaf(pt[a], inv, b);
                        const float t = q + 12582912.0f;
                        u[a] = (t - 12582912.0f) - q;
                        uint32_t bits;
                        std::memcpy(&bits, &t, 4);
                        const int32_t local = (int32_t)bits + k[a] + (int32_t)ok - 0x4B400000;
                        const long double v = ((long double)(c64[a] + s[a]) - g.gso) / g.diameter;
                        const long double r = std::rint(v), w = std::fabs(r - v);
                        same = same && r == (long double)local + (long double)k0[a];
                        d2 += w * w;
                        // either rounding of a coordinate by a half-way plane
                        low += w * w;
                        high += w > 0.49999L ? (1 - w) * (1 - w) : w * w;
                    }
                    const float dist = std::fmaf(u[0], u[0], std::fmaf(u[1], u[1], u[2] * u[2]));
                    const long double r2 = 0.25L;
                    if (dist < bk.sure32) {
                        ++sure;
                        if (!same || !(d2 < r2)) {
                            std::printf("wrong inside: D %g spread %g point %d\n", gd[1], spread, p);
                            return 1;
                        }
                    } else if (dist > bk.maybe32) {
                        ++outside;
                        if (!(std::min(low, high) > r2)) {
                            std::printf("wrong outside: D %g spread %g point %d\n", gd[1], spread, p);
                            return 1;
                        }
                    } else {
                        ++near;
                    }
                }
            }
        }
    }
    std::printf("ok: %lld inside, %lld outside, %lld in doubt\n", sure, outside, near);
    return sure > 100000 && outside > 100000 ? 0 : 1;
}
