// The boxes that the positions of a system's rows are cut into. The cuts hold
// equal row counts, so any number of boxes per axis serves.
#pragma once

#include <algorithm>
#include <cmath>

namespace astg {

// Boxes per axis, near cubes, at most K in all, over the coordinate extents
// (axes of extent 1 are not cut). Rounding each axis by the cube's edge leaves
// fewer than K: 1 of 2 or 3, 4 of 5 to 7, 8 of 15, 216 of 256 over a cube. While
// the boxes are small that is right, a boundary less on the chain is worth more
// than smaller boxes. us per iteration with these and with most(): octrees FP64
// 28^3 48 / 53 (1 / 3 boxes of 6.4 / 2.1 k rows), 52^3 78 / 85 (12 / 16), 96^3
// 130 / 135 and mixed 86 / 92 (80 / 96), 136^3 198 / 205 (216 / 252, 2.5 / 2.2 k
// rows). At 112^3 (125 / 150) two runs gave either form up to 15 % over the other.
inline void cubes(int K, const int* ext, int* k) {
    double vol = 1.0;
    int dims = 0;
    for (int a = 0; a < 3; ++a)
        if (ext[a] > 1) {
            vol *= ext[a];
            ++dims;
        }
    const double edge = dims ? std::pow(vol / K, 1.0 / dims) : 1.0;
    for (int a = 0; a < 3; ++a) k[a] = ext[a] > 1 ? std::max(1, (int)std::lround(ext[a] / edge)) : 1;
    while ((long)k[0] * k[1] * k[2] > K) {
        int m = 0;
        for (int a = 1; a < 3; ++a)
            if (k[a] > k[m]) m = a;
        --k[m];
    }
}

// The most boxes against their shape: the product k0 k1 k2 times the root of
// the shortest over the longest edge is largest (252 of 256 over a cube).
inline void most(int K, const int* ext, int* k) {
    double best = -1.0;
    for (int x = 1; x <= (ext[0] > 1 ? K : 1); ++x)
        for (int y = 1; y <= (ext[1] > 1 ? K / x : 1); ++y)
            for (int z = 1; z <= (ext[2] > 1 ? K / (x * y) : 1); ++z) {
                const int c[3] = {x, y, z};
                double lo = 1e300, hi = 0.0;
                for (int a = 0; a < 3; ++a)
                    if (ext[a] > 1) {
                        lo = std::min(lo, (double)ext[a] / c[a]);
                        hi = std::max(hi, (double)ext[a] / c[a]);
                    }
                const double score = (double)x * y * z * (hi > 0.0 ? std::sqrt(lo / hi) : 1.0);
                if (score > best) {
                    best = score;
                    std::copy(c, c + 3, k);
                }
            }
}

// Boxes for n rows on a device of `units` compute units. With a box per unit
// asked for and more than 3000 rows in each of the cubes, the units that cubes
// leave idle are worth more than their shape: 160^3 FP64 264 / 259 us per
// iteration (cubes / most), 176^3 314 / 301, 192^3 370 / 354 and mixed 191 / 184,
// 224^3 mixed 245 / 245; slabs (the product alone) 1.5 times as long.
inline void tileGrid(int K, long long n, int units, const int* ext, int* k) {
    cubes(K, ext, k);
    if (K == units && n > 3000ll * k[0] * k[1] * k[2]) most(K, ext, k);
}

}  // namespace astg
