// fqsl_route.h -- which kernels a call runs and what they may touch.
//
// Plain host C++ without HIP, so that the CPU tests build and check the rules.
#pragma once

namespace fqsl {

// Sides up to which an RKF45 launch is traced by quads alone, two per resident
// quad.  On the multipole 256^3 field (s_len 1/8, tol_coef 0.5; ms by quads /
// tangent lines by quads and the rest by lanes): 65 k sides 0.72 / 0.73, 131 k
// 0.68 / 0.70, 262 k 0.90 / 0.84, 1.0 M 1.57 / 1.25, 2.1 M 2.38 / 1.74.  RK4
// lines have no tangent class and all go by quads, whose two loads a stage touch
// a third of the cache lines of a lane's six (2.1 M sides 10.4 against 11.9 ms).
constexpr unsigned long long kPlainQuadSides = 131072;

// Lines for which a plain trace keeps a place in the list and the marks of its
// tangent lines (0: no list, all by quads).  `lines` is how many the kernels
// trace, or, with `counted` false, a mere cap on a grid's size: the count is
// then read on the device, nothing bounds it, and every line a kernel may index
// needs its place.
inline unsigned long long plain_listed_lines(bool rkf45, unsigned long long lines, bool counted) {
    const bool list = rkf45 && counted && lines > kPlainQuadSides / 2 && lines < (1ull << 32);
    return list ? lines : 0ull;
}

}  // namespace fqsl
