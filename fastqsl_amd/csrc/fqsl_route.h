// fqsl_route.h -- which kernels a call runs and what they may touch.
//
// Plain host C++ without HIP, so that the CPU tests build and check the rules.
#pragma once

#include <vector>

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

// RK4 lines go by quads of lanes on any layout, but on component arrays a side's stage
// point touches twelve cache lines and not one record.  Two resident wavefronts a SIMD of
// 16 sides are 6.3 MB of lines for each 4 MiB L2 cache (FP32 has four), and sides that
// start anywhere in the box drive each other out of it.  From this count on the seeds
// tell (vote_near: the lines of most neighbouring lanes begin within a few cells or not);
// where they lie far apart, one wavefront a SIMD traces.  ms all / one / the kernels
// before quads, one lane a line: FP64 160 x 128 x 128, 24,576 lines 6.5 / 4.3 / 8.9, 65,536
// 19.9 / 9.0 / 16.9, 262,144 82 / 32.6 / 66; 64^3 262,144 13.0 / 11.9 / 12.9; FP32 160 x 128 x
// 128, 16,384 lines 3.2 / 2.6 / 6.9, 65,536 14.8 / 7.4 / 12.8, 600,000 148 / 60 / 123; 64^3
// 600,000 25.3 / 25.6 / 28.6.
constexpr unsigned long long kPlainRk4VoteLines = 16384;
// Close together no cache is short, and one side a lane takes fewer instructions: from
// this count on near lines go by lanes (ms by quads / by lanes / before: maps on 160 x
// 128 x 128, FP64 65,536 lines 2.9 / 2.3 / 3.2, 131,072 4.4 / 3.3 / 3.9, 1 M 21 / 11.9 / 17;
// FP32 65,536 2.7 / 2.45 / 2.7, 262,144 6.7 / 4.3 / 4.9, 600,000 13.0 / 6.6 / 7.9; 32,768 lines
// FP64 2.1 / 2.1 / 3.3, FP32 1.6 / 1.75 / 3.0).
constexpr unsigned long long kPlainRk4PickLines = 65536;
// One side a lane, from this count on half the resident grid, for the caches too (all /
// half: RK4 maps FP64 131,072 lines on 160 x 128 x 128 3.8 / 3.3, FP32 600,000 on 200 x 160 x
// 128 8.4 / 7.8, RKF45 maps 1.95 / 1.58, seeds anywhere 13.6 / 13.4; 65,536 FP64 2.3 / 2.9).
constexpr unsigned long long kPlainHalfSidesLines = 98304;

// Whether a plain trace writes a result where it reads its seeds.  The forward
// and the backward side of a line are separate tasks, each of which reads the
// seed when it begins, and the outputs that belong to the line are written
// before either: only one thread that traces both sides, and writes when they
// have ended, may overwrite them.
inline bool plain_in_place(const void* const* seeds, int nseeds, const void* const* out, int nout) {
    for (int i = 0; i < nout; ++i)
        for (int k = 0; k < nseeds; ++k)
            if (out[i] && out[i] == seeds[k]) return true;
    return false;
}

// Whether a plain trace runs one thread per line.  The other kernels draw their
// work from a counter in a ring that later launches share; a captured launch
// keeps its counter, and a replay may meet a launch that the ring has come round
// to.  The per-line schedule has no such counter to be captured.
inline bool plain_by_lines(bool in_place, bool per_line, bool capturing) {
    return in_place || (per_line && capturing);
}

// Most FP64 RK4 Scott lines' worth of work, counted in longest lines of the launch
// by the queue order's estimate, that go by quads of lanes.  By lanes a launch that
// fits the chip takes as long as its longest line (3.3 us an evaluation on a field of
// 6 or 9 MiB, 5.0 on one of 50 or 90); by quads the chip does an
// evaluation every 0.12-0.15 ns, so the two meet where the work is that many longest
// lines.  ms by quads / by lanes: 64^3 seeds anywhere, 24,576 lines (14,500 longest)
// 3.8 / 4.3, 32,768 (19,400) 4.5 / 4.4, 65,536 (38,600) 6.6 / 4.4, a 256^2 map (13,300)
// 2.7 / 3.5; 128^3 49,152 lines (31,900) 11.7 / 13.1, 57,344 (36,900) 13.3 / 13.0, a
// 256^2 map (18,400) 4.8 / 7.7.  RKF45 lines go by quads up to the full count: 15 of 16
// such launches gain 1.03-1.5, one takes 1.05 times as long.
inline unsigned long long scott_fp64_quad_work(unsigned long long field_bytes) {
    return field_bytes <= (32ull << 20) ? 19000ull : 34000ull;
}

// Consecutive requests of a batch and their lines: those of one layout, which a
// launch by quads takes together, or of one field and method, which a launch by
// lanes takes.  `counter` is the work counter of that launch.  Layouts of one
// run go either way, each by its own line count, so both kinds of launches draw
// from one numbering: a group's counter is its place among the groups, a
// layout's that of its first group, which is not launched beside it.
struct BatchSpan {
    int r0, r1, counter;
    unsigned long long base, n;
};

// Spans of requests in batch order: request k has n[k] lines on layout kind[k];
// other[k]: its field or method is another than request k - 1's.
inline void batch_spans(int nreq, const int* kind, const char* other, const unsigned long long* n,
                        std::vector<BatchSpan>& layouts, std::vector<BatchSpan>& groups) {
    unsigned long long lines = 0;
    for (int k = 0; k < nreq; ++k) {
        const bool layout = k == 0 || kind[k] != kind[k - 1];
        const int next = (int)groups.size();
        if (layout) layouts.push_back(BatchSpan{k, k, next, lines, 0});
        if (layout || other[k]) groups.push_back(BatchSpan{k, k, next, lines, 0});
        for (BatchSpan* s : {&layouts.back(), &groups.back()}) {
            s->r1 = k + 1;
            s->n += n[k];
        }
        lines += n[k];
    }
}

// Whether one launch by quads takes all requests of a batch's layout.  By lanes each
// (field, method) group is a launch of its own.
// FP32c: lines of which a quad has hundreds leave no tail to shorten, and a launch per
// group keeps to one field at a time; fixed-step lines hold on longer (three fields, ms by
// quads / by lanes: 1.9 M lines RKF45 23.7 / 28.7, 7.7 M 87 / 89 and seeds anywhere 138 /
// 136, 15.4 M 171 / 167 and 275 / 265; RK4 1.9 M 23.9 / 28.5, 15.4 M 167 / 168 and 325 /
// 348; both 16.6 M 183 / 186; 50.5 M in 256 requests 1.55 s / 1.46).
inline bool batch_fp32_by_quads(unsigned long long rkf45_lines, unsigned long long rk4_lines) {
    return rkf45_lines + rk4_lines / 2 <= (1ull << 23);
}
// FP64: of several groups each would wait for its longest line in turn; one alone does
// so once, and its lines are not ordered (ms by quads / by lanes: one RK4 request on 96^3
// of 16,384 map pixels 2.9 / 5.0, 24,576 5.6 / 5.3, 65,536 7.8 / 5.1; RKF45 24,576 7.8 / 9.0,
// 40,000 9.2 / 9.0; two of 32,000 RK4 10.8 / 12.9, RKF45 11.0 / 20.4; twelve of 5,000 9.2 / 24.8).
inline bool batch_fp64_by_quads(unsigned long long lines, int groups, bool rk4) {
    return lines <= (groups > 1 ? 65536ull : rk4 ? 20000ull : 32768ull);
}

// An allocation that may find the memory in what the library keeps: `alloc` is
// tried again when it fails for want of memory (`full`) and `give_back` has freed
// some.
template <typename E, class Alloc, class GiveBack>
E alloc_or_give_back(E full, Alloc alloc, GiveBack give_back) {
    const E e = alloc();
    return e == full && give_back() ? alloc() : e;
}

}  // namespace fqsl
