// Test-only CPU build of fastqsl_amd/csrc/fqsl_route.h.
#include "fqsl_route.h"

extern "C" unsigned long long rt_plain_listed_lines(int rkf45, unsigned long long lines, int counted) {
    return fqsl::plain_listed_lines(rkf45 != 0, lines, counted != 0);
}

// Counter and first request of every launch of a batch in which layouts of at
// most `quad_lines` lines are launched whole and larger ones group by group;
// returns how many there are.
extern "C" int rt_batch_launches(int nreq, const int* kind, const char* other, const unsigned long long* n,
                                 unsigned long long quad_lines, int* counter, int* first, unsigned long long* lines) {
    std::vector<fqsl::BatchSpan> layouts, groups;
    fqsl::batch_spans(nreq, kind, other, n, layouts, groups);
    int m = 0;
    auto launch = [&](const fqsl::BatchSpan& v) {
        counter[m] = v.counter;
        first[m] = v.r0;
        lines[m++] = v.n;
    };
    for (const fqsl::BatchSpan& s : layouts) {
        if (s.n <= quad_lines) launch(s);
        else
            for (const fqsl::BatchSpan& g : groups)
                if (g.r0 >= s.r0 && g.r0 < s.r1) launch(g);
    }
    return m;
}
extern "C" int rt_batch_groups(int nreq, const int* kind, const char* other, const unsigned long long* n) {
    std::vector<fqsl::BatchSpan> layouts, groups;
    fqsl::batch_spans(nreq, kind, other, n, layouts, groups);
    return (int)groups.size();
}

extern "C" int rt_plain_in_place(const void* const* seeds, int nseeds, const void* const* out, int nout) {
    return fqsl::plain_in_place(seeds, nseeds, out, nout) ? 1 : 0;
}

extern "C" int rt_plain_by_lines(int in_place, int per_line, int capturing) {
    return fqsl::plain_by_lines(in_place != 0, per_line != 0, capturing != 0) ? 1 : 0;
}

// An allocator that fails with `code` until its `ok_at`-th call, with blocks to give back or
// none; returns the code of the last call and how often it was called.
extern "C" int rt_alloc_or_give_back(int full, int code, int ok_at, int has_blocks, int* calls) {
    *calls = 0;
    return fqsl::alloc_or_give_back(
        full, [&] { return ++*calls >= ok_at ? 0 : code; }, [&] { return has_blocks != 0; });
}

extern "C" unsigned long long rt_scott_fp64_quad_work(unsigned long long bytes) { return fqsl::scott_fp64_quad_work(bytes); }

extern "C" int rt_batch_fp32_by_quads(unsigned long long rkf45, unsigned long long rk4) {
    return fqsl::batch_fp32_by_quads(rkf45, rk4) ? 1 : 0;
}
extern "C" int rt_batch_fp64_by_quads(unsigned long long lines, int groups, int rk4) {
    return fqsl::batch_fp64_by_quads(lines, groups, rk4 != 0) ? 1 : 0;
}
