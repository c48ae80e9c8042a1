// Test-only CPU build of fastqsl_amd/csrc/fqsl_route.h.
#include "fqsl_route.h"

extern "C" unsigned long long rt_plain_listed_lines(int rkf45, unsigned long long lines, int counted) {
    return fqsl::plain_listed_lines(rkf45 != 0, lines, counted != 0);
}
