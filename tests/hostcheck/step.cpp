// Test-only CPU build of fastqsl_amd/csrc/fqsl_step.h.
#define FQSL_HD static inline
#define FQSL_COLD static
#include "fqsl_step.h"

// The step after an attempt: as next_step takes it, from the estimates
// (1 / sqrt(e2)) (1 + eps) and (float)(q^0.2 (1 + eps5)), and as written.
extern "C" void st_steps(long n, const double* s, const double* tol, const double* e2, const double* eps,
                         const double* eps5, double* got, int* got_ok, double* written, int* written_ok) {
    for (long i = 0; i < n; ++i) {
        const fqsl::Step w = fqsl::step_of_scale(s[i], pow(tol[i] / sqrt(e2[i]) / 11.09, 0.2));
        const bool plain = fqsl::step_is_plain(tol[i], e2[i], fqsl::step_tol_limit(s[i]));
        const double q = plain ? fqsl::scale_argument(tol[i], e2[i], 1.0 / sqrt(e2[i]) * (1.0 + eps[i]))
                               : fqsl::scale_argument_wide(tol[i], e2[i]);
        const float root = plain ? (float)(pow((double)(float)q, 0.2) * (1.0 + eps5[i])) : NAN;
        const fqsl::Step g = fqsl::step_of_argument(s[i], q, root);
        got[i] = g.s;
        got_ok[i] = g.accepted;
        written[i] = w.s;
        written_ok[i] = w.accepted;
    }
}

extern "C" void st_arguments(long n, const double* tol, const double* e2, const double* eps, double* got,
                             double* written, int* plain) {
    for (long i = 0; i < n; ++i) {
        plain[i] = fqsl::step_is_plain(tol[i], e2[i], fqsl::step_tol_limit(1.0));
        got[i] = fqsl::scale_argument(tol[i], e2[i], 1.0 / sqrt(e2[i]) * (1.0 + eps[i]));
        written[i] = tol[i] / sqrt(e2[i]) / 11.09;
    }
}
