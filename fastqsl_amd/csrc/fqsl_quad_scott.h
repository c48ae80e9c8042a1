// fqsl_quad_scott.h -- the Scott tracer with one line per quad of lanes.
//
// As in fqsl_quad.h: lane q = 0, 1, 2 of a quad owns axis q of the position and
// component q of x, u and v, lane 3 repeats lane 0.  A stage evaluation takes two
// 16-byte loads and ~100 instructions a lane where one lane doing all three
// components takes six and ~250, and a lane holds a third of the state: all
// stage derivatives stay in registers.  What a launch of few lines waits for is
// the chain of its longest line, so such launches are traced this way.  Every
// value is formed by the same expression on the same operands as in
// scott_attempt (fqsl_tracer.h).
#pragma once

#include "fqsl_quad.h"

namespace fqsl {

#if defined(__HIP_DEVICE_COMPILE__)

// Value and the three edge derivatives of one component (coef_eval / cell_eval).
template <typename R>
__device__ __forceinline__ void coef_eval1(const R c[8], R x, R y, R z, R& B, R d[3]) {
    const R t = c[1] + c[4] * y, u = c[6] + c[7] * y;
    const R A = (c[0] + c[2] * y) + x * t;
    const R C = (c[3] + c[5] * y) + x * u;
    B = A + z * C;
    d[2] = C;
    d[0] = t + z * u;
    d[1] = (c[2] + c[4] * x) + z * (c[5] + c[7] * x);
}
// coef_eval1 with the weight each lane of the quad holds: 2 + 11 instructions.
// (The first products go to new registers; as DPP operands they would overwrite
// coefficients, which the compiler copies out of the loads' registers first.)
__device__ __forceinline__ void quad_coef_eval(const float c[8], float w, float& B, float d[3]) {
    const float x = quad_lane<0>(w), y = quad_lane<1>(w);
    float t = c[1] + c[4] * y, u = c[6] + c[7] * y;
    float A = (c[0] + c[2] * y) + x * t;
    const float C = (c[3] + c[5] * y) + x * u;
    float e = c[2] + c[4] * x;
    const float f = c[5] + c[7] * x;
    asm("s_nop 1\n\t"
        "v_fmac_f32_dpp %2, %3, %4" FQSL_Q2  // d1
        "v_fmac_f32_dpp %1, %3, %5" FQSL_Q2  // d0 = t + z u
        "v_fmac_f32_dpp %0, %3, %6" FQSL_Q2  // A + z C
        : "+v"(A), "+v"(t), "+v"(e) : "v"(w), "v"(f), "v"(u), "v"(C));
    B = A;
    d[0] = t; d[1] = e; d[2] = C;
}

// dot3(k, v_j) of three vectors v_j, whose component each lane holds.
__device__ __forceinline__ void quad_dots(const float v[3], const float k[3], float out[3]) {
    asm("s_nop 1\n\t"
        "v_mul_f32_dpp %0, %3, %7" FQSL_Q1
        "v_mul_f32_dpp %1, %4, %7" FQSL_Q1
        "v_mul_f32_dpp %2, %5, %7" FQSL_Q1
        "v_fmac_f32_dpp %0, %3, %6" FQSL_Q0
        "v_fmac_f32_dpp %1, %4, %6" FQSL_Q0
        "v_fmac_f32_dpp %2, %5, %6" FQSL_Q0
        "v_fmac_f32_dpp %0, %3, %8" FQSL_Q2
        "v_fmac_f32_dpp %1, %4, %8" FQSL_Q2
        "v_fmac_f32_dpp %2, %5, %8" FQSL_Q2
        : "=&v"(out[0]), "=&v"(out[1]), "=&v"(out[2]) : "v"(v[0]), "v"(v[1]), "v"(v[2]), "v"(k[0]), "v"(k[1]), "v"(k[2]));
}
__device__ __forceinline__ void quad_dots(const double v[3], const double k[3], double out[3]) {
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        double a[3];
        all_axes<1>(&v[j], a);
        out[j] = dot3(k, a);
    }
}
// u_0 J_0 + u_1 J_1 + u_2 J_2 for two vectors whose component each lane holds.
__device__ __forceinline__ void quad_rows(float u, float v, const float J[3], float& ju, float& jv) {
    asm("s_nop 1\n\t"
        "v_mul_f32_dpp %0, %2, %5" FQSL_Q1
        "v_mul_f32_dpp %1, %3, %5" FQSL_Q1
        "v_fmac_f32_dpp %0, %2, %4" FQSL_Q0
        "v_fmac_f32_dpp %1, %3, %4" FQSL_Q0
        "v_fmac_f32_dpp %0, %2, %6" FQSL_Q2
        "v_fmac_f32_dpp %1, %3, %6" FQSL_Q2
        : "=&v"(ju), "=&v"(jv) : "v"(u), "v"(v), "v"(J[0]), "v"(J[1]), "v"(J[2]));
}
__device__ __forceinline__ void quad_rows(double u, double v, const double J[3], double& ju, double& jv) {
    double a[3], b[3];
    all_axes<1>(&u, a);
    all_axes<1>(&v, b);
    ju = a[0] * J[0] + a[1] * J[1] + a[2] * J[2];
    jv = b[0] * J[0] + b[1] * J[1] + b[2] * J[2];
}

template <typename R>
__device__ __forceinline__ void cell_eval1(const R c[8], R wx, R wy, R wz, R& B, R d[3]) {
    const R dx00 = c[1] - c[0], dx10 = c[3] - c[2];
    const R dx01 = c[5] - c[4], dx11 = c[7] - c[6];
    const R e00 = c[0] + wx * dx00, e10 = c[2] + wx * dx10;
    const R e01 = c[4] + wx * dx01, e11 = c[6] + wx * dx11;
    const R dy0 = e10 - e00, dy1 = e11 - e01;
    const R f0 = e00 + wy * dy0, f1 = e01 + wy * dy1;
    const R gx0 = dx00 + wy * (dx10 - dx00), gx1 = dx01 + wy * (dx11 - dx01);
    const R dz = f1 - f0;
    B = f0 + wz * dz;
    d[2] = dz;
    d[1] = dy0 + wz * (dy1 - dy0);
    d[0] = gx0 + wz * (gx1 - gx0);
}
// Edge derivative along axis J of one component (coef_edge / cell_edge).
template <class F, int J, typename R>
__device__ __forceinline__ R edge1(const R c[8], R x, R y, R z) {
    if constexpr (F::kCoef) {
        if (J == 0) return (c[1] + c[4] * y) + z * (c[6] + c[7] * y);
        if (J == 1) return (c[2] + c[4] * x) + z * (c[5] + c[7] * x);
        return (c[3] + c[5] * y) + x * (c[6] + c[7] * y);
    } else {
        constexpr int bj = 1 << J, bu = J == 0 ? 2 : 1, bv = J == 2 ? 2 : 4;
        const R wu = J == 0 ? y : x, wv = J == 2 ? y : z;
        const R e00 = c[bj] - c[0], e10 = c[bj + bu] - c[bu];
        const R e01 = c[bj + bv] - c[bv], e11 = c[bj + bu + bv] - c[bu + bv];
        const R f0 = e00 + wu * (e10 - e00), f1 = e01 + wu * (e11 - e01);
        return f0 + wv * (f1 - f0);
    }
}

// A value rounded here: what follows is not fused with the product behind it.
__device__ __forceinline__ float rounded(float v) {
    asm("" : "+v"(v));
    return v;
}
__device__ __forceinline__ double rounded(double v) {
    asm("" : "+v"(v));
    return v;
}

// pend: kSideIdle, kSideActive, or the class of the ended side; for a face exit
// x, u, v are the last state inside, xb, iu, iv the step's end and increments.
template <typename R>
struct QuadLine {
    Coord<R> x, xb;
    R p0, u, v, iu, iv, b;
    double s, len, tw, tw_rate, bend;
    int steps, attempts, dir, pend;
    uint32_t evals;
};

template <typename R, class F, class FJ>
struct QuadScott {
    SideField<1, F> f;
    int n[3], na, len_lim;
    float top;  // the last cell of the lane's axis
    const ScottParams& P;

    __device__ __forceinline__ QuadScott(const F& ff, const ScottParams& p, int a) : f(ff, a), P(p) { set_box(ff, a); }
    // another field, for this lane's quad (lines of several fields in one launch)
    __device__ __forceinline__ void set_field(const F& ff, int a) {
        f = SideField<1, F>(ff, a);
        set_box(ff, a);
    }
    __device__ __forceinline__ void set_box(const F& ff, int a) {
        na = axis_of(ff.n[0], ff.n[1], ff.n[2], a);
        top = (float)(na - 2);
        len_lim = scott_len_lim(ff);
        n[0] = ff.n[0]; n[1] = ff.n[1]; n[2] = ff.n[2];
    }

    template <class FX>
    __device__ __forceinline__ void raw_all(const SideField<1, FX>& fx, double x, double out[3]) const {
        const double fl = floor(x);
        int c;
        R w, B, v[3];
        clamp_cell<R>(to_int(fl), (R)(x - fl), na, c, w);
        side_value<1, FX, R>(fx, &c, &w, &B);
        all_axes<1>(&B, v);
        out[0] = v[0]; out[1] = v[1]; out[2] = v[2];
    }

    // The quotient row J of scott_axis: ax is this lane's own axis.
    template <int J>
    __device__ __forceinline__ R quotient(const Axis<R>& own, unsigned cell, const R x[3], R B, R dj) const {
        const R ax_ap = quad_lane<J>(own.ap), ax_am = quad_lane<J>(own.am);
        const R ax_apn = quad_lane<J>(own.apn), ax_amp = quad_lane<J>(own.amp);
        R ap = rounded(ax_ap * dj), am = rounded(ax_am * dj);
        if (ax_apn != (R)0 || ax_amp != (R)0) {  // the +-h sample crosses a grid plane
            const bool up = ax_apn != (R)0;
            const int step = quad_lane<J>(f.stride[0]);
            R c[1][8];
            f.template load<R>(up ? cell + (unsigned)step : cell - (unsigned)step, c);
            const R dn = edge1<F, J, R>(c[0], x[0], x[1], x[2]);
            if (up) ap += ax_apn * dn;
            else am += ax_amp * dn;
            ap = rounded(ap);
            am = rounded(am);
        }
        const R Bp = B + ap, Bm = B - am, D = ap + am, S = Bp + Bm;
        R vp[3], vm[3], vd[3], vs[3];
        all_axes<1>(&Bp, vp);
        all_axes<1>(&Bm, vm);
        all_axes<1>(&D, vd);
        all_axes<1>(&S, vs);
        const R np2 = dot3(vp, vp), nm2 = dot3(vm, vm);
        const R ip = rsq(np2), im = rsq(nm2);
        const R np = np2 * ip, nm = nm2 * im;
        const R inv2h = (R)(0.5 / kFdH);
        const R t1 = (R)0.5 * (ip + im) * inv2h;
        // which of the two products the sum is fused with, as the one-lane kernels are compiled
        const R both = sizeof(R) == 4 ? fma(nm2, im, np) : np + nm;
        const R t2 = (R)0.5 * dot3(vs, vd) * ip * im * rcp(both) * inv2h;
        return D * t1 - S * t2;
    }

    // Rows of the axes whose +-h samples leave the cell, every place being inside
    // the box: axis_setup_sel's values without its places beyond the faces (at
    // x = 0 its lower sample is clamped to weight 0, as r = 0 gives).
    __device__ __forceinline__ void near_plane(unsigned cell, int i, R r, R w, R B, const R d[3], R J[3]) const {
        const R h = (R)kFdH;
        const bool down = !(r >= h), up = !(r + h <= (R)1);
        Axis<R> own;
        own.am = down ? r : h;
        own.amp = (down && i >= 1) ? h - r : (R)0;
        own.ap = up ? (R)1 - r : h;
        own.apn = (up && i + 1 <= na - 2) ? (r + h) - (R)1 : (R)0;
        const int code = down || up ? 1 : 0;
        int codes[3];
        all_axes<1>(&code, codes);
        R x[3];
        all_axes<1>(&w, x);
        if (codes[0]) J[0] = quotient<0>(own, cell, x, B, d[0]);
        if (codes[1]) J[1] = quotient<1>(own, cell, x, B, d[1]);
        if (codes[2]) J[2] = quotient<2>(own, cell, x, B, d[2]);
    }
    // The same for places anywhere (NaN among them), and every axis in FP64.
    __device__ __forceinline__ void any_place(unsigned cell, int i, R r, R w, const R bd[3], R& B, R& b, const R d[3],
                                              R J[3]) const {
        constexpr bool kExact = sizeof(R) == 8;
        const R h = (R)kFdH;
        int code = 2, codes[3] = {2, 2, 2};
        if constexpr (!kExact) {
            const bool odd = !((unsigned)i < (unsigned)(na - 1) && r >= h && r + h <= (R)1);
            const bool below = i < -1 || (i == -1 && !(r > (R)1 - h));          // x <= -h
            const bool above = i >= na - 1 && !(((R)(i - (na - 1)) + r) < h);  // x >= N-1+h
            code = odd ? (r == r && (below || above) ? 1 : 2) : 0;
            all_axes<1>(&code, codes);
            const R bad = r - r;  // 0, or NaN, which the clamped weight does not keep
            R bads[3];
            all_axes<1>(&bad, bads);
            const R any = bads[0] + bads[1] + bads[2];
            if (any != any) B = b = any;
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                if (codes[a] == 1) J[a] = (d[a] - b * bd[a]) * (R)0;
                if (any != any) J[a] = any;
            }
        }
        if (kExact || any_lane(code == 2)) {
            const Axis<R> own = axis_setup_sel<R>(i, r, na);
            R x[3];
            all_axes<1>(&w, x);
            if (codes[0] == 2) J[0] = quotient<0>(own, cell, x, B, d[0]);
            if (codes[1] == 2) J[1] = quotient<1>(own, cell, x, B, d[1]);
            if (codes[2] == 2) J[2] = quotient<2>(own, cell, x, B, d[2]);
        }
    }

    // scott_stage for this lane's components; b receives the unit field.
    __device__ __forceinline__ void stage(const QuadLine<R>& L, R dx, R du, R dv, R sc, R& kx, R& ku, R& kv, R& b) const {
        constexpr bool kExact = sizeof(R) == 8;
        const R h = (R)kFdH;
        int i, c;
        R r, w;
        float fh, fq;
        if constexpr (sizeof(R) == 4) {
            fh = floorf(L.x.hi);
            const float q = (L.x.hi - fh) + (L.x.lo + dx);
            fq = floorf(q);
            r = q - fq;
            clamp_cell_f(fh + fq, r, top, c, w);
        } else {
            const double q = L.x.x + dx;
            const double f0 = floor(q);
            i = to_int(f0);
            r = q - f0;
            clamp_cell<R>(i, r, na, c, w);
        }
        const unsigned cell = record_index<1, F>(f, &c);
        R cc[1][8], B, d[3];
        f.template load<R>(cell, cc);
        if constexpr (F::kCoef && sizeof(R) == 4) {
            quad_coef_eval(cc[0], w, B, d);
        } else {
            R x[3];
            all_axes<1>(&w, x);
            if constexpr (F::kCoef) coef_eval1<R>(cc[0], x[0], x[1], x[2], B, d);
            else cell_eval1<R>(cc[0], x[0], x[1], x[2], B, d);
        }
        R Bv[3], bv[3], bd[3], J[3];
        all_axes<1>(&B, Bv);
        const R inb = rsq(dot3(Bv, Bv));
        b = B * inb;
        if (!kExact) {  // the closed form on every axis
#pragma unroll
            for (int a = 0; a < 3; ++a) bv[a] = Bv[a] * inb;
            quad_dots(d, bv, bd);
#pragma unroll
            for (int a = 0; a < 3; ++a) J[a] = (d[a] - b * bd[a]) * inb;
        }
        // axes whose rows are another: zero (both samples beyond one face) or the
        // exact quotient; few stages of a wavefront have any
        // (a weight nearer to a face than h + 1e-6, which NaN and places outside
        // have too, for the exact test to follow)
        if (kExact || any_lane(!(fabsf((float)w - 0.5f) <= (float)(0.5 - kFdH - 1e-6)))) {
            if constexpr (!kExact) {
                i = sum_int(fh, fq);
                if (!any_lane(!((unsigned)i < (unsigned)(na - 1) && r == r))) {
                    near_plane(cell, i, r, w, B, d, J);
                } else {
                    any_place(cell, i, r, w, bd, B, b, d, J);
                }
            } else {
                any_place(cell, i, r, w, bd, B, b, d, J);
            }
        }
        kx = sc * b;
        R ju, jv;
        quad_rows(L.u + du, L.v + dv, J, ju, jv);
        ku = sc * ju;
        kv = sc * jv;
    }

    __device__ __forceinline__ bool can_step(const QuadLine<R>& L) const {
        return L.len < (double)len_lim && L.steps < kScottStepLim && L.attempts < kAttemptCap;
    }

    // One integrator attempt (scott_attempt).
    __device__ __forceinline__ void attempt(QuadLine<R>& L, const SideField<1, FJ>& fj) const {
        const R sc = (R)(L.s * L.dir);
        R incx, incu, incv;
        L.attempts += 1;
        if (P.method == kRKF45) {
            R x[6], u[6], v[6], tx, tu, tv, b;
            stage(L, (R)0, (R)0, (R)0, sc, x[0], u[0], v[0], L.b);
            tx = (R)Tab::a21 * x[0]; tu = (R)Tab::a21 * u[0]; tv = (R)Tab::a21 * v[0];
            stage(L, tx, tu, tv, sc, x[1], u[1], v[1], b);
            tx = (R)Tab::a31 * x[0] + (R)Tab::a32 * x[1];
            tu = (R)Tab::a31 * u[0] + (R)Tab::a32 * u[1];
            tv = (R)Tab::a31 * v[0] + (R)Tab::a32 * v[1];
            stage(L, tx, tu, tv, sc, x[2], u[2], v[2], b);
            tx = (R)Tab::a41 * x[0] + (R)Tab::a42 * x[1] + (R)Tab::a43 * x[2];
            tu = (R)Tab::a41 * u[0] + (R)Tab::a42 * u[1] + (R)Tab::a43 * u[2];
            tv = (R)Tab::a41 * v[0] + (R)Tab::a42 * v[1] + (R)Tab::a43 * v[2];
            stage(L, tx, tu, tv, sc, x[3], u[3], v[3], b);
            tx = (R)Tab::a51 * x[0] + (R)Tab::a52 * x[1] + (R)Tab::a53 * x[2] + (R)Tab::a54 * x[3];
            tu = (R)Tab::a51 * u[0] + (R)Tab::a52 * u[1] + (R)Tab::a53 * u[2] + (R)Tab::a54 * u[3];
            tv = (R)Tab::a51 * v[0] + (R)Tab::a52 * v[1] + (R)Tab::a53 * v[2] + (R)Tab::a54 * v[3];
            stage(L, tx, tu, tv, sc, x[4], u[4], v[4], b);
            tx = (R)Tab::a61 * x[0] + (R)Tab::a62 * x[1] + (R)Tab::a63 * x[2] + (R)Tab::a64 * x[3] +
                 (R)Tab::a65 * x[4];
            tu = (R)Tab::a61 * u[0] + (R)Tab::a62 * u[1] + (R)Tab::a63 * u[2] + (R)Tab::a64 * u[3] +
                 (R)Tab::a65 * u[4];
            tv = (R)Tab::a61 * v[0] + (R)Tab::a62 * v[1] + (R)Tab::a63 * v[2] + (R)Tab::a64 * v[3] +
                 (R)Tab::a65 * v[4];
            stage(L, tx, tu, tv, sc, x[5], u[5], v[5], b);
            incx = (R)Tab::b1 * x[0] + (R)Tab::b3 * x[2] + (R)Tab::b4 * x[3] + (R)Tab::b5 * x[4] + (R)Tab::b6 * x[5];
            incu = (R)Tab::b1 * u[0] + (R)Tab::b3 * u[2] + (R)Tab::b4 * u[3] + (R)Tab::b5 * u[4] + (R)Tab::b6 * u[5];
            incv = (R)Tab::b1 * v[0] + (R)Tab::b3 * v[2] + (R)Tab::b4 * v[3] + (R)Tab::b5 * v[4] + (R)Tab::b6 * v[5];
            const double ec = Tab::e1 * (double)x[0] + Tab::e3 * (double)x[2] + Tab::e4 * (double)x[3] +
                              Tab::e5 * (double)x[4] + Tab::e6 * (double)x[5];
            double ev[3], e2 = 0.0;
            all_axes<1>(&ec, ev);
#pragma unroll
            for (int a = 0; a < 3; ++a) e2 += ev[a] * ev[a];
            L.evals += 6;
            const double scale = sizeof(R) == 4 ? P.ctl * pow_minus_tenth(e2) : pow(P.tol / sqrt(e2) / 11.09, 0.2);
            if (scale < 0.618) {
                L.s = L.s * 0.618;
                if (!can_step(L)) L.pend = kClassLimit;
                return;
            }
            L.s = L.s * scale;
            if (L.s > 100.) L.s = 100.;
            if (L.s < 1. / 10.) L.s = 1. / 10.;
        } else {
            const R half = (R)0.5;
            R kx, ku, kv, tx, tu, tv, b;
            stage(L, (R)0, (R)0, (R)0, sc, kx, ku, kv, L.b);
            incx = kx; incu = ku; incv = kv;
            tx = half * kx; tu = half * ku; tv = half * kv;
            stage(L, tx, tu, tv, sc, kx, ku, kv, b);
            incx += (R)2 * kx; incu += (R)2 * ku; incv += (R)2 * kv;
            tx = half * kx; tu = half * ku; tv = half * kv;
            stage(L, tx, tu, tv, sc, kx, ku, kv, b);
            incx += (R)2 * kx; incu += (R)2 * ku; incv += (R)2 * kv;
            stage(L, kx, ku, kv, sc, tx, tu, tv, b);
            incx = (incx + tx) * (R)(1.0 / 6.0);
            incu = (incu + tu) * (R)(1.0 / 6.0);
            incv = (incv + tv) * (R)(1.0 / 6.0);
            L.evals += 4;
        }
        const Coord<R> xb = L.x.add(incx);
        R iv[3];
        all_axes<1>(&incx, iv);
        const double dL = sizeof(R) == 4 ? (double)sqrtf((float)(iv[0] * iv[0] + iv[1] * iv[1] + iv[2] * iv[2]))
                                         : sqrt((double)iv[0] * iv[0] + (double)iv[1] * iv[1] + (double)iv[2] * iv[2]);
        L.len += dL;
        double tw_rate = 0.0, Bend[3] = {0.0, 0.0, 0.0};
        if constexpr (has_current<FJ>()) {  // at the step's end point (TraceBlineScott.cu:423-427)
            double Jc[3];
            const double xe = xb.get();
            raw_all<FJ>(fj, xe, Jc);
            raw_all<F>(f, xe, Bend);
            tw_rate = dot3(Jc, Bend) / dot3(Bend, Bend) * kQuarterOverPi;
            L.tw += tw_rate * dL;
        }
        const int in = xb.inside(na) ? 1 : 0;
        int in_all[3];
        all_axes<1>(&in, in_all);
        if ((in_all[0] & in_all[1] & in_all[2]) == 0) {
            const double xe = xb.get();
            double p[3];
            all_axes<1>(&xe, p);
            const int flag = check_flag(n, p);
            if (flag > 0) {
                L.len -= dL;
                if constexpr (has_current<FJ>()) {
                    L.tw -= tw_rate * dL;  // :432-434
                    L.tw_rate = tw_rate;
                    L.bend = flag <= 6 ? (flag <= 2 ? Bend[0] : (flag <= 4 ? Bend[1] : Bend[2])) : 0.0;
                }
                L.pend = flag;
                L.xb = xb;
                L.iu = incu;
                L.iv = incv;
                return;
            }
        }
        L.x = xb;
        L.u += incu;
        L.v += incv;
        L.steps += 1;
        if (!can_step(L)) L.pend = kClassLimit;
    }

    // Footpoint (x, u, v) of an ended side, this lane's components.
    __device__ __forceinline__ void land(QuadLine<R>& L, R& fx, R& fu, R& fv) const {
        const double xa = L.x.get();
        fx = (R)xa; fu = L.u; fv = L.v;
        if (L.pend < 1 || L.pend > 6) return;
        L.steps += 1;
        const double xb = L.xb.get();
        const int dim = (L.pend - 1) / 2;
        const double p1 = pick_axis<1>(&xa, dim), p2 = pick_axis<1>(&xb, dim);
        if (!(fabs(p1 - p2) > 0)) return;
        // linear landing of the 9-vector on the face (TraceBlineScott.cu:442-448);
        // max faces land on index N
        const double pm = (L.pend % 2 == 1) ? 0.0 : (double)axis_of(n[0], n[1], n[2], dim);
        const double wa = (p2 - pm) / (p2 - p1), wb = (pm - p1) / (p2 - p1);
        fx = (R)(fma(xa, p2 - pm, xb * (pm - p1)) / (p2 - p1));
        fu = (R)((double)L.u * wa + (double)(L.u + L.iu) * wb);
        fv = (R)((double)L.v * wa + (double)(L.v + L.iv) * wb);
        double bdim;
        if constexpr (has_current<FJ>()) bdim = L.bend;
        else bdim = (double)pick_axis<1>(&L.b, dim);
        const double arc = fabs(pm - p1) / (1e-4 + fabs(bdim));
        L.len += arc;
        if constexpr (has_current<FJ>()) L.tw += L.tw_rate * arc;
    }
};

#endif  // __HIP_DEVICE_COMPILE__

}  // namespace fqsl
