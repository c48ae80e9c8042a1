// fqsl_quad.h -- the position-only tracers on the device, one line side per lane
// or per four lanes.
//
// A line of a plain (position-only) trace is a serial chain: six stage
// evaluations per attempt, each a cell load that waits for the stage point and
// a stage point that waits for the load.  A map's time has two parts: the
// chain of its longest side (thousands of evaluations; the average side takes
// fifty), and the instructions of all of them.
//
// K = 1 shortens the chain.  Lane q = 0, 1, 2 of a quad owns axis q and
// component q: it forms its own coordinate's stage point and cell, loads its
// own component's eight coefficients (two 16-byte loads, adjacent to its
// neighbours'), evaluates its own component, and the three weights, the cell
// index and the three components of B pass between the lanes by quad permutes
// (DPP).  Lane 3 repeats lane 0, so control flow is the same on all four.  A
// stage is ~42 instructions long.  K = 3 keeps the three axes in one lane: ~80
// instructions a stage, but for 64 sides and not 16.
//
// Forward and backward sides do not depend on each other in these tracers
// (each starts from the seed with the initial step), so they are separate
// tasks of the queue.  Every value is formed by the same expression on the same
// operands as in the one-thread-per-line code of fqsl_tracer.h /
// fqsl_stretch.h, which the CPU tests build.  FP32 lines have the same bits; of
// FP64 lines on uniform grids, where the compiler fuses products and sums in
// another order, one length in twenty differs in its last place; and the twists
// of the two sides are summed apart, not one after the other.
#pragma once

#include "fqsl_stretch.h"
#include "fqsl_tracer.h"
#include "fqsl_step.h"

namespace fqsl {

// Geometry of the plain tracer: grid-index coordinates, a stretched grid
// (StretchRef), or a float stretched grid whose compact lookup table each
// workgroup copies to LDS at the start (`lds_bytes` of dynamic shared memory):
// the bin record of a stage point is then an LDS read instead of a global load
// that the cell load has to wait for.
struct UniformGrid {};
struct StretchLds {
    const StretchGrid<float>* g;
    int lds_bytes;
};

#if defined(__HIP_DEVICE_COMPILE__)

// ------------------------------------------------------- lanes of a side
template <int kLane>
__device__ __forceinline__ int quad_lane(int v) {
    return __builtin_amdgcn_mov_dpp(v, kLane * 0x55, 0xf, 0xf, true);
}
template <int kLane>
__device__ __forceinline__ float quad_lane(float v) {
    return __int_as_float(quad_lane<kLane>(__float_as_int(v)));
}
template <int kLane>
__device__ __forceinline__ double quad_lane(double v) {
    return __hiloint2double(quad_lane<kLane>(__double2hiint(v)), quad_lane<kLane>(__double2loint(v)));
}

// The three axes' values, on every lane of the side, from the K that this lane
// holds.
template <int K, typename T>
__device__ __forceinline__ void all_axes(const T* v, T out[3]) {
    if constexpr (K == 1) {
        out[0] = quad_lane<0>(v[0]);
        out[1] = quad_lane<1>(v[0]);
        out[2] = quad_lane<2>(v[0]);
    } else {
        out[0] = v[0]; out[1] = v[1]; out[2] = v[2];
    }
}
template <int K, typename T>
__device__ __forceinline__ T pick_axis(const T* v, int dim) {
    T a[3];
    all_axes<K>(v, a);
    return dim == 0 ? a[0] : (dim == 1 ? a[1] : a[2]);
}
// Float arithmetic on values of the quad's other lanes, as DPP operands of the
// multiply-adds themselves.  (The compiler moves such operands to registers
// first: it selects the three-address multiply-add, which has no DPP form.)  Two
// wait states separate a register's last write from its reading by DPP; the
// compiler cannot see into the block, so each begins with them.
#define FQSL_Q0 " quad_perm:[0,0,0,0] row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
#define FQSL_Q1 " quad_perm:[1,1,1,1] row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
#define FQSL_Q2 " quad_perm:[2,2,2,2] row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"

// Sum over the three axes, on every lane.
__device__ __forceinline__ int quad_sum(int v) {
    int r;
    asm("s_nop 1\n\t"
        "v_add_u32_dpp %0, %1, %1 quad_perm:[1,2,0,1] row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
        "v_add_u32_dpp %0, %1, %0 quad_perm:[2,0,1,2] row_mask:0xf bank_mask:0xf bound_ctrl:1"
        : "=&v"(r) : "v"(v));
    return r;
}
// coef_value1 with this lane's component c and the weight each lane holds.
__device__ __forceinline__ float quad_coef_value(const float c[8], float w) {
    float c0 = c[0], c1 = c[1], c3 = c[3], c6 = c[6];
    asm("s_nop 1\n\t"
        "v_fmac_f32_dpp %0, %4, %5" FQSL_Q1  // c0 + c2 y
        "v_fmac_f32_dpp %1, %4, %6" FQSL_Q1  // c1 + c4 y
        "v_fmac_f32_dpp %3, %4, %8" FQSL_Q1  // c6 + c7 y
        "v_fmac_f32_dpp %2, %4, %7" FQSL_Q1  // c3 + c5 y
        "v_fmac_f32_dpp %0, %4, %1" FQSL_Q0  // A
        "v_fmac_f32_dpp %2, %4, %3" FQSL_Q0  // C
        "v_fmac_f32_dpp %0, %4, %2" FQSL_Q2  // A + z C
        : "+v"(c0), "+v"(c1), "+v"(c3), "+v"(c6) : "v"(w), "v"(c[2]), "v"(c[4]), "v"(c[5]), "v"(c[7]));
    return c0;
}

// First of the axes a lane holds: its own of a quad (lane 3 repeats axis 0), 0
// when it holds all.
template <int K>
__device__ __forceinline__ int first_axis() {
    if constexpr (K == 3) return 0;
    const int q = __lane_id() & 3;
    return q == 3 ? 0 : q;
}
template <typename T>
__device__ __forceinline__ T axis_of(T x, T y, T z, int a) {
    return a == 0 ? x : (a == 1 ? y : z);
}

// ------------------------------------------------------- field views
// What a lane needs of the field: the components it evaluates, its axes' node
// counts and the distance in the record index between neighbours along them.
template <int K, class F>
struct SideField;

template <int K>
struct SideField<K, NoCurrent> {
    __device__ __forceinline__ SideField(const NoCurrent&, int) {}
};

template <int K>
struct SideField<K, FieldCell32> {
    const FQSL_GLOBAL float4* base;  // first record of this lane's first component
    int stride[K];
    __device__ __forceinline__ SideField(const FieldCell32& f, int a) : base((const FQSL_GLOBAL float4*)f.cells + 2 * a) {
        const int s[3] = {1, f.n[0] - 1, (f.n[0] - 1) * (f.n[1] - 1)};
#pragma unroll
        for (int q = 0; q < K; ++q) stride[q] = K == 3 ? s[q] : axis_of(s[0], s[1], s[2], a);
    }
    template <typename R>
    __device__ __forceinline__ void load(unsigned cell, R c[K][8]) const {
        const FQSL_GLOBAL float4* p = base + 8 * (unsigned long long)cell;
#pragma unroll
        for (int q = 0; q < K; ++q) {
            const float4 lo = p[2 * q], hi = p[2 * q + 1];
            c[q][0] = lo.x; c[q][1] = lo.y; c[q][2] = lo.z; c[q][3] = lo.w;
            c[q][4] = hi.x; c[q][5] = hi.y; c[q][6] = hi.z; c[q][7] = hi.w;
        }
    }
};

template <int K, typename T>
struct SideField<K, FieldSoA<T>> {
    const FQSL_GLOBAL T* base[K];
    int stride[K], nx, nxy;
    __device__ __forceinline__ SideField(const FieldSoA<T>& f, int a) : nx(f.n[0]), nxy(f.n[0] * f.n[1]) {
        const T* b[3] = {f.bx, f.by, f.bz};
        const int s[3] = {1, nx, nxy};
#pragma unroll
        for (int q = 0; q < K; ++q) {
            base[q] = (const FQSL_GLOBAL T*)(K == 3 ? b[q] : axis_of(b[0], b[1], b[2], a));
            stride[q] = K == 3 ? s[q] : axis_of(s[0], s[1], s[2], a);
        }
    }
    template <typename R>
    __device__ __forceinline__ void load(unsigned node, R c[K][8]) const {
#pragma unroll
        for (int q = 0; q < K; ++q) {
            const FQSL_GLOBAL T* p = base[q] + (unsigned long long)node;
#pragma unroll
            for (int k = 0; k < 8; ++k) c[q][k] = (R)p[(k & 1) + ((k >> 1) & 1) * nx + ((k >> 2) & 1) * (long)nxy];
        }
    }
};

template <>
struct SideField<1, FieldPairs> {
    const FQSL_GLOBAL float2* base;
    int stride[1], nx, nxy;
    __device__ __forceinline__ SideField(const FieldPairs& f, int a)
        : base((const FQSL_GLOBAL float2*)f.pairs + a), nx(f.n[0]), nxy(f.n[0] * f.n[1]) {
        stride[0] = axis_of(1, nx, nxy, a);
    }
    template <typename R>
    __device__ __forceinline__ void load(unsigned node, R c[1][8]) const {
        const FQSL_GLOBAL float2* p = base + 4 * (unsigned long long)node;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const float2 v = p[4 * ((k & 1) * (long)nx + (k >> 1) * (long)nxy)];
            c[0][2 * k] = (R)v.x;
            c[0][2 * k + 1] = (R)v.y;
        }
    }
};

// Index of the record at the cells the lanes hold.
template <int K, class F>
__device__ __forceinline__ unsigned record_index(const SideField<K, F>& f, const int* c) {
    if constexpr (K == 1) return (unsigned)quad_sum(c[0] * f.stride[0]);
    else return (unsigned)(c[0] * f.stride[0] + c[1] * f.stride[1] + c[2] * f.stride[2]);
}

// This lane's components of B at the cells and weights the lanes hold.
template <int K, class F, typename R>
__device__ __forceinline__ void side_value(const SideField<K, F>& f, const int* c, const R* w, R B[K]) {
    R k[K][8], x[3];
    f.template load<R>(record_index<K, F>(f, c), k);
    if constexpr (K == 1 && F::kCoef && sizeof(R) == 4) {
        B[0] = quad_coef_value(k[0], w[0]);
        return;
    }
    all_axes<K>(w, x);
#pragma unroll
    for (int q = 0; q < K; ++q) {
        if constexpr (F::kCoef) B[q] = coef_value1<R>(k[q], x[0], x[1], x[2]);
        else B[q] = cell_value1<R>(k[q], x[0], x[1], x[2]);
    }
}

template <int K, typename R>
__device__ __forceinline__ void side_unit(const R B[K], R b[K]) {
    R v[3];
    all_axes<K>(B, v);
    const R inb = rsq(dot3(v, v));
#pragma unroll
    for (int q = 0; q < K; ++q) b[q] = B[q] * inb;
}

__device__ __forceinline__ float clamp01(float t) { return fminf(fmaxf(t, 0.f), 1.f); }
__device__ __forceinline__ double clamp01(double t) { return fmin(fmax(t, 0.), 1.); }

// Cell and weight of x = i + r by the Interp3dxyzn clamp rule, as axis_setup's
// c and w without its branches: outside the box the distance to the clamped
// cell saturates the weight at 0 or 1, and r - r carries a NaN through.
template <typename R>
__device__ __forceinline__ void clamp_cell(int i, R r, int n, int& c, R& w) {
    c = max(min(i, n - 2), 0);
    w = clamp01(r + (R)(i - c)) + (r - r);
}

// The same for x = f + r with the whole part held as a float (exact below 2^24;
// beyond, only its side of the box counts), top = n - 2: a NaN gives weight 0.
__device__ __forceinline__ void clamp_cell_f(float f, float r, float top, int& c, float& w) {
    const float cf = __builtin_amdgcn_fmed3f(f, 0.f, top);
    c = (int)cf;
    w = clamp01(r + (f - cf));
}

// a + b of two whole numbers held as floats, as an integer.  The conversion and
// the sum saturate (to_int's limits lie in the same direction of the array), and
// NaN gives 0: its weight is NaN in any cell.
__device__ __forceinline__ int cvt_int(float v) {
    int i;
    asm("v_cvt_i32_f32_e32 %0, %1" : "=v"(i) : "v"(v));
    return i;
}
__device__ __forceinline__ int sum_int(float a, float b) { return __builtin_elementwise_add_sat(cvt_int(a), cvt_int(b)); }
__device__ __forceinline__ bool any_lane(bool v) { return __builtin_amdgcn_ballot_w64(v) != 0ull; }

// ------------------------------------------------------- positions
// One coordinate: a compensated float pair, or a double.
template <typename R>
struct Coord;
template <>
struct Coord<float> {
    float hi, lo;
    __device__ __forceinline__ void set_f(float v) { hi = v; lo = 0.f; }
    __device__ __forceinline__ double get() const { return (double)hi + (double)lo; }
    __device__ __forceinline__ Coord add(float inc) const {
        const float t = lo + inc;
        const float s = hi + t;
        const float bb = s - hi;
        const float err = (hi - (s - bb)) + (t - bb);
        return Coord{s, err};
    }
    // strictly inside (0, n - 1): then so is hi + lo, which check_flag compares
    __device__ __forceinline__ bool inside(int n) const { return hi > 0.f && hi < (float)(n - 1); }
};
template <>
struct Coord<double> {
    double x;
    __device__ __forceinline__ void set_f(float v) { x = v; }
    __device__ __forceinline__ double get() const { return x; }
    __device__ __forceinline__ Coord add(double inc) const { return Coord{x + inc}; }
    __device__ __forceinline__ bool inside(int n) const { return x > 0. && x < n - 1.; }
};

// ------------------------------------------------------- geometries
// cell(): cell and weight, along axis q of this lane, of the stage point x + d;
// cell_at(): of a double position; inside(): a sufficient test for class 0;
// flag(): the exit class from the three coordinates.
template <int K, class G, typename R>
struct SideGeom;

template <int K, typename R>
struct SideGeom<K, UniformGrid, R> {
    int n[3], na[K];
    __device__ __forceinline__ SideGeom(const UniformGrid&, const int* nn, int a) {
        n[0] = nn[0]; n[1] = nn[1]; n[2] = nn[2];
#pragma unroll
        for (int q = 0; q < K; ++q) na[q] = K == 3 ? nn[q] : axis_of(nn[0], nn[1], nn[2], a);
    }
    __device__ __forceinline__ void cell(int q, const Coord<R>& x, R d, int& c, R& w) const {
        if constexpr (sizeof(R) == 4) {
            const float fh = floorf(x.hi);
            const float u = (x.hi - fh) + (x.lo + d);
            const float fu = floorf(u);
            clamp_cell<R>(sum_int(fh, fu), u - fu, na[q], c, w);
        } else {
            const double v = x.x + d;
            const double f = floor(v);
            clamp_cell<R>(to_int(f), v - f, na[q], c, w);
        }
    }
    __device__ __forceinline__ void cell_at(int q, double x, int& c, R& w) const {
        const double f = floor(x);
        clamp_cell<R>(to_int(f), (R)(x - f), na[q], c, w);
    }
    __device__ __forceinline__ bool inside(int q, const Coord<R>& x) const { return x.inside(na[q]); }
    __device__ __forceinline__ int flag(const double* p) const { return check_flag(n, p); }
    __device__ __forceinline__ double land(int flag, int dim) const {
        return (flag % 2 == 1) ? 0.0 : (double)axis_of(n[0], n[1], n[2], dim);
    }
    // Interp3d's clamp of b_clamped, in float as the reference
    __device__ __forceinline__ double out_point(int q, float v) const {
        v = (v > 0.f) ? v : 0.0001f;
        v = (v < (float)(na[q] - 1)) ? v : (float)((double)na[q] - 1 - 0.0001);
        return v;
    }
    __device__ __forceinline__ double len_lim(int method) const {
        return (method == kRKF45 ? kPlainRkf45LenRatio : kPlainRk4LenRatio) * (n[0] + n[1] + n[2]);
    }
    __device__ __forceinline__ int step_lim(int method) const {
        return method == kRKF45 ? kPlainRkf45StepLim : kPlainRk4StepLim;
    }
    static constexpr bool kLandTwist = false;  // RKF45's landing twist
};

template <int K, typename R, bool kL>
struct SideStretch {
    const FQSL_CONST StretchGrid<R>& g;
    const FQSL_CONST StretchAxis<R>* ax;
    StretchAxis<R> A[K];  // what a lookup reads of this lane's axes
    int rule;
    double lo[K], hi[K];
    __device__ __forceinline__ SideStretch(const FQSL_CONST StretchGrid<R>* gp, int a)
        : g(*gp), ax(gp->ax + a), rule(gp->rule) {
#pragma unroll
        for (int q = 0; q < K; ++q) {
            A[q].brec = ax[q].brec;
            A[q].lo = ax[q].lo; A[q].hi = ax[q].hi; A[q].clo = ax[q].clo; A[q].chi = ax[q].chi;
            A[q].bin_scale = ax[q].bin_scale;
            A[q].nbins = ax[q].nbins; A[q].lbin = ax[q].lbin; A[q].lcell = ax[q].lcell;
            lo[q] = gp->lo[a + q];
            hi[q] = gp->hi[a + q];
        }
    }
    __device__ __forceinline__ void locate(int q, R phi, R plo, int& c, R& w) const {
        if constexpr (kL) stretch_locate_lds(A[q], ax + q, rule, phi, plo, c, w);
        else stretch_locate<R>(A[q], ax + q, rule, phi, plo, c, w);
    }
    __device__ __forceinline__ void cell(int q, const Coord<R>& x, R d, int& c, R& w) const {
        if constexpr (sizeof(R) == 4) locate(q, x.hi, x.lo + d, c, w);
        else locate(q, x.x, d, c, w);
    }
    __device__ __forceinline__ void cell_at(int q, double x, int& c, R& w) const {
        const R phi = (R)x;
        locate(q, phi, (R)(x - (double)phi), c, w);
    }
    __device__ __forceinline__ bool inside(int q, const Coord<R>& x) const {
        const double p = x.get();
        return p > lo[q] && p < hi[q];
    }
    __device__ __forceinline__ int flag(const double* p) const {
        const double l[3] = {g.lo[0], g.lo[1], g.lo[2]}, h[3] = {g.hi[0], g.hi[1], g.hi[2]};
        return check_flag_box(l, h, p);
    }
    __device__ __forceinline__ double land(int flag, int dim) const {
        return (flag % 2 == 1) ? g.land_lo[dim] : g.land_hi[dim];
    }
    __device__ __forceinline__ double out_point(int, float v) const { return v; }
    __device__ __forceinline__ double len_lim(int) const { return g.len_lim; }
    __device__ __forceinline__ int step_lim(int) const { return INT_MAX; }
    static constexpr bool kLandTwist = true;
};

template <int K, typename R>
struct SideGeom<K, StretchRef<R>, R> : SideStretch<K, R, false> {
    __device__ __forceinline__ SideGeom(const StretchRef<R>& r, const int*, int a)
        : SideStretch<K, R, false>((const FQSL_CONST StretchGrid<R>*)r.g, a) {}
};
template <int K>
struct SideGeom<K, StretchLds, float> : SideStretch<K, float, true> {
    __device__ __forceinline__ SideGeom(const StretchLds& r, const int*, int a)
        : SideStretch<K, float, true>((const FQSL_CONST StretchGrid<float>*)r.g, a) {}
};

// ------------------------------------------------------- one line side
constexpr int kSideActive = -1, kSideIdle = -2;

// pend is kSideActive while the side is traced; then its class, and x is the
// recorded point or, for a face exit (1..6), the last point inside with xb the
// first one outside.
template <int K, typename R>
struct Side {
    Coord<R> x[K], xb[K];
    double s, len, tw;
    double tol;  // RKF45: the line's tolerance
    int steps, attempts, dir, pend;
    uint32_t evals;
};

// The RKF45 tolerance of a line (TraceBlineAdaptive.cu:354-359), out of line.
FQSL_COLD double plain_tol(double bn, double tol_coef) {
    return (bn <= 0.05 ? kTolBase / 8e3 : kTolBase * pow(bn, 1.5)) * tol_coef;
}

// Step control (TraceBlineAdaptive.cu:365-370) with the hardware's estimates: scales s,
// false when the step is rejected.
__device__ __forceinline__ bool next_step(double& s, double tol, double e2, double limit) {
    double q;
    float g;
    if (step_is_plain(tol, e2, limit)) {
        q = scale_argument(tol, e2, __builtin_amdgcn_rsq(e2));
        g = __builtin_amdgcn_exp2f(0.2f * __builtin_amdgcn_logf((float)q));
    } else {
        q = scale_argument_wide(tol, e2);
        g = NAN;
    }
    const Step n = step_of_argument(s, q, g);
    s = n.s;
    return n.accepted;
}

template <int K, typename R, class F, class FJ, class G>
struct SideTracer {
    SideField<K, F> f;
    SideGeom<K, G, R> geo;
    const PlainParams& P;
    double len_lim, tol_limit;
    int step_lim;

    __device__ __forceinline__ SideTracer(const F& ff, const G& g, const PlainParams& p, int a)
        : f(ff, a), geo(g, ff.n, a), P(p), len_lim(geo.len_lim(p.method)),
          tol_limit(step_tol_limit(p.s0)), step_lim(geo.step_lim(p.method)) {}

    __device__ __forceinline__ void unit(const Coord<R>* x, const R* d, R b[K]) const {
        int c[K];
        R w[K], B[K];
#pragma unroll
        for (int q = 0; q < K; ++q) geo.cell(q, x[q], d[q], c[q], w[q]);
        side_value<K, F, R>(f, c, w, B);
        side_unit<K, R>(B, b);
    }
    template <class FX>
    __device__ __forceinline__ void raw_at(const SideField<K, FX>& fx, const double* x, R B[K]) const {
        int c[K];
        R w[K];
#pragma unroll
        for (int q = 0; q < K; ++q) geo.cell_at(q, x[q], c[q], w[q]);
        side_value<K, FX, R>(fx, c, w, B);
    }
    __device__ __forceinline__ void unit_at(const double* x, R b[K]) const {
        R B[K];
        raw_at<F>(f, x, B);
        side_unit<K, R>(B, b);
    }
    // the raw field at x, all components, in double
    template <class FX>
    __device__ __forceinline__ void raw_all(const SideField<K, FX>& fx, const double* x, double out[3]) const {
        R B[K], v[3];
        raw_at<FX>(fx, x, B);
        all_axes<K>(B, v);
        out[0] = v[0]; out[1] = v[1]; out[2] = v[2];
    }
    __device__ __forceinline__ bool can_step(const Side<K, R>& L) const {
        return L.len < len_lim && L.steps < step_lim && L.attempts < kAttemptCap;
    }

    // |b.n| at a seed, which sets the RKF45 tolerance.
    __device__ __forceinline__ double slope(const float* p0) const {
        double x[K];
        R b[K], v[3];
#pragma unroll
        for (int q = 0; q < K; ++q) x[q] = (double)p0[q];
        unit_at(x, b);
        all_axes<K>(b, v);
        return fabs((double)v[0] * P.ncross[0] + (double)v[1] * P.ncross[1] + (double)v[2] * P.ncross[2]);
    }

    __device__ __forceinline__ void init(Side<K, R>& L, const float* p0, int dir) const {
        L.tol = P.method == kRKF45 ? plain_tol(slope(p0), P.tol_coef) : 0.0;
#pragma unroll
        for (int q = 0; q < K; ++q) L.x[q].set_f(p0[q]);
        L.s = P.s0;
        L.len = 0.0;
        L.tw = 0.0;
        L.steps = 0;
        L.attempts = 0;
        L.dir = dir;
        L.pend = kSideActive;
        L.evals = 0;
    }

    // One integrator attempt (plain_attempt / stretch_attempt).
    __device__ __forceinline__ void attempt(Side<K, R>& L, const SideField<K, FJ>& fj) const {
        const R sc = (R)(L.s * L.dir);
        R inc[K];
        const R zero[K] = {};
        L.attempts += 1;
        if (P.method == kRKF45) {
            R k[6][K], t[K];
            unit(L.x, zero, k[0]);
#pragma unroll
            for (int a = 0; a < K; ++a) { k[0][a] *= sc; t[a] = (R)Tab::a21 * k[0][a]; }
            unit(L.x, t, k[1]);
#pragma unroll
            for (int a = 0; a < K; ++a) { k[1][a] *= sc; t[a] = (R)Tab::a31 * k[0][a] + (R)Tab::a32 * k[1][a]; }
            unit(L.x, t, k[2]);
#pragma unroll
            for (int a = 0; a < K; ++a) {
                k[2][a] *= sc;
                t[a] = (R)Tab::a41 * k[0][a] + (R)Tab::a42 * k[1][a] + (R)Tab::a43 * k[2][a];
            }
            unit(L.x, t, k[3]);
#pragma unroll
            for (int a = 0; a < K; ++a) {
                k[3][a] *= sc;
                t[a] = (R)Tab::a51 * k[0][a] + (R)Tab::a52 * k[1][a] + (R)Tab::a53 * k[2][a] + (R)Tab::a54 * k[3][a];
            }
            unit(L.x, t, k[4]);
#pragma unroll
            for (int a = 0; a < K; ++a) {
                k[4][a] *= sc;
                t[a] = (R)Tab::a61 * k[0][a] + (R)Tab::a62 * k[1][a] + (R)Tab::a63 * k[2][a] +
                       (R)Tab::a64 * k[3][a] + (R)Tab::a65 * k[4][a];
            }
            unit(L.x, t, k[5]);
            double ec[K], ev[3], e2 = 0.0;
#pragma unroll
            for (int a = 0; a < K; ++a) {
                k[5][a] *= sc;
                inc[a] = (R)Tab::b1 * k[0][a] + (R)Tab::b3 * k[2][a] + (R)Tab::b4 * k[3][a] +
                         (R)Tab::b5 * k[4][a] + (R)Tab::b6 * k[5][a];
                ec[a] = Tab::e1 * (double)k[0][a] + Tab::e3 * (double)k[2][a] + Tab::e4 * (double)k[3][a] +
                        Tab::e5 * (double)k[4][a] + Tab::e6 * (double)k[5][a];
            }
            all_axes<K>(ec, ev);
#pragma unroll
            for (int a = 0; a < 3; ++a) e2 += ev[a] * ev[a];
            L.evals += 6;
            bool accept;
            if constexpr (sizeof(R) == 4) {
                accept = next_step(L.s, L.tol, e2, tol_limit);
            } else {
                const double scale = pow(L.tol / sqrt(e2) / 11.09, 0.2);
                accept = !(scale < 0.618);
                L.s = L.s * (accept ? scale : 0.618);
                if (accept) {
                    if (L.s > 100.) L.s = 100.;
                    if (L.s < 1. / 10.) L.s = 1. / 10.;
                }
            }
            if (!accept) {
                if (!can_step(L)) L.pend = kClassLimit;
                return;
            }
        } else {
            R k[K], t[K];
            unit(L.x, zero, k);
#pragma unroll
            for (int a = 0; a < K; ++a) { inc[a] = k[a]; t[a] = sc * k[a] * (R)0.5; }
            unit(L.x, t, k);
#pragma unroll
            for (int a = 0; a < K; ++a) { inc[a] += (R)2 * k[a]; t[a] = sc * k[a] * (R)0.5; }
            unit(L.x, t, k);
#pragma unroll
            for (int a = 0; a < K; ++a) { inc[a] += (R)2 * k[a]; t[a] = sc * k[a]; }
            unit(L.x, t, k);
#pragma unroll
            for (int a = 0; a < K; ++a) inc[a] = (R)(1.0 / 6.0) * sc * (inc[a] + k[a]);
            L.evals += 4;
        }
        Coord<R> xb[K];
        R iv[3];
        bool in = true;
        int in_all[3];
        {
            int in_q[K];
#pragma unroll
            for (int a = 0; a < K; ++a) {
                xb[a] = L.x[a].add(inc[a]);
                in_q[a] = geo.inside(a, xb[a]) ? 1 : 0;
            }
            all_axes<K>(in_q, in_all);
            in = (in_all[0] & in_all[1] & in_all[2]) != 0;
        }
        all_axes<K>(inc, iv);
        const double dl = sqrt((double)iv[0] * iv[0] + (double)iv[1] * iv[1] + (double)iv[2] * iv[2]);
        double tw_rate = 0.0;
        if constexpr (has_current<FJ>()) {  // at the step's start point (TraceBline.cu:325-329)
            double xa[K], J[3], B[3];
#pragma unroll
            for (int a = 0; a < K; ++a) xa[a] = L.x[a].get();
            raw_all<FJ>(fj, xa, J);
            raw_all<F>(f, xa, B);
            tw_rate = dot3(J, B) / dot3(B, B) * kQuarterOverPi;
        }
        L.steps += 1;
        if (!in) {
            double xq[K], p[3];
#pragma unroll
            for (int a = 0; a < K; ++a) xq[a] = xb[a].get();
            all_axes<K>(xq, p);
            const int flag = geo.flag(p);
            if (flag > 0) {
                L.pend = flag;
#pragma unroll
                for (int a = 0; a < K; ++a) {
                    if (flag <= 6) L.xb[a] = xb[a];
                    else L.x[a] = xb[a];  // "ignore": the outside point itself
                }
                // the step's length and twist, added and taken back as the
                // reference does: the rounding of len + dl - dl stays
                L.len += dl;
                L.len -= dl;
                if constexpr (has_current<FJ>()) { L.tw += tw_rate * dl; L.tw -= tw_rate * dl; }
                return;
            }
        }
        L.len += dl;
        if constexpr (has_current<FJ>()) L.tw += tw_rate * dl;
#pragma unroll
        for (int a = 0; a < K; ++a) L.x[a] = xb[a];
        if (!can_step(L)) L.pend = kClassLimit;
    }

    // Footpoint of an ended side, this lane's coordinates.
    __device__ __forceinline__ void land(Side<K, R>& L, const SideField<K, FJ>& fj, double out[K]) const {
        double xa[K], xb[K];
#pragma unroll
        for (int a = 0; a < K; ++a) { xa[a] = L.x[a].get(); out[a] = xa[a]; }
        if (L.pend < 1 || L.pend > 6) return;
#pragma unroll
        for (int a = 0; a < K; ++a) xb[a] = L.xb[a].get();
        const int dim = (L.pend - 1) / 2;
        const double pa = pick_axis<K>(xa, dim), pb = pick_axis<K>(xb, dim);
        if (!(fabs(pa - pb) > 1e-3)) return;  // TraceBlineAdaptive.cu:391-405
        const double pm = geo.land(L.pend, dim);
        R b1[K], b2[K];
        unit_at(xa, b1);
        unit_at(xb, b2);
        const double b1d = (double)pick_axis<K>(b1, dim), b2d = (double)pick_axis<K>(b2, dim);
        if (fabs(b1d) < 0.2 || fabs(b2d) < 0.2) {
#pragma unroll
            for (int a = 0; a < K; ++a) out[a] = fma(xa[a], pb - pm, xb[a] * (pm - pa)) / (pb - pa);
        } else {  // RK4_boundary: dx/dx_dim = b / b_dim over pm - pa
            const double s = pm - pa;
            double k[4][K], t[K];
#pragma unroll
            for (int st = 0; st < 4; ++st) {
                const double cf = st == 0 ? 0.0 : (st == 3 ? 1.0 : 0.5);
#pragma unroll
                for (int a = 0; a < K; ++a) t[a] = st == 0 ? xa[a] : xa[a] + s * k[st - 1][a] * cf;
                R b[K];
                unit_at(t, b);
                const double bd = (double)pick_axis<K>(b, dim);
#pragma unroll
                for (int a = 0; a < K; ++a) k[st][a] = (double)b[a] / bd;
            }
#pragma unroll
            for (int a = 0; a < K; ++a)
                out[a] = xa[a] + (1. / 6.) * s * (k[0][a] + 2.0 * k[1][a] + 2.0 * k[2][a] + k[3][a]);
            L.evals += 4;
        }
        const double arc = fabs(pm - pa) / (1e-4 + fabs(b1d));
        L.len += arc;
        // landing twist J.b/|b|^2, b the normalised B at the last point inside
        // (TraceBline.cu:362-365, TraceBlineAdaptiveStretch.cu:403-406; the
        // uniform RKF45 tracer's term is commented out)
        if constexpr (has_current<FJ>()) {
            if (SideGeom<K, G, R>::kLandTwist || P.method == kRK4) {
                double J[3], bd[3];
                R bv[3];
                raw_all<FJ>(fj, xa, J);
                all_axes<K>(b1, bv);
                bd[0] = bv[0]; bd[1] = bv[1]; bd[2] = bv[2];
                L.tw += dot3(J, bd) / dot3(bd, bd) * kQuarterOverPi * arc;
            }
        }
    }
};

#endif  // __HIP_DEVICE_COMPILE__

}  // namespace fqsl
