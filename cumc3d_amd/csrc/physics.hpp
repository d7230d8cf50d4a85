// Device-side physics of the MHD update step: reconstruction, EOS, face
// states, Riemann solvers.  Everything is templated on the arithmetic type T
// (double for the FP64 mode, float for the FP32 split) and, where the normal
// direction matters, on the sweep direction D (0=x, 1=y, 2=z) so that the
// component permutation is resolved at compile time and every state vector
// lives in registers.
//
// Operation order follows the reference expression by expression (Fortran
// evaluates a*b*c as (a*b)*c and a+b+c as (a+b)+c); together with
// -ffp-contract=off and IEEE division/square root this makes the FP64 mode
// reproduce the reference bit for bit.
#pragma once
#include <hip/hip_runtime.h>

namespace cumc3d {

template <class T> __device__ __forceinline__ T fsign1(T b) { return __builtin_copysign(T(1), b); }
// Fortran MIN/MAX as flang evaluates them: MIN(a,b) = a < b ? a : b, so a
// NaN or a tie yields the second argument.
template <class T> __device__ __forceinline__ T fmin2(T a, T b) { return (a < b) ? a : b; }
template <class T> __device__ __forceinline__ T fmax2(T a, T b) { return (a > b) ? a : b; }
// MIN(a, 0.0) as the reference evaluates it: (a < 0) ? a : +0.  The backend
// turns that select into v_min (and drops a following + 0), which returns -0
// for a = -0; a condition the compiler cannot see through keeps the select.
template <class T> __device__ __forceinline__ T fmin_zero(T a) {
    int lt = a < T(0);
    __asm__("" : "+v"(lt));
    return lt ? a : T(0);
}
template <class T> __device__ __forceinline__ T fabsT(T a) { return __builtin_fabs(a); }
__device__ __forceinline__ float fabsT(float a) { return __builtin_fabsf(a); }
__device__ __forceinline__ float fsign1(float b) { return __builtin_copysignf(1.0f, b); }
__device__ __forceinline__ double fmaT(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ __forceinline__ float fmaT(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double sqrtT(double a) { return __builtin_sqrt(a); }
__device__ __forceinline__ float sqrtT(float a) { return __builtin_sqrtf(a); }

// Divides and square roots of the sweeps.  The FP64 sweeps are bound by VALU
// issue, and IEEE division is over half of their instructions: 11 per
// quotient as the compiler expands it (two v_div_scale, v_rcp_f64 at a quarter
// of the rate, five refining fma/mul, residual, v_div_fmas, v_div_fixup).
// Den<double> forms the refined reciprocal once per denominator (4
// instructions: the seed, its error e, e + e^2, and the cubic correction, in
// place of two Newton steps) and each quotient takes 4 more (product, residual,
// correction, v_div_fixup): the compiler's own without the range scaling.  They
// give the same bits wherever scaling would not have acted: numerator 0 or
// from 2^-969 up (below it the residual underflows), denominator and quotient
// clear of the ends of the range.  Zeros, infinities and NaN are
// v_div_fixup's, as they are the compiler's.
//   operator()  for numerators that are 0 or ordinary (densities, pressures,
//               energies), or whose quotient only enters a sum with such a
//               value, where a last bit at 2^-969 is lost;
//   tiny()      for velocities, fields and what is proportional to them: at the
//               front of a field spreading through an empty region these fall
//               through 1e-292 and the denormals to 0.  Numerators below
//               2^-900 are scaled by 2^128 and v_div_fmas scales the quotient
//               back with its one rounding: three more instructions, the IEEE
//               bits down to the last denormal.
// The square root is likewise the compiler's sequence (a v_rsq_f64 seed, one
// coupled Newton step, two residual corrections) without the scaling that
// acts below 2^-767; its arguments are densities and sums with a squared sound
// speed.  Denominators here are densities, differences of signal speeds and
// the like, from 2^-700 up or 0.  In single precision all of these are the
// plain operators, which the FP32 unit turns into reciprocals that it shares.
// (MI355X, FP64, HLLD + WENO-Z at 256^3: x sweep 1.92 -> 1.58 ms, y 2.70 ->
// 2.05, z 2.33 -> 1.95; HLLD + PPM at 128^3: x 0.162 -> 0.150 ms; HLL + MC at
// 150 x 130 x 110: x 0.100 -> 0.091 ms.)
template <class T> struct Den {
    T d;
    __device__ __forceinline__ explicit Den(T x) : d(x) {}
    __device__ __forceinline__ T operator()(T n) const { return n / d; }
    __device__ __forceinline__ T tiny(T n) const { return n / d; }
};
template <> struct Den<double> {
    double d, y;
    __device__ __forceinline__ explicit Den(double x) : d(x) {
        y = __builtin_amdgcn_rcp(x);
        const double e = __builtin_fma(-x, y, 1.0);
        y = __builtin_fma(__builtin_fma(e, e, e), y, y);
    }
    // a denominator with its correctly rounded reciprocal
    __device__ __forceinline__ Den(double x, double inv) : d(x), y(inv) {}
    __device__ __forceinline__ double operator()(double n) const {
        const double q = n * y;
        return __builtin_amdgcn_div_fixup(__builtin_fma(__builtin_fma(-d, q, n), y, q), d, n);
    }
    __device__ __forceinline__ double tiny(double n) const {
        const bool low = __builtin_fabs(n) < 0x1p-900;
        const double m = n * (low ? 0x1p128 : 1.0);
        const double q = m * y;
        return __builtin_amdgcn_div_fixup(__builtin_amdgcn_div_fmas(__builtin_fma(-d, q, m), y, q, low), d, n);
    }
};
// n / 3.  The residual n - 3q is a multiple of n's last denormal place, so it
// is exact for every n and no scaling is needed; taken as -(3q - n) it keeps
// the sign of a zero without v_div_fixup.  An infinite n gives NaN: its one
// caller's WENO weights are NaN then (inf / inf) whatever this returns.
__device__ __forceinline__ double third(double n) {
    const double q = n * (1.0 / 3.0);
    return __builtin_fma(-__builtin_fma(3.0, q, -n), 1.0 / 3.0, q);
}
__device__ __forceinline__ double sqrtS(double a) {
    const double y = __builtin_amdgcn_rsq(a);
    double h = 0.5 * y, s = a * y;
    double r = __builtin_fma(-h, s, 0.5);
    h = __builtin_fma(h, r, h);
    s = __builtin_fma(s, r, s);
    r = __builtin_fma(-s, s, a);
    s = __builtin_fma(r, h, s);
    r = __builtin_fma(-s, s, a);
    s = __builtin_fma(r, h, s);
    return __builtin_amdgcn_class(a, 0x260) ? a : s;   // +-0, +inf
}
__device__ __forceinline__ float sqrtS(float a) { return sqrtT(a); }

// Permutation (normal, transverse 1, transverse 2) of BUILDSTATES
// (solver/mhd/spatial.f90:307-331): x -> (x,y,z), y -> (y,z,x), z -> (z,x,y).
template <int D> struct Perm {
    static constexpr int n = D, t1 = (D + 1) % 3, t2 = (D + 2) % 3;
};

// Primitive face state: natural component order for v and B.
template <class T> struct Q {
    T rho, v[3], p, b[3];
};
// Conserved vector / flux in the reference's variable order
// (rho, mx, my, mz, tau, Bx, By, Bz) = indices 1..8 of SETUP_EQNS.
template <class T> struct V8 {
    T a[8];
};

// ---------------------------------------------------------------------------
// EOS hooks: EOSEPSILON_NM and EOSSOUNDSPEED (model/riemann/src/getepsilon.f90:4-17,
// soundspeed.f90:4-21), ideal gas.
// ---------------------------------------------------------------------------
template <class T> __device__ __forceinline__ T eos_eps(T g1, T rho, T p) {
    return Den<T>(g1)(Den<T>(rho)(p));
}
template <class T> __device__ __forceinline__ T eos_cs(T g1, T p, T rho, T eps) {
    T dpdden = eps * g1;
    T dpdint = rho * g1;
    return sqrtS(dpdden + Den<T>(rho * rho)(dpdint * p));
}

// ---------------------------------------------------------------------------
// Reconstruction of one cell's two faces from its stencil.
// ---------------------------------------------------------------------------

// TVD slope limiters (tvd_module.f90:279-344); lim 0 minmod, 1 van Leer, 2 MC.
template <class T, int LIM>
__device__ __forceinline__ void recon_tvd(T cf, T cb, T vm, T vc, T vp, T &vm_out, T &vp_out) {
    if constexpr (sizeof(T) == 4 && LIM != 1) {
        // Single precision: the same limiters without a divide or a branch.
        // dqf = 2 df / cf and dqb = 2 db / cb carry the signs of df and db
        // (cf, cb > 0).  When dqf dqb > 0, minmod is sign(df) min(|dqf|, |dqb|)
        // and MC's dqf max(0, min((1 + r) / 2, cf, cb r)), r = dqb / dqf, is
        // sign(df) min(|df / cf + db / cb|, 2 |df|, 2 |db|); both are 0
        // otherwise.  (On gfx950 v_rcp_f32 issues at a third of a multiply's
        // rate, and each range-checked divide adds four instructions.)
        const T df = vp - vc, db = vc - vm;
        const T icf = __builtin_amdgcn_rcpf(cf), icb = __builtin_amdgcn_rcpf(cb);
        T m;
        if constexpr (LIM == 0)
            m = T(2) * __builtin_fminf(__builtin_fabsf(df * icf), __builtin_fabsf(db * icb));
        else
            m = __builtin_fminf(__builtin_fabsf(df * icf + db * icb),
                                T(2) * __builtin_fminf(__builtin_fabsf(df), __builtin_fabsf(db)));
        const T slope = (df * db > T(0)) ? __builtin_copysignf(m, df) : T(0);
        vp_out = vc + T(0.5) * slope;
        vm_out = vc - T(0.5) * slope;
        return;
    }
    T dqf = Den<T>(cf).tiny(T(2) * (vp - vc));
    T dqb = Den<T>(cb).tiny(T(2) * (vc - vm));
    T slope;
    if constexpr (LIM == 0) {
        slope = T(0.5) * (fsign1(dqf) + fsign1(dqb)) * fmin2(fabsT(dqf), fabsT(dqb));
    } else if constexpr (LIM == 1) {
        T dq2 = dqf * dqb;
        if (dq2 <= T(0)) slope = T(0);
        else slope = (dq2 * (cf * dqb + cb * dqf) / (dqb * dqb + dqf * dqf + dq2 * (cf + cb - T(2))));
    } else {
        if (dqf == T(0)) {
            slope = T(0);
        } else {
            T r = dqb / dqf;
            slope = fmax2(T(0), fmin2(fmin2(T(0.5) * (T(1) + r), cf), cb * r));
            slope = dqf * slope;
        }
    }
    vp_out = vc + T(0.5) * slope;
    vm_out = vc - T(0.5) * slope;
}

// PPM without steepening/flattening (ppmc_module.f90:359-464); w = 14
// interpolation weights of PPM_INTERPOLANT, in pieces that neighbouring cells
// can share: the limited slope of a cell, the value at its upper edge (the
// lower edge of the next cell), and the limiter of the two edges.  The weights
// of a shared piece are the same expressions of the same widths seen from
// either cell, so it has the same bits; products by 2 fused into a sum too.
template <class T> __device__ __forceinline__ T ppm_slope(T wb, T wa, T a, T b) {
    const T d = wb * b + wa * a;
    const T m = __builtin_elementwise_min(fabsT(d), T(2) * __builtin_elementwise_min(fabsT(a), fabsT(b)));
    return b * a > T(0) ? __builtin_elementwise_copysign(m, d) : T(0);
}
// upper edge of cell c: w = its weights 4..7, b = v(c+1) - v(c), dc and dp the slopes of c and c+1
template <class T> __device__ __forceinline__ T ppm_edge(const T *w, T vc, T b, T dc, T dp) {
    return vc + w[0] * b + w[1] * b + w[2] * dp + w[3] * dc;
}
template <class T> __device__ __forceinline__ void ppm_limit(T vc, T vl, T vr, T &vm_out, T &vp_out) {
    const T c3 = T(3) * vc, lo = fmaT(T(-2), vr, c3), hi = fmaT(T(-2), vl, c3);
    const T vm = (vr - vl) * fmaT(T(2), vr, vl - c3) < T(0) ? lo : vl;
    const T vp = (vr - vm) * (hi - vr) < T(0) ? hi : vr;
    const bool flat = (vr - vc) * (vc - vl) <= T(0);
    vm_out = flat ? vc : vm;
    vp_out = flat ? vc : vp;
}
// Both edges of a cell from its whole stencil, and the slope of the next cell
template <class T>
__device__ __forceinline__ void ppm_edges(const T *__restrict__ w, const T s[5], T &low, T &high, T &dp) {
    const T a = s[2] - s[1], b = s[3] - s[2];
    const T dm = ppm_slope(w[8], w[9], s[1] - s[0], a), dc = ppm_slope(w[10], w[11], a, b);
    dp = ppm_slope(w[12], w[13], b, s[4] - s[3]);
    low = ppm_edge(w, s[1], a, dm, dc);
    high = ppm_edge(w + 4, s[2], b, dc, dp);
}
// WENO-Z, q=2, eps=1e-40 (weno_module.f90:315-408); w = 10 weights of
// WENO_INTERPOLANT.  In single precision eps is 1e-30 (1e-40 is below the
// normal range) and tau5/(eps+beta) is capped at 4e17 so that its square times
// a face value stays finite; both change nothing unless a smoothness indicator
// is within 17 decades of zero while tau5 is not.
// The face from the candidates P (three times the faces of the sub-stencils)
// and the smoothness indicators B.
__device__ __forceinline__ double weno_face(double P1, double P2, double P3, double B1, double B2, double B3) {
    const double sp = 1.0e-40, tau5 = fabsT(B1 - B3);
    double q = Den<double>(sp + B1)(tau5);
    const double w1 = (1.0 / 10.0) * (1.0 + q * q);
    q = Den<double>(sp + B2)(tau5);
    const double w2 = (6.0 / 10.0) * (1.0 + q * q);
    q = Den<double>(sp + B3)(tau5);
    const double w3 = (3.0 / 10.0) * (1.0 + q * q);
    return Den<double>(w1 + w2 + w3)(w1 * third(P1) + w2 * third(P2) + w3 * third(P3));
}
// Single precision: weights relative to the middle one, y2 = 1/(eps + B2)
__device__ __forceinline__ float weno_face(float P1, float P2, float P3, float B1, float y2, float B3) {
    const float tau5 = fabsT(B1 - B3), cap = 4.0e17f;
    const float q1 = fmin2(tau5 / B1, cap), q2 = fmin2(tau5 * y2, cap), q3 = fmin2(tau5 / B3, cap);
    const float w1 = fmaT(q1 * float(1.0 / 6.0), q1, float(1.0 / 6.0)), w2 = fmaT(q2, q2, 1.0f),
                w3 = fmaT(q3 * 0.5f, q3, 0.5f);
    return fmaT(w1, P1, fmaT(w2, P2, w3 * P3)) / (3.0f * (w1 + w2 + w3));
}

// The reference's sums with common powers of two taken out of t and s (beta =
// 13/12 t^2 + s^2/4 = 13/3 (t/2)^2 + (s/2)^2) and products by powers of two
// fused into the additions: neither changes a bit.  What bounds a WENO-Z sweep
// is VALU issue.  Per variable this takes 72 operations to the indicators
// instead of 97 (double precision); in single precision the two faces also
// share the middle indicator, which differs in rounding only.  256^3, HLLD,
// x / y / z sweep: FP64 1.54 / 1.51 / 1.56 -> 1.49 / 1.42 / 1.49 ms, FP32
// 0.54 / 0.61 / 0.60 -> 0.48 / 0.53 / 0.54 ms.
template <class T>
__device__ __forceinline__ void recon_weno(const T *__restrict__ w, T vm2, T vm1, T vc, T vp1, T vp2, T &vm_out,
                                           T &vp_out) {
    const T r = T(13.0 / 12.0) * T(4);
    const T U01 = w[0] * vc + w[1] * vp1;
    const T U12 = w[2] * vp1 + w[3] * vp2;
    const T U10 = w[4] * vm1 + w[5] * vc;
    const T U21 = w[6] * vm2 + w[7] * vm1;
    const T U00 = vm1 + w[8] * (vm1 - vm2);
    const T U11 = vp1 + w[9] * (vp1 - vp2);
    const T X = fmaT(T(2), vc, -U10), Y = fmaT(T(2), vc, -U01);
    // single precision: eps enters with the indicator, where it is free
    auto sq = [](T s) { return sizeof(T) == 4 ? fmaT(s, s, T(1.0e-30)) : s * s; };
    auto beta = [&](T t, T s2) { return r * (t * t) + s2; };
    const T s2 = sq(U01 - U10);
    const T B1p = beta(U10 - U00, sq(X - U00)), B1m = beta(U01 - U11, sq(Y - U11));
    const T B3p = beta(fmaT(T(-2), vp1, U01) + U12, sq(fmaT(T(4), vp1, -(T(3) * U01)) - U12));
    const T B3m = beta(fmaT(T(-2), vm1, U10) + U21, sq(fmaT(T(4), vm1, -(T(3) * U10)) - U21));
    T B2p = beta(U01 - X, s2), B2m;
    if constexpr (sizeof(T) == 4) B2m = B2p = T(1) / B2p;   // the two differ in rounding only
    else B2m = beta(U10 - Y, s2);
    vp_out = weno_face(fmaT(T(-2), U00, T(6) * vc - U10), fmaT(T(2), U01, X), fmaT(T(2), U01 + vp1, -U12), B1p, B2p, B3p);
    vm_out = weno_face(fmaT(T(-2), U11, T(6) * vc - U01), fmaT(T(2), U10, Y), fmaT(T(2), U10 + vm1, -U21), B1m, B2m, B3m);
}

// Scheme ids as in the build descriptor: 0 minmod, 1 van Leer, 2 MC, 3 PPM, 4 WENO-Z.
template <class T, int R>
__device__ __forceinline__ void recon1(const T *__restrict__ w, const T s[5], T &vm_out, T &vp_out) {
    if constexpr (R <= 2) recon_tvd<T, R>(w[0], w[1], s[1], s[2], s[3], vm_out, vp_out);
    else if constexpr (R == 3) {
        T low, high, dp;
        ppm_edges(w, s, low, high, dp);
        ppm_limit(s[2], low, high, vm_out, vp_out);
    }
    else recon_weno<T>(w, s[0], s[1], s[2], s[3], s[4], vm_out, vp_out);
}

// Both faces of one cell: 5 hydro primitives and the 2 transverse cell-centred
// fields, then the EOS at each face (TVD_reconx etc., tvd_module.f90:97-113).
// Face "m" is the cell's left face (reference primR(c-1)), face "p" its right
// face (primL(c)).  The normal field component is filled in by the caller.
template <class T> struct Face {
    T rho, v[3], p, bt1, bt2, eps, cs;
};

// epsilon and the sound speed at both faces
template <class T> __device__ __forceinline__ void face_eos(T g1, Face<T> &fm, Face<T> &fp) {
    if constexpr (sizeof(T) == 4) {
        // single precision: one reciprocal per face.  eps = (p / rho) / g1 and
        // eps g1 + rho g1 p / rho^2 = (g1 + 1) p / rho, the ideal-gas c_s^2
        const T ig1 = __builtin_amdgcn_rcpf(g1);
        const T prm = fm.p * __builtin_amdgcn_rcpf(fm.rho), prp = fp.p * __builtin_amdgcn_rcpf(fp.rho);
        fm.eps = prm * ig1;
        fp.eps = prp * ig1;
        fm.cs = sqrtT((g1 + T(1)) * prm);
        fp.cs = sqrtT((g1 + T(1)) * prp);
    } else {
        fm.eps = eos_eps(g1, fm.rho, fm.p);
        fp.eps = eos_eps(g1, fp.rho, fp.p);
        fm.cs = eos_cs(g1, fm.p, fm.rho, fm.eps);
        fp.cs = eos_cs(g1, fp.p, fp.rho, fp.eps);
    }
}

template <class T, int R>
__device__ __forceinline__ void recon_cell(const T *__restrict__ w, const T st[7][5], T g1, Face<T> &fm,
                                           Face<T> &fp) {
    recon1<T, R>(w, st[0], fm.rho, fp.rho);
    recon1<T, R>(w, st[1], fm.v[0], fp.v[0]);
    recon1<T, R>(w, st[2], fm.v[1], fp.v[1]);
    recon1<T, R>(w, st[3], fm.v[2], fp.v[2]);
    recon1<T, R>(w, st[4], fm.p, fp.p);
    face_eos(g1, fm, fp);
    recon1<T, R>(w, st[5], fm.bt1, fp.bt1);
    recon1<T, R>(w, st[6], fm.bt2, fp.bt2);
}

// Face -> full primitive state with the normal field of the interface.
// bt1/bt2 in Face are the two transverse components in the reconstruction
// order of the sweep: x -> (By,Bz), y -> (Bx,Bz), z -> (Bx,By)
// (tvd_module.f90:108-109, 181-182, 254-255).
template <class T, int D>
__device__ __forceinline__ Q<T> to_q(const Face<T> &f, T bn) {
    Q<T> q;
    q.rho = f.rho;
    q.v[0] = f.v[0]; q.v[1] = f.v[1]; q.v[2] = f.v[2];
    q.p = f.p;
    if constexpr (D == 0) { q.b[0] = bn; q.b[1] = f.bt1; q.b[2] = f.bt2; }
    else if constexpr (D == 1) { q.b[0] = f.bt1; q.b[1] = bn; q.b[2] = f.bt2; }
    else { q.b[0] = f.bt1; q.b[1] = f.bt2; q.b[2] = bn; }
    return q;
}

template <class T> __device__ __forceinline__ T dot3(const T *a, const T *b) {
    return a[0] * b[0] + a[1] * b[1] + a[2] * b[2];
}

// BUILDSTATES for one face state (spatial.f90:342-388): u (conserved) and f
// (physical flux along D).  Index layout of u/f: 0 rho, 1-3 momentum (x,y,z),
// 4 tau, 5-7 B (x,y,z).
template <class T, int D>
__device__ __forceinline__ void build_state(const Q<T> &q, T eps, T u[8], T f[8]) {
    constexpr int n = Perm<D>::n, t1 = Perm<D>::t1, t2 = Perm<D>::t2;
    T b2 = dot3(q.b, q.b), v2 = dot3(q.v, q.v), vb = dot3(q.b, q.v);
    u[0] = q.rho;
    u[1] = q.v[0] * q.rho;
    u[2] = q.v[1] * q.rho;
    u[3] = q.v[2] * q.rho;
    u[5] = q.b[0]; u[6] = q.b[1]; u[7] = q.b[2];
    u[4] = q.rho * (T(0.5) * v2 + eps) + T(0.5) * b2;
    T vn = q.v[n];
    for (int i = 0; i < 5; ++i) f[i] = u[i] * vn;
    f[1 + n] = f[1 + n] + q.p + T(0.5) * (b2) - q.b[n] * q.b[n];
    f[1 + t1] = f[1 + t1] - q.b[n] * q.b[t1];
    f[1 + t2] = f[1 + t2] - q.b[n] * q.b[t2];
    f[4] = f[4] + (q.p + T(0.5) * (b2)) * vn - q.b[n] * vb;
    f[5 + n] = T(0);
    f[5 + t1] = (vn * q.b[t1] - q.v[t1] * q.b[n]);
    f[5 + t2] = (vn * q.b[t2] - q.v[t2] * q.b[n]);
}

// rsolver_module.f90:32-93
template <class T>
__device__ __forceinline__ T signalspeed(T cs, T bn, T bt1, T bt2, T rho) {
    T a2 = cs * cs, a4 = a2 * a2;
    const Den<T> dr(rho);
    T b2n = dr(bn * bn), b2t1 = dr(bt1 * bt1), b2t2 = dr(bt2 * bt2);
    T b2 = b2n + b2t1 + b2t2, b4 = b2 * b2;
    return sqrtS(T(0.5) * (a2 + b2 + sqrtS(fmax2((a4 + b4 + T(2) * b2 * a2) - T(4) * a2 * b2n, T(0)))));
}
// ds: the denominator sr - sl
template <class T> __device__ __forceinline__ T hll_state(T ul, T ur, T fl, T fr, T sl, T sr, const Den<T> &ds) {
    return ds.tiny(sr * ur - sl * ul - (fr - fl));
}
template <class T>
__device__ __forceinline__ T hll_flux(T yl, T yr, T xl, T xr, T sl, T sr, const Den<T> &ds) {
    return ds.tiny(sr * yl - sl * yr + sl * sr * (xr - xl));
}
// ql, qr: square roots of the two densities, dq: the denominator ql + qr
template <class T> __device__ __forceinline__ T roe_avg(T xl, T xr, T ql, T qr, const Den<T> &dq) {
    return dq.tiny(ql * xl + qr * xr);
}
template <class T>
__device__ __forceinline__ T sstar_hllc(T pl, T pr, T rl, T rr, T vl, T vr, T sl, T sr, T bl, T br) {
    return Den<T>(rr * (sr - vr) - rl * (sl - vl))
        .tiny(rr * vr * (sr - vr) - rl * vl * (sl - vl) + pl - pr + br * br - bl * bl);
}

// Riemann solver ids: 0 LF, 1 HLL, 2 HLLC, 3 HLLD.
// Result of one interface.  ds: the HLLD double-star branch was taken;
// uss_t1/uss_t2: the transverse fields of that double-star state, needed to
// reproduce the reference's carried usstar(ibn) (see riemann()).
// none: HLL took none of its branches (a NaN signal speed) and assigned no flux.
template <class T> struct RiemannOut {
    T f[8];
    bool ds;
    bool none;
    T uss_t1, uss_t2;
};

// bn_mode: 0 -> usstar(ibn)=0, 1 -> Bn, 2 -> carried value `carry`.
template <class T, int D, int S>
__device__ __forceinline__ void riemann(const Q<T> &qL, const Q<T> &qR, T epsL, T epsR, T csL, T csR, int bn_mode,
                                        T carry, RiemannOut<T> &out) {
    constexpr int n = Perm<D>::n, t1 = Perm<D>::t1, t2 = Perm<D>::t2;
    T uL[8], uR[8], fL[8], fR[8];
    build_state<T, D>(qL, epsL, uL, fL);
    build_state<T, D>(qR, epsR, uR, fR);
    out.ds = false;
    out.none = false;
    out.uss_t1 = T(0);
    out.uss_t2 = T(0);
    T cfsL = signalspeed(csL, qL.b[n], qL.b[t1], qL.b[t2], qL.rho);
    T cfsR = signalspeed(csR, qR.b[n], qR.b[t1], qR.b[t2], qR.rho);
    if constexpr (S == 0) {   // LFNM, rsolver_module.f90:199-207
        T sL = fabsT(qL.v[n]) + cfsL, sR = fabsT(qR.v[n]) + cfsR, splus = fmax2(sL, sR);
        for (int i = 0; i < 8; ++i) out.f[i] = T(0.5) * (fL[i] + fR[i] - splus * (uR[i] - uL[i]));
        return;
    }
    const T wL = sqrtS(qL.rho), wR = sqrtS(qR.rho);
    const Den<T> dw(wL + wR);
    T ubar = roe_avg(qL.v[n], qR.v[n], wL, wR, dw);
    T cbar = roe_avg(cfsL, cfsR, wL, wR, dw);
    T sL = fmin2(qL.v[n] - cfsL, ubar - cbar);
    T sR = fmax2(qR.v[n] + cfsR, ubar + cbar);
    if constexpr (S == 1) {   // HLLNM, rsolver_module.f90:303-311 (no ELSE branch)
        if (sL >= T(0)) { for (int i = 0; i < 8; ++i) out.f[i] = fL[i]; }
        else if (sL <= T(0) && sR >= T(0)) {
            const Den<T> ds(sR - sL);
            for (int i = 0; i < 8; ++i) out.f[i] = hll_flux(fL[i], fR[i], uL[i], uR[i], sL, sR, ds);
        }
        else if (sR <= T(0)) { for (int i = 0; i < 8; ++i) out.f[i] = fR[i]; }
        else out.none = true;
        return;
    }
    if (sL >= T(0)) { for (int i = 0; i < 8; ++i) out.f[i] = fL[i]; return; }
    if (sR <= T(0)) { for (int i = 0; i < 8; ++i) out.f[i] = fR[i]; return; }
    T b2L = dot3(qL.b, qL.b), b2R = dot3(qR.b, qR.b);
    T pLt = qL.p + T(0.5) * b2L, pRt = qR.p + T(0.5) * b2R;
    if constexpr (S == 2) {   // HLLCNM, rsolver_module.f90:425-499
        T sstar = sstar_hllc(pLt, pRt, qL.rho, qR.rho, qL.v[n], qR.v[n], sL, sR, qL.b[n], qR.b[n]);
        T bh[3], vh[3];
        const Den<T> dlr(sR - sL);
        bh[n] = qL.b[n];
        bh[t1] = hll_state(qL.b[t1], qR.b[t1], fL[5 + t1], fR[5 + t1], sL, sR, dlr);
        bh[t2] = hll_state(qL.b[t2], qR.b[t2], fL[5 + t2], fR[5 + t2], sL, sR, dlr);
        T rh = hll_state(qL.rho, qR.rho, fL[0], fR[0], sL, sR, dlr);
        T mh1 = hll_state(uL[1 + t1], uR[1 + t1], fL[1 + t1], fR[1 + t1], sL, sR, dlr);
        T mh2 = hll_state(uL[1 + t2], uR[1 + t2], fL[1 + t2], fR[1 + t2], sL, sR, dlr);
        vh[n] = sstar;
        const Den<T> drh(rh);
        vh[t1] = drh.tiny(mh1);
        vh[t2] = drh.tiny(mh2);
        const bool left = sstar >= T(0);
        const Q<T> &q = left ? qL : qR;
        const T *u = left ? uL : uR;
        const T *f = left ? fL : fR;
        T s = left ? sL : sR, pt = left ? pLt : pRt;
        T us[8];
        const Den<T> dss(s - sstar);
        us[0] = dss(u[0] * (s - q.v[n]));
        T vb = dot3(q.b, q.v);
        T vbhll = dot3(bh, vh);
        T ps = q.rho * (s - q.v[n]) * (sstar - q.v[n]) + pt;
        us[5 + n] = bh[n];
        us[5 + t1] = bh[t1];
        us[5 + t2] = bh[t2];
        us[1 + n] = us[0] * sstar;
        us[1 + t1] = dss.tiny(u[1 + t1] * (s - q.v[n]) - (us[5 + n] * us[5 + t1] - q.b[n] * q.b[t1]));
        us[1 + t2] = dss.tiny(u[1 + t2] * (s - q.v[n]) - (us[5 + n] * us[5 + t2] - q.b[n] * q.b[t2]));
        us[4] = dss(u[4] * (s - q.v[n]) + (ps * sstar - pt * q.v[n]) - ((vbhll * us[5 + n] - vb * q.b[n])));
        for (int i = 0; i < 8; ++i) out.f[i] = f[i] + s * (us[i] - u[i]);
        return;
    }
    // HLLDNM, rsolver_module.f90:615-752
    T sM = sstar_hllc(pLt, pRt, qL.rho, qR.rho, qL.v[n], qR.v[n], sL, sR, qL.b[n], qR.b[n]);
    T usL[8], usR[8], psL[3], psR[3];
    const Den<T> dL(sL - sM), dR(sR - sM);
    usL[0] = dL(uL[0] * (sL - qL.v[n]));
    usL[1 + t1] = dL.tiny(uL[1 + t1] * (sL - qL.v[n]));
    usL[1 + t2] = dL.tiny(uL[1 + t2] * (sL - qL.v[n]));
    usL[4] = dL(uL[4] * (sL - qL.v[n]));
    usR[0] = dR(uR[0] * (sR - qR.v[n]));
    usR[1 + t1] = dR.tiny(uR[1 + t1] * (sR - qR.v[n]));
    usR[1 + t2] = dR.tiny(uR[1 + t2] * (sR - qR.v[n]));
    usR[4] = dR(uR[4] * (sR - qR.v[n]));
    T sstarL = sM - Den<T>(sqrtS(usL[0])).tiny(fabsT(qL.b[n]));
    T sstarR = sM + Den<T>(sqrtS(usR[0])).tiny(fabsT(qR.b[n]));
    if (((sstarL - sL) < T(1.0e-4) * (sM - sL)) || ((sstarR - sR) > -T(1.0e-4) * (sR - sM))) {
        const Den<T> dlr(sR - sL);
        usL[5 + n] = qL.b[n];
        usL[5 + t1] = hll_state(qL.b[t1], qR.b[t1], fL[5 + t1], fR[5 + t1], sL, sR, dlr);
        usL[5 + t2] = hll_state(qL.b[t2], qR.b[t2], fL[5 + t2], fR[5 + t2], sL, sR, dlr);
        usR[5 + n] = qR.b[n];
        usR[5 + t1] = usL[5 + t1];
        usR[5 + t2] = usL[5 + t2];
        sstarL = sM;
        sstarR = sM;
    } else {
        const Den<T> dfL(qL.rho * (sL - qL.v[n]) * (sL - sM) - qL.b[n] * qL.b[n]);
        usL[5 + n] = qL.b[n];
        usL[5 + t1] = dfL.tiny(qL.b[t1] * (qL.rho * (sL - qL.v[n]) * (sL - qL.v[n]) - qL.b[n] * qL.b[n]));
        usL[5 + t2] = dfL.tiny(qL.b[t2] * (qL.rho * (sL - qL.v[n]) * (sL - qL.v[n]) - qL.b[n] * qL.b[n]));
        const Den<T> dfR(qR.rho * (sR - qR.v[n]) * (sR - sM) - qR.b[n] * qR.b[n]);
        usR[5 + n] = qR.b[n];
        usR[5 + t1] = dfR.tiny(qR.b[t1] * (qR.rho * (sR - qR.v[n]) * (sR - qR.v[n]) - qR.b[n] * qR.b[n]));
        usR[5 + t2] = dfR.tiny(qR.b[t2] * (qR.rho * (sR - qR.v[n]) * (sR - qR.v[n]) - qR.b[n] * qR.b[n]));
    }
    usL[1 + n] = usL[0] * sM;
    usL[1 + t1] = usL[1 + t1] - dL.tiny(usL[5 + n] * usL[5 + t1] - qL.b[n] * qL.b[t1]);
    usL[1 + t2] = usL[1 + t2] - dL.tiny(usL[5 + n] * usL[5 + t2] - qL.b[n] * qL.b[t2]);
    usR[1 + n] = usR[0] * sM;
    usR[1 + t1] = usR[1 + t1] - dR.tiny(usR[5 + n] * usR[5 + t1] - qR.b[n] * qR.b[t1]);
    usR[1 + t2] = usR[1 + t2] - dR.tiny(usR[5 + n] * usR[5 + t2] - qR.b[n] * qR.b[t2]);
    const Den<T> duL(usL[0]), duR(usR[0]);
    psL[n] = sM;
    psL[t1] = duL.tiny(usL[1 + t1]);
    psL[t2] = duL.tiny(usL[1 + t2]);
    psR[n] = sM;
    psR[t1] = duR.tiny(usR[1 + t1]);
    psR[t2] = duR.tiny(usR[1 + t2]);
    T pLs = qL.rho * (sL - qL.v[n]) * (sM - qL.v[n]) + pLt;
    T pRs = qR.rho * (sR - qR.v[n]) * (sM - qR.v[n]) + pRt;
    T bdotu = dot3(qL.b, qL.v);
    T bdotus = dot3(&usL[5], psL);
    usL[4] = usL[4] + dL((pLs * sM - pLt * qL.v[n]) - (bdotus - bdotu) * qL.b[n]);
    bdotu = dot3(qR.b, qR.v);
    bdotus = dot3(&usR[5], psR);
    usR[4] = usR[4] + dR((pRs * sM - pRt * qR.v[n]) - (bdotus - bdotu) * qR.b[n]);
    if (sstarL >= T(0)) {
        for (int i = 0; i < 8; ++i) out.f[i] = fL[i] + sL * (usL[i] - uL[i]);
        return;
    }
    if (sstarR <= T(0)) {
        for (int i = 0; i < 8; ++i) out.f[i] = fR[i] + sR * (usR[i] - uR[i]);
        return;
    }
    // double-star states.  usstar(ibn) is never assigned by the reference
    // (rsolver_module.f90:704-741): its value is selected by bn_mode.
    T ussL[8], ussR[8], pss[3];
    T bnL = (bn_mode == 1) ? qL.b[n] : ((bn_mode == 2) ? carry : T(0));
    T bnR = (bn_mode == 1) ? qR.b[n] : ((bn_mode == 2) ? carry : T(0));
    ussL[5 + n] = bnL;
    ussR[5 + n] = bnR;
    ussL[0] = usL[0];
    ussR[0] = usR[0];
    T f1 = Den<T>(sqrtS(usL[0]) + sqrtS(usR[0]))(T(1));
    T f2 = fsign1(qL.b[n]);
    pss[n] = sM;
    pss[t1] = f1 * (sqrtS(usL[0]) * psL[t1] + sqrtS(usR[0]) * psR[t1] + (usR[5 + t1] - usL[5 + t1]) * f2);
    pss[t2] = f1 * (sqrtS(usL[0]) * psL[t2] + sqrtS(usR[0]) * psR[t2] + (usR[5 + t2] - usL[5 + t2]) * f2);
    ussL[5 + t1] = f1 * (sqrtS(usL[0]) * usR[5 + t1] + sqrtS(usR[0]) * usL[5 + t1] +
                         sqrtS(usL[0] * usR[0]) * (psR[t1] - psL[t1]) * f2);
    ussL[5 + t2] = f1 * (sqrtS(usL[0]) * usR[5 + t2] + sqrtS(usR[0]) * usL[5 + t2] +
                         sqrtS(usL[0] * usR[0]) * (psR[t2] - psL[t2]) * f2);
    ussL[1 + n] = ussL[0] * pss[n];
    ussL[1 + t1] = ussL[0] * pss[t1];
    ussL[1 + t2] = ussL[0] * pss[t2];
    bdotus = dot3(&usL[5], psL);
    T bdotuss = dot3(&ussL[5], pss);
    ussL[4] = usL[4] - sqrtS(usL[0]) * (bdotus - bdotuss) * f2;
    ussR[5 + t1] = ussL[5 + t1];
    ussR[5 + t2] = ussL[5 + t2];
    ussR[1 + n] = ussR[0] * pss[n];
    ussR[1 + t1] = ussR[0] * pss[t1];
    ussR[1 + t2] = ussR[0] * pss[t2];
    bdotus = dot3(&usR[5], psR);
    bdotuss = dot3(&ussR[5], pss);
    ussR[4] = usR[4] + sqrtS(usR[0]) * (bdotus - bdotuss) * f2;
    out.ds = true;
    out.uss_t1 = ussL[5 + t1];
    out.uss_t2 = ussL[5 + t2];
    if (sM >= T(0)) {
        for (int i = 0; i < 8; ++i) out.f[i] = fL[i] + sL * (usL[i] - uL[i]) + sstarL * (ussL[i] - usL[i]);
    } else {
        for (int i = 0; i < 8; ++i) out.f[i] = fR[i] + sR * (usR[i] - uR[i]) + sstarR * (ussR[i] - usR[i]);
    }
}

}  // namespace cumc3d
