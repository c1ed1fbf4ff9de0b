// swe_physics.hpp — per-cell and per-face arithmetic of the practical 2D
// shallow-water scheme, as device functions for gfx950.
//
// Every expression keeps the reference's operation order and rounding points
// so that FP64 results are bitwise equal to the reference's CPU path; the
// library is built with -ffp-contract=off (no a*b+c fusion) and without
// fast-math (IEEE NaN / signed-zero behaviour).  Storage type S is double
// (Float64 backend) or float (Float32 storage); values read from S buffers
// stay S and parameters stay double, so C++ promotion reproduces Julia's.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace sfv {

// Julia max/min on IEEE floats (base/math.jl): NaN-propagating, -0.0 < +0.0.
template <class T>
__device__ __forceinline__ T jl_max(T x, T y) {
    if (x != x) return x;
    if (y != y) return y;
    if (x > y) return x;
    if (y > x) return y;
    return __builtin_signbit(x) ? y : x;
}
template <class T>
__device__ __forceinline__ T jl_min(T x, T y) {
    if (x != x) return x;
    if (y != y) return y;
    if (x < y) return x;
    if (y < x) return y;
    return __builtin_signbit(x) ? x : y;
}

// max / min of two values neither of which is -0.0 (wave speeds and
// eigenvalues: u +- c with c > 0 rounds to +0.0 at worst, dry sides give
// +0.0): one hardware max/min, and Julia's NaN propagation kept by an
// unordered check.  For such inputs this equals jl_max / jl_min.
__device__ __forceinline__ double nz_max(double a, double b) { return (a > b || a != a) ? a : b; }
__device__ __forceinline__ double nz_min(double a, double b) { return (a < b || a != a) ? a : b; }

// linearreconstruction.jl:28-35: min(a,b,c) if all > 0, max(a,b,c) if all
// < 0, else +0.0 (also when any is NaN, as every comparison is then false).
// Evaluated as max(lo, 0) + min(hi, 0) (+0.0) with lo/hi the hardware
// min/max: all > 0 gives lo, all < 0 gives hi, mixed signs or zeros give a
// sum of two zeros, and the trailing +0.0 turns -0.0 + -0.0 into +0.0.
// NaN: with `regular` (θ finite and nonzero) a NaN in a or c implies one in b
// (a = θ·fwd, c = θ·bwd, b = (fwd + bwd)/2), so checking b suffices.
__device__ __forceinline__ double minmod(double a, double b, double c, bool regular = false) {
    const double lo = __builtin_fmin(__builtin_fmin(a, b), c);
    const double hi = __builtin_fmax(__builtin_fmax(a, b), c);
    const double r = (__builtin_fmax(lo, 0.0) + __builtin_fmin(hi, 0.0)) + 0.0;
    const bool nan = regular ? (b != b) : (__builtin_isunordered(a, b) || c != c);
    return nan ? 0.0 : r;
}

// equation.jl:56 (Brodtkorb & Holm 2021, eq. 26).  When |h| >= κ the inner
// min(...) is <= κ <= |h|, so max(|h|, ...) = |h| and h* = copysign(1,h)*|h|
// = h exactly; the divide is only evaluated where it can matter.
template <class H>
__device__ __forceinline__ double desingularize(H h, double kappa) {
    const double ah = (double)__builtin_fabs(h);
    if (!(ah < kappa)) return (double)h;          // |h| >= κ, or NaN (which propagates)
    const H h2 = h * h;
    const double sgn = __builtin_signbit(h) ? -1.0 : 1.0;
    // |h| < κ here, and h^2/(2κ) + κ/2 >= κ/2 > 0: no NaN or -0.0 reaches max/min
    return sgn * __builtin_fmax(ah, __builtin_fmin(h2 / (2 * kappa) + kappa / 2.0, kappa));
}

struct PhysParams {
    double g, rho, cutoff, kappa;
};

// swe_2D.jl:43-81: flux and eigenvalues of one wet face state in direction d
// (0 = x, 1 = y).
template <class S>
__device__ __forceinline__ void phys_flux(int d, S h, S hu, S hv, const PhysParams& p,
                                          double f[3], double e[2]) {
    const double hs = desingularize(h, p.kappa);
    const double u = hu / hs;
    const double v = hv / hs;
    const S h2 = h * h;
    const double c = sqrt(p.g * h);
    if (d == 0) {
        f[0] = p.rho * h * u;
        f[1] = p.rho * h * u * u + 0.5 * p.rho * p.g * h2;
        f[2] = p.rho * h * u * v;
        e[0] = u + c;
        e[1] = u - c;
    } else {
        f[0] = p.rho * h * v;
        f[1] = p.rho * h * u * v;
        f[2] = p.rho * h * v * v + 0.5 * p.rho * p.g * h2;
        e[0] = v + c;
        e[1] = v - c;
    }
}

// centralupwind.jl:48-77 (practical SWE variant).  m = faceminus (right face
// of the left cell), q = faceplus (left face of the right cell).  Returns the
// face wave speed; F receives the numerical flux.
template <class S>
__device__ __forceinline__ double central_upwind(int d, const S m[3], const S q[3], const PhysParams& p,
                                                 double F[3]) {
    double fm[3] = {0.0, 0.0, 0.0}, em[2] = {0.0, 0.0};
    double fp[3] = {0.0, 0.0, 0.0}, ep[2] = {0.0, 0.0};
    if (m[0] > p.cutoff) phys_flux(d, m[0], m[1], m[2], p, fm, em);
    if (q[0] > p.cutoff) phys_flux(d, q[0], q[1], q[2], p, fp, ep);
    const double aplus = nz_max(nz_max(ep[0], em[0]), 0.0);
    const double aminus = nz_min(nz_min(ep[1], em[1]), 0.0);
    const double da = aplus - aminus;
    if (__builtin_fabs(da) < p.kappa) {
        F[0] = F[1] = F[2] = 0.0;
        return 0.0;
    }
    const double pm = (aplus * aminus) / da;
#pragma unroll
    for (int v = 0; v < 3; ++v) {
        const S diff = q[v] - m[v];
        F[v] = (aplus * fm[v] - aminus * fp[v]) / da + pm * diff;
    }
    if (m[0] < p.cutoff && q[0] < p.cutoff) return 0.0;
    return nz_max(__builtin_fabs(aplus), __builtin_fabs(aminus));
}

// minmod_slope + the SWE dry-face slope fix + face values
// (linearreconstruction.jl:37-43, 73-100).  Given the cell and its two
// neighbours along the sweep, and the cell's two face bottoms, writes the
// left and right face states (h, hu, hv) — variable 1 becomes a depth.
template <class S>
__device__ __forceinline__ void reconstruct_cell(const S l[3], const S c[3], const S r[3], double theta,
                                                 double Bl, double Br, S L[3], S R[3], bool known_regular = false) {
    const bool regular = known_regular || (__builtin_isfinite(theta) && theta != 0.0);
    double slope[3];
#pragma unroll
    for (int v = 0; v < 3; ++v) {
        const S fwd = r[v] - c[v];
        const S bwd = c[v] - l[v];
        const double central = (fwd + bwd) / 2.0;
        slope[v] = minmod(theta * fwd, central, theta * bwd, regular);
    }
    const S w = c[0];
    if (w - 0.5 * slope[0] < Bl) slope[0] = 2.0 * (w - Bl);
    else if (w + 0.5 * slope[0] < Br) slope[0] = 2.0 * (Br - w);
#pragma unroll
    for (int v = 0; v < 3; ++v) {
        L[v] = (S)(c[v] - 0.5 * slope[v]);
        R[v] = (S)(c[v] + 0.5 * slope[v]);
    }
    L[0] = (S)(L[0] - Bl);
    R[0] = (S)(R[0] - Br);
}

// friction.jl:30-43
__device__ __forceinline__ double friction_law(int law, double c, double h, double speed) {
    if (law == 2) { const double denom = cbrt(h) * h; return -c * speed / denom; }
    if (law == 3) { const double denom = cbrt(h) * h * h; return -c * speed / denom; }
    const double denom = h * h;
    return -c * speed / denom;
}

// implicit_friction's `out ./ (1 .- dt .* [0, f, f])` (friction.jl:77).  For
// the w component the divisor 1 - dt*0.0 is exactly 1.0 for finite dt and NaN
// otherwise, so multiplying by it is the same as dividing.
template <class S>
__device__ __forceinline__ void apply_friction(S o[3], S dt_s, double fs) {
    o[0] = (S)(o[0] * (1 - dt_s * 0.0));
    o[1] = (S)(o[1] / (1 - dt_s * fs));
    o[2] = (S)(o[2] / (1 - dt_s * fs));
}

// (B_R - B_L)/Δ of the bottom source (source_term_bottom.jl:38).  When Δ is a
// power of two, x/Δ and x*(1/Δ) are the same correctly rounded value.
__device__ __forceinline__ double slope_div(double x, double d, double inv_d, int pow2) {
    return pow2 ? x * inv_d : x / d;
}

// friction.jl:62-78: the implicit friction scalar from the substep input
// state (w, hu, hv) and B_cell.
template <class S>
__device__ __forceinline__ double friction_scalar(int law, double Cz, double kappa, S w, S hu, S hv, double Bm) {
    const double hs = desingularize(w - Bm, kappa);
    const double u = hu / hs, v = hv / hs;
    double speed = sqrt(u * u + v * v);
    if (speed == 0.0) speed = 0.0;
    return friction_law(law, Cz, hs, speed);
}


// ---------------------------------------------------------------------------
// Face evaluation on operands in a proven range.
//
// The compiler's correctly rounded FP64 quotient x/d on gfx950 is
//   ds = div_scale(d; d, x), xs = div_scale(x; d, x, flag),
//   r = rcp(ds), then twice r = fma(r, fma(-ds, r, 1), r),
//   q = xs*r, e = fma(-ds, q, xs), q = div_fmas(e, r, q, flag),
//   result = div_fixup(q, d, x).
// div_scale returns its operand unchanged and clears the flag, and div_fmas
// is then a plain fma, unless an operand or the quotient nears the ends of
// the exponent range (d or 1/d subnormal, x/d subnormal, |x| < 2^-969, or
// exponent(x) - exponent(d) >= 768).  div_fixup decides the result from x
// and d alone when either is zero, infinite or NaN.  So for d in
// [2^-40, 2^94] and x = 0 or |x| in [2^-800, 2^340] (or x, d special), the
// steps without the scaling give the hardware quotient bit for bit, and one
// refined reciprocal serves every numerator over the same d: 4 instructions
// per quotient after 5 for the reciprocal, against 11 per quotient.
//
// The compiler's sqrt scales x < 2^-767 by 2^256 before its rsq-based
// Newton steps (and the result back) and passes +-0 and +Inf through; for x
// in [2^-767, DBL_MAX] both are no-ops, and sqrt_rng is the same steps
// without them: 10 instructions against 17.
//
// The *_rng functions below are the functions above with these forms.  They
// are used only by waves whose inputs lie in band: every stage input (w, hu,
// hv of every cell the face stencils read) and bottom corner is 0 or of
// magnitude in [2^-120, 2^40) (checked as the rows arrive, in_band), with θ
// (linear reconstruction), ρ and g in [2^-10, 2^10], depth_cutoff and κ in
// [2^-39, 2^10] and the spacings in [2^-60, 2^100] (KParams::ranged).  Then
// (exact differences of such values are multiples of 2^-172, rounded products
// keep their exponent sums, and cancellation in u +- c leaves at least an ulp
// of c >= sqrt(g*cutoff)):
//   face values:   0 or [2^-235, 2^51]; wet depths h > cutoff >= 2^-39
//   velocity quotient hu/h*:  x in {0} U [2^-235, 2^51], d = h* in [2^-40, 2^51]
//   c = sqrt(g h):  g h in [2^-49, 2^61]
//   a+, a-:         0 or [2^-78, 2^92];  da = a+ - a- in [κ, 2^93] unless degenerate
//   flux quotients: numerators 0 or [2^-752, 2^336], (a+ a-) in [2^-156, 2^184]
//   h^2/(2κ) below κ: x = 0 or [2^-470, 2^20], d in [2^-38, 2^11]
//   bottom slopes:  x = 0 or [2^-173, 2^41], d in [2^-60, 2^100]
// which is inside the range above, or clear of every scaling condition where
// d reaches beyond it (no operand is subnormal, |x| > 2^-969, the exponents
// of x and d are less than 768 apart).  A degenerate face (|da| < κ) discards
// its quotients, as the reference's early return does.
struct Recip {
    double d, r;
};
__device__ __forceinline__ Recip recip_rng(double d) {
    double r = __builtin_amdgcn_rcp(d);
    double t = __builtin_fma(-d, r, 1.0);
    r = __builtin_fma(r, t, r);
    t = __builtin_fma(-d, r, 1.0);
    r = __builtin_fma(r, t, r);
    return {d, r};
}
__device__ __forceinline__ double div_rng(double x, const Recip& R) {
    const double q = x * R.r;
    const double e = __builtin_fma(-R.d, q, x);
    return __builtin_amdgcn_div_fixup(__builtin_fma(e, R.r, q), R.d, x);
}
__device__ __forceinline__ double sqrt_rng(double x) {
    double y = __builtin_amdgcn_rsq(x);
    double g = x * y;
    double h = y * 0.5;
    const double r = __builtin_fma(-h, g, 0.5);
    g = __builtin_fma(g, r, g);
    h = __builtin_fma(h, r, h);
    double d = __builtin_fma(-g, g, x);
    g = __builtin_fma(d, h, g);
    d = __builtin_fma(-g, g, x);
    return __builtin_fma(d, h, g);
}
// Every value is 0 or of magnitude at least 2^-120, and their magnitudes add
// up to less than 2^40 (false for NaN and Inf, whose sums are not less).  The
// lower bound is tested through the hardware's frexp exponent e (v = m 2^e
// with |m| in [0.5, 1); 0 for 0, the true exponent for subnormals): integer
// minima combine it over the values, and one addition per value covers the
// rest.
__device__ __forceinline__ bool in_band(double a, double b, double c, double d) {
    const int lo = min(min(__builtin_amdgcn_frexp_exp(a), __builtin_amdgcn_frexp_exp(b)),
                       min(__builtin_amdgcn_frexp_exp(c), __builtin_amdgcn_frexp_exp(d)));
    const double s = (__builtin_fabs(a) + __builtin_fabs(b)) + (__builtin_fabs(c) + __builtin_fabs(d));
    return lo >= -119 && s < 0x1p40;
}

// What the ranged forms need of a run's constants, the same on every lane:
// refined reciprocals and products formed once per wave.
struct RngK {
    Recip k2, dx, dy;          // 2κ and the spacings
    double half_kappa, hrg;    // κ/2, (0.5 ρ) g
    double theta2;             // 2 θ
    double bx, by;             // -g (1/Δ) / 2 (power-of-two spacings)
};

// equation.jl:56 as desingularize.
template <class H>
__device__ __forceinline__ double desingularize_rng(H h, double kappa, const RngK& K) {
    const double ah = (double)__builtin_fabs(h);
    if (!(ah < kappa)) return (double)h;
    const H h2 = h * h;
    return __builtin_copysign(__builtin_fmax(ah, __builtin_fmin(div_rng(h2, K.k2) + K.half_kappa, kappa)), (double)h);
}

// swe_2D.jl:43-81 for direction D with the ranged quotients and square root
// (h > cutoff).  UNIT_RHO: ρ is 1.
template <int D, bool UNIT_RHO, class S>
__device__ __forceinline__ void phys_flux_rng(S h, S hu, S hv, const PhysParams& p, const RngK& K, double f[3],
                                              double e[2]) {
    const Recip R = recip_rng(desingularize_rng(h, p.kappa, K));
    const double u = div_rng(hu, R);
    const double v = div_rng(hv, R);
    const S h2 = h * h;
    const double c = sqrt_rng(p.g * h);
    const double rh = UNIT_RHO ? (double)h : p.rho * h;
    const double ph = K.hrg * h2;
    f[0] = rh * (D == 0 ? u : v);
    f[1] = D == 0 ? rh * u * u + ph : rh * u * v;
    f[2] = D == 0 ? rh * u * v : rh * v * v + ph;
    e[0] = (D == 0 ? u : v) + c;
    e[1] = (D == 0 ? u : v) - c;
}

// centralupwind.jl:48-77 as central_upwind.  No NaN and no -0.0 reaches
// max/min here (finite inputs; see nz_max), so they are the hardware's.
template <int D, bool UNIT_RHO, class S>
__device__ __forceinline__ double central_upwind_rng(const S m[3], const S q[3], const PhysParams& p, const RngK& K,
                                                     double F[3]) {
    double fm[3] = {0.0, 0.0, 0.0}, em[2] = {0.0, 0.0};
    double fp[3] = {0.0, 0.0, 0.0}, ep[2] = {0.0, 0.0};
    if (m[0] > p.cutoff) phys_flux_rng<D, UNIT_RHO>(m[0], m[1], m[2], p, K, fm, em);
    if (q[0] > p.cutoff) phys_flux_rng<D, UNIT_RHO>(q[0], q[1], q[2], p, K, fp, ep);
    const double aplus = __builtin_fmax(__builtin_fmax(ep[0], em[0]), 0.0);
    const double aminus = __builtin_fmin(__builtin_fmin(ep[1], em[1]), 0.0);
    const double da = aplus - aminus;
    if (__builtin_fabs(da) < p.kappa) {
        F[0] = F[1] = F[2] = 0.0;
        return 0.0;
    }
    const Recip R = recip_rng(da);
    const double pm = div_rng(aplus * aminus, R);
#pragma unroll
    for (int v = 0; v < 3; ++v) {
        const S diff = q[v] - m[v];
        F[v] = div_rng(aplus * fm[v] - aminus * fp[v], R) + pm * diff;
    }
    if (m[0] < p.cutoff && q[0] < p.cutoff) return 0.0;
    return __builtin_fmax(aplus, -aminus);
}

// minmod_slope + the SWE dry-face slope fix + face values
// (linearreconstruction.jl:37-43, 73-100) as reconstruct_cell: no NaN, and
// scaling by a power of two is exact.  Slopes are kept doubled (s2 = 2
// slope, theta2 = 2 θ), so (fwd + bwd)/2 needs no product, and c -+ slope/2 is
// one fma, its product exact.  With lo = max(min(a, e), 0) and hi =
// min(max(a, e), 0), minmod(a, b, e) is b clamped to [hi, lo]: both positive
// gives hi = 0 and min(b, lo), both negative lo = 0 and max(b, hi), else lo =
// hi = 0.  The added +0.0 keeps a and e from being -0.0, so a zero slope is
// +0.0 as the reference's is.
template <class S>
__device__ __forceinline__ void reconstruct_cell_rng(const S l[3], const S c[3], const S r[3], double theta2,
                                                     double Bl, double Br, S L[3], S R[3]) {
    double s2[3];
#pragma unroll
    for (int v = 0; v < 3; ++v) {
        const S fwd = r[v] - c[v];
        const S bwd = c[v] - l[v];
        const S sum = fwd + bwd;
        const double a = __builtin_fma(theta2, (double)fwd, 0.0), e = __builtin_fma(theta2, (double)bwd, 0.0);
        const double lo = __builtin_fmax(__builtin_fmin(a, e), 0.0), hi = __builtin_fmin(__builtin_fmax(a, e), 0.0);
        s2[v] = __builtin_fmin(__builtin_fmax((double)sum, hi), lo);
    }
    // w's faces before the bottoms are taken off; the dry-face fix makes the
    // half slope w - Bl or Br - w
    const double w = (double)c[0];
    double wl = __builtin_fma(-0.25, s2[0], w), wr = __builtin_fma(0.25, s2[0], w);
    if (wl < Bl || wr < Br) {
        const double half = wl < Bl ? w - Bl : Br - w;
        wl = w - half;
        wr = w + half;
    }
    L[0] = (S)((S)wl - Bl);
    R[0] = (S)((S)wr - Br);
#pragma unroll
    for (int v = 1; v < 3; ++v) {
        L[v] = (S)__builtin_fma(-0.25, s2[v], (double)c[v]);
        R[v] = (S)__builtin_fma(0.25, s2[v], (double)c[v]);
    }
}

// friction.jl:40-43, 62-78: the bh2021 friction scalar from a substep input in
// band, with Cz 0 or in [2^-60, 2^10].  hs in [2^-40, 2^41], so u, v are 0 or in
// [2^-161, 2^80], u^2 + v^2 0 or in [2^-322, 2^161], the denominator in
// [2^-80, 2^82].  Adding 2^-700 leaves a nonzero u^2 + v^2 as it is and turns 0
// into a speed of 2^-350: the caller's 1 - dt*fs is then 1, as it is for 0
// (dt <= 2^100).
template <class S>
__device__ __forceinline__ double friction_scalar_rng(double Cz, double kappa, const RngK& K, S w, S hu, S hv,
                                                      double Bm) {
    const double hs = desingularize_rng(w - Bm, kappa, K);
    const Recip R = recip_rng(hs);
    const double u = div_rng(hu, R), v = div_rng(hv, R);
    const double speed = sqrt_rng((u * u + v * v) + 0x1p-700);
    return div_rng(-Cz * speed, recip_rng(hs * hs));
}

}  // namespace sfv
