// swe_rows.hpp — what the wave-march and workgroup-march kernels share: lane
// shifts, row access through buffer descriptors, the stage-1 result of a
// cell, the domain's corner cells and the tile order over the XCDs.
#pragma once

#include <type_traits>

#include "swe_common.hpp"

namespace sfv {

// Lane shifts by one across the whole wave with DPP (wave_shr:1 / wave_shl:1,
// VALU latency instead of an LDS round trip): lane i receives lane i-1
// (shfl_up1) or lane i+1 (shfl_dn1).  Lane 0 (shfl_up1) / lane 63
// (shfl_dn1) have no source lane and read zero; both are halo lanes whose
// shifted values feed no output.  With no old value to keep, each shift is a
// single DPP move into a fresh register.
template <int CTRL>
__device__ __forceinline__ int dpp_shift(int v) {
    return __builtin_amdgcn_mov_dpp(v, CTRL, 0xf, 0xf, true);
}
template <int CTRL>
__device__ __forceinline__ double dpp_shift(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = dpp_shift<CTRL>((int)(unsigned long long)b);
    const int hi = dpp_shift<CTRL>((int)((unsigned long long)b >> 32));
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}
template <int CTRL>
__device__ __forceinline__ float dpp_shift(float v) { return __int_as_float(dpp_shift<CTRL>(__float_as_int(v))); }
constexpr int DPP_WAVE_SHR1 = 0x138, DPP_WAVE_SHL1 = 0x130;
template <class T>
__device__ __forceinline__ T shfl_up1(T v) { return dpp_shift<DPP_WAVE_SHR1>(v); }
template <class T>
__device__ __forceinline__ T shfl_dn1(T v) { return dpp_shift<DPP_WAVE_SHL1>(v); }

__device__ __forceinline__ double Bload(const KParams& P, const double* __restrict__ B, int i, int j) {
    return (i <= P.nxT && j <= P.nyT) ? B[(size_t)i + (size_t)(P.nxT + 1) * j] : 0.0;
}

// Row access through a raw buffer resource: the descriptor (SGPRs) spans one
// row, base at its first element and `len` elements long, and a lane's
// access is its 32-bit byte offset (a loop-invariant VGPR).  That keeps the
// per-lane 64-bit address arithmetic of a global access out of the row loop,
// and the hardware range check reads zero for (and drops a store to) an
// offset past the row.  validate_config caps a row at 2^27 elements, so the
// byte offsets and lengths fit in 31 bits.  The row pointer must be the same for the whole wave.
constexpr int RSRC_WORD3 = 0x00020000;   // gfx9 raw buffer: 32-bit data format
template <class T>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t row_rsrc(const T* row, int len) {
    return __builtin_amdgcn_make_buffer_rsrc((void*)row, (short)0, len * (int)sizeof(T), RSRC_WORD3);
}
__device__ __forceinline__ double rsrc_ld(__amdgpu_buffer_rsrc_t r, unsigned off, double) {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
}
__device__ __forceinline__ float rsrc_ld(__amdgpu_buffer_rsrc_t r, unsigned off, float) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
}
template <class T>
__device__ __forceinline__ T row_ld(const T* row, int len, int col) {
    return rsrc_ld(row_rsrc(row, len), (unsigned)col * (unsigned)sizeof(T), T());
}
// columns col and col + 1: one offset register, the second load's is immediate
__device__ __forceinline__ void row_ld2(const double* row, int len, int col, double& a, double& b) {
    const __amdgpu_buffer_rsrc_t r = row_rsrc(row, len);
    const unsigned off = (unsigned)col * 8u;
    a = rsrc_ld(r, off, double());
    b = rsrc_ld(r, off + 8u, double());
}
// Bload for a row j that is the same for the whole wave (the descriptor's
// length does Bload's range check: zero past column nxT or row nyT)
__device__ __forceinline__ double Bload_row(const KParams& P, const double* __restrict__ B, int i, int j) {
    return row_ld(B + (size_t)(P.nxT + 1) * j, j <= P.nyT ? P.nxT + 1 : 0, i);
}
// columns i and i + 1 of corner row j
__device__ __forceinline__ void Bload_row2(const KParams& P, const double* __restrict__ B, int i, int j, double& a,
                                           double& b) {
    row_ld2(B + (size_t)(P.nxT + 1) * j, j <= P.nyT ? P.nxT + 1 : 0, i, a, b);
}
__device__ __forceinline__ void row_st(double* row, int len, int col, double v) {
    using V = decltype(__builtin_amdgcn_raw_buffer_load_b64(__amdgpu_buffer_rsrc_t(), 0u, 0, 0));
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(V, v), row_rsrc(row, len), (unsigned)col * 8u, 0, 0);
}
__device__ __forceinline__ void row_st(float* row, int len, int col, float v) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), row_rsrc(row, len), (unsigned)col * 4u, 0, 0);
}

// Stage-1 result of one cell (rungekutta.jl:38-41 with the Float64 dt,
// friction.jl:80-84 from U0 with the stored dt, timestepper.jl:53-63).
// FAST: the friction law is none or bh2021.
template <class S, bool FAST = false>
__device__ __forceinline__ void stage1_cell(const KParams& P, const S x[3], const S r[3], double Bm, double dt_d,
                                            S dt_s, S o[3]) {
    o[0] = (S)(x[0] + dt_d * r[0]);
    o[1] = (S)(x[1] + dt_d * r[1]);
    o[2] = (S)(x[2] + dt_d * r[2]);
    if (P.friction) {
        const double fs = friction_scalar(FAST ? 1 : P.friction, P.Cz, P.phys.kappa, x[0], x[1], x[2], Bm);
        apply_friction(o, dt_s, fs);
    }
    if (o[0] - Bm < P.phys.cutoff) {
        o[0] = (S)jl_max((double)o[0], Bm);
        o[1] = (S)0.0;
        o[2] = (S)0.0;
    }
}

// Rain and infiltration on the w component where both are uniform in space,
// in source-list order (apply_sources).
template <class S>
__device__ __forceinline__ S uniform_sources(const KParams& P, const StepRates& sl, S w) {
    auto infil = [&](S x) -> S { return P.infil_kind ? (S)(x - sl.infil_tfac) : x; };
    auto rain = [&](S x) -> S { return P.rain_kind ? (S)(x + sl.rain_now) : x; };
    return P.rain_first ? infil(rain(w)) : rain(infil(w));
}

// A value that is the same on every lane, moved to scalar registers.
__device__ __forceinline__ double wave_uniform(double v) {
    const long long b = __double_as_longlong(v);
    const unsigned lo = __builtin_amdgcn_readfirstlane((int)(unsigned long long)b);
    const unsigned hi = __builtin_amdgcn_readfirstlane((int)((unsigned long long)b >> 32));
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// The specialised kernels (FAST): linear reconstruction with a finite nonzero
// θ, ρ = 1, the 2D cell-bottom lookup, no friction or bh2021, and rain and
// infiltration uniform in space; MODE_POW2 also has power-of-two spacings.
enum { MODE_GENERAL = 0, MODE_FAST = 1, MODE_POW2 = 2 };

__device__ __forceinline__ RngK rng_constants(const KParams& P) {
    RngK K;
    auto uni = [](const Recip& R) { return Recip{R.d, wave_uniform(R.r)}; };
    K.k2 = uni(recip_rng(wave_uniform(2 * P.phys.kappa)));
    K.dx = uni(recip_rng(P.dx));
    K.dy = uni(recip_rng(P.dy));
    K.half_kappa = wave_uniform(P.phys.kappa / 2.0);
    K.hrg = wave_uniform(0.5 * P.phys.rho * P.phys.g);
    K.theta2 = wave_uniform(2.0 * P.theta);
    K.bx = wave_uniform(-P.phys.g * P.inv_dx * 0.5);
    K.by = wave_uniform(-P.phys.g * P.inv_dy * 0.5);
    return K;
}
template <int MODE>
__device__ __forceinline__ double cell_bottom(const KParams& P, double a, double b, double c, double d) {
    return MODE ? 0.25 * (((a + b) + c) + d) : bcell4(P, a, b, c, d);
}
// The bottom source of one direction (source_term_bottom.jl:38):
// -g (dB/Δ) (hsum/2).  With a power-of-two spacing (and no underflow: in
// band) the exact scalings by 1/Δ and 1/2 move into the constant.
template <int MODE, bool RNG, class S>
__device__ __forceinline__ double bottom_term(const KParams& P, const RngK& K, int dir, double dB, S hsum) {
    if (RNG && MODE == MODE_POW2) return ((dir == 0 ? K.bx : K.by) * dB) * hsum;
    const double s = RNG ? div_rng(dB, dir == 0 ? K.dx : K.dy)
                         : slope_div(dB, dir == 0 ? P.dx : P.dy, dir == 0 ? P.inv_dx : P.inv_dy,
                                     dir == 0 ? P.dx_pow2 : P.dy_pow2);
    return -P.phys.g * s * (hsum / 2.0);
}

// x part minus the y flux difference (numericalflux.jl:27): with a
// power-of-two spacing the product with 1/Δ is exact (in band), so it may be
// fused into the subtraction.
template <int MODE, bool RNG, class S>
__device__ __forceinline__ S y_part(const KParams& P, S accx, double dF) {
    if (RNG && MODE == MODE_POW2) return (S)__builtin_fma(-P.inv_dy, dF, (double)accx);
    return (S)(accx - P.inv_dy * dF);
}

// Is dt in the range the ranged friction form needs?
__device__ __forceinline__ bool dt_in_range(double dt) { return dt > 0.0 && dt <= 0x1p100; }

// stage1_cell with the ranged friction form, for a wave in band so far: the
// stage-1 result o and whether this lane's values allow it and keep the wave in
// band (b0: a bottom corner of the row).  With friction the substep input x and
// the momenta before the division by D = 1 - dt*fs >= 1 are checked too:
// magnitudes of at least 2^-80 over D < 2^40 leave at least 2^-120.
template <class S, bool FRICTION>
__device__ __forceinline__ bool stage1_cell_rng(const KParams& P, const RngK& K, const S x[3], const S r[3], double Bm,
                                                double b0, double dt_d, S dt_s, S o[3]) {
    o[0] = (S)(x[0] + dt_d * r[0]);
    o[1] = (S)(x[1] + dt_d * r[1]);
    o[2] = (S)(x[2] + dt_d * r[2]);
    bool ok = true;
    if (FRICTION) {
        const double fs = friction_scalar_rng(P.Cz, P.phys.kappa, K, x[0], x[1], x[2], Bm);
        const double D = 1 - dt_s * fs;
        const double p1 = (double)o[1], p2 = (double)o[2];
        const Recip R = recip_rng(D);
        o[1] = (S)div_rng(p1, R);
        o[2] = (S)div_rng(p2, R);
        const int ep = min(__builtin_amdgcn_frexp_exp(p1), __builtin_amdgcn_frexp_exp(p2));
        const int ex = min(min(__builtin_amdgcn_frexp_exp((double)x[0]), __builtin_amdgcn_frexp_exp((double)x[1])),
                           __builtin_amdgcn_frexp_exp((double)x[2]));
        const double s = (__builtin_fabs(p1) + __builtin_fabs(p2)) +
                         ((__builtin_fabs((double)x[0]) + __builtin_fabs((double)x[1])) +
                          (__builtin_fabs((double)x[2]) + D));
        ok = ep >= -79 && ex >= -119 && s < 0x1p40;
    }
    if (o[0] - Bm < P.phys.cutoff) {
        o[0] = (S)__builtin_fmax((double)o[0], Bm);
        o[1] = (S)0.0;
        o[2] = (S)0.0;
    }
    if (FRICTION) {
        const int e = min(__builtin_amdgcn_frexp_exp((double)o[0]), __builtin_amdgcn_frexp_exp(b0));
        return ok && e >= -119 && __builtin_fabs((double)o[0]) + __builtin_fabs(b0) < 0x1p40;
    }
    return in_band((double)o[0], (double)o[1], (double)o[2], b0);
}

// The stage-1 result o of one cell per lane, by the ranged friction form while
// the wave is in band (and its dt in range); returns whether it still is.
template <class S, int MODE>
__device__ __forceinline__ bool stage1_any(const KParams& P, const RngK& K, const S x[3], const S r[3], double Bm,
                                           double b0, double dt_d, S dt_s, bool band, S o[3]) {
    if (band) {
        bool ok;
        if (MODE && P.friction) {
            ok = stage1_cell_rng<S, true>(P, K, x, r, Bm, b0, dt_d, dt_s, o);
        } else if (MODE) {
            ok = stage1_cell_rng<S, false>(P, K, x, r, Bm, b0, dt_d, dt_s, o);
        } else {
            stage1_cell<S>(P, x, r, Bm, dt_d, dt_s, o);
            return __all(in_band((double)o[0], (double)o[1], (double)o[2], b0));
        }
        if (__all(ok)) return true;
    }
    stage1_cell<S, MODE != 0>(P, x, r, Bm, dt_d, dt_s, o);
    return false;
}

// The RK2 result of an output cell of stage 2 (rungekutta.jl:43-47, friction
// from the stage input u1, the dry clamp): x0 is U^n, acc L(U1) + sources.
// RNG: u1 and the bottom are in band and dt in range.
template <class S, int MODE, bool RNG>
__device__ __forceinline__ void stage2_cell(const KParams& P, const RngK& K, const S x0[3], const S u1[3],
                                            const S acc[3], double Bm, S dt_s, S o[3]) {
#pragma unroll
    for (int v = 0; v < 3; ++v) o[v] = (S)(u1[v] + dt_s * acc[v]);
#pragma unroll
    for (int v = 0; v < 3; ++v) o[v] = (S)(0.5 * (x0[v] + o[v]));
    if (P.friction) {
        if (RNG && MODE) {
            const double D = 1 - dt_s * friction_scalar_rng(P.Cz, P.phys.kappa, K, u1[0], u1[1], u1[2], Bm);
            o[1] = (S)(o[1] / D);                   // o[0] * (1 - dt*0.0) is o[0]: dt is finite
            o[2] = (S)(o[2] / D);
        } else {
            apply_friction(o, dt_s, friction_scalar(MODE ? 1 : P.friction, P.Cz, P.phys.kappa, u1[0], u1[1], u1[2], Bm));
        }
    }
    if (o[0] - Bm < P.phys.cutoff) {
        o[0] = (S)jl_max((double)o[0], Bm);
        o[1] = (S)0.0;
        o[2] = (S)0.0;
    }
}

// Raise a maximum speed kept as the bit pattern of a non-negative double (or
// a NaN, which orders above every number) to at least sp.  RNG: neither is a
// NaN, so the hardware maximum of the doubles serves.
template <bool RNG>
__device__ __forceinline__ void raise_speed(unsigned long long& sm, double sp) {
    if (RNG) {
        sm = (unsigned long long)__double_as_longlong(__builtin_fmax(__longlong_as_double((long long)sm), sp));
    } else {
        const unsigned long long bits = (unsigned long long)__double_as_longlong(sp);
        sm = bits > sm ? bits : sm;
    }
}

// v with its sign bit flipped where mask has bit 31 set.
__device__ __forceinline__ double flip_sign(double v, unsigned mask) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    return __longlong_as_double((long long)(((unsigned long long)((unsigned)(b >> 32) ^ mask) << 32) | (unsigned)b));
}
__device__ __forceinline__ float flip_sign(float v, unsigned mask) {
    return __int_as_float(__float_as_int(v) ^ (int)mask);
}

// Stage 2 on the gc x gc corner cells of the domain, by `lanes` threads:
// never written by the boundary condition (bc.jl:92-109) nor read by a
// stencil, but part of the state; both stages run sources, RK update,
// friction and clamp on them.  ONE_STAGE: the ForwardEuler step, which is the
// first of the two.
template <class S, bool FAST, bool ONE_STAGE>
__device__ __forceinline__ void finish_corners(const KParams& P, const StepRates& sl, const S* __restrict__ U0,
                                               S* __restrict__ OUT, const double* __restrict__ B, double dt_d, S dt_s,
                                               int lane, int lanes) {
    const int gc = P.gc, nxT = P.nxT, nyT = P.nyT;
    const size_t n = (size_t)nxT * nyT;
    for (int e = lane; e < 4 * gc * gc; e += lanes) {
        const int corner = e / (gc * gc), rr = e % (gc * gc);
        const int ci = (corner & 1) ? nxT - gc + rr % gc : rr % gc;
        const int cj = (corner >> 1) ? nyT - gc + rr / gc : rr / gc;
        const size_t k = (size_t)ci + (size_t)nxT * cj;
        const double Bm = bcell4(P, Bload(P, B, ci, cj), Bload(P, B, ci + 1, cj), Bload(P, B, ci, cj + 1),
                                 Bload(P, B, ci + 1, cj + 1));
        const S src = FAST ? uniform_sources<S>(P, sl, S(0)) : apply_sources(P, sl, S(0), k);
        const S x[3] = {U0[k], U0[n + k], U0[2 * n + k]};
        const S rs[3] = {src, S(0), S(0)};
        S u1[3];
        stage1_cell<S, FAST>(P, x, rs, Bm, dt_d, dt_s, u1);
        if (ONE_STAGE) {
            OUT[k] = u1[0];
            OUT[n + k] = u1[1];
            OUT[2 * n + k] = u1[2];
            continue;
        }
        S o[3];
#pragma unroll
        for (int v = 0; v < 3; ++v) o[v] = (S)(u1[v] + dt_s * rs[v]);
#pragma unroll
        for (int v = 0; v < 3; ++v) o[v] = (S)(0.5 * (x[v] + o[v]));
        if (P.friction) {
            const double fs = friction_scalar(FAST ? 1 : P.friction, P.Cz, P.phys.kappa, u1[0], u1[1], u1[2], Bm);
            apply_friction(o, dt_s, fs);
        }
        if (o[0] - Bm < P.phys.cutoff) {
            o[0] = (S)jl_max((double)o[0], Bm);
            o[1] = (S)0.0;
            o[2] = (S)0.0;
        }
        OUT[k] = o[0];
        OUT[n + k] = o[1];
        OUT[2 * n + k] = o[2];
    }
}

// What a stage launch (2 to 4) does once, by one wave of a workgroup of its
// own: dt for the host, the step's closing (t += dt, next slot armed; the other
// waves read only this step's slot, and the next one is read only by the next
// launches) and the domain's corners.  An inactive step passes inactivity on,
// so steps launched past the end of a run stay no-ops.  At the end of the first
// tile's wave this chain of memory latencies made small launches longer: a 1D
// run of 1024 cells took 7.35 ms, now 6.77, 107x145 ForwardEuler 1.27, now 1.19.
// The workgroup comes last, so that it takes no tile's place.
template <class S, int STAGE, bool FAST>
__device__ __forceinline__ void close_stage(const KParams& P, StepCtl* ctl, int slot, const S* __restrict__ U0,
                                            S* __restrict__ UN, const double* __restrict__ B, int close) {
    const StepSlot& sl = ctl->slot[slot];
    const int next = STAGE == 3 ? next_of_three(slot) : 1 - slot, lane = threadIdx.x;
    if (!sl.active) {
        if (close && lane == 0) ctl->slot[next].active = 0;
        return;
    }
    const double dt_d = wave_uniform(stage1_dt<S>(P, ctl, sl));
    const S dt_s = (S)dt_d;
    if (lane == 0) {
        ctl->dt = (double)dt_s;
        ctl->dt_stage1 = dt_d;
        // stage 3 raises the next slot's speeds meanwhile, and clears the third's
        if (close) close_step<S, FAST>(P, ctl, slot, next, STAGE == 3 ? next_of_three(next) : next);
    }
    finish_corners<S, FAST, (STAGE >= 3)>(P, sl, U0, UN, B, dt_d, dt_s, lane, 64);
}

// The hardware hands workgroup L of a launch to XCD L mod 8, and each XCD
// has its own L2.  Block L therefore takes logical tile
//   prefix(L mod 8) + L div 8,
// so the blocks of one XCD work on one contiguous run of tiles, where
// neighbouring segments (which share 4 halo rows) are resident together.
constexpr int N_XCD = 8;
__device__ __forceinline__ int xcd_tile(int L, int N) {
    const int x = L % N_XCD, k = L / N_XCD, q = N / N_XCD, r = N % N_XCD;
    return x * q + min(x, r) + k;
}

// kernel(stage, mode) for a run-time stage (1 to STAGES) and mode.
template <int STAGES, class F>
inline void by_stage_mode(int stage, int mode, F&& go) {
    auto with = [&](auto st) {
        if (mode == MODE_POW2) go(st, std::integral_constant<int, MODE_POW2>{});
        else if (mode == MODE_FAST) go(st, std::integral_constant<int, MODE_FAST>{});
        else go(st, std::integral_constant<int, MODE_GENERAL>{});
    };
    if (stage == 1) return with(std::integral_constant<int, 1>{});
    if constexpr (STAGES >= 3)
        if (stage == 3) return with(std::integral_constant<int, 3>{});
    if constexpr (STAGES >= 4)
        if (stage == 4) return with(std::integral_constant<int, 4>{});
    with(std::integral_constant<int, 2>{});
}
// The stages a launch of storage type S has: the adjoint, whose steps take
// stage 4, is double only.
template <class S>
constexpr int LAUNCH_STAGES = std::is_same<S, double>::value ? 4 : 3;

}  // namespace sfv
