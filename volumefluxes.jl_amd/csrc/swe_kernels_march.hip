// swe_kernels_march.hip — RK2 stage kernels, one wavefront per strip.
//
// A wave owns MX = 60 output columns (lanes 2..61 of its 64; lanes 0, 1,
// 62, 63 are the x halo) and a segment of MY rows, and marches up the
// segment one row per iteration.  x neighbours come from the adjacent lanes
// (LDS reads and cross-lane moves), y neighbours from a sliding window of rows
// that the wave keeps for itself in LDS, so every cell is loaded once per
// wave, every reconstruction (linearreconstruction.jl:58-102) is evaluated
// once per cell and direction, and every face flux (centralupwind.jl:48-77)
// once per face — the reference evaluates each face from both sides with
// identical arguments (numericalflux.jl:25-26), so sharing it is bit-exact.
// No block-level barriers: waves are independent.
//
// FP64 issue bounds these kernels at sizes that fill the device, so what
// counts is instructions per row and waves to cover their latencies.  Against
// a window in registers (141-168 VGPRs, three waves per SIMD, the first rows
// peeled: 44-60 KB of code), one loop over the LDS window has 118-122 VGPRs and
// 14-21 KB; with the ranged reconstruction and friction of swe_physics.hpp a
// 2048^2 step issues 32.0 M (stage 1) and 46.8 M (stage 2) VALU instructions
// instead of 38.0 M and 55.1 M.  Per step, same box, before and after: 2048^2
// f64 251 and 240 us, with f32 storage 240 and 211 us, with spacings that are
// no power of two and infiltration 282 and 239 us, 1024^2 82 and 74 us.
//
// The segment height is chosen per grid by the host so that the waves fill
// the GPU's resident wave slots in whole rounds.  Per iteration r the wave
// takes row jr = j0-2+r and
//   1. y-reconstructs row jr-1 from rows jr-2..jr,
//   2. evaluates the y face between rows jr-2 and jr-1,
//   3. finishes row jr-2 (its x part was done one iteration earlier, its
//      y faces are now both known): flux difference in the reference's
//      X-then-Y order, bottom source, rain/infiltration, then either stores
//      the stage right-hand side (stage 1) or the RK2 result (stage 2),
//   4. x-reconstructs row jr-1 and evaluates its x faces (the x part).
// Stage 2 rebuilds U1 = clamp(friction(U0 + dt*RHS1)) for every loaded cell
// (ghost cells through the boundary-condition source maps), so the stage-1
// state never touches HBM.
#include <algorithm>
#include <cmath>
#include <mutex>
#include <type_traits>
#include <utility>

#include "swe_kernels.hpp"
#include "swe_rows.hpp"

namespace sfv {

// Build-time tuning knobs (defaults are the measured best on MI355X):
//   SFV_MARCH_ROWS        rows per wave segment (0: chosen per grid)
//   SFV_MARCH_MIN_WAVES   minimum waves per SIMD the register allocation must allow
//   SFV_MARCH_XCD         block order: 1 = each XCD gets a contiguous run of tiles,
//                         segments fastest (vertical halos stay in one L2);
//                         2 = same, strips fastest
//   SFV_MARCH_PRIO        1 = waves with more rows left issue first; 0 = hardware order
//                         (oldest wave first)
//   SFV_MARCH_PRIO_DIV    the priority steps down every 1/DIV of a wave's rows, over
//                         its last 3/DIV
//   SFV_MARCH_LINEAR      1 = waves numbered across the launch (no per-strip padding of
//                         segments to whole workgroups); 0 = a workgroup per 4 segments of a strip
//   SFV_MARCH_TIMELINE    measurement build (`make timeline`): the single-grid kernels record
//                         each wave's start, end, hardware slot and row start times
#ifndef SFV_MARCH_ROWS
#define SFV_MARCH_ROWS 0
#endif
#ifndef SFV_MARCH_MIN_WAVES
#define SFV_MARCH_MIN_WAVES 4
#endif
#ifndef SFV_MARCH_XCD
#define SFV_MARCH_XCD 2
#endif
#ifndef SFV_MARCH_PRIO
#define SFV_MARCH_PRIO 1
#endif
#ifndef SFV_MARCH_PRIO_DIV
#define SFV_MARCH_PRIO_DIV 8
#endif
#ifndef SFV_MARCH_TIMELINE
#define SFV_MARCH_TIMELINE 0
#endif
#if SFV_MARCH_TIMELINE
// Wave timeline of the last single-grid launch of each stage (the 100 MHz
// real-time counter): [stage][wave] = {start, end, HW_ID, XCC_ID << 32 |
// strip << 16 | segment}, and the start of each of the first 32 row
// iterations.  Read with sfv_probe_timeline (this build only).
constexpr int TL_WAVES = 16384, TL_ROWS = 32;
__device__ unsigned long long tl_wave[2][TL_WAVES][4];
__device__ unsigned long long tl_rows[2][TL_WAVES][TL_ROWS];
#endif

// s_setprio takes an immediate: one branch per level
__device__ __forceinline__ void set_issue_priority(int lvl) {
    switch (lvl) {
        case 0: __builtin_amdgcn_s_setprio(0); break;
        case 1: __builtin_amdgcn_s_setprio(1); break;
        case 2: __builtin_amdgcn_s_setprio(2); break;
        default: __builtin_amdgcn_s_setprio(3); break;
    }
}

constexpr int MW = 64;                // lanes
constexpr int MX = MARCH_COLS;        // output columns per wave
constexpr int MWAVES = MARCH_WAVES;   // waves per block

// Stage 1's wave-speed maxima of one block (its 4 waves) into the step slot.
// Every wave of the block calls this exactly once per tile, also a wave whose
// segment lies past the grid (with zeros): the maxima meet in LDS behind a
// barrier and one lane raises the slot's line of this XCD.  `par` alternates
// between consecutive tiles of a persistent block so the next tile's writes
// never meet this tile's reads.
__device__ __forceinline__ void block_max_to_slot_m(unsigned long long smx, unsigned long long smy, StepSlot* s,
                                                    int par) {
    __shared__ unsigned long long red[2][MWAVES][2];
    smx = wave_max_u64(smx);
    smy = wave_max_u64(smy);
    const int lane = threadIdx.x & (MW - 1), w = threadIdx.x / MW;
    if (lane == 0) {
        red[par][w][0] = smx;
        red[par][w][1] = smy;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 1; k < MWAVES; ++k) {
            smx = red[par][k][0] > smx ? red[par][k][0] : smx;
            smy = red[par][k][1] > smy ? red[par][k][1] : smy;
        }
        raise_wsmax(s, smx, smy);
    }
}

// A wave's window of past rows, in LDS and private to the wave: its lanes
// write and read it in program order, so no barrier is involved (march_fence
// keeps the compiler to that order).  Held in registers instead, the window
// alone takes 40-50 VGPRs and its shifting about 60 moves per row; in LDS the
// kernels fit 128 VGPRs, four waves per SIMD instead of three.
template <class S>
struct MarchWin {
    S ry[4][MW];                   // the row below's upper y face state and lower face depth
    S u[3][3][MW];                 // stage input of the last three rows
    S ax[3][MW];                   // x part of the row below
    double fy[3][MW];              // y flux below it
};
__device__ __forceinline__ void march_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// One wave's work: output columns gc + 60*strip .. +59 (lanes 2..61) of rows
// gc + seg*my .. +my-1.  Shared by the single-grid kernel (strip, seg from
// the block index) and the batched kernel (from the batch's tile table).
// Every wave is independent.
// MODE: what is known of the configuration (march_mode), so that its run-time
// checks fold away.
template <class S, int STAGE, int MODE = MODE_GENERAL, bool BATCH = false>
__device__ __forceinline__ void march_tile(const KParams& P, StepCtl* ctl, int slot, int my, int strip, int seg,
                                           const S* __restrict__ U0, const S* __restrict__ RHS1,
                                           S* __restrict__ OUT, S* __restrict__ UO, const double* __restrict__ B,
                                           MarchWin<S>& win, int remap, int par = 0, int close = 0,
                                           int prio_after = 0, int prio_total = 0, int prio_cap = 3) {
    const StepSlot& sl = ctl->slot[slot];
    // the slot of the step whose speeds are found here
    const int rslot = STAGE == 3 ? next_of_three(slot) : slot;
    const int lane = threadIdx.x & (MW - 1);
    if (!sl.active) {                              // the same for every wave of the block
        // an inactive step passes inactivity on, so steps launched past the
        // end of a run stay no-ops (close_stage in a launch of one grid)
        if (BATCH && STAGE == 2 && close && strip == 0 && seg == 0 && lane == 0) ctl->slot[1 - slot].active = 0;
        return;
    }
    const int gc = P.gc, nxT = P.nxT, nyT = P.nyT;
    const int j0 = gc + seg * my;
    if (j0 >= nyT - gc) {                          // whole wave: past the grid
        if (STAGE == 1 || STAGE == 3) block_max_to_slot_m(0ull, 0ull, &ctl->slot[rslot], par);
        return;
    }
    const int th = min(my, nyT - gc - j0);
    const int i = gc + strip * MX + lane - 2;      // this lane's column (>= 0 since gc >= 2)
    const bool in_dom = i < nxT;
    const bool out_col = lane >= 2 && lane < MX + 2 && i < nxT - gc;
    const size_t n = (size_t)nxT * nyT;
    const bool rec_linear = MODE || P.rec == 1;
    const RngK K = rng_constants(P);

    double dt_d = 0.0;
    S dt_s = S(0);
    if (STAGE >= 2) {
        dt_d = wave_uniform(stage1_dt<S>(P, ctl, sl));
        dt_s = (S)dt_d;
    }
    // the source rates of the right-hand side: this step's, in STAGE 3 the
    // next one's (close_step gives its slot the same values)
    StepRates nrates;
    if (STAGE == 3) {
        set_rates<MODE != 0>(P, nrates, (double)(S)((S)sl.t + dt_s));
        nrates.rain_now = wave_uniform(nrates.rain_now);
        nrates.infil_tfac = wave_uniform(nrates.infil_tfac);
    }
    const StepRates& rates = STAGE == 3 ? nrates : static_cast<const StepRates&>(sl);

    // Ghost cells are read through the boundary-condition maps (stage 2
    // always, stage 1 with remap): a ghost's value is its source's, with the
    // sign flip, as update_bc! would have stored it; corners, which the
    // boundary condition never writes, feed no output.  Only the edge strips
    // and segments hold ghost columns or rows; the test is the same for the
    // whole wave.  The lanes span columns gc + strip*MX - 2 .. +61, the rows
    // loaded are j0 - 2 .. j0 + th + 1.
    const bool rmp = STAGE >= 2 || remap;
    const bool xedge = rmp && (strip == 0 || gc + strip * MX + MW - 3 >= nxT - gc);
    const bool yedge = rmp && (j0 - 2 < gc || j0 + th + 1 >= nyT - gc);
    int sci = i;
    unsigned fxb = 0u;                             // the sign bit if this column's hu is negated
    if (xedge && in_dom) {
        if (i < gc) { sci = P.src_lo_x[i]; fxb = P.flip_lo_x[i] ? 0x80000000u : 0u; }
        else if (i >= nxT - gc) { sci = P.src_hi_x[i - (nxT - gc)]; fxb = P.flip_hi_x[i - (nxT - gc)] ? 0x80000000u : 0u; }
    }
    // ranged face evaluation (central_upwind_rng) while the wave's inputs allow it
    bool band = P.ranged && (STAGE == 1 || dt_in_range(dt_d));
    double Blyp = 0.0, bcp = 0.0;                  // row jr-2's lower face bottom and B_cell
    unsigned long long smx = 0, smy = 0;

    // a row's stage input as loaded: the state, with stage 2 the right-hand
    // side and the upper bottom corners of the source cell
    struct Raw {
        S x[3], r[STAGE >= 2 ? 3 : 1];
        double c2, c3;
        int sj;
        unsigned fyb;
    };
    auto fetch = [&](int jr, Raw& o) {
        int sj = jr;
        unsigned fyb = 0u;
        if (yedge) {
            if (jr < gc) { sj = P.src_lo_y[jr]; fyb = P.flip_lo_y[jr] ? 0x80000000u : 0u; }
            else if (jr >= nyT - gc) { sj = P.src_hi_y[jr - (nyT - gc)]; fyb = P.flip_hi_y[jr - (nyT - gc)] ? 0x80000000u : 0u; }
        }
        o.sj = sj;
        o.fyb = fyb;
        const size_t ro = (size_t)nxT * sj;        // row sj (uniform), column sci (per lane)
#pragma unroll
        for (int v = 0; v < 3; ++v) o.x[v] = row_ld(U0 + v * n + ro, nxT, sci);
        if (STAGE >= 2) {
#pragma unroll
            for (int v = 0; v < 3; ++v) o.r[v] = row_ld(RHS1 + v * n + ro, nxT, sci);
            Bload_row2(P, B, sci, sj + 1, o.c2, o.c3);
        }
        if constexpr (STAGE == 3 && MODE == MODE_GENERAL) {
            // a source that is a ghost has the non-directional sources only
            if (P.ghost_self && in_dom && (sci >= nxT - gc || sj >= nyT - gc)) {
                o.r[0] = apply_sources(P, sl, S(0), (size_t)sci + ro);
                o.r[1] = o.r[2] = S(0);
            }
        }
    };
    Raw raw;

    // Row loop r = 0..th+3 over input rows jr = j0-2+r.  Row q = jr-1 is
    // worked on only where it feeds an output row: its x part when q is an
    // output row, i.e. 3 <= r <= th+2; the y face below it when it borders
    // one, i.e. r >= 3; row jr-2 is finished for r >= 4.
    int s0 = 0, s1 = 2, s2 = 1;                    // window slots of rows jr, jr-1, jr-2
    for (int r = 0; r < th + 4; ++r) {
        const int jr = j0 - 2 + r;
#if SFV_MARCH_TIMELINE
        if (!BATCH && r < TL_ROWS && lane == 0) {
            const int tw = blockIdx.x * MWAVES + threadIdx.x / MW;
            if (tw < TL_WAVES) tl_rows[STAGE == 1 ? 0 : 1][tw][r] = __builtin_amdgcn_s_memrealtime();
        }
#endif
        // Issue priority by iterations left (this segment's and, in the
        // persistent batch kernel, those of the wave's later tiles): 3 until
        // the last 3/DIV of the wave's total, then one step lower every
        // 1/DIV.  The waves sharing a SIMD then progress together and end
        // together, instead of the oldest finishing first and the youngest
        // running on alone at the end of the launch.  prio_after < 0: the
        // caller keeps its own priority; prio_cap: the highest level used.
        if (SFV_MARCH_PRIO && prio_after >= 0) {
            const int left = th + 3 - r + prio_after,
                      q = max(1, (prio_total > 0 ? prio_total : th + 4) / SFV_MARCH_PRIO_DIV);
            set_issue_priority(min(prio_cap, left >= 3 * q ? 3 : left >= 2 * q ? 2 : left >= q ? 1 : 0));
        }
        // bottom corner rows jr-1 and jr, columns i and i+1 (row j0-3 is not read)
        const int jb = r >= 1 ? jr - 1 : jr;
        double bm1, nm1, b0, n0;
        Bload_row2(P, B, i, jb, bm1, nm1);
        Bload_row2(P, B, i, jr, b0, n0);
        fetch(jr, raw);
        // stage input of row jr
        S cC[3];
        const S x[3] = {raw.x[0], raw.x[1], raw.x[2]};
        const unsigned fyb = raw.fyb;
        if (STAGE == 1) {
            cC[0] = x[0]; cC[1] = x[1]; cC[2] = x[2];
        } else {
            double c0 = b0, c1 = n0;
            if (xedge || raw.sj != jr) Bload_row2(P, B, sci, raw.sj, c0, c1);
            const double Bm = cell_bottom<MODE>(P, c0, c1, raw.c2, raw.c3);      // the source cell's bottom
            // the ranged forms apply while every stage input and bottom corner
            // this wave has taken in lies in band; the faces of this iteration
            // read rows up to jr and corner rows up to jr
            band = stage1_any<S, MODE>(P, K, x, raw.r, Bm, b0, dt_d, dt_s, band, cC);
        }
        // (a lane past the grid feeds no output)
        cC[1] = flip_sign(cC[1], fxb);
        cC[2] = flip_sign(cC[2], fyb);
        if (STAGE == 1) band = band && __all(in_band(cC[0], cC[1], cC[2], b0));
        if constexpr (STAGE == 3 && MODE == MODE_GENERAL) {
            // ghosts on the high sides whose values live on in memory (gc = 2)
            const bool gx = in_dom && i >= nxT - gc && jr >= j0 && jr < j0 + th;
            const bool gy = out_col && jr >= nyT - gc && j0 + th == nyT - gc;
            if (P.ghost_self && (gx || gy)) {
                S* urow = UO + (size_t)nxT * jr;
#pragma unroll
                for (int v = 0; v < 3; ++v) row_st(urow + v * n, nxT, i, cC[v]);
            }
        }
#pragma unroll
        for (int v = 0; v < 3; ++v) win.u[s0][v][lane] = cC[v];
        const double Bly = 0.5 * (bm1 + nm1), Bry = 0.5 * (b0 + n0);
        const double bcq = cell_bottom<MODE>(P, bm1, nm1, b0, n0);           // B_cell of row jr-1
        const S* ub = &win.u[s1][0][lane];                         // row jr-1
        const S* ua = &win.u[s2][0][lane];                         // row jr-2
        auto work = [&](auto rng_tag) {
            constexpr bool RNG = decltype(rng_tag)::value;         // every input of these faces is in band
            // y reconstruction of row m = jr-1
            S Ly[3], Ry[3];
            {
                const S cA[3] = {ua[0], ua[MW], ua[2 * MW]}, cB[3] = {ub[0], ub[MW], ub[2 * MW]};
                if (rec_linear) {
                    if (RNG) reconstruct_cell_rng(cA, cB, cC, K.theta2, Bly, Bry, Ly, Ry);
                    else reconstruct_cell(cA, cB, cC, P.theta, Bly, Bry, Ly, Ry, MODE != 0);
                } else {
#pragma unroll
                    for (int v = 0; v < 3; ++v) Ly[v] = Ry[v] = cB[v];
                    Ly[0] = Ry[0] = (S)(cB[0] - bcq);
                }
            }
            S Ryp[3], Lyp0;
#pragma unroll
            for (int v = 0; v < 3; ++v) { Ryp[v] = win.ry[v][lane]; win.ry[v][lane] = Ry[v]; }
            Lyp0 = win.ry[3][lane];
            win.ry[3][lane] = Ly[0];
            if (r >= 3) {
                // the y face between rows jr-2 and jr-1
                double Fy[3], Fyp[3];
                const double spy = RNG ? central_upwind_rng<1, MODE != 0>(Ryp, Ly, P.phys, K, Fy)
                                       : central_upwind(1, Ryp, Ly, P.phys, Fy);
                if (STAGE == 1 || STAGE == 3) raise_speed<RNG>(smy, (double)(S)spy);
#pragma unroll
                for (int v = 0; v < 3; ++v) { Fyp[v] = win.fy[v][lane]; win.fy[v][lane] = Fy[v]; }
                // finish row p = jr-2: y part on top of its x part, then sources
                if (r >= 4 && out_col) {
                    const int p = jr - 2;
                    S* orow = OUT + (size_t)nxT * p;               // row p (uniform), column i (per lane)
                    S acc[3];
#pragma unroll
                    for (int v = 0; v < 3; ++v) acc[v] = y_part<MODE, RNG>(P, win.ax[v][lane], Fy[v] - Fyp[v]);
                    if (P.bottom)
                        acc[2] = (S)(acc[2] + bottom_term<MODE, RNG>(P, K, 1, Bly - Blyp, Ryp[0] + Lyp0));
                    acc[0] = MODE ? uniform_sources<S>(P, rates, acc[0])
                                  : apply_sources(P, rates, acc[0], (size_t)i + (size_t)nxT * p);
                    if (STAGE != 2) {
#pragma unroll
                        for (int v = 0; v < 3; ++v) row_st(orow + v * n, nxT, i, acc[v]);
                        if (STAGE >= 3) {                          // the new state, from the window
                            S* urow = UO + (size_t)nxT * p;
#pragma unroll
                            for (int v = 0; v < 3; ++v) row_st(urow + v * n, nxT, i, ua[v * MW]);
                        }
                    } else {
                        // U1 of row p from the window; U0 (output rows are
                        // interior) once more from the cache
                        const S cA[3] = {ua[0], ua[MW], ua[2 * MW]};
                        S x0[3], o[3];
#pragma unroll
                        for (int v = 0; v < 3; ++v) x0[v] = row_ld(U0 + v * n + (size_t)nxT * p, nxT, i);
                        stage2_cell<S, MODE, RNG>(P, K, x0, cA, acc, bcp, dt_s, o);
#pragma unroll
                        for (int v = 0; v < 3; ++v) row_st(orow + v * n, nxT, i, o[v]);
                    }
                }
                if (r < th + 3) {
                    // x part of row q = jr-1 (finished next iteration)
                    const double Blx = 0.5 * (bm1 + b0), Brx = 0.5 * (nm1 + n0);
                    S Lx[3], Rx[3], Rxl[3];
                    const S cB[3] = {ub[0], ub[MW], ub[2 * MW]};
                    if (rec_linear) {
                        const S cl[3] = {ub[-1], ub[MW - 1], ub[2 * MW - 1]};
                        const S cr[3] = {ub[1], ub[MW + 1], ub[2 * MW + 1]};
                        if (RNG) reconstruct_cell_rng(cl, cB, cr, K.theta2, Blx, Brx, Lx, Rx);
                        else reconstruct_cell(cl, cB, cr, P.theta, Blx, Brx, Lx, Rx, MODE != 0);
                    } else {
#pragma unroll
                        for (int v = 0; v < 3; ++v) Lx[v] = Rx[v] = cB[v];
                        Lx[0] = Rx[0] = (S)(cB[0] - bcq);
                    }
#pragma unroll
                    for (int v = 0; v < 3; ++v) Rxl[v] = shfl_up1(Rx[v]);
                    double Fxm[3];
                    const double spx = RNG ? central_upwind_rng<0, MODE != 0>(Rxl, Lx, P.phys, K, Fxm)
                                           : central_upwind(0, Rxl, Lx, P.phys, Fxm);
                    if (STAGE == 1 || STAGE == 3) raise_speed<RNG>(smx, (double)(S)spx);
                    S ax[3];
#pragma unroll
                    for (int v = 0; v < 3; ++v)
                        ax[v] = (S)__builtin_fma(-P.inv_dx, shfl_dn1(Fxm[v]) - Fxm[v], 0.0);   // 0 - inv*diff
                    if (P.bottom)
                        ax[1] = (S)(ax[1] + bottom_term<MODE, RNG>(P, K, 0, Brx - Blx, Rx[0] + Lx[0]));
#pragma unroll
                    for (int v = 0; v < 3; ++v) win.ax[v][lane] = ax[v];
                }
            }
        };
        if (r >= 2) {
            if (band) work(std::true_type{});
            else work(std::false_type{});
        }
        march_fence();
        Blyp = Bly;
        bcp = bcq;
        const int free = s2;
        s2 = s1;
        s1 = s0;
        s0 = free;
    }
    if (STAGE == 1 || STAGE == 3) {
        // x faces this lane evaluated (its left face) that border an output cell
        const bool face_x_ok = in_dom && lane >= 2 && lane <= MX + 2 && (lane == 2 ? i < nxT - gc : i - 1 < nxT - gc);
        block_max_to_slot_m(face_x_ok ? smx : 0ull, out_col ? smy : 0ull, &ctl->slot[rslot], par);
    }

    // a batch member's dt for the host and its step's closing (t += dt, next
    // slot armed), by one lane: the other waves read only this step's slot, and
    // the next slot is read only by the next launches
    if (BATCH && STAGE == 2 && strip == 0 && seg == 0) {
        if (lane == 0) {
            ctl->dt = (double)dt_s;
            ctl->dt_stage1 = dt_d;
            if (close) close_step_call<S, MODE != 0>(P, ctl, slot);
        }
        finish_corners<S, MODE != 0, false>(P, sl, U0, OUT, B, dt_d, dt_s, lane, MW);
    }
}

// Grid of march_blocks(strips, segs) blocks of MWAVES waves (swe_kernels.hpp).
// With SFV_MARCH_LINEAR a wave's number is the block's logical tile times
// MWAVES plus the wave, and a workgroup's waves are neighbouring strips of
// one segment row.
template <class S, int STAGE, int MODE>
__global__ void __launch_bounds__(MW* MWAVES)
__attribute__((amdgpu_waves_per_eu(SFV_MARCH_MIN_WAVES)))
k_march(KParams P, StepCtl* ctl, int slot, int my, int strips, int segs, const S* __restrict__ U0,
        const S* __restrict__ RHS1, S* __restrict__ OUT, S* __restrict__ UO, const double* __restrict__ B, int close,
        int remap) {
    // stages 2 to 4: the last block closes, the others are tiles
    if (STAGE >= 2 && (int)blockIdx.x == march_blocks(strips, segs)) {
        if (threadIdx.x < MW) close_stage<S, STAGE, MODE != 0>(P, ctl, slot, U0, STAGE >= 3 ? UO : OUT, B, close);
        return;
    }
    const int t = xcd_tile(blockIdx.x, march_blocks(strips, segs));
    // the same for every lane of the wave; readfirstlane tells the compiler so
#if SFV_MARCH_LINEAR
    const int w = __builtin_amdgcn_readfirstlane(t * MWAVES + threadIdx.x / MW);
    const bool idle = w >= strips * segs;          // past the last tile: seg = segs is past the grid
#if SFV_MARCH_XCD == 2
    const int strip = idle ? 0 : w % strips, seg = idle ? segs : w / strips;
#else
    const int strip = idle ? 0 : w / segs, seg = idle ? segs : w % segs;
#endif
#else
    const int seggroups = (segs + MWAVES - 1) / MWAVES;
#if SFV_MARCH_XCD == 2
    const int strip = t % strips, sg = t / strips;
#else
    const int strip = t / seggroups, sg = t % seggroups;
#endif
    const int seg = __builtin_amdgcn_readfirstlane(sg * MWAVES + threadIdx.x / MW);
#endif
#if SFV_MARCH_TIMELINE
    const unsigned long long tl0 = __builtin_amdgcn_s_memrealtime();
#endif
    __shared__ MarchWin<S> win[MWAVES];
    march_tile<S, STAGE, MODE>(P, ctl, slot, my, strip, seg, U0, RHS1, OUT, UO, B, win[threadIdx.x / MW], remap, 0, close);
#if SFV_MARCH_TIMELINE
    const unsigned long long tl1 = __builtin_amdgcn_s_memrealtime();
    const int tw = blockIdx.x * MWAVES + threadIdx.x / MW;
    if ((threadIdx.x & (MW - 1)) == 0 && tw < TL_WAVES) {
        unsigned long long* o = tl_wave[STAGE == 1 ? 0 : 1][tw];
        o[0] = tl0;
        o[1] = tl1;
        o[2] = __builtin_amdgcn_s_getreg((31 << 11) | 4);                       // HW_ID
        o[3] = ((unsigned long long)__builtin_amdgcn_s_getreg((15 << 11) | 20) << 32) |   // XCC_ID
               ((unsigned long long)(strip & 0xFFFF) << 16) | (unsigned)(seg & 0xFFFF);
    }
#endif
}

// Batched stage kernel: a persistent grid (a multiple of 8 workgroups) walks
// the tiles of every member.  The tile order is split into 8 contiguous
// chunks, one per XCD, and the workgroups of XCD x (blockIdx mod 8 == x) walk
// chunk x, so a member's neighbouring tiles share that XCD's L2.  With
// hdr->prio == 1 (a batch of small grids stepping beside another batch) the
// waves take the highest issue priority: their short serial chains issue
// first and the other batch's waves fill the gaps; that other batch runs with
// hdr->prio == 2, its rows-left priority capped one level below.  Where the
// member table's values around the tile loop would push the tile's registers
// into scratch at four waves per SIMD (18-37 spilled), three are asked for.
template <class S, int STAGE, int MODE>
__global__ void __launch_bounds__(MW* MWAVES)
__attribute__((amdgpu_waves_per_eu(sizeof(S) == 4 || (STAGE == 1 && MODE == MODE_GENERAL) ? 3 : SFV_MARCH_MIN_WAVES)))
k_march_batch(const BatchMember* __restrict__ mem, const BatchHeader* __restrict__ hdr, int lp) {
    __shared__ MarchWin<S> win[MWAVES];
    const int members = hdr->members, tiles = hdr->tiles;
    if (hdr->prio == 1) __builtin_amdgcn_s_setprio(3);
    const int cap = hdr->prio == 2 ? 2 : 3;          // a host engine's waves stay below its guest's
    const int x = blockIdx.x % N_XCD, k = blockIdx.x / N_XCD, per = gridDim.x / N_XCD;
    const int q = tiles / N_XCD, r = tiles % N_XCD;
    const int c0 = x * q + min(x, r), c1 = c0 + q + (x < r ? 1 : 0);
    int par = 0;
    // this wave's tiles: c0 + k, c0 + k + per, ... below c1
    const int ntiles = c1 > c0 + k ? (c1 - 1 - c0 - k) / per + 1 : 0;
    for (int t = c0 + k; t < c1; t += per, par ^= 1) {
        const int m = batch_find(mem, members, t);
        const BatchMember& M = mem[m];
        const int local = t - M.tile0;
        const int cur = (M.cur0 ^ lp) & 1, slot = (M.slot0 ^ lp) & 1;
        // the same for every lane of the wave; readfirstlane tells the compiler so
#if SFV_MARCH_LINEAR
        const int w = __builtin_amdgcn_readfirstlane(local * MWAVES + threadIdx.x / MW);
        const bool idle = w >= M.strips * M.segs;  // past the member's last tile: seg = segs is past its grid
        const int strip = idle ? 0 : w % M.strips, seg = idle ? M.segs : w / M.strips;
#else
        const int strip = local % M.strips, sg = local / M.strips;
        const int seg = __builtin_amdgcn_readfirstlane(sg * MWAVES + threadIdx.x / MW);
#endif
        const S* U0 = (const S*)M.U[cur];
        // iterations of this wave's later tiles, counted at this member's height
        const int after = hdr->prio == 1 ? -1 : ((c1 - 1 - t) / per) * (M.my + 4);
        const int total = ntiles * (M.my + 4);
        march_tile<S, STAGE, MODE, true>(M.P, M.ctl, slot, M.my, strip, seg, U0, STAGE == 1 ? nullptr : (const S*)M.RHS,
                                         STAGE == 1 ? (S*)M.RHS : (S*)M.U[cur ^ 1], nullptr, M.B, win[threadIdx.x / MW], 1, par,
                                         1, after, total, cap);
    }
}

// What the specialised kernels may take for granted of a configuration.
int march_mode(const KParams& P) {
    const bool fast = P.rec == 1 && std::isfinite(P.theta) && P.theta != 0.0 && P.phys.rho == 1.0 && !P.bcell_1d &&
                      (P.friction == 0 || P.friction == 1) && P.infil_kind <= 1 && P.rain_kind <= 2;
    return !fast ? MODE_GENERAL : P.dx_pow2 && P.dy_pow2 ? MODE_POW2 : MODE_FAST;
}

// The kernels of a stage: the ones that write ghosts are the general ones.
static int stage_mode(const KParams& P, int stage) {
    return stage == 3 && P.ghost_self ? MODE_GENERAL : march_mode(P);
}

// Rows per wave segment for this grid.  With w waves on each SIMD a launch
// lasts about w (my + 4) / f(w): every wave marches my + 4 rows, the SIMD's
// issue is shared, and fewer than four waves leave part of it idle.  Measured
// at 600^2 to 2048^2: f = 0.43, 0.70, 0.92 and 1 for one to four waves (1024^2: 116.8 us
// at 20 rows, 84.1 at 10, 76.8 at 7, 74.8 at 5; 2048^2: 255 us at 24, 245 at 18;
// 1777x1409: 144.9 at 14, 147.3 at 11).  Further waves come in further
// rounds.  The height in [1, 64] that minimises it wins (the smallest on a tie).
template <class S, int STAGE, int MODE>
static int march_resident_blocks() {
    int blocks = 0;
    const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, k_march<S, STAGE, MODE>, MW * MWAVES, 0);
    return (e == hipSuccess && blocks > 0) ? blocks : 2;
}
int march_rows_per_wave(const KParams& P, int stage, int precision) {
    if (SFV_MARCH_ROWS > 0) return SFV_MARCH_ROWS;
    static int cus = 0, bpc[2][3][3];       // [precision][stage - 1][mode]
    static std::once_flag once;
    std::call_once(once, [] {
        int dev = 0;
        hipDeviceProp_t prop;
        if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&prop, dev) == hipSuccess)
            cus = prop.multiProcessorCount;
        if (cus <= 0) cus = 256;
        auto fill = [](auto s, int (&b)[3][3]) {
            using S = decltype(s);
            b[0][0] = march_resident_blocks<S, 1, 0>();
            b[0][1] = march_resident_blocks<S, 1, 1>();
            b[0][2] = march_resident_blocks<S, 1, 2>();
            b[1][0] = march_resident_blocks<S, 2, 0>();
            b[1][1] = march_resident_blocks<S, 2, 1>();
            b[1][2] = march_resident_blocks<S, 2, 2>();
            b[2][0] = march_resident_blocks<S, 3, 0>();
            b[2][1] = march_resident_blocks<S, 3, 1>();
            b[2][2] = march_resident_blocks<S, 3, 2>();
        };
        fill(double(), bpc[0]);
        fill(float(), bpc[1]);
    });
    // a workgroup puts one wave on each SIMD of its CU
    const long resident = bpc[precision ? 1 : 0][std::min(stage, 3) - 1][stage_mode(P, stage)];
    const long strips = (P.nx + MX - 1) / MX;
    static const double f[5] = {1.0, 0.43, 0.70, 0.92, 1.0};
    auto round_time = [&](long w) { return (double)w / f[std::min(w, 4L)]; };
    int best = 1;
    double best_cost = -1.0;
    for (int my = 1; my <= 64; ++my) {
        const long blocks = march_blocks((int)strips, (P.ny + my - 1) / my);
        const long w = (blocks + cus - 1) / cus;
        const double cost = ((double)(w / resident) * round_time(resident) + round_time(w % resident)) * (my + 4);
        if (best_cost < 0 || cost < best_cost) { best_cost = cost; best = my; }
    }
    return best;
}

template <class S>
hipError_t launch_march(hipStream_t st, const KParams& P, StepCtl* ctl, int slot, int stage, const S* U0,
                        const S* RHS1, S* OUT, const double* B, int close, int remap_halo, S* UO) {
    if (stage > LAUNCH_STAGES<S>) return hipErrorInvalidValue;
    const int my = P.rows > 0 ? P.rows : march_rows_per_wave(P, stage, std::is_same<S, float>::value ? 1 : 0);
    const int segs = (P.ny + my - 1) / my;
    const int strips = (P.nx + MX - 1) / MX;
    by_stage_mode<LAUNCH_STAGES<S>>(stage, stage_mode(P, stage), [&](auto stg, auto mode) {
        hipLaunchKernelGGL((k_march<S, decltype(stg)::value, decltype(mode)::value>), dim3(march_blocks(strips, segs) + (decltype(stg)::value >= 2 ? 1 : 0)),
                           dim3(MW * MWAVES), 0, st, P, ctl, slot, my, strips, segs, U0, RHS1, OUT, UO, B, close,
                           remap_halo);
    });
    return hipPeekAtLastError();
}
template <class S>
hipError_t launch_march_batch(hipStream_t st, int stage, const BatchMember* mem, const BatchHeader* hdr, int lp,
                              int blocks, int mode) {
    if (blocks < N_XCD || blocks % N_XCD) return hipErrorInvalidValue;
    by_stage_mode<2>(stage, mode, [&](auto stg, auto m) {
        hipLaunchKernelGGL((k_march_batch<S, decltype(stg)::value, decltype(m)::value>), dim3(blocks),
                           dim3(MW * MWAVES), 0, st, mem, hdr, lp);
    });
    return hipPeekAtLastError();
}

int march_batch_blocks_per_cu(int precision, int stage, int mode) {
    int blocks = 0;
    hipError_t e = hipErrorUnknown;
    by_stage_mode<2>(stage, mode, [&](auto stg, auto m) {
        constexpr int ST = decltype(stg)::value, M = decltype(m)::value;
        e = precision == 0 ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, k_march_batch<double, ST, M>, MW * MWAVES, 0)
                           : hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, k_march_batch<float, ST, M>, MW * MWAVES, 0);
    });
    return (e == hipSuccess && blocks > 0) ? blocks : 2;
}

template hipError_t launch_march_batch<double>(hipStream_t, int, const BatchMember*, const BatchHeader*, int, int,
                                               int);
template hipError_t launch_march_batch<float>(hipStream_t, int, const BatchMember*, const BatchHeader*, int, int,
                                              int);
template hipError_t launch_march<double>(hipStream_t, const KParams&, StepCtl*, int, int, const double*,
                                         const double*, double*, const double*, int, int, double*);
template hipError_t launch_march<float>(hipStream_t, const KParams&, StepCtl*, int, int, const float*, const float*,
                                        float*, const double*, int, int, float*);

}  // namespace sfv

#if SFV_MARCH_TIMELINE
// Measurement build only: copy the timeline buffers out (waves: 2 x 16384 x 4,
// rows: 2 x 16384 x 32 unsigned 64-bit words) or clear them.
extern "C" int sfv_probe_timeline(unsigned long long* waves, unsigned long long* rows) {
    hipError_t e = hipMemcpyFromSymbol(waves, HIP_SYMBOL(sfv::tl_wave), sizeof(sfv::tl_wave), 0, hipMemcpyDeviceToHost);
    if (e == hipSuccess)
        e = hipMemcpyFromSymbol(rows, HIP_SYMBOL(sfv::tl_rows), sizeof(sfv::tl_rows), 0, hipMemcpyDeviceToHost);
    return (int)e;
}
extern "C" int sfv_probe_timeline_clear() {
    void* p = nullptr;
    hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(sfv::tl_wave));
    if (e == hipSuccess) e = hipMemset(p, 0, sizeof(sfv::tl_wave));
    if (e == hipSuccess) e = hipGetSymbolAddress(&p, HIP_SYMBOL(sfv::tl_rows));
    if (e == hipSuccess) e = hipMemset(p, 0, sizeof(sfv::tl_rows));
    return (int)e;
}
#endif
