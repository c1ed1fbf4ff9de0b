// swe_kernels_block.hip — RK2 stage kernels, one workgroup per strip segment,
// for grids too small to fill the device.
//
// A workgroup of BW waves owns BCOLS = 60 output columns (lanes 2..61 of each
// wave; lanes 0, 1, 62, 63 are the x halo) and a segment of H rows.  It marches
// up the segment in chunks of BW rows, one row per wave: wave w of a chunk
// takes input row r = a + w and works on
//   1. the stage input of row r (stage 2 rebuilds U1 = clamp(friction(U0 +
//      dt*RHS1)) there), which goes to LDS,
//   -- barrier --
//   2. the y reconstruction of row m = r-1 (rows r-2, r-1 from LDS), whose
//      upper face state goes to LDS, and the whole x part of row p = r-2,
//   -- barrier --
//   3. the y face between rows p and m, whose flux goes to LDS,
//   -- barrier --
//   4. the finish of row p: its lower y flux is wave w-1's.
// What a row hands to the next chunk stays in LDS, in slots of alternating
// parity.  Ghost cells are read through the boundary-condition maps, as in
// the wave-march kernels (swe_kernels_march.hip), and every arithmetic step
// is theirs, so results are bitwise the same.
//
// What bounds a small grid is the serial chain of a launch: a wave-march wave
// of one output row works through five input rows one after the other, a
// workgroup here through as many at once, and its halo rows are shared by H
// output rows instead of one or two (block_suits has the times).
#include <cmath>
#include <mutex>
#include <type_traits>

#include "swe_kernels.hpp"
#include "swe_rows.hpp"

namespace sfv {

constexpr int BL = 64;                // lanes
constexpr int BCOLS = MARCH_COLS;     // output columns per workgroup

template <class S, int BW>
struct BlockSmem {
    S pad[2];                         // lane 0 reads one element before a row
    S u[BW + 2][3][BL];               // stage input; the chunk's last two rows alternate between two slots
    S ry[BW + 1][4][BL];              // upper y face state of a row and its lower face depth
    double fy[BW + 1][3][BL];         // y flux below a row
    unsigned long long red[BW][2];
    int bad;                          // serial of the last tile with a value out of band
};
// LDS slots of wave w in a chunk of parity par
template <int BW>
__device__ __forceinline__ int u_slot(int w, int par) { return w < BW - 2 ? w : w + 2 * par; }
template <int BW>
__device__ __forceinline__ int y_slot(int w, int par) { return w < BW - 1 ? w : w + par; }

// MODE: what is known of the configuration (march_mode), so that its run-time
// checks fold away.
template <class S, int STAGE, int MODE, int BW>
__device__ __forceinline__ void block_tile(const KParams& P, StepCtl* ctl, int slot, int H, int strip, int seg,
                                           const S* __restrict__ U0, const S* __restrict__ RHS1,
                                           S* __restrict__ OUT, S* __restrict__ UO, const double* __restrict__ B,
                                           BlockSmem<S, BW>& sm, int serial, int remap) {
    const StepSlot& sl = ctl->slot[slot];
    // the slot of the step whose speeds are found here
    const int rslot = STAGE == 3 ? next_of_three(slot) : slot;
    const int lane = threadIdx.x & (BL - 1);
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / BL);
    if (!sl.active) return;                        // the same for the whole workgroup
    const int gc = P.gc, nxT = P.nxT, nyT = P.nyT;
    const int j0 = gc + seg * H;
    const int th = min(H, nyT - gc - j0);          // >= 1: the launch has no empty segments
    const int i = gc + strip * BCOLS + lane - 2;   // this lane's column
    const bool in_dom = i < nxT;
    const bool out_col = lane >= 2 && lane < BCOLS + 2 && i < nxT - gc;
    const size_t n = (size_t)nxT * nyT;
    const bool rec_linear = MODE || P.rec == 1;
    const RngK K = rng_constants(P);
    auto bc4 = [&](double a, double b, double c, double d) { return cell_bottom<MODE>(P, a, b, c, d); };

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
    // ghost columns read their boundary-condition source; a wall's negated
    // normal momentum flips the sign bit
    const bool rmp = STAGE >= 2 || remap;
    const bool xedge = rmp && (strip == 0 || gc + strip * BCOLS + BL - 3 >= nxT - gc);
    int sci = i;
    unsigned fx = 0u;
    if (xedge && in_dom) {
        if (i < gc) { sci = P.src_lo_x[i]; fx = P.flip_lo_x[i] ? 0x80000000u : 0u; }
        else if (i >= nxT - gc) { sci = P.src_hi_x[i - (nxT - gc)]; fx = P.flip_hi_x[i - (nxT - gc)] ? 0x80000000u : 0u; }
    }
    // x faces this lane evaluates (its left face) that border an output cell
    const bool face_x_ok = in_dom && lane >= 2 && lane <= BCOLS + 2 && (lane == 2 ? i < nxT - gc : i - 1 < nxT - gc);
    unsigned long long smx = 0, smy = 0;
    const bool ranged = P.ranged && (STAGE == 1 || dt_in_range(dt_d));
    const int rows = th + 4;                       // input rows j0-2 .. j0+th+1
    int par = 0;
    for (int q0 = 0; q0 < rows; q0 += BW, par ^= 1) {
        const int q = q0 + w;                      // input row r = j0 - 2 + q
        const int r = j0 - 2 + q;
        const bool has = q < rows, yrec = q >= 2 && has, yface = q >= 3 && has, fin = q >= 4 && has;
        // ---- 1. the stage input of row r
        S cC[3] = {S(0), S(0), S(0)}, cA[3], cB[3], x0[3];
        double b0 = 0.0, n0 = 0.0, bm = 0.0, nm = 0.0, bp = 0.0, np = 0.0;   // corner rows r, r-1, r-2 (columns i, i+1)
        if (has) {
            int sj = r;
            unsigned fyb = 0u;
            if (!rmp) {
            } else if (r < gc) { sj = P.src_lo_y[r]; fyb = P.flip_lo_y[r] ? 0x80000000u : 0u; }
            else if (r >= nyT - gc) { sj = P.src_hi_y[r - (nyT - gc)]; fyb = P.flip_hi_y[r - (nyT - gc)] ? 0x80000000u : 0u; }
            const size_t ro = (size_t)nxT * sj;
            S x[3];
            x[0] = row_ld(U0 + ro, nxT, sci); x[1] = row_ld(U0 + n + ro, nxT, sci);
            x[2] = row_ld(U0 + 2 * n + ro, nxT, sci);
            b0 = Bload_row(P, B, i, r);
            n0 = Bload_row(P, B, i + 1, r);
            bool ok = true;
            if (STAGE >= 2) {
                S rr[3];
                rr[0] = row_ld(RHS1 + ro, nxT, sci); rr[1] = row_ld(RHS1 + n + ro, nxT, sci);
                rr[2] = row_ld(RHS1 + 2 * n + ro, nxT, sci);
                if constexpr (STAGE == 3 && MODE == MODE_GENERAL) {
                    // a source that is a ghost has the non-directional sources only
                    if (P.ghost_self && in_dom && (sci >= nxT - gc || sj >= nyT - gc)) {
                        rr[0] = apply_sources(P, sl, S(0), (size_t)sci + ro);
                        rr[1] = rr[2] = S(0);
                    }
                }
                double c0 = b0, c1 = n0;
                if (xedge || sj != r) { c0 = Bload_row(P, B, sci, sj); c1 = Bload_row(P, B, sci + 1, sj); }
                const double c2 = Bload_row(P, B, sci, sj + 1), c3 = Bload_row(P, B, sci + 1, sj + 1);
                if (yrec) { bm = Bload_row(P, B, i, r - 1); nm = Bload_row(P, B, i + 1, r - 1); }
                if (fin) { bp = Bload_row(P, B, i, r - 2); np = Bload_row(P, B, i + 1, r - 2); }
                const double Bm = bc4(c0, c1, c2, c3);
                ok = stage1_any<S, MODE>(P, K, x, rr, Bm, b0, dt_d, dt_s, ranged, cC);
            } else {
                if (yrec) { bm = Bload_row(P, B, i, r - 1); nm = Bload_row(P, B, i + 1, r - 1); }
                if (fin) { bp = Bload_row(P, B, i, r - 2); np = Bload_row(P, B, i + 1, r - 2); }
                cC[0] = x[0]; cC[1] = x[1]; cC[2] = x[2];
            }
            cC[1] = flip_sign(cC[1], fx);
            cC[2] = flip_sign(cC[2], fyb);
            if (STAGE == 1) ok = __all(in_band((double)cC[0], (double)cC[1], (double)cC[2], b0));
            if constexpr (STAGE == 3 && MODE == MODE_GENERAL) {
                // ghosts on the high sides whose values live on in memory (gc = 2)
                const bool gx = in_dom && i >= nxT - gc && r >= j0 && r < j0 + th;
                const bool gy = out_col && r >= nyT - gc && j0 + th == nyT - gc;
                if (P.ghost_self && (gx || gy)) {
                    S* urow = UO + (size_t)nxT * r;
#pragma unroll
                    for (int v = 0; v < 3; ++v) row_st(urow + v * n, nxT, i, cC[v]);
                }
            }
            const int s = u_slot<BW>(w, par);
#pragma unroll
            for (int v = 0; v < 3; ++v) sm.u[s][v][lane] = cC[v];
            if (ranged && !ok && lane == 0) sm.bad = serial;
        }
        __syncthreads();
        const bool band = ranged && __builtin_amdgcn_readfirstlane(sm.bad) != serial;
        // ---- 2. y reconstruction of row m = r-1, x part of row p = r-2
        S Ly[3] = {S(0), S(0), S(0)}, Ry[3] = {S(0), S(0), S(0)};
        S accx[3] = {S(0), S(0), S(0)};
        double bcp = 0.0;
        const double Bly = 0.5 * (bm + nm);
        if (yrec) {
            const int sa = w >= 2 ? u_slot<BW>(w - 2, par) : u_slot<BW>(w - 2 + BW, par ^ 1);
            const int sb = w >= 1 ? u_slot<BW>(w - 1, par) : u_slot<BW>(BW - 1, par ^ 1);
#pragma unroll
            for (int v = 0; v < 3; ++v) { cA[v] = sm.u[sa][v][lane]; cB[v] = sm.u[sb][v][lane]; }
            if (rec_linear) {
                if (band) reconstruct_cell_rng(cA, cB, cC, K.theta2, Bly, 0.5 * (b0 + n0), Ly, Ry);
                else reconstruct_cell(cA, cB, cC, P.theta, Bly, 0.5 * (b0 + n0), Ly, Ry, MODE != 0);
            } else {
                const double bcm = bc4(bm, nm, b0, n0);
#pragma unroll
                for (int v = 0; v < 3; ++v) Ly[v] = Ry[v] = cB[v];
                Ly[0] = Ry[0] = (S)(cB[0] - bcm);
            }
            const int s = y_slot<BW>(w, par);
#pragma unroll
            for (int v = 0; v < 3; ++v) sm.ry[s][v][lane] = Ry[v];
            sm.ry[s][3][lane] = Ly[0];
            if (fin) {
                S Lx[3], Rx[3], Rxl[3];
                const double Blx = 0.5 * (bp + bm), Brx = 0.5 * (np + nm);
                bcp = bc4(bp, np, bm, nm);
                double Fxm[3];
                auto xpart = [&](auto rng_tag) {
                    constexpr bool RNG = decltype(rng_tag)::value;
                    if (rec_linear) {
                        S cl[3], cr[3];
#pragma unroll
                        for (int v = 0; v < 3; ++v) { cl[v] = (&sm.u[sa][v][lane])[-1]; cr[v] = (&sm.u[sa][v][lane])[1]; }
                        if (RNG) reconstruct_cell_rng(cl, cA, cr, K.theta2, Blx, Brx, Lx, Rx);
                        else reconstruct_cell(cl, cA, cr, P.theta, Blx, Brx, Lx, Rx, MODE != 0);
                    } else {
#pragma unroll
                        for (int v = 0; v < 3; ++v) Lx[v] = Rx[v] = cA[v];
                        Lx[0] = Rx[0] = (S)(cA[0] - bcp);
                    }
#pragma unroll
                    for (int v = 0; v < 3; ++v) Rxl[v] = shfl_up1(Rx[v]);
                    const double spx = RNG ? central_upwind_rng<0, MODE != 0>(Rxl, Lx, P.phys, K, Fxm)
                                           : central_upwind(0, Rxl, Lx, P.phys, Fxm);
                    if (STAGE == 1 || STAGE == 3) raise_speed<RNG>(smx, (double)(S)spx);
#pragma unroll
                    for (int v = 0; v < 3; ++v)
                        accx[v] = (S)__builtin_fma(-P.inv_dx, shfl_dn1(Fxm[v]) - Fxm[v], 0.0);   // 0 - inv*diff
                    if (P.bottom)
                        accx[1] = (S)(accx[1] + bottom_term<MODE, RNG>(P, K, 0, Brx - Blx, Rx[0] + Lx[0]));
                };
                if (band) xpart(std::true_type{});
                else xpart(std::false_type{});
            }
        }
        __syncthreads();
        // ---- 3. the y face between rows p and m
        double Fy[3] = {0.0, 0.0, 0.0};
        S Ryp[4];
        if (yface) {
            const int s = w >= 1 ? y_slot<BW>(w - 1, par) : y_slot<BW>(BW - 1, par ^ 1);
#pragma unroll
            for (int v = 0; v < 4; ++v) Ryp[v] = sm.ry[s][v][lane];
            const S Rlow[3] = {Ryp[0], Ryp[1], Ryp[2]};
            if (band) {
                const double spy = central_upwind_rng<1, MODE != 0>(Rlow, Ly, P.phys, K, Fy);
                if (STAGE == 1 || STAGE == 3) raise_speed<true>(smy, (double)(S)spy);
            } else {
                const double spy = central_upwind(1, Rlow, Ly, P.phys, Fy);
                if (STAGE == 1 || STAGE == 3) raise_speed<false>(smy, (double)(S)spy);
            }
            const int t = y_slot<BW>(w, par);
#pragma unroll
            for (int v = 0; v < 3; ++v) sm.fy[t][v][lane] = Fy[v];
            if (STAGE == 2 && fin) {               // U0 of row p, for the RK combination
                const size_t ro = (size_t)nxT * (r - 2);
#pragma unroll
                for (int v = 0; v < 3; ++v) x0[v] = row_ld(U0 + v * n + ro, nxT, i);
            }
        }
        __syncthreads();
        // ---- 4. finish row p
        if (fin && out_col) {
            const int p = r - 2;
            const int s = w >= 1 ? y_slot<BW>(w - 1, par) : y_slot<BW>(BW - 1, par ^ 1);
            const size_t k = (size_t)i + (size_t)nxT * p;
            S* orow = OUT + (size_t)nxT * p;
            auto finish = [&](auto rng_tag) {
                constexpr bool RNG = decltype(rng_tag)::value;
                S acc[3];
#pragma unroll
                for (int v = 0; v < 3; ++v) acc[v] = y_part<MODE, RNG>(P, accx[v], Fy[v] - sm.fy[s][v][lane]);
                if (P.bottom)
                    acc[2] = (S)(acc[2] + bottom_term<MODE, RNG>(P, K, 1, Bly - 0.5 * (bp + np), Ryp[0] + Ryp[3]));
                acc[0] = MODE ? uniform_sources<S>(P, rates, acc[0]) : apply_sources(P, rates, acc[0], k);
                if (STAGE != 2) {
#pragma unroll
                    for (int v = 0; v < 3; ++v) row_st(orow + v * n, nxT, i, acc[v]);
                    if (STAGE >= 3) {              // the new state
                        S* urow = UO + (size_t)nxT * p;
#pragma unroll
                        for (int v = 0; v < 3; ++v) row_st(urow + v * n, nxT, i, cA[v]);
                    }
                } else {
                    S o[3];
                    stage2_cell<S, MODE, RNG>(P, K, x0, cA, acc, bcp, dt_s, o);
#pragma unroll
                    for (int v = 0; v < 3; ++v) row_st(orow + v * n, nxT, i, o[v]);
                }
            };
            if (band) finish(std::true_type{});
            else finish(std::false_type{});
        }
    }
    if (STAGE == 1 || STAGE == 3) {
        smx = wave_max_u64(face_x_ok ? smx : 0ull);
        smy = wave_max_u64(out_col ? smy : 0ull);
        if (lane == 0) { sm.red[w][0] = smx; sm.red[w][1] = smy; }
        __syncthreads();
        if (threadIdx.x == 0) {
#pragma unroll
            for (int k = 1; k < BW; ++k) {
                smx = sm.red[k][0] > smx ? sm.red[k][0] : smx;
                smy = sm.red[k][1] > smy ? sm.red[k][1] : smy;
            }
            raise_wsmax(&ctl->slot[rslot], smx, smy);
        }
    }
}

// Grid of strips x segs workgroups in XCD-contiguous order, strips fastest.
template <class S, int STAGE, int MODE, int BW>
__global__ void __launch_bounds__(BL* BW) __attribute__((amdgpu_waves_per_eu(4)))
k_block(KParams P, StepCtl* ctl, int slot, int H, int strips, int segs, const S* __restrict__ U0,
        const S* __restrict__ RHS1, S* __restrict__ OUT, S* __restrict__ UO, const double* __restrict__ B, int remap,
        int close) {
    __shared__ BlockSmem<S, BW> sm;
    // stages 2 to 4: the last block closes, the others are tiles
    if (STAGE >= 2 && (int)blockIdx.x == strips * segs) {
        if (threadIdx.x < BL) close_stage<S, STAGE, MODE != 0>(P, ctl, slot, U0, STAGE >= 3 ? UO : OUT, B, close);
        return;
    }
    if (threadIdx.x == 0) sm.bad = 0;
    __syncthreads();
    const int t = xcd_tile(blockIdx.x, strips * segs);
    block_tile<S, STAGE, MODE, BW>(P, ctl, slot, H, t % strips, t / strips, U0, RHS1, OUT, UO, B, sm, 1, remap);
}

// Rows per workgroup: the smallest height at which every workgroup, the
// closing one of stages 2 to 4 included, has a CU of its own (0: the strips
// alone are more than the CUs).
static int block_height(const KParams& P) {
    static int cus = 0;
    static std::once_flag once;
    std::call_once(once, [] {
        int dev = 0, n = 0;
        if (hipGetDevice(&dev) == hipSuccess &&
            hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess)
            cus = n;
        if (cus <= 0) cus = 256;
    });
    const int strips = (P.nx + BCOLS - 1) / BCOLS;
    return strips >= cus ? 0 : (P.ny + (cus - 1) / strips - 1) / ((cus - 1) / strips);
}

// These kernels against the wave-march kernels, us per step (f64, same box):
// 64x48 15.1 and 22.1, 256^2 18.3 and 23.6, 420^2 22.8 and 28.0, 512^2 31 and 35,
// 700^2 (36 rows per workgroup) 46 and 44, 1024^2 86 and 74.  A workgroup's 6,
// 10 or 16 rows in flight beat a wave's one after the other until a CU's rows are
// more than about 24, the four-rows-in-flight limit per SIMD of either kernel.
// Near the limit the order depends on the grid more than on the type, options
// or stage (f64; f32 storage; general options; ForwardEuler, where the launch is
// stage 3): at 19 rows 30.5 and 34.6; 29.8 and 34.7; 32.0 and 37.4; 18.7 and 20.1;
// at 24 rows (600^2) 36.9 and 36.1; 38.5 and 36.3; 40.1 and 39.0; 21.0 and 20.6;
// at 27 rows (619x610) 37.1 and 41.1; 41.8 and 43.9; 43.0 and 46.1; 25.2 and 25.7,
// but (4000x80) 43.4 and 38.9; 41.9 and 38.7; 44.7 and 42.2; 25.1 and 23.4.
bool block_suits(const KParams& P) {
    const int H = block_height(P);
    return P.gc >= 2 && H > 0 && H <= BLOCK_MAX_ROWS;
}

// A chunk of BW rows takes about 9 + BW units of time (two launches of one
// chunk each: 15.0 us at 6 rows, 17.5 at 10, 22 at 16).  Three sizes, so that
// each stage and mode is built three times; sizes between were not measured.
template <class F>
static void by_waves(int H, F&& go) {
    int best = 6, cost = 1 << 30;
    for (int bw : {6, 10, 16}) {
        const int c = (H + 4 + bw - 1) / bw * (9 + bw);
        if (c < cost) { cost = c; best = bw; }
    }
    if (best == 6) go(std::integral_constant<int, 6>{});
    else if (best == 10) go(std::integral_constant<int, 10>{});
    else go(std::integral_constant<int, 16>{});
}

template <class S>
hipError_t launch_block(hipStream_t st, const KParams& P, StepCtl* ctl, int slot, int stage, const S* U0,
                        const S* RHS1, S* OUT, const double* B, int close, int remap_halo, S* UO) {
    if (stage > LAUNCH_STAGES<S>) return hipErrorInvalidValue;
    int H = block_height(P);
    if (H <= 0 || H > BLOCK_MAX_ROWS) H = BLOCK_MAX_ROWS;   // asked for on a larger grid: several rounds
    const int strips = (P.nx + BCOLS - 1) / BCOLS, segs = (P.ny + H - 1) / H;
    by_waves(H, [&](auto waves) {
        constexpr int BW = decltype(waves)::value;
        by_stage_mode<LAUNCH_STAGES<S>>(stage, stage == 3 && P.ghost_self ? MODE_GENERAL : march_mode(P), [&](auto stg, auto mode) {
            hipLaunchKernelGGL((k_block<S, decltype(stg)::value, decltype(mode)::value, BW>), dim3(strips * segs + (decltype(stg)::value >= 2 ? 1 : 0)),
                               dim3(BL * BW), 0, st, P, ctl, slot, H, strips, segs, U0, RHS1, OUT, UO, B, remap_halo,
                               close);
        });
    });
    return hipPeekAtLastError();
}
template hipError_t launch_block<double>(hipStream_t, const KParams&, StepCtl*, int, int, const double*,
                                         const double*, double*, const double*, int, int, double*);
template hipError_t launch_block<float>(hipStream_t, const KParams&, StepCtl*, int, int, const float*, const float*,
                                        float*, const double*, int, int, float*);

}  // namespace sfv
