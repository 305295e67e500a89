// jfa_walk.h -- what the stage kernels share: the face flux from a register window, the arguments of a
// stage's finish, and the walk over rows that evaluates two axes in one pass and finishes the stage
// (the FINAL kernel of jfa_fused.h, the batched 2-D kernel of jfa_batch.h).
#pragma once

#include "jfa_common.h"

namespace jfa {

// Face flux from a register window (cell k-h relative to the cell right of the face, k < n; 6 cells,
// 8 for WENO7-JS).
// CHAR-CONSERVATIVE also needs the primitives of the two cells adjacent to the face.
// CARRY: face_states' states shared by consecutive faces, in carry.  after_states runs once the
// window's lowest cell is no longer needed.
struct Nothing {
    __device__ __forceinline__ void operator()() const {}
};
template <class T, int AXIS, int VAR, int STENCIL, int RIEMANN, bool FLIM, bool CARRY = false, class After = Nothing>
__device__ __forceinline__ void window_flux(const double (&win)[Win<STENCIL>::n][5], const T* __restrict__ W,
                                            const T* __restrict__ U, int64_t b_right, int64_t sa, int64_t fs,
                                            const Params& prm, double F[5], double* carry = nullptr,
                                            After after_states = After()) {
    if constexpr (RIEMANN == kFluxSplit) {
        flux_split_face<AXIS, STENCIL>(win, prm, F);
        after_states();
    } else {
        double wl[5], wr[5];
        if constexpr (VAR == JFA_CHAR_CONSERVATIVE) {
#pragma unroll
            for (int i = 0; i < 5; ++i) {
                wl[i] = ld(W, i * fs + b_right - sa);
                wr[i] = ld(W, i * fs + b_right);
            }
        }
        double WL[5], WR[5], UL[5], UR[5];
        face_states<AXIS, VAR, STENCIL, CARRY>(win, wl, wr, prm, WL, WR, UL, UR, carry);
        after_states();
        if (prm.limiter) {
            double c[5];
#pragma unroll
            for (int i = 0; i < 5; ++i) c[i] = ld(W, i * fs + b_right - sa);
            limit_side<VAR>(c, prm, WL, UL);
#pragma unroll
            for (int i = 0; i < 5; ++i) c[i] = ld(W, i * fs + b_right);
            limit_side<VAR>(c, prm, WR, UR);
        }
        riemann<AXIS, RIEMANN, VAR == JFA_PRIMITIVE || VAR == JFA_CHAR_PRIMITIVE>(WL, WR, UL, UR, prm, F);
    }
    if constexpr (FLIM) {  // positivity flux limiter, with the step's dt (space_solver.py:530-541)
        double wl_[5], wr_[5], ul_[5], ur_[5];
#pragma unroll
        for (int i = 0; i < 5; ++i) {
            wl_[i] = ld(W, i * fs + b_right - sa);
            wr_[i] = ld(W, i * fs + b_right);
            ul_[i] = ld(U, i * fs + b_right - sa);
            ur_[i] = ld(U, i * fs + b_right);
        }
        const double dt = prm.dt_ptr ? *prm.dt_ptr : prm.dt_val;
        limit_flux<AXIS>(F, wl_, wr_, ul_, ur_, flux_lambda<AXIS>(prm, dt), prm);
    }
}

// The options most simulations run with, as constants: kernels compiled for them drop the run-time
// switches and the scalar registers these hold.
__device__ __forceinline__ Params common_options(Params p) {
    p.signal_speed = JFA_SS_EINFELDT;
    p.frozen = JFA_FROZEN_ARITHMETIC;
    p.limiter = 0;
    return p;
}
template <int VAR, int RIEMANN>
inline bool common_scheme(const Params& p) {
    return !p.limiter && (VAR == JFA_PRIMITIVE || p.frozen == JFA_FROZEN_ARITHMETIC) &&
           (RIEMANN == JFA_RUSANOV || p.signal_speed == JFA_SS_EINFELDT);
}

template <class T>
struct InnerArgs {
    const double* R;        // RHS of the previous sweeps (valid when accumulate)
    int accumulate;
    int mode;               // 0: write rhs to rhs_out; 1: finish the RK3 stage
    T* rhs_out;             // (5, N0, N1, N2) when mode 0
    const T* Uin;
    const T* Un;
    T* Wout;
    T* Uout;
    BC6 bc;
    int stage;
    const double* dt_dev;
    double dt_host;
    double* cfl_part;       // per-block partial max of the new state's wave speed, or null
};

// ------------------------------------------------------------------ FINAL kernel
// The last two sweeps of a stage and its finish in one pass (the common schemes, kFinal): along A,
// the last active axis below IN, and along IN.  It takes the place of MARCH<A> + INNER and with them
// of a write and two reads of the scratch RHS (a third of a 3-D stage's traffic; a 2-D stage needs no
// scratch RHS at all), and of every re-read of a face window through the caches.
//
// A wavefront holds 64 consecutive cells of rows along IN and walks along A.  Rows live in LDS, NW - 1
// of them in a ring (5 fields each): the A window of a lane is its own column of the ring, the IN
// window of the row that is finished is the row beside the lane's cell, so every cell is loaded from
// memory once (plus H rows per chunk).  How rows are cut:
//   packed = 0: each wave takes 64 cells of one row; five cells beside them are loaded as well, and
//     the flux above its last cell is evaluated for all rows of the chunk before the walk (lane k: row
//     a0 + k).  No lane idles where the row length is a multiple of 64.
//   packed = 1: rows of N + 6 positions (with the windows' halo cells) after one another; a wave takes
//     64 positions, of which the middle 58 have their whole window, and the next wave starts 58 on.
//     For ragged rows: a row of 80 cells keeps 84 % of the lanes, against 62 %.
// Loads run ahead: the finish's (scratch RHS, U, U_n) at the top of the row, two faces before their
// use; the next row's during the A face, once the reconstruction is done with the window.
//
// Bound: FP64 issue of two waves per SIMD (250 VGPRs; three spill) at the clock the card holds under it
// (58 % of the cycles issue; 1.97 GHz), 3.1 GB read and 1.6 GB written per stage at 256^3.
// Measured there (FP64, sustained, us per stage with the x sweep): CHAR-PRIMITIVE WENO5-Z HLLC 2000
// with MARCH + INNER, 1460 with this kernel (windows through the caches instead of LDS 1680, the
// finish's loads after the IN face 1490); PRIMITIVE WENO5-JS 1770 and 1425.  256 x 256: 22.8 and
// 12.9, 65 x 64 x 63: 64 and 47 us.
// The shared left states along A (CARRY) pay in CHAR-PRIMITIVE (1500 without); PRIMITIVE's five
// spill (1860 against 1415).
template <int VAR, int STENCIL, int RIEMANN, bool DISS, bool FLIM>
constexpr bool kFinal = kCarry<VAR, STENCIL> && (RIEMANN == JFA_HLLC || RIEMANN == JFA_RUSANOV) && !DISS && !FLIM;

// A wavefront's rows in LDS, a ring of window rows: H cells below its first cell, H - 1 above its last.
template <int STENCIL>
using WalkRows = double[Win<STENCIL>::n - 1][5][64 + Win<STENCIL>::n + 2];

// The walk of one wavefront: rows a0 .. a1 - 1 along A of its 64 cells along IN; lane l owns cell
// f of row io of axis O if vcell (io0: the wave's first row).  Aligned walks own cells f0 + lane of one
// row, packed ones 64 positions of rows with their halo cells.  Returns the lane's maximum of the new
// state's wave speeds.
template <class T, int A, int IN, int VAR, int STENCIL, int RIEMANN>
__device__ __forceinline__ double walk_rows(const T* __restrict__ W, const T* __restrict__ U, const Geo& G,
                                            const Params& prm, const InnerArgs<T>& args, bool packed, int io0, int io,
                                            int f0, int f, bool vcell, int a0, int a1, WalkRows<STENCIL>& rows,
                                            double (&top)[5][64]) {
    constexpr int O = 3 - A - IN;
    constexpr int NW = Win<STENCIL>::n, H = Win<STENCIL>::h;
    constexpr int RW = 64 + NW - 1;
    constexpr bool CARRY = VAR == JFA_CHAR_PRIMITIVE;
    const int lane = threadIdx.x & 63;
    const int N = G.n[IN];
    double vmax = 0.0;
    const int fc = f < N + H - 1 ? f : N + H - 1;  // columns past the row read its last halo cell
    const int64_t sa = G.s[A], fs = G.fs;
    // wave-uniform part of the buffer index: H cells below the first of row io0, coordinate 0 along A
    const int64_t brow = (int64_t)(io0 + G.off[O]) * G.s[O] + (int64_t)G.off[A] * sa + G.off[IN] - H;
    const int bl = (io - io0) * (int)G.s[O] + fc + H;  // the lane's part
    const uint32_t voff = (uint32_t)bl * (uint32_t)sizeof(T);
    // lanes 0 .. NW - 2 also hold the row's cells beside the wave's 64: H below, H - 1 above (the
    // other lanes repeat the last of them into the row's padding; packed waves do not read them)
    const int hl = lane < NW - 1 ? lane : NW - 2;
    const int fh = hl < H ? f0 - H + hl : f0 + 64 + hl - H;
    const uint32_t hoff = (uint32_t)((fh < N + H - 1 ? fh : N + H - 1) + H) * (uint32_t)sizeof(T);
    const int hpos = lane < H ? lane : (lane < NW - 1 ? 64 + lane : RW);
    const int64_t ncell = (int64_t)G.n[0] * G.n[1] * G.n[2];
    const int64_t rsA = A == 0 ? (int64_t)G.n[1] * G.n[2] : (int64_t)G.n[2];
    const int64_t rsO = O == 0 ? (int64_t)G.n[1] * G.n[2] : (O == 1 ? (int64_t)G.n[2] : 1);
    const int64_t r0 = (int64_t)io0 * rsO;
    const uint32_t roff = vcell ? (uint32_t)((io - io0) * (int)rsO + f) * (uint32_t)sizeof(double) : 0u;

    // upper face of the wave's last cell, for the row a0 + lane
    if (!packed && f0 + 64 <= N && lane < a1 - a0) {
        const int64_t b = brow + (int64_t)a0 * sa + f0 + 64 + H;
        const uint32_t v = (uint32_t)lane * (uint32_t)sa * (uint32_t)sizeof(T);
        double win[NW][5], Ft[5];
#pragma unroll
        for (int k = 0; k < NW; ++k)
#pragma unroll
            for (int i = 0; i < 5; ++i) win[k][i] = ldo(W + (i * fs + b + (k - H)), v);
        window_flux<T, IN, VAR, STENCIL, RIEMANN, false>(win, W, U, b + (int64_t)lane * sa, 1, fs, prm, Ft);
#pragma unroll
        for (int i = 0; i < 5; ++i) top[i][lane] = Ft[i];
    }
    double carry[5], Fp[5], nxt[5], hal[5];
    {
        double win[NW][5];
#pragma unroll
        for (int k = 0; k < NW; ++k)
#pragma unroll
            for (int i = 0; i < 5; ++i) win[k][i] = ldo(W + (i * fs + brow + (int64_t)(a0 - H + k) * sa), voff);
#pragma unroll
        for (int k = 0; k < NW - 1; ++k)
#pragma unroll
            for (int i = 0; i < 5; ++i) rows[k][i][H + lane] = win[k + 1][i];
#pragma unroll
        for (int k = H; k < NW; ++k)  // rows a0 .. a0 + H - 1
#pragma unroll
            for (int i = 0; i < 5; ++i)
                rows[k - 1][i][hpos] = ldo(W + (i * fs + brow + (int64_t)(a0 - H + k) * sa), hoff);
        if constexpr (CARRY) carry_start<A, VAR, STENCIL>(win, prm, carry);
        window_flux<T, A, VAR, STENCIL, RIEMANN, false, CARRY>(win, W, U, bl + brow + (int64_t)a0 * sa, sa, fs, prm,
                                                               Fp, carry);
    }
#pragma unroll
    for (int i = 0; i < 5; ++i) {
        nxt[i] = ldo(W + (i * fs + brow + (int64_t)(a0 + H) * sa), voff);
        hal[i] = ldo(W + (i * fs + brow + (int64_t)(a0 + H) * sa), hoff);
    }
    double c0, c1, m;
    rk3_coeffs(args.stage, c0, c1, m);
    const double ts = args.mode == 0 ? 0.0 : (args.dt_dev ? args.dt_dev[0] : args.dt_host) * m;  // RK3.py:60
    int slot = 0;  // ring position of row a - H + 1
    for (int a = a0; a < a1; ++a) {
        uint32_t vo = voff, ro = roff, ho = hoff;
        JFA_OPAQUE(vo);
        JFA_OPAQUE(ro);
        JFA_OPAQUE(ho);
        int64_t fso = fs;  // opaque: multiples of it are formed again, not kept in (spilled) scalar registers
        JFA_OPAQUE_S(fso);
        const int64_t rb = brow + (int64_t)a * sa;
        const int64_t rr0 = r0 + a * rsA;
        auto row = [&](int k) { return slot + k >= NW - 1 ? slot + k - (NW - 1) : slot + k; };
        // what the finish of this row needs from memory, two faces ahead
        double rr[5], ui[5], un[5];
#pragma unroll
        for (int i = 0; i < 5; ++i) {
            rr[i] = args.accumulate ? ldo(args.R + (i * ncell + rr0), ro) : 0.0;
            if (args.mode) {
                ui[i] = ldo(args.Uin + (i * fso + rb), vo);
                if (args.stage > 0) un[i] = ldo(args.Un + (i * fso + rb), vo);
            }
        }
        JFA_SCHED_BARRIER();
        JFA_WAVE_FENCE();
        double dz[5];
        {
            double zw[NW][5], Fz[5];
            const int q = row(H - 1);
#pragma unroll
            for (int k = 0; k < NW; ++k)
#pragma unroll
                for (int i = 0; i < 5; ++i) zw[k][i] = rows[q][i][lane + k];
            window_flux<T, IN, VAR, STENCIL, RIEMANN, false>(zw, W, U, bl + rb, 1, fs, prm, Fz);
#pragma unroll
            for (int i = 0; i < 5; ++i) {
                const double e = top[i][a - a0];
                const double up = __shfl_down(Fz[i], 1, 64);
                dz[i] = G.one_dx[IN] * (Fz[i] - (lane == 63 ? e : up));
            }
        }
        JFA_WAVE_FENCE();
        double Fn[5];
        {
            double win[NW][5];
#pragma unroll
            for (int k = 0; k < NW - 1; ++k) {
                const int q = row(k);
#pragma unroll
                for (int i = 0; i < 5; ++i) win[k][i] = rows[q][i][H + lane];
            }
#pragma unroll
            for (int i = 0; i < 5; ++i) win[NW - 1][i] = nxt[i];
            const int64_t nb = rb + (a + 1 < a1 ? H + 1 : H) * sa;
            window_flux<T, A, VAR, STENCIL, RIEMANN, false, CARRY>(
                win, W, U, bl + rb + sa, sa, fs, prm, Fn, carry, [&]() {
                    // the new row takes the place of the lowest; the next one is loaded ahead (the
                    // last step repeats its own)
#pragma unroll
                    for (int i = 0; i < 5; ++i) {
                        rows[slot][i][H + lane] = nxt[i];
                        rows[slot][i][hpos] = hal[i];
                        nxt[i] = ldo(W + (i * fso + nb), vo);
                        hal[i] = ldo(W + (i * fso + nb), ho);
                    }
                    JFA_SCHED_BARRIER();
                });
        }
        slot = slot == NW - 2 ? 0 : slot + 1;
        double rhs[5];
#pragma unroll
        for (int i = 0; i < 5; ++i) {
            rhs[i] = (rr[i] + G.one_dx[A] * (Fp[i] - Fn[i])) + dz[i];  // space_solver.py:314
            Fp[i] = Fn[i];
        }
        if (vcell) {
            if (args.mode == 0) {
#pragma unroll
                for (int i = 0; i < 5; ++i)
                    args.rhs_out[i * ncell + rr0 + (roff / (uint32_t)sizeof(double))] = static_cast<T>(rhs[i]);
            } else {
                double u[5], wn[5];
#pragma unroll
                for (int i = 0; i < 5; ++i) {
                    const double x = args.stage > 0 ? c0 * ui[i] + c1 * un[i] : ui[i];  // RK3.py:49-50
                    u[i] = x + ts * rhs[i];                                             // time_integrator.py:57
                }
                prim_from_cons(u, prm, wn);
#pragma unroll
                for (int i = 0; i < 5; ++i) {
                    sto(args.Wout + (i * fso + rb), vo, wn[i]);
                    sto(args.Uout + (i * fso + rb), vo, u[i]);
                }
                double uh[5];
                cons_from_prim(wn, prm, uh);
                int c[3];
                c[A] = a;
                c[O] = io;
                c[IN] = f;
                halo_scatter(args.Wout, args.Uout, G, args.bc, c, bl + rb, wn, uh, prm);
                if (args.cfl_part) vmax = nan_max(vmax, wave_sum(wn, G.active, prm.gamma));
            }
        }
    }
    return vmax;
}

}  // namespace jfa
