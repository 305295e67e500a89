// jfa_dissipative.h -- second-order central viscous and heat fluxes at one face, added to the
// convective face flux inside the fused sweeps (solvers/source_term_solver.py:188-350,414-448,
// 504-580; flux assembly space_solver.py:565-587).
//
// Face f along AXIS lies between the cells L = f-1 and R = f:
//   T_f  = (T_L + T_R)/2,  T = p/(rho R)                          (central_2, ideal_gas.py:81-83)
//   mu   = mu(T_f) (POWER or SUTHERLAND law),  mu2 = mu_b - 2/3 mu   (material.py:82-101, :527)
//   g[k][i] = d u_k / d x_i at the face: i == AXIS: (u_R - u_L)/dx (deriv_face_2);
//            i != AXIS: the central derivative (u(+e_i) - u(-e_i))/(2 dx_i) at L and at R
//            (deriv_center_2), averaged (central_2); inactive i: 0
//   tau_k = mu (g[AXIS][k] + g[k][AXIS]) (active k), tau_AXIS += mu2 sum_k g[k][k]
//   F[1+k] += -tau_k;  F[4] += -sum_k tau_k u_f,k + q,  q = -kappa(T_f) (T_R - T_L)/dx,
//   kappa = cp mu / Pr (PRANDTL) or its own POWER / SUTHERLAND law      (material.py:103-124)
// The two cells are those of the convective window.  On periodic domains their transverse neighbours wrap
// onto the interior (the edge halos there may be unwritten; they would be periodic copies); otherwise
// (prm.diss_halos) they are read from the buffer's face and edge halos, which the stage's halo scatter
// and edge-halo fill wrote.
#pragma once

#include "jfa_common.h"

namespace jfa {

// A series coefficient, with SCALAR in scalar registers and formed where it is used.  The compiler copies
// each into vector registers before its fma, or keeps them all in scalar registers around a loop and
// spills others for it: a viscous sweep takes 223 VGPRs so and 177 with SCALAR.  Where many faces stand
// in one block the asm keeps them from being interleaved: the reverse's cell kernel spills with SCALAR
// (128^3, us: 331 against 257).
template <bool SCALAR>
__device__ __forceinline__ double coef(double c) {
    if constexpr (!SCALAR) return c;
    long long bits = __double_as_longlong(c);
    JFA_OPAQUE_S(bits);
    return __longlong_as_double(bits);
}
// x^p as exp(p log x) with the logarithm in two doubles: log x = k ln 2 + log m, m in [sqrt(1/2), sqrt(2)),
// log m = 2 artanh(s), s = (m - 1)/(m + 1) (its series to s^27); exp by its series on half a binade, the first
// terms summed with their errors.  86 instructions against 226 for pow(x, p), which a viscous face
// otherwise spends a quarter of its time in (128^3 PRIMITIVE WENO5-Z HLLC, us per x sweep: 129 with pow
// and an index computation per neighbour, 109 with this and the neighbours as offsets).  Error against
// extended precision on the GPU, 4e5 values each of x in [e^-300, e^300] and p of -0.7 .. 3: below
// 0.57 ulp, mean 0.25 (pow: 1.33 and up to 0.35).
// Outside 0 < x < infinity as pow; SIGNED: x may be negative, which has a power only for a whole p (NaN
// otherwise, so a cell of negative temperature shows in the time step).  The faces' temperatures are
// clamped to positive ones: their power leaves that branch out (it costs 0.5 .. 2.7 % of a viscous stage).
constexpr double kLn2Hi = 0x1.62e42fefa0000p-1, kLn2Lo = 0x1.cf79abc9e3b3ap-40;

// x^p (p != 0) for x <= 0, an infinite x and NaN, where v = |x|^p if x is finite and not 0
__device__ __forceinline__ double power_special(double x, double p, double v) {
    const double h = 0.5 * p, a = fabs(x);
    const bool whole = rint(p) == p, odd = whole && rint(h) != h;
    double r = v;
    if (!(a > 0.0 && a < __builtin_inf())) r = p > 0.0 ? a : __builtin_amdgcn_rcp(a);  // 0, infinity, NaN
    else if (!whole) r = __builtin_nan("");
    return odd ? copysign(r, x) : r;
}

template <bool SCALAR, bool SIGNED>
__device__ __forceinline__ double power(double x, double p) {
#pragma clang fp contract(off)
    int k;
    double m = frexp(SIGNED ? fabs(x) : x, &k);
    const bool low = m < 0.70710678118654757;
    m = low ? m + m : m;
    k = low ? k - 1 : k;
    const double f = m - 1.0, d = m + 1.0, dl = m - (d - 1.0);
    const double r = rcp(d);
    const double s = f * r;
    const double sl = r * fma(-s, dl, fma(-s, d, f));
    const double z = s * s;
    double P = coef<SCALAR>(1.0 / 27.0);
    P = fma(P, z, coef<SCALAR>(1.0 / 25.0));
    P = fma(P, z, coef<SCALAR>(1.0 / 23.0));
    P = fma(P, z, coef<SCALAR>(1.0 / 21.0));
    P = fma(P, z, coef<SCALAR>(1.0 / 19.0));
    P = fma(P, z, coef<SCALAR>(1.0 / 17.0));
    P = fma(P, z, coef<SCALAR>(1.0 / 15.0));
    P = fma(P, z, coef<SCALAR>(1.0 / 13.0));
    P = fma(P, z, coef<SCALAR>(1.0 / 11.0));
    P = fma(P, z, coef<SCALAR>(1.0 / 9.0));
    P = fma(P, z, coef<SCALAR>(1.0 / 7.0));
    P = fma(P, z, coef<SCALAR>(1.0 / 5.0));
    P = fma(P, z, coef<SCALAR>(1.0 / 3.0));
    const double t = s * (z * P);
    const double n1 = (double)k;
    const double A = n1 * kLn2Hi, S = s + s;
    const double h0 = A + S;
    const double l0 = (S - (h0 - A)) + fma(n1, kLn2Lo, 2.0 * (sl + t));
    const double h = h0 + l0;
    const double y = p * h;
    const double yl = fma(p, l0 - (h - h0), fma(p, h, -y));
    const double n2 = rint(y * 1.4426950408889634);
    const double q0 = fma(-n2, kLn2Hi, y);
    const double qr = fma(-n2, kLn2Lo, yl);
    const double q = q0 + qr, ql = qr - (q - q0);
    double E = coef<SCALAR>(1.0 / 87178291200.0);
    E = fma(E, q, coef<SCALAR>(1.0 / 6227020800.0));
    E = fma(E, q, coef<SCALAR>(1.0 / 479001600.0));
    E = fma(E, q, coef<SCALAR>(1.0 / 39916800.0));
    E = fma(E, q, coef<SCALAR>(1.0 / 3628800.0));
    E = fma(E, q, coef<SCALAR>(1.0 / 362880.0));
    E = fma(E, q, coef<SCALAR>(1.0 / 40320.0));
    E = fma(E, q, coef<SCALAR>(1.0 / 5040.0));
    E = fma(E, q, coef<SCALAR>(1.0 / 720.0));
    E = fma(E, q, coef<SCALAR>(1.0 / 120.0));
    E = fma(E, q, coef<SCALAR>(1.0 / 24.0));
    E = fma(E, q, coef<SCALAR>(1.0 / 6.0));
    const double hq = 0.5 * q, b = hq * q, be = fma(hq, q, -b);
    const double u = q + b, w = 1.0 + u;
    const double c = fma(b * q, E + E, fma(q, ql, ql) + be);
    const double v = ldexp(w + ((u - (w - 1.0)) + ((b - (u - q)) + c)), (int)n2);
    const bool finite = x > 0.0 && x < __builtin_inf();
    if constexpr (SIGNED) {
        if (!finite) return power_special(x, p, v);
        return v;
    } else {
        return finite ? v : (p > 0.0 ? x : __builtin_amdgcn_rcp(x));  // 0, infinity, NaN
    }
}

template <bool SCALAR = false, bool SIGNED = false>
__device__ __forceinline__ double law_value(double T, const Law& l) {
    if (l.kind == JFA_LAW_SUTHERLAND) {  // material.py:94-96, power3_2 (math/power_functions.py:29-30)
        const double x = T * l.inv_T_ref;
        return l.ref * ((l.T_ref + l.param) / (T + l.param)) * (x * sqrt(x));
    }
    return l.param == 0.0 ? l.ref : l.ref * power<SCALAR, SIGNED>(T * l.inv_T_ref, l.param);
}

template <bool SCALAR = false, bool SIGNED = false>
__device__ __forceinline__ double viscosity(double T, const Params& prm) {
    return law_value<SCALAR, SIGNED>(T, prm.mu);
}

// thermal conductivity at temperature T, where mu = viscosity(T)
template <bool SCALAR = false, bool SIGNED = false>
__device__ __forceinline__ double conductivity(double T, double mu, const Params& prm) {
    return prm.kappa.kind == JFA_LAW_PRANDTL ? prm.kappa_fac * mu : law_value<SCALAR, SIGNED>(T, prm.kappa);
}

// Offsets from a cell at coordinate c along axis i to its neighbours above and below: on periodic
// domains they wrap onto [0, n), otherwise (halos) the neighbours past the ends are halo cells.
__device__ __forceinline__ int64_t offset_up(const Geo& G, int i, int c, int halos) {
    return !halos && c == G.n[i] - 1 ? (1 - (int64_t)G.n[i]) * G.s[i] : G.s[i];
}
__device__ __forceinline__ int64_t offset_down(const Geo& G, int i, int c, int halos) {
    return !halos && c == 0 ? ((int64_t)G.n[i] - 1) * G.s[i] : -G.s[i];
}

// buffer index of the interior cell c
__device__ __forceinline__ int64_t cell_index(const Geo& G, const int c[3]) {
    return (int64_t)(c[0] + G.off[0]) * G.s[0] + (int64_t)(c[1] + G.off[1]) * G.s[1] +
           (int64_t)(c[2] + G.off[2]) * G.s[2];
}

template <class T>
__device__ __forceinline__ void load_velocity(const T* __restrict__ W, int64_t fs, int64_t b, double u[3]) {
#pragma unroll
    for (int k = 0; k < 3; ++k) u[k] = ld(W, (k + 1) * fs + b);
}

// Face state of the dissipative flux: the two cells' primitives, their temperatures, the face
// temperature (clamped: T_f <= 0 replaced by the precision eps), the viscosity there and, for
// viscous fluxes, the velocity-gradient tensor g[k][i] = d u_k / d x_i at the face.
struct DissState {
    double wl[5], wr[5];
    double TL, TR, Tf;
    bool clamped;
    double mu;
    double g[3][3];
};

// temperature of a cell (ideal_gas.py:81-83)
__device__ __forceinline__ double temperature(const double w[5], const Params& prm) {
    return w[4] / (w[0] * prm.R);
}

// central derivative of the velocity along axis i at cell b, from its neighbours at the given offsets
template <class T>
__device__ __forceinline__ void velocity_derivative(const T* __restrict__ W, const Geo& G, int i, int64_t b, int64_t up,
                                                    int64_t down, double d[3]) {
    double u[3], v[3];
    load_velocity(W, G.fs, b + up, u);
    load_velocity(W, G.fs, b + down, v);
#pragma unroll
    for (int k = 0; k < 3; ++k) d[k] = (u[k] - v[k]) * (0.5 * G.one_dx[i]);
}

// Face state along AXIS between two cells given by their primitives, temperatures and transverse velocity
// derivatives d[i][k] = d u_k / d x_i (i != AXIS; read with viscous fluxes only).
template <int AXIS, bool SCALAR = false>
__device__ __forceinline__ void dissipative_state_between(const Geo& G, const Params& prm, const double wl[5],
                                                          double TL, const double (&dl)[3][3], const double wr[5],
                                                          double TR, const double (&dr)[3][3], DissState& s) {
#pragma unroll
    for (int i = 0; i < 5; ++i) {
        s.wl[i] = wl[i];
        s.wr[i] = wr[i];
    }
    s.TL = TL;
    s.TR = TR;
    s.Tf = 0.5 * (s.TL + s.TR);
    s.clamped = s.Tf <= 0.0;
    if (s.clamped) s.Tf = 2.220446049250313e-16;  // source_term_solver.py:301 (precision eps)
    s.mu = viscosity<SCALAR>(s.Tf, prm);
    if (!(prm.dissip & 1)) return;
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            if (!G.active[i]) s.g[k][i] = 0.0;
            else if (i == AXIS) s.g[k][i] = (s.wr[1 + k] - s.wl[1 + k]) * G.one_dx[i];
            else s.g[k][i] = 0.5 * (dl[i][k] + dr[i][k]);
        }
}

// Transverse velocity derivatives d[i][k], i != AXIS, at cell b, whose coordinates across AXIS are c's.
template <class T, int AXIS>
__device__ __forceinline__ void transverse_derivatives(const T* __restrict__ W, const Geo& G, const Params& prm,
                                                       const int c[3], int64_t b, double (&d)[3][3]) {
    if (!(prm.dissip & 1)) return;
#pragma unroll
    for (int i = 0; i < 3; ++i)
        if (i != AXIS && G.active[i])
            velocity_derivative(W, G, i, b, offset_up(G, i, c[i], prm.diss_halos), offset_down(G, i, c[i], prm.diss_halos),
                                d[i]);
}

// Buffer indices of the cells beside the face whose right cell is cr; faces 0 and n of a periodic domain
// lie between the same two cells.
template <int AXIS>
__device__ __forceinline__ void face_cells(const Geo& G, const Params& prm, const int cr[3], int64_t& bl, int64_t& br) {
    br = cell_index(G, cr);
    bl = br - G.s[AXIS];
    if (!prm.diss_halos) {
        const int64_t row = (int64_t)G.n[AXIS] * G.s[AXIS];
        if (cr[AXIS] == 0) bl += row;
        if (cr[AXIS] == G.n[AXIS]) br -= row;
    }
}

// adds the dissipative flux of a face state to F
template <int AXIS, bool SCALAR = false>
__device__ __forceinline__ void dissipative_flux(const DissState& s, const Geo& G, const Params& prm, double F[5]) {
    double d4 = 0.0;
    if (prm.dissip & 1) {
        const double mu2 = prm.bulk - 2.0 / 3.0 * s.mu;
        double tau[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) tau[k] = G.active[k] ? s.mu * (s.g[AXIS][k] + s.g[k][AXIS]) : 0.0;
        double div = 0.0;
#pragma unroll
        for (int k = 0; k < 3; ++k)
            if (G.active[k]) div = div + s.g[k][k];
        tau[AXIS] = tau[AXIS] + mu2 * div;
        double vel_tau = 0.0;
#pragma unroll
        for (int k = 0; k < 3; ++k)
            if (G.active[k]) vel_tau = vel_tau + tau[k] * (0.5 * (s.wl[1 + k] + s.wr[1 + k]));
#pragma unroll
        for (int k = 0; k < 3; ++k) F[1 + k] = F[1 + k] + (-tau[k]);
        d4 = -vel_tau;
    }
    if (prm.dissip & 2) d4 = d4 + (-conductivity<SCALAR>(s.Tf, s.mu, prm) * ((s.TR - s.TL) * G.one_dx[AXIS]));
    F[4] = F[4] + d4;
}

// adds the dissipative flux of the face whose right cell has interior coordinates cr and whose cells hold
// the primitives wl, wr to F
template <class T, int AXIS>
__device__ __forceinline__ void dissipative_face(const T* __restrict__ W, const Geo& G, const Params& prm,
                                                 const int cr[3], const double wl[5], const double wr[5], double F[5]) {
    int64_t bl, br;
    face_cells<AXIS>(G, prm, cr, bl, br);
    double dl[3][3], dr[3][3];
    transverse_derivatives<T, AXIS>(W, G, prm, cr, bl, dl);
    transverse_derivatives<T, AXIS>(W, G, prm, cr, br, dr);
    DissState s;
    dissipative_state_between<AXIS, true>(G, prm, wl, temperature(wl, prm), dl, wr, temperature(wr, prm), dr, s);
    dissipative_flux<AXIS, true>(s, G, prm, F);
}

// cell diffusivities for the time-step limits: nu = mu/rho, alpha = kappa/(rho cp)
__device__ __forceinline__ void diffusivities(const double w[5], const Params& prm, double& nu, double& alpha) {
    const double T = w[4] / (w[0] * prm.R);
    const double mu = viscosity<true, true>(T, prm);
    nu = (prm.dissip & 1) ? mu / w[0] : 0.0;
    alpha = (prm.dissip & 2) ? conductivity<true, true>(T, mu, prm) / w[0] * prm.inv_cp : 0.0;
}

}  // namespace jfa
