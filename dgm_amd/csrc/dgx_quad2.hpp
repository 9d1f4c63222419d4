// One stage of an affine 2D domain in one pass over its elements: residual,
// register update and the face traces of the new state.
//
// One wavefront owns EPW elements (one, or quad_epw on large meshes of low
// order); every phase after the loads is a batch of pencils over LDS tensors
// of all fields of all its elements.  The kernel is bound by latency, the
// chain of dependent loads and LDS phases of its few wavefronts per SIMD, not
// by bandwidth (a stage of 64^2 quads at p = 5 moves 25 MB).  Hence: a side's
// neighbour, side and orientation come in one word (Geo::link2), so its traces
// are two loads away; the links, the state and the update's inputs are all
// issued before the first LDS phase; the state stays in registers for the
// update; and the new state's traces are taken from LDS in the same pass, so
// that a stage of any integrator is one launch.  A stage of 32^2 quads at
// p = 4 under RK4 went from 13.4 us (traces, residual and two or three flat
// updates) to 4.1 us, the acoustic adjoint's stages at 64^2, p = 5 from 19 to
// 12 us.
#pragma once
#include "dgx_kernels.hpp"

namespace dgx {

template <int P, int NF, int EPW> struct Q2S {
  static constexpr int L = P + 1, Q = P + 2, QF = P + 1, L2 = L * L, Q2 = Q * Q, NT = 64;
  static constexpr int EF = EPW * NF;                    // fields of the wavefront's elements
  static constexpr int NM = EF * L2, NX = EF * Q * L, NN = EF * Q2, NFP = EPW * 4 * QF;
  static constexpr int NU = (NM + NT - 1) / NT;          // modal entries per lane
  static constexpr int NPT = (EPW * Q2 + NT - 1) / NT;   // nodes per lane
  // M [EF][L2] modal; X1, X2 [EF][Q][L]; N1, N2 [EF][Q2] nodal state, fluxes
  // (N1 later the traces' end values [EF][4][L]); gF [EF][4][QF]; H [EF][4][L]
  static constexpr int size = NM + 2 * NX + 2 * NN + EF * 4 * QF + EF * 4 * L;
  static constexpr int traces = NM + EF * 4 * L;         // of which the traces alone need M and the end values
  static_assert(NFP <= NT, "one face point per lane");
  static_assert(4 * L <= Q2, "the end values fit in N1");
};

// Physics of a stage.  flux: Cartesian fluxes of a nodal state; face: the
// correction Fhat - F(U-).n of a face point; ghost: the state beyond a
// boundary side.
struct QuadEuler {
  static constexpr int NF = 4;
  static constexpr bool scaled = false;
  const Phys &ph;
  __device__ __forceinline__ void flux(const double *U, double *fx, double *fy) const {
    const double r = U[0], ru = U[1], rv = U[2], rE = U[3];
    const double ir = 1.0 / r, u = ru * ir, vv = rv * ir;
    const double p = (ph.gamma - 1.0) * (rE - 0.5 * (ru * u + rv * vv)), h = rE + p;
    fx[0] = ru; fx[1] = ru * u + p; fx[2] = rv * u; fx[3] = u * h;
    fy[0] = rv; fy[1] = ru * vv; fy[2] = rv * vv + p; fy[3] = vv * h;
  }
  __device__ __forceinline__ void face(const double *UL, const double *UR, double nx, double ny, double *g,
                                       bool &bad) const {
    double FL[4], FR[4], Fh[4], lL, lR;
    bool bl, br;
    euler_normal_flux2(UL, nx, ny, ph.gamma - 1.0, FL, lL, bl);
    euler_normal_flux2(UR, nx, ny, ph.gamma - 1.0, FR, lR, br);
    bad |= bl | br;
    if (ph.flux == 1) {
      roe_flux2(UL, UR, nx, ny, ph.gamma, FL, Fh);
    } else {
      const double lmax = fmax(lL, lR);
#pragma unroll
      for (int v = 0; v < 4; ++v) Fh[v] = 0.5 * (FL[v] + FR[v] + lmax * (UL[v] - UR[v]));
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) g[v] = Fh[v] - FL[v];
  }
  __device__ __forceinline__ void ghost(int bc, const double *UL, double nx, double ny, double *UR) const {
    ghost2(bc, UL, nx, ny, ph.bcU, UR);
  }
};

// Shallow water (Shallow::time_derivative, src/Shallow.cpp:255-336).
struct QuadShallow {
  static constexpr int NF = 3;
  static constexpr bool scaled = false;
  const Phys &ph;
  __device__ __forceinline__ void flux(const double *U, double *fx, double *fy) const {
    const double phi = U[0], mx = U[1], my = U[2];
    const double u = mx / phi, vv = my / phi, p = 0.5 * (phi * phi);
    fx[0] = mx; fx[1] = mx * u + p; fx[2] = my * u;
    fy[0] = my; fy[1] = mx * vv; fy[2] = my * vv + p;
  }
  __device__ __forceinline__ void face(const double *UL, const double *UR, double nx, double ny, double *g,
                                       bool &bad) const {
    double FL[3], FR[3], lL, lR;
    bad |= shallow_normal_flux2(UL, nx, ny, FL, lL);
    bad |= shallow_normal_flux2(UR, nx, ny, FR, lR);
    const double lmax = fmax(lL, lR);
#pragma unroll
    for (int v = 0; v < 3; ++v) g[v] = 0.5 * (FL[v] + FR[v] + lmax * (UL[v] - UR[v])) - FL[v];
  }
  __device__ __forceinline__ void ghost(int bc, const double *UL, double nx, double ny, double *UR) const {
    ghost_shallow2(bc, UL, nx, ny, ph.bcU, UR);
  }
};

// A linear system with constant Jacobians Ax, Ay and the Lax-Friedrichs speed
// |u0 nx + v0 ny| + c0.  SC: the state is scaled by 1 / J of its element (the
// adjoint system acts on V / J).
template <bool SC> struct QuadLinear {
  static constexpr int NF = 4;
  static constexpr bool scaled = SC;
  const LinArgs &a;
  __device__ __forceinline__ void flux(const double *U, double *fx, double *fy) const {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      double sx = 0.0, sy = 0.0;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        sx = fma(a.Ax[4 * v + j], U[j], sx);
        sy = fma(a.Ay[4 * v + j], U[j], sy);
      }
      fx[v] = sx; fy[v] = sy;
    }
  }
  __device__ __forceinline__ void face(const double *UL, const double *UR, double nx, double ny, double *g,
                                       bool &) const {
    const double lam = fabs(a.u0 * nx + a.v0 * ny) + a.c0;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      double fl = 0.0, fr = 0.0;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const double An = nx * a.Ax[4 * v + j] + ny * a.Ay[4 * v + j];
        fl = fma(An, UL[j], fl);
        fr = fma(An, UR[j], fr);
      }
      g[v] = 0.5 * (fl + fr + lam * (UL[v] - UR[v])) - fl;
    }
  }
  __device__ __forceinline__ void ghost(int, const double *, double, double, double *) const {}   // periodic meshes
};

// What a stage does with its residual r: x is the stage's own state, pre the
// inputs loaded with it; returns the state whose traces the stage writes.
struct QuadUpdate {
  static constexpr int NPRE = 2;
  StageStep s;
  __device__ __forceinline__ void pre(size_t o, int, int, double *p) const {
    p[0] = stage_reads_acc(s.mode) ? s.acc[o] : 0.0;
    p[1] = s.mode >= ST_RK4_MID ? s.base[o] : 0.0;
  }
  __device__ __forceinline__ double post(size_t o, int, int, int, double r, double x, const double *p) const {
    return stage_update(s, o, r, x, p[0], p[1]);
  }
};

// Shallow water's balance term (src/Shallow.cpp:251-266) before the update:
// bal 1 stores the residual and returns R - R, bal 2 returns R - Bal.
struct QuadBalanced {
  static constexpr int NPRE = 2;
  QuadUpdate u;
  double *Bal;
  int bal;
  __device__ __forceinline__ void pre(size_t o, int e, int v, double *p) const { u.pre(o, e, v, p); }
  __device__ __forceinline__ double post(size_t o, int e, int v, int m, double r, double x, const double *p) const {
    if (bal) {
      double b = r;
      if (bal == 1) Bal[o] = r;
      else b = Bal[o];
      r = -1.0 * b + r;
    }
    return u.post(o, e, v, m, r, x, p);
  }
};

// The linear system's LSRK stage with the source theta g(t) in the energy
// equation, and one reversed stage of its discrete adjoint: the state's
// adjoint Y -= dt J Fadj(X / J), the source gradient, then the register's next
// value ca X, to which the next reversed stage's Bn Y is added when it
// follows at once (bn).
struct LinearForward {
  static constexpr int NPRE = 1;
  const LinArgs &a;
  __device__ __forceinline__ void pre(size_t o, int, int, double *p) const { p[0] = a.Yt[o]; }
  __device__ __forceinline__ double post(size_t o, int e, int v, int m, double r, double x, const double *p) const {
    if (v == 3 && m == 0) r -= 2.0 * a.theta[e] * a.g;   // source: mode 0 of the constant theta_e
    const double ut = a.ca * p[0] - a.dt * r, y = fma(a.cb, ut, x);
    a.Yt[o] = ut;
    a.Y[o] = y;
    return y;
  }
};
struct LinearAdjoint {
  static constexpr int NPRE = 2;
  const LinArgs &a;
  __device__ __forceinline__ void pre(size_t o, int e, int, double *p) const {
    const double *m = a.geo.metric + 9 * (size_t)e;
    p[0] = a.Y[o];
    p[1] = m[0] * m[4] - m[1] * m[3];   // 1 / J_e
  }
  __device__ __forceinline__ double post(size_t o, int e, int v, int m, double r, double x, const double *p) const {
    const double y = fma(-a.dt, r / p[1], p[0]);
    a.Y[o] = y;
    if (v == 3 && m == 0) a.gtheta[e] += 2.0 * a.g * a.dt * x;
    double xt = a.ca * x;
    if (a.Tn) xt = fma(a.bn, y, xt);
    a.Yt[o] = xt;
    return xt;
  }
};

// y = M x of one pencil, for the two forms of a table: even-odd, or the plain
// rows M [NO][NI] with sums in ascending order.
template <int K, int NI, int NO, typename T>
__device__ __forceinline__ void table_apply(EoMat<K, T> M, const T (&x)[NI], T (&y)[NO]) {
  eo_apply<K, NI, NO>(M.h, x, y);
}
template <int NI, int NO, typename T>
__device__ __forceinline__ void table_apply(const T *__restrict__ M, const T (&x)[NI], T (&y)[NO]) {
#pragma unroll
  for (int o = 0; o < NO; ++o) {
    T s = 0;
#pragma unroll
    for (int i = 0; i < NI; ++i) s = fma(M[o * NI + i], x[i], s);
    y[o] = s;
  }
}
// the full rows of a table whose even-odd form holds them (EO_MN), or of a plain one
template <typename T> __device__ __forceinline__ const T *table_rows(EoMat<EO_MN, T> M) { return M.h; }
template <typename T> __device__ __forceinline__ const T *table_rows(const T *M) { return M; }

// The state's end values [EF][4][L] on the four edges from M, then its values
// at their Gauss points, into T of elements e0 .. (those below ne).
template <int P, int NF, int EPW, typename R, class TE>
__device__ __forceinline__ void quad_traces(const R *M, R *K, double *__restrict__ T, int e0, int ne, int tid) {
  using S = Q2S<P, NF, EPW>;
  constexpr int L = S::L, QF = S::QF, EF = S::EF, NT = S::NT;
  R *Kb = K, *Ka = K + 2 * EF * L;
  contract<EF, L, L, 2, 2, NT>(TE::Bend(), M, Kb, tid);   // [EF][L][2]
  contract<EF, L, L, 1, 2, NT>(TE::Bend(), M, Ka, tid);   // [EF][2][L]
  __syncthreads();
  double *Te = T + (size_t)e0 * 4 * NF * QF;
  for (int pc = tid; pc < 4 * EF; pc += NT) {
    const int el = pc / (4 * NF), s = (pc / NF) & 3, f = el * NF + pc % NF;
    const R *k = (s & 1) ? Ka + (f * 2 + (s == 1)) * L : Kb + f * L * 2 + (s == 2);
    const int st = (s & 1) ? 1 : 2;
    R x[L], y[QF];
#pragma unroll
    for (int l = 0; l < L; ++l) x[l] = k[l * st];
    table_apply(TE::Bg(), x, y);
    if (e0 + el < ne) {
#pragma unroll
      for (int q = 0; q < QF; ++q) Te[pc * QF + q] = y[q];
    }
  }
}

// One stage of elements e0 .. e0 + EPW - 1 (those below ne).  X modal state and
// T its traces; NS: V, TV the BR1 viscous terms; Tn: if set, the traces of the
// state `up` returns.  sm: Q2S::size values of LDS.
template <int P, int EPW, typename R, class TE, bool NS, class PH, class UP>
__device__ __forceinline__ void quad_stage(const double *X, const double *__restrict__ T,
                                           const double *__restrict__ V, const double *__restrict__ TV,
                                           const Geo &geo, int ne, int e0, int *__restrict__ flag, const PH &ph,
                                           const UP &up, double *__restrict__ Tn, R *sm) {
  constexpr int NF = PH::NF;
  using S = Q2S<P, NF, EPW>;
  constexpr int L = S::L, Q = S::Q, QF = S::QF, L2 = S::L2, Q2 = S::Q2, NT = S::NT, EF = S::EF;
  R *M = sm, *X1 = M + S::NM, *X2 = X1 + S::NX, *N1 = X2 + S::NX, *N2 = N1 + S::NN, *gF = N2 + S::NN,
    *H = gF + EF * 4 * QF;
  const int tid = threadIdx.x;
  // the lane's face point: side s, Gauss point a of element fe
  const bool fp = tid < S::NFP;
  const int fel = fp ? tid / (4 * QF) : 0, fsd = fp ? (tid / QF) & 3 : 0, fa = fp ? tid % QF : 0;
  const int fe = min(e0 + fel, ne - 1), es = fe * 4 + fsd;
  const int link = geo.link2[es];
  const double nx = geo.fnorm[3 * es], ny = geo.fnorm[3 * es + 1], jr = geo.fjr[es];
  // the state and the update's inputs
  double x[S::NU], pre[S::NU][UP::NPRE], vv[NS ? S::NU : 1];
#pragma unroll
  for (int k = 0; k < S::NU; ++k) {
    const int i = tid + k * NT, el = i / (NF * L2), r = i - el * NF * L2, v = r / L2;
    const size_t o = ((size_t)v * ne + min(e0 + el, ne - 1)) * L2 + (r - v * L2);
    x[k] = i < S::NM ? X[o] : 0.0;
  }
  // the face traces of both sides
  double UL[NF], UR[NF], gv[NS ? NF - 1 : 1];
  {
    const double *tl = T + (size_t)es * NF * QF + fa;
#pragma unroll
    for (int v = 0; v < NF; ++v) UL[v] = tl[v * QF];
    const int ns = link < 0 ? es : link >> 1, an = (link >= 0 && (link & 1)) ? QF - 1 - fa : fa;
    const double *tr = T + (size_t)ns * NF * QF + an;
#pragma unroll
    for (int v = 0; v < NF; ++v) UR[v] = tr[v * QF];
    if constexpr (NS) {
      const double *vl = TV + (size_t)es * (NF - 1) * QF + fa, *vr = TV + (size_t)ns * (NF - 1) * QF + an;
#pragma unroll
      for (int v = 0; v < NF - 1; ++v) gv[v] = link >= 0 ? vl[v * QF] + vr[v * QF] : 0.0;
    }
    if constexpr (PH::scaled) {
      auto inv = [&](int e) {
        const double *m = geo.metric + 9 * (size_t)e;
        return m[0] * m[4] - m[1] * m[3];
      };
      const double sl = inv(fe), sr = inv(ns >> 2);
#pragma unroll
      for (int v = 0; v < NF; ++v) { UL[v] *= sl; UR[v] *= sr; }
    }
  }
  // the lane's nodes and their elements' metric terms
  double mt[S::NPT][4];
#pragma unroll
  for (int r = 0; r < S::NPT; ++r) {
    const int k = tid + r * NT;
    const double *m = geo.metric + 9 * (size_t)min(e0 + k / Q2, ne - 1);
    mt[r][0] = m[0]; mt[r][1] = m[1]; mt[r][2] = m[3]; mt[r][3] = m[4];
  }
#pragma unroll
  for (int k = 0; k < S::NU; ++k) {
    const int i = tid + k * NT, el = i / (NF * L2), r = i - el * NF * L2, v = r / L2, m = r - v * L2;
    const int e = min(e0 + el, ne - 1);
    const size_t o = ((size_t)v * ne + e) * L2 + m;
    if (i < S::NM) up.pre(o, e, v, pre[k]);
    if constexpr (NS) vv[k] = (i < S::NM && v > 0) ? V[((size_t)e * (NF - 1) + (v - 1)) * L2 + m] : 0.0;
  }
  // modes -> nodes
#pragma unroll
  for (int k = 0; k < S::NU; ++k)
    if (tid + k * NT < S::NM) M[tid + k * NT] = (R)x[k];
  __syncthreads();
  contract<EF, L, L, 1, Q, NT>(TE::BT(), M, X1, tid);
  __syncthreads();
  contract<EF, Q, L, 2, Q, NT>(TE::BT(), X1, N1, tid);
  __syncthreads();
  double un[S::NPT][NF];
#pragma unroll
  for (int r = 0; r < S::NPT; ++r) {
    const int k = tid + r * NT, el = k / Q2, n = k - el * Q2;
#pragma unroll
    for (int v = 0; v < NF; ++v) un[r][v] = k < EPW * Q2 ? (double)N1[(el * NF + v) * Q2 + n] : 1.0;
  }
  // face corrections g = J_side/J_vol (Fhat - F(U-).n) [+ the BR1 viscous part]
  if (fp) {
    bool bad = false;
    double g[NF];
    if (link < 0) ph.ghost(-1 - link, UL, nx, ny, UR);
    ph.face(UL, UR, nx, ny, g, bad);
    if (bad && e0 + fel < ne) atomicOr(flag, 1);
#pragma unroll
    for (int v = 0; v < NF; ++v) {
      double t = jr * g[v];
      if (NS && v > 0) t += 0.5 * jr * gv[v - 1];
      gF[((fel * NF + v) * 4 + fsd) * QF + fa] = (R)t;
    }
  }
  // contravariant fluxes at the nodes
#pragma unroll
  for (int r = 0; r < S::NPT; ++r) {
    const int k = tid + r * NT, el = k / Q2, n = k - el * Q2;
    if (k >= EPW * Q2) continue;
    double u[NF], fx[NF], fy[NF];
    const double sc = PH::scaled ? mt[r][0] * mt[r][3] - mt[r][1] * mt[r][2] : 1.0;   // 1 / J
#pragma unroll
    for (int v = 0; v < NF; ++v) u[v] = PH::scaled ? sc * un[r][v] : un[r][v];
    ph.flux(u, fx, fy);
#pragma unroll
    for (int v = 0; v < NF; ++v) {
      N1[(el * NF + v) * Q2 + n] = (R)(mt[r][0] * fx[v] + mt[r][1] * fy[v]);
      N2[(el * NF + v) * Q2 + n] = (R)(mt[r][2] * fx[v] + mt[r][3] * fy[v]);
    }
  }
  __syncthreads();
  // projected divergence: (QD (x) BW) N1 + (BW (x) QD) N2, and the face blocks
  contract<EF, Q, Q, 2, L, NT>(TE::BW(), N1, X1, tid);
  contract<EF, Q, Q, 2, L, NT>(TE::QD(), N2, X2, tid);
  contract<EF, 4, QF, 2, L, NT>(TE::PW(), gF, H, tid);
  __syncthreads();
  for (int pc = tid; pc < EF * L; pc += NT) {
    const int f = pc / L, c = pc - f * L;
    R a[Q], b[Q], y[L], z[L];
#pragma unroll
    for (int i = 0; i < Q; ++i) { a[i] = X1[(f * Q + i) * L + c]; b[i] = X2[(f * Q + i) * L + c]; }
    table_apply(TE::QD(), a, y);
    table_apply(TE::BW(), b, z);
#pragma unroll
    for (int l = 0; l < L; ++l) M[(f * L + l) * L + c] = y[l] + z[l];
  }
  __syncthreads();
  const double cw[4] = {1.0, 1.0, 1.0, 1.0};
#pragma unroll
  for (int k = 0; k < S::NU; ++k) {
    const int i = tid + k * NT, el = i / (NF * L2), rr = i - el * NF * L2, v = rr / L2, m = rr - v * L2, l = m / L;
    if (i >= S::NM) continue;
    double r = M[i] + face_add2<P, R>(table_rows(TE::Bend()), H + (el * NF + v) * 4 * L, l, m - l * L, cw);
    if constexpr (NS) r -= vv[k];
    const int e = e0 + el;
    const size_t o = ((size_t)v * ne + e) * L2 + m;
    if (e < ne) M[i] = (R)up.post(o, e, v, m, r, x[k], pre[k]);
  }
  if (!Tn) return;
  __syncthreads();
  quad_traces<P, NF, EPW, R, TE>(M, N1, Tn, e0, ne, tid);
}

}  // namespace dgx
