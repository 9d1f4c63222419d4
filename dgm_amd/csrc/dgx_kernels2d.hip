// Quad (2D) kernels of the DG residual; same structure as the hex kernels:
// one workgroup per element, LDS tensors, register-blocked pencil contractions.
//   face traces      Quad::fill_sides                 src/Quad.cpp:845-869
//   volume term      Euler::convection                src/Euler.cpp:296-390
//   numerical flux   Euler::convective_flux (LF, Roe) src/Euler.cpp:399-757
//   lift + project   Quad::lift, Element::project     src/Quad.cpp:1971-2038, src/Element.hpp:427-437
//   BR1 viscous      Navier_Stokes::diffusion         src/Navier_Stokes.cpp:113-258
//   shallow water    Shallow::convection, LF flux     src/Shallow.cpp:251-525
//   linear system    LinEuler_quasi::convection       src/LinEuler_quasi.cpp:151-495
//                    and its discrete adjoint
#include <hip/hip_cooperative_groups.h>

#include <algorithm>
#include <type_traits>
#include <vector>

#include "dgx_quad2.hpp"

namespace dgx {

// Float copies of the basis tables for the mixed quad kernels, which hold
// their LDS tensors and run their contractions in FP32 while the state, face
// traces, LSRK registers and pointwise physics stay FP64; filled beside c_tab
// at upload.  TE<R, P> gives the even-odd tables of arithmetic type R.
static __constant__ float c_tabf[kTabTotal];
struct EoBaseF {
  using R = float;
  __device__ static __forceinline__ const float *base() { return c_tabf; }
};
template <typename R, int P> using TE = EOx<std::conditional_t<std::is_same<R, double>::value, EoBaseD, EoBaseF>, P>;

template <int P> struct H2 {
  static constexpr int L = P + 1, Q = P + 2, QF = P + 1;
  static constexpr int L2 = L * L, Q2 = Q * Q;
  static constexpr int NT = 64;
};

template <int P>
__device__ __forceinline__ void backward2(const Tab &tb, const double *m, double *s1, double *out,
                                          int tid) {
  constexpr int L = H2<P>::L, Q = H2<P>::Q, NT = H2<P>::NT;
  contract<1, L, L, 1, Q, NT>(CT<P>::BT(), m, s1, tid);
  __syncthreads();
  contract<1, Q, L, 2, Q, NT>(CT<P>::BT(), s1, out, tid);
  __syncthreads();
}

// Gauss-point traces of a state's NF fields on the elements' edges.
template <int P, int NF, int EPW, class TT, typename R>
__device__ __forceinline__ void load_traces2(const double *__restrict__ U, double *__restrict__ T, int ne, int e0,
                                             R *sm) {
  using S = Q2S<P, NF, EPW>;
  constexpr int L2 = S::L2, NT = S::NT;
  R *M = sm, *K = M + S::NM;
  const int tid = threadIdx.x;
#pragma unroll
  for (int k = 0; k < S::NU; ++k) {
    const int i = tid + k * NT, el = i / (NF * L2), r = i - el * NF * L2, v = r / L2;
    if (i < S::NM) M[i] = (R)U[((size_t)v * ne + min(e0 + el, ne - 1)) * L2 + (r - v * L2)];
  }
  __syncthreads();
  quad_traces<P, NF, EPW, R, TT>(M, K, T, e0, ne, tid);
}

// TT: the tables (CT<P> for Navier-Stokes, see k_quad2).  EPW as for the stage;
// LDS for the traces alone.  With every mesh packed and the whole stage's block
// (42 KB at p = 10, three wavefronts a CU) a residual of Euler quads took 6.84 us
// on 32^2 at p = 2, 47.6 us on 256^2 at p = 2, 58.9 us on 64^2 at p = 10; now
// 6.57, 38.8 and 45.5.
template <int P, int EPW, int NF, class TT, typename R>
__global__ void __launch_bounds__(64)
k_traces2(const double *__restrict__ U, double *__restrict__ T, int ne) {
  __shared__ R sm[Q2S<P, NF, EPW>::traces];
  load_traces2<P, NF, EPW, TT, R>(U, T, ne, blockIdx.x * EPW, sm);
}

// One stage of an affine domain (quad_stage): EQ 0 Euler, 1 Navier-Stokes with
// the BR1 viscous terms V, TV, 2 shallow water.  Navier-Stokes takes the plain
// tables, like its traces, k_grad2 and k_visc2: explicit steps may exceed the
// viscous limit dt ~ h^2 / (nu (p + 1)^4) for a while, and there each step
// multiplies a difference in the last bit by ten and more (p = 10, 134^2
// quads, five RK4 steps: a million times), so that the even-odd sums' other
// rounding shows in the eleventh digit.  It costs time: ten TVD-RK3 steps of
// four quads at p = 10 take 0.94 ms, with even-odd sums 0.63 ms.
template <int P, int EPW, typename R, int EQ>
__global__ void __launch_bounds__(64)
k_quad2(const double *X, const double *__restrict__ T, const double *__restrict__ V, const double *__restrict__ TV,
        Geo geo, Phys ph, int ne, int *__restrict__ flag, StageStep s, double *Bal, int bal, double *__restrict__ Tn) {
  constexpr int NF = EQ == 2 ? 3 : 4;
  __shared__ R sm[Q2S<P, NF, EPW>::size];
  const int e0 = xcd_element(blockIdx.x, gridDim.x) * EPW;
  const QuadUpdate up{s};
  if constexpr (EQ == 2)
    quad_stage<P, EPW, R, TE<R, P>, false>(X, T, V, TV, geo, ne, e0, flag, QuadShallow{ph}, QuadBalanced{up, Bal, bal},
                                           Tn, sm);
  else
    quad_stage<P, EPW, R, std::conditional_t<EQ == 1, CT<P>, TE<R, P>>, EQ == 1>(X, T, V, TV, geo, ne, e0, flag,
                                                                                QuadEuler{ph}, up, Tn, sm);
}

// lifted, projected gradients of (u, v, e): G[e][2*prim + dir][L2]
template <int P>
__global__ void __launch_bounds__(64)
k_grad2(const double *__restrict__ U, const double *__restrict__ T, double *__restrict__ G, Tab tb,
        Geo geo, int ne) {
  using S = H2<P>;
  constexpr int L = S::L, Q = S::Q, QF = S::QF, L2 = S::L2, Q2 = S::Q2, NT = S::NT;
  __shared__ double Un[4 * Q2], Jq[12 * QF], Fb[Q2], Xa[Q * L], Xc[Q * L], D2[2 * L2], H[4 * L];
  const int e = blockIdx.x, tid = threadIdx.x;
  for (int v = 0; v < 4; ++v) {
    copy_block<NT>(U + ((size_t)v * ne + e) * L2, D2, L2, tid);
    __syncthreads();
    backward2<P>(tb, D2, Xa, Un + v * Q2, tid);
  }
  for (int i = tid; i < 4 * QF; i += NT) {
    const int s = i / QF, a = i - s * QF;
    const int es = e * 4 + s;
    const int nb = geo.nbr[es], ns = geo.nside[es];
    const int an = geo.perm[geo.permid[es] * QF + a];
    const double jr = geo.fjr[es];
    const double *tl = T + ((size_t)e * 4 + s) * 4 * QF;
    const double *tr = T + ((size_t)nb * 4 + ns) * 4 * QF;
    double pl[3], pr[3];
    {
      const double r = tl[a], u = tl[QF + a] / r, v = tl[2 * QF + a] / r;
      double en = tl[3 * QF + a] / r;
      double wk = u * u; wk = v * v + wk;
      pl[0] = u; pl[1] = v; pl[2] = -0.5 * wk + en;
    }
    {
      const double r = tr[an], u = tr[QF + an] / r, v = tr[2 * QF + an] / r;
      double en = tr[3 * QF + an] / r;
      double wk = u * u; wk = v * v + wk;
      pr[0] = u; pr[1] = v; pr[2] = -0.5 * wk + en;
    }
#pragma unroll
    for (int q = 0; q < 3; ++q) Jq[(q * 4 + s) * QF + a] = jr * (0.5 * (pl[q] + pr[q]) - pl[q]);
  }
  __syncthreads();
  const double *mt = geo.metric + 9 * (size_t)e;
  for (int q = 0; q < 3; ++q) {
    for (int k = tid; k < Q2; k += NT) {
      const double r = Un[k], u = Un[Q2 + k] / r, v = Un[2 * Q2 + k] / r;
      double val;
      if (q == 0) val = u;
      else if (q == 1) val = v;
      else {
        double en = Un[3 * Q2 + k] / r;
        double wk = u * u; wk = v * v + wk;
        val = -0.5 * wk + en;
      }
      Fb[k] = val;
    }
    __syncthreads();
    contract<1, Q, Q, 2, L, NT>(CT<P>::BW(), Fb, Xa, tid);
    contract<1, Q, Q, 2, L, NT>(CT<P>::QD(), Fb, Xc, tid);
    contract<1, 4, QF, 2, L, NT>(CT<P>::PW(), Jq + q * 4 * QF, H, tid);
    __syncthreads();
    contract<1, Q, L, 1, L, NT>(CT<P>::QD(), Xa, D2, tid);
    contract<1, Q, L, 1, L, NT>(CT<P>::BW(), Xc, D2 + L2, tid);
    __syncthreads();
    for (int k = tid; k < L2; k += NT) {
      const int l = k / L, m = k - l * L;
#pragma unroll
      for (int d = 0; d < 2; ++d) {
        double c[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) c[s] = geo.fnorm[3 * (e * 4 + s) + d];
        G[((size_t)e * 6 + 2 * q + d) * L2 + k] =
            mt[d] * D2[k] + mt[3 + d] * D2[L2 + k] + face_add2<P>(CT<P>::Bend(), H, l, m, c);
      }
    }
    __syncthreads();
  }
}

template <int P>
__global__ void __launch_bounds__(64)
k_visc2(const double *__restrict__ U, const double *__restrict__ G, double *__restrict__ V,
        double *__restrict__ TV, Tab tb, Geo geo, Phys ph, int ne) {
  using S = H2<P>;
  constexpr int L = S::L, Q = S::Q, QF = S::QF, L2 = S::L2, Q2 = S::Q2, NT = S::NT;
  __shared__ double Un[4 * Q2], Gn[6 * Q2], M0[L2], S1[Q * L], Lay[12 * Q], Wf[12 * QF], X1[Q * L],
      X2[Q * L], Vo[L2];
  const int e = blockIdx.x, tid = threadIdx.x;
  for (int v = 0; v < 10; ++v) {
    const double *src = v < 4 ? U + ((size_t)v * ne + e) * L2 : G + ((size_t)e * 6 + (v - 4)) * L2;
    double *dst = v < 4 ? Un + v * Q2 : Gn + (v - 4) * Q2;
    copy_block<NT>(src, M0, L2, tid);
    __syncthreads();
    backward2<P>(tb, M0, S1, dst, tid);
  }
  const double mu = ph.vis, kap = ph.vis * ph.gamma / ph.Pr;
  auto vflux = [&](int k, double out[3][2]) {
    const double r = Un[k], u = Un[Q2 + k] / r, v = Un[2 * Q2 + k] / r;
    const double ux = Gn[k], uy = Gn[Q2 + k], vx = Gn[2 * Q2 + k], vy = Gn[3 * Q2 + k];
    const double ex = Gn[4 * Q2 + k], ey = Gn[5 * Q2 + k];
    const double t12 = mu * (uy + vx);
    const double t11 = mu * ((2.0 / 3.0) * (2.0 * ux - vy));
    const double t22 = mu * ((2.0 / 3.0) * (2.0 * vy - ux));
    out[0][0] = t11; out[0][1] = t12;
    out[1][0] = t12; out[1][1] = t22;
    out[2][0] = t11 * u + t12 * v + kap * ex;
    out[2][1] = t12 * u + t22 * v + kap * ey;
  };
  for (int i = tid; i < 4 * Q; i += NT) {
    const int s = i / Q, j = i - s * Q;
    int k;
    switch (s) {
      case 0: k = j * Q; break;
      case 1: k = (Q - 1) * Q + j; break;
      case 2: k = j * Q + Q - 1; break;
      default: k = j; break;
    }
    const double *nn = geo.fnorm + 3 * (e * 4 + s);
    double f[3][2];
    vflux(k, f);
#pragma unroll
    for (int q = 0; q < 3; ++q) Lay[(s * 3 + q) * Q + j] = f[q][0] * nn[0] + f[q][1] * nn[1];
  }
  __syncthreads();
  contract<1, 12, Q, 2, QF, NT>(CT<P>::Ig(), Lay, Wf, tid);
  __syncthreads();
  copy_block<NT>(Wf, TV + (size_t)e * 12 * QF, 12 * QF, tid);
  const double *mt = geo.metric + 9 * (size_t)e;
  for (int k = tid; k < Q2; k += NT) {
    double f[3][2];
    vflux(k, f);
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      Gn[(2 * q) * Q2 + k] = mt[0] * f[q][0] + mt[1] * f[q][1];
      Gn[(2 * q + 1) * Q2 + k] = mt[3] * f[q][0] + mt[4] * f[q][1];
    }
  }
  __syncthreads();
  for (int q = 0; q < 3; ++q) {
    contract<1, Q, Q, 2, L, NT>(CT<P>::BW(), Gn + 2 * q * Q2, X1, tid);
    contract<1, Q, Q, 2, L, NT>(CT<P>::QD(), Gn + (2 * q + 1) * Q2, X2, tid);
    __syncthreads();
    contract<1, Q, L, 1, L, NT>(CT<P>::QD(), X1, Vo, tid);
    __syncthreads();
    contract<1, Q, L, 1, L, NT, true>(CT<P>::BW(), X2, Vo, tid);
    __syncthreads();
    copy_block<NT>(Vo, V + ((size_t)e * 3 + q) * L2, L2, tid);
    __syncthreads();
  }
}

template <int P>
__global__ void __launch_bounds__(64)
k_forward2(const double *__restrict__ Fn, double *__restrict__ Fm, Tab tb, int ne) {
  using S = H2<P>;
  constexpr int L = S::L, Q = S::Q, L2 = S::L2, Q2 = S::Q2, NT = S::NT;
  __shared__ double A[Q2], X[Q * L], O[L2];
  const int e = blockIdx.x % ne, v = blockIdx.x / ne, tid = threadIdx.x;
  copy_block<NT>(Fn + ((size_t)v * ne + e) * Q2, A, Q2, tid);
  __syncthreads();
  contract<1, Q, Q, 2, L, NT>(CT<P>::BW(), A, X, tid);
  __syncthreads();
  contract<1, Q, L, 1, L, NT>(CT<P>::BW(), X, O, tid);
  __syncthreads();
  copy_block<NT>(O, Fm + ((size_t)v * ne + e) * L2, L2, tid);
}

template <int P>
__global__ void __launch_bounds__(64)
k_backward2(const double *__restrict__ Fm, double *__restrict__ Fn, Tab tb, int ne) {
  using S = H2<P>;
  constexpr int L = S::L, Q = S::Q, L2 = S::L2, Q2 = S::Q2, NT = S::NT;
  __shared__ double A[L2], X[Q * L], O[Q2];
  const int e = blockIdx.x % ne, v = blockIdx.x / ne, tid = threadIdx.x;
  copy_block<NT>(Fm + ((size_t)v * ne + e) * L2, A, L2, tid);
  __syncthreads();
  backward2<P>(tb, A, X, O, tid);
  copy_block<NT>(O, Fn + ((size_t)v * ne + e) * Q2, Q2, tid);
}

// Linear system residual, Lax-Friedrichs flux 1/2 (An UL + An UR) + 1/2 lam
// (UL - UR), lam = |u0.n| + c0 (LinEuler_quasi::convection / convective_flux,
// src/LinEuler_quasi.cpp:161-495, for a uniform mean flow), fused with its
// LSRK14 stage.  ADJ: the same residual of the adjoint system applied to
// X / J_e and multiplied by J_e is the transpose of the forward residual in
// modal coordinates (exact quadrature throughout), and the kernel performs one
// reversed stage: Ubar += -dt L^T X, dJ/dtheta_e += 2 g dt X[E][e][0],
// Ubar_t = ca X.
template <int P, int EPW, bool ADJ, typename R = double>
__global__ void __launch_bounds__(64)
k_lin2(LinArgs a) {
  __shared__ R sm[Q2S<P, 4, EPW>::size];
  const int e0 = xcd_element(blockIdx.x, gridDim.x) * EPW;
  if constexpr (ADJ)
    quad_stage<P, EPW, R, TE<R, P>, false>(a.X, a.T, nullptr, nullptr, a.geo, a.ne, e0, nullptr, QuadLinear<true>{a},
                                           LinearAdjoint{a}, a.Tn, sm);
  else
    quad_stage<P, EPW, R, TE<R, P>, false>(a.X, a.T, nullptr, nullptr, a.geo, a.ne, e0, nullptr, QuadLinear<false>{a},
                                           LinearForward{a}, a.Tn, sm);
}

// Observations (one workgroup per receiver) and the objective's adjoint (one
// workgroup, receivers in order, so that receivers sharing an element never
// race).
__global__ void __launch_bounds__(64)
k_observe(const double *__restrict__ U, const int *__restrict__ rec_e, const double *__restrict__ rec_w,
          const double *__restrict__ cobs, int ne, int L2, double *__restrict__ y) {
  __shared__ double red[64];
  const int r = blockIdx.x, tid = threadIdx.x, e = rec_e[r];
  double s = 0.0;
  for (int i = tid; i < 4 * L2; i += 64) {
    const int f = i / L2, m = i - f * L2;
    s = fma(cobs[f] * rec_w[(size_t)r * L2 + m], U[((size_t)f * ne + e) * L2 + m], s);
  }
  red[tid] = s;
  __syncthreads();
  for (int w = 32; w > 0; w >>= 1) {
    if (tid < w) red[tid] += red[tid + w];
    __syncthreads();
  }
  if (tid == 0) y[r] = red[0];
}

__global__ void __launch_bounds__(64)
k_observe_adjoint(const double *__restrict__ U, double *__restrict__ Ubar, const int *__restrict__ rec_e,
                  const double *__restrict__ rec_w, const double *__restrict__ cobs, int nrec, int ne, int L2,
                  const double *__restrict__ d, double dt, double *__restrict__ J) {
  __shared__ double red[64];
  const int tid = threadIdx.x;
  double jsum = 0.0;
  for (int r = 0; r < nrec; ++r) {
    const int e = rec_e[r];
    double s = 0.0;
    for (int i = tid; i < 4 * L2; i += 64) {
      const int f = i / L2, m = i - f * L2;
      s = fma(cobs[f] * rec_w[(size_t)r * L2 + m], U[((size_t)f * ne + e) * L2 + m], s);
    }
    red[tid] = s;
    __syncthreads();
    for (int w = 32; w > 0; w >>= 1) {
      if (tid < w) red[tid] += red[tid + w];
      __syncthreads();
    }
    const double res = red[0] - d[r];
    __syncthreads();
    jsum += res * res;
    for (int i = tid; i < 4 * L2; i += 64) {
      const int f = i / L2, m = i - f * L2;
      const size_t gi = ((size_t)f * ne + e) * L2 + m;
      Ubar[gi] = fma(dt * res * cobs[f], rec_w[(size_t)r * L2 + m], Ubar[gi]);
    }
    __syncthreads();
  }
  if (tid == 0) *J += 0.5 * dt * jsum;
}

// Batched serving (dgx_server with batching): one launch per stage runs every
// member request of a group (same order and physics).  A fixed grid of
// workgroups walks the flat list of (request, element) work items; members
// are in work-item order, b[r].off their first item.  The step kernel fuses
// the LSRK14 register update of the direct path (vField axpby, axpy:
// Ut = A Ut - dt R, U += B Ut) into the residual's store.
template <int P, int E, int NF, typename R = double>
__global__ void __launch_bounds__(64)
k_batch_traces2(const Batch2 *__restrict__ b, int nreq, int nwork) {
  __shared__ R sm[Q2S<P, NF, E>::traces];
  int r = 0;
  for (int w = blockIdx.x; w < nwork; w += gridDim.x) {
    while (r + 1 < nreq && b[r + 1].off <= w) ++r;
    load_traces2<P, NF, E, TE<R, P>, R>(b[r].U, b[r].T, b[r].ne, (w - b[r].off) * E, sm);
    __syncthreads();
  }
}

// Work item w - off of member m: a stage of its elements.
template <int P, int E, bool SHALLOW, typename R>
__device__ __forceinline__ void batch_stage2(const Batch2 &m, int w, const double *Tc, double *Tn, double A, double B,
                                             R *sm) {
  const Geo geo = m.geo;
  const Phys ph = m.phys;
  StageStep s;
  s.mode = ST_LSRK; s.Xn = m.U; s.acc = m.Ut; s.a = A; s.b = B; s.dt = m.dt;
  const int e0 = (w - m.off) * E;
  if constexpr (SHALLOW)
    quad_stage<P, E, R, TE<R, P>, false>(m.U, Tc, nullptr, nullptr, geo, m.ne, e0, m.flag, QuadShallow{ph},
                                         QuadBalanced{QuadUpdate{s}, m.Bal, m.bal}, Tn, sm);
  else
    quad_stage<P, E, R, TE<R, P>, false>(m.U, Tc, nullptr, nullptr, geo, m.ne, e0, m.flag, QuadEuler{ph},
                                         QuadUpdate{s}, Tn, sm);
  __syncthreads();
}

// odd: the stage reads the traces of T2 and writes the next ones into T
// (else T and T2); next: write the next stage's traces at all.
template <int P, int E, bool SHALLOW, typename R = double>
__global__ void __launch_bounds__(64)
k_batch_step2(const Batch2 *__restrict__ b, int nreq, int nwork, double A, double B, int odd, int next) {
  constexpr int NF = SHALLOW ? 3 : 4;
  __shared__ R sm[Q2S<P, NF, E>::size];
  int r = 0;
  for (int w = blockIdx.x; w < nwork; w += gridDim.x) {
    while (r + 1 < nreq && b[r + 1].off <= w) ++r;
    batch_stage2<P, E, SHALLOW, R>(b[r], w, odd ? b[r].T2 : b[r].T, next ? (odd ? b[r].T : b[r].T2) : nullptr, A, B,
                                   sm);
  }
}

struct LsrkTab {
  double A[14], B[14];
};

// A persistent slice of a batched group: nsteps LSRK14 steps of every member
// in one cooperative launch, whose workgroups are all resident at once.  The
// face traces of the slice's first state are computed first; then each stage
// is one pass over the members' elements, in which an element takes its
// residual from the current traces, updates its register and state in place
// and writes the traces of its new state into the other trace buffer,
// followed by one grid-wide barrier.  The buffers alternate T, T2, T, ... so
// that no element overwrites traces a neighbour may still be reading; after
// the even number of stages of a step the current traces are in T again.
// Each element's arithmetic is that of k_batch_traces2 and k_batch_step2, so
// the results are bitwise those of the per-stage launches.
template <int P, int E, bool SHALLOW, typename R = double>
__global__ void __launch_bounds__(64)
k_batch_persist2(const Batch2 *__restrict__ b, int nreq, int nwork, int nsteps, LsrkTab c) {
  constexpr int NF = SHALLOW ? 3 : 4;
  __shared__ R sm[Q2S<P, NF, E>::size];
  cooperative_groups::grid_group grid = cooperative_groups::this_grid();
  {
    int r = 0;
    for (int w = blockIdx.x; w < nwork; w += gridDim.x) {
      while (r + 1 < nreq && b[r + 1].off <= w) ++r;
      load_traces2<P, NF, E, TE<R, P>, R>(b[r].U, b[r].T, b[r].ne, (w - b[r].off) * E, sm);
      __syncthreads();
    }
  }
  grid.sync();
  for (int step = 0; step < nsteps; ++step)
    for (int st = 0; st < 14; ++st) {
      const bool odd = st & 1, last = step == nsteps - 1 && st == 13;
      int r = 0;
      for (int w = blockIdx.x; w < nwork; w += gridDim.x) {
        while (r + 1 < nreq && b[r + 1].off <= w) ++r;
        batch_stage2<P, E, SHALLOW, R>(b[r], w, odd ? b[r].T2 : b[r].T, last ? nullptr : (odd ? b[r].T : b[r].T2),
                                       c.A[st], c.B[st], sm);
      }
      grid.sync();
    }
}

template <int P, int E, bool SHALLOW, typename R>
static hipError_t launch_persist2(BatchLaunch &a) {
  const void *kern = reinterpret_cast<const void *>(&k_batch_persist2<P, E, SHALLOW, R>);
  int dev = 0, ncu = 0, per = 0;
  hipError_t e;
  if ((e = hipGetDevice(&dev)) != hipSuccess) return e;
  if ((e = hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev)) != hipSuccess) return e;
  if ((e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kern, 64, 0)) != hipSuccess) return e;
  // every workgroup must be resident at once for the grid-wide barriers: keep
  // well inside the occupancy the runtime reports, counting a CU's LDS as
  // 64 KiB
  hipFuncAttributes fa;
  if ((e = hipFuncGetAttributes(&fa, kern)) != hipSuccess) return e;
  per = std::min(per, (int)(65536 / std::max<size_t>(fa.sharedSizeBytes, 1)));
  if (per < 1 || ncu < 1) return hipErrorInvalidConfiguration;
  const int grid = std::max(1, std::min(a.nwork, per * ncu));
  LsrkTab c;
  for (int s = 0; s < 14; ++s) { c.A[s] = a.lsrkA[s]; c.B[s] = a.lsrkB[s]; }
  const Batch2 *b = a.b;
  int nreq = a.nreq, nwork = a.nwork, nsteps = a.nsteps;
  void *args[] = {&b, &nreq, &nwork, &nsteps, &c};
  a.grid = grid;
  return hipLaunchCooperativeKernel(kern, dim3(grid), dim3(64), args, 0, a.stream);
}

template <int P, int E, bool SHALLOW, typename R>
static hipError_t launch_batch2_k(BatchLaunch &a) {
  if (a.op == 2) return launch_persist2<P, E, SHALLOW, R>(a);
  const int grid = std::max(1, std::min(a.nwork, kBatchGrid));
  if (a.op == 0)
    hipLaunchKernelGGL((k_batch_traces2<P, E, SHALLOW ? 3 : 4, R>), dim3(grid), dim3(64), 0, a.stream, a.b, a.nreq,
                       a.nwork);
  else
    hipLaunchKernelGGL((k_batch_step2<P, E, SHALLOW, R>), dim3(grid), dim3(64), 0, a.stream, a.b, a.nreq, a.nwork,
                       a.A, a.B, a.odd, a.next);
  return hipGetLastError();
}

template <int P, bool SHALLOW, typename R>
static hipError_t launch_batch2_e(BatchLaunch &a) {
  constexpr int E = quad_epw(P, SHALLOW ? 3 : 4);
  return a.packed ? launch_batch2_k<P, E, SHALLOW, R>(a) : launch_batch2_k<P, 1, SHALLOW, R>(a);
}

template <int P>
static hipError_t launch_batch2_p(BatchLaunch &a) {
  if (a.mixed) return a.shallow ? launch_batch2_e<P, true, float>(a) : launch_batch2_e<P, false, float>(a);
  return a.shallow ? launch_batch2_e<P, true, double>(a) : launch_batch2_e<P, false, double>(a);
}

hipError_t launch_batch2(BatchLaunch &a) {
  if (a.nreq < 1 || a.nwork < 1 || !a.b || (a.op == 2 && a.nsteps < 1)) return hipErrorInvalidValue;
  switch (a.p) {
#define DGX_CASE(PP) case PP: return launch_batch2_p<PP>(a);
    DGX_CASE(1) DGX_CASE(2) DGX_CASE(3) DGX_CASE(4) DGX_CASE(5)
    DGX_CASE(6) DGX_CASE(7) DGX_CASE(8) DGX_CASE(9) DGX_CASE(10)
#undef DGX_CASE
    default: return hipErrorInvalidValue;
  }
}

template <int P, int EPW>
static hipError_t launch_lin2_pe(const LinArgs &a) {
  const dim3 grid((a.ne + EPW - 1) / EPW);
  if (a.adjoint && a.mixed) hipLaunchKernelGGL((k_lin2<P, EPW, true, float>), grid, dim3(64), 0, a.stream, a);
  else if (a.adjoint) hipLaunchKernelGGL((k_lin2<P, EPW, true>), grid, dim3(64), 0, a.stream, a);
  else if (a.mixed) hipLaunchKernelGGL((k_lin2<P, EPW, false, float>), grid, dim3(64), 0, a.stream, a);
  else hipLaunchKernelGGL((k_lin2<P, EPW, false>), grid, dim3(64), 0, a.stream, a);
  return hipGetLastError();
}

template <int P>
static hipError_t launch_lin2_p(const LinArgs &a) {
  constexpr int E = quad_epw(P, 4);
  return quad_packed(P, a.ne) ? launch_lin2_pe<P, E>(a) : launch_lin2_pe<P, 1>(a);
}

hipError_t launch_lin2(const LinArgs &a) {
  switch (a.p) {
#define DGX_CASE(PP) case PP: return launch_lin2_p<PP>(a);
    DGX_CASE(1) DGX_CASE(2) DGX_CASE(3) DGX_CASE(4) DGX_CASE(5)
    DGX_CASE(6) DGX_CASE(7) DGX_CASE(8) DGX_CASE(9) DGX_CASE(10)
#undef DGX_CASE
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_observe(const double *U, const int *rec_e, const double *rec_w, const double *cobs, int nrec,
                          int ne, int L2, double *y, hipStream_t s) {
  hipLaunchKernelGGL(k_observe, dim3(nrec), dim3(64), 0, s, U, rec_e, rec_w, cobs, ne, L2, y);
  return hipGetLastError();
}

hipError_t launch_observe_adjoint(const double *U, double *Ubar, const int *rec_e, const double *rec_w,
                                  const double *cobs, int nrec, int ne, int L2, const double *d, double dt,
                                  double *J, hipStream_t s) {
  hipLaunchKernelGGL(k_observe_adjoint, dim3(1), dim3(64), 0, s, U, Ubar, rec_e, rec_w, cobs, nrec, ne, L2, d,
                     dt, J);
  return hipGetLastError();
}

template <int P, int EPW, typename R, int EQ>
static hipError_t launch_quad2_k(const LaunchArgs &a, const StageStep &s, double *Tn) {
  hipLaunchKernelGGL((k_quad2<P, EPW, R, EQ>), dim3((a.ne + EPW - 1) / EPW), dim3(64), 0, a.stream, a.U, a.T, a.V,
                     a.TV, a.geo, a.phys, a.ne, a.flag, s, a.Bal, a.bal, Tn);
  return hipGetLastError();
}

template <int P, typename R, int EQ>
static hipError_t launch_quad2_e(const LaunchArgs &a, const StageStep &s, double *Tn) {
  constexpr int E = quad_epw(P, EQ == 2 ? 3 : 4);
  return quad_packed(P, a.ne) ? launch_quad2_k<P, E, R, EQ>(a, s, Tn) : launch_quad2_k<P, 1, R, EQ>(a, s, Tn);
}

template <int P>
static hipError_t launch_quad2(const LaunchArgs &a, const StageStep &s, double *Tn) {
  if (a.eqn == 30) return a.mixed ? launch_quad2_e<P, float, 2>(a, s, Tn) : launch_quad2_e<P, double, 2>(a, s, Tn);
  if (a.mixed) return launch_quad2_e<P, float, 0>(a, s, Tn);
  return a.ns ? launch_quad2_e<P, double, 1>(a, s, Tn) : launch_quad2_e<P, double, 0>(a, s, Tn);
}

template <int P, int EPW, int NF, class TT, typename R>
static hipError_t launch_traces2_k(const LaunchArgs &a) {
  hipLaunchKernelGGL((k_traces2<P, EPW, NF, TT, R>), dim3((a.ne + EPW - 1) / EPW), dim3(64), 0, a.stream, a.U, a.T,
                     a.ne);
  return hipGetLastError();
}

template <int P, int NF, class TT, typename R>
static hipError_t launch_traces2(const LaunchArgs &a) {
  constexpr int E = quad_epw(P, NF);
  return quad_packed(P, a.ne) ? launch_traces2_k<P, E, NF, TT, R>(a) : launch_traces2_k<P, 1, NF, TT, R>(a);
}

template <int P>
static hipError_t launch2(const LaunchArgs &a) {
  const int ne = a.ne;
  switch (a.op) {
    case OP_TRACES:
      if (a.mixed)
        return a.nfield == 3 ? launch_traces2<P, 3, TE<float, P>, float>(a) : launch_traces2<P, 4, TE<float, P>, float>(a);
      if (a.ns) return launch_traces2<P, 4, CT<P>, double>(a);
      return a.nfield == 3 ? launch_traces2<P, 3, EO<P>, double>(a) : launch_traces2<P, 4, EO<P>, double>(a);
    case OP_RHS: {
      StageStep s;
      s.Xn = a.R;
      return launch_quad2<P>(a, s, nullptr);
    }
    case OP_STAGE: return launch_quad2<P>(a, a.step, a.Tn);
    case OP_GRAD:
      hipLaunchKernelGGL(k_grad2<P>, dim3(ne), dim3(64), 0, a.stream, a.U, a.T, a.G, a.tab, a.geo, ne);
      break;
    case OP_VISC:
      hipLaunchKernelGGL(k_visc2<P>, dim3(ne), dim3(64), 0, a.stream, a.U, a.G, a.V, a.TV, a.tab,
                         a.geo, a.phys, ne);
      break;
    case OP_FORWARD:
      hipLaunchKernelGGL(k_forward2<P>, dim3(ne * a.nfield), dim3(64), 0, a.stream, a.X, a.Y, a.tab, ne);
      break;
    case OP_BACKWARD:
      hipLaunchKernelGGL(k_backward2<P>, dim3(ne * a.nfield), dim3(64), 0, a.stream, a.X, a.Y, a.tab, ne);
      break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

int lds_bytes2(int p, int which) { return (p >= 1 && p <= 10) ? 0 : -1; }

hipError_t launch_2d(const LaunchArgs &a) {
  switch (a.p) {
#define DGX_CASE(PP) case PP: return launch2<PP>(a);
    DGX_CASE(1) DGX_CASE(2) DGX_CASE(3) DGX_CASE(4) DGX_CASE(5)
    DGX_CASE(6) DGX_CASE(7) DGX_CASE(8) DGX_CASE(9) DGX_CASE(10)
#undef DGX_CASE
    default: return hipErrorInvalidValue;
  }
}

hipError_t upload_tables_2d(const double *h) {
  hipError_t e = hipMemcpyToSymbol(HIP_SYMBOL(c_tab), h, sizeof(double) * kTabTotal);
  if (e != hipSuccess) return e;
  std::vector<float> f(h, h + kTabTotal);
  return hipMemcpyToSymbol(HIP_SYMBOL(c_tabf), f.data(), sizeof(float) * kTabTotal);
}

}  // namespace dgx
