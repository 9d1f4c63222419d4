// Sum-factorization contractions over LDS tensors, shared by the hex kernels
// (FP64; FP32 in the mixed curved residual).  One thread owns one pencil at a time and computes all of its
// outputs with the even-odd form of the matrix (dgx_device.hpp), whose
// coefficients come from constant memory as scalar operands.
#pragma once
#include "dgx_device.hpp"

namespace dgx {

constexpr int round64(int n) { return (n + 63) / 64 * 64; }
// Wavefronts per SIMD that the LDS of workgroups of nt threads allows, at
// most `most`: the register budget to ask the compiler for.
constexpr int lds_waves(int lds, int nt, int most = 4) {
  const int w = (160 * 1024 / lds) * (nt / 64) / 4;
  return w < 1 ? 1 : (w > most ? most : w);
}
constexpr int odd(int n) { return n | 1; }
template <int V> struct IC { static constexpr int value = V; };
constexpr int cmax(int a, int b) { return a > b ? a : b; }


// [A][N][B][C] (last-dim pitch PI) -> [A][NO][B][C] (pitch PO), contracting N
// with an even-odd matrix; one thread computes all outputs of a pencil.
template <int A, int N, int B, int C, int NO, int PI, int PO, int NT, bool ACC = false, int K, typename T>
__device__ __forceinline__ void con_mid(EoMat<K, T> M, const T *in, T *out, int tid) {
  constexpr int NP = A * B * C;
  const T *h = uniform_const(M.h);
  auto pencil = [&](int pc) {
    const int c = pc % C, t = pc / C, b = t % B, a = t / B;
    T x[N], y[NO];
#pragma unroll
    for (int i = 0; i < N; ++i) x[i] = in[((a * N + i) * B + b) * PI + c];
    eo_apply<K, N, NO>(h, x, y);
#pragma unroll
    for (int o = 0; o < NO; ++o) {
      T *dst = out + ((a * NO + o) * B + b) * PO + c;
      if (ACC) *dst += y[o]; else *dst = y[o];
    }
  };
  if constexpr (NP <= NT) {
    if (tid < NP) pencil(tid);
  } else {
    for (int pc = tid; pc < NP; pc += NT) pencil(pc);
  }
}

// [R][NI] (pitch PI) -> [R][NO] (pitch PO), contracting the last dimension.
template <int R, int NI, int NO, int PI, int PO, int NT, int K, typename T>
__device__ __forceinline__ void con_last(EoMat<K, T> M, const T *in, T *out, int tid) {
  const T *h = uniform_const(M.h);
  auto pencil = [&](int r) {
    T x[NI], y[NO];
#pragma unroll
    for (int i = 0; i < NI; ++i) x[i] = in[r * PI + i];
    eo_apply<K, NI, NO>(h, x, y);
#pragma unroll
    for (int o = 0; o < NO; ++o) out[r * PO + o] = y[o];
  };
  if constexpr (R <= NT) {
    if (tid < R) pencil(tid);
  } else {
    for (int r = tid; r < R; r += NT) pencil(r);
  }
}

// Values at the Gauss points of an element's six faces, Te [6][5][QF^2], of the
// modal state in A ([5][L][L][L], last pitch odd(L)): the end values across
// each direction in B (20 L odd(L) + 15 L^2 values), then Bg (x) Bg per pair of
// faces in A (10 QF max(odd(L), 3 L) + 15 QF^2 values).
template <int P, int NT>
__device__ __forceinline__ void face_traces3(double *A, double *B, double *__restrict__ Te, int tid) {
  constexpr int L = P + 1, QF = P + 1, L2 = L * L, QF2 = QF * QF, LP = odd(L), FP = odd(QF);
  constexpr int KP = 3;   // pitch of the [..][2] collapse
  double *K0 = B, *K1 = B + 10 * L * LP, *K2 = B + 20 * L * LP;
  con_mid<5, L, L, L, 2, LP, LP, NT>(EO<P>::Bend(), A, K0, tid);       // [5][2][L][L]
  con_mid<5 * L, L, 1, L, 2, LP, LP, NT>(EO<P>::Bend(), A, K1, tid);   // [5][L][2][L]
  con_last<5 * L2, L, 2, LP, KP, NT>(EO<P>::Bend(), A, K2, tid);       // [5][L][L][2]
  __syncthreads();
  double *W = A, *O = A + 10 * QF * cmax(LP, KP * L);
  // faces 4 / 2: [5][2][QF][QF]
  con_mid<10, L, 1, L, QF, LP, LP, NT>(EO<P>::Bg(), K0, W, tid);      // [10][QF][L]
  __syncthreads();
  con_last<10 * QF, L, QF, LP, FP, NT>(EO<P>::Bg(), W, O, tid);       // [10][QF][QF]
  __syncthreads();
  for (int i = tid; i < 10 * QF2; i += NT) {
    const int ve = i / QF2, q = i - ve * QF2, v = ve >> 1, end = ve & 1;
    Te[((end ? 2 : 4) * 5 + v) * QF2 + q] = O[(ve * QF + q / QF) * FP + q % QF];
  }
  // faces 1 / 3: [5][QF][2][QF]
  con_mid<5, L, 2, L, QF, LP, LP, NT>(EO<P>::Bg(), K1, W, tid);       // [5][QF][2][L]
  __syncthreads();
  con_last<10 * QF, L, QF, LP, FP, NT>(EO<P>::Bg(), W, O, tid);       // [5][QF][2][QF]
  __syncthreads();
  for (int i = tid; i < 10 * QF2; i += NT) {
    const int v = i / (2 * QF2), r = i - v * 2 * QF2, end = r / QF2, q = r - end * QF2;
    const int ia = q / QF, ic = q - ia * QF;
    Te[((end ? 3 : 1) * 5 + v) * QF2 + q] = O[((v * QF + ia) * 2 + end) * FP + ic];
  }
  // faces 0 / 5: [5][QF][QF][2]
  con_mid<5, L, L, 2, QF, KP, KP, NT>(EO<P>::Bg(), K2, W, tid);       // [5][QF][L][2]
  __syncthreads();
  con_mid<5 * QF, L, 1, 2, QF, KP, KP, NT>(EO<P>::Bg(), W, O, tid);   // [5][QF][QF][2]
  __syncthreads();
  for (int i = tid; i < 10 * QF2; i += NT) {
    const int v = i / (2 * QF2), r = i - v * 2 * QF2, end = r / QF2, q = r - end * QF2;
    Te[((end ? 5 : 0) * 5 + v) * QF2 + q] = O[(v * QF2 + q) * KP + end];
  }
}

// BR2 correction of the normal viscous flux at GLL node (i, j, k) on face f of
// an affine hex (faces: 0 z-, 1 y-, 2 x+, 3 y+, 4 x-, 5 z+).  The nodal
// stresses come from the gradient lifted over all six faces,
// G = grad_h q + sum_d r_d; BR2 evaluates the face flux with grad_h q + eta r_f
// instead, so fd receives the flux (equations 1..4, contracted with n) of the
// velocity / energy gradient increment
//   -sum_d r_d + eta (lifting of face f alone).
// Hn[(c*6 + s)][Q][Q] (pitch QP) holds the nodal values, at face s's GLL
// points, of the modal face lift of primitive c (u, v, w, e) on face s, without
// the 1/|grad xi_d| factor; KE[2][Q] = sum_l phi_l(-+1) phi_l(xi_i).  The
// lifting across reference direction d at a node is then
//   r_d = (KE[1][xi_d] Hn[face d+] - KE[0][xi_d] Hn[face d-]) / |grad xi_d|,
// with physical components grad(xi_d) r_d; gs[3d + x] = grad(xi_d)_x / |grad xi_d|.
// A gradient increment g (x) a (du_i/dx_j = g_j a_i) has stress . n
//   mu (a_i (g.n) + g_i (a.n)) - 2/3 mu (g.a) n_i
// and heat flux . n = kappa a_e (g.n).
template <int Q, int QP, typename R, typename RT>
__device__ __forceinline__ void br2_flux(R (&fd)[4], const R *Hn, const RT *KE, int f, int i, int j, int k,
                                         const R *gs, R mu, R kap, R eta, R u, R v, R w, R n0, R n1, R n2) {
  const int df = (f == 2 || f == 4) ? 0 : ((f == 1 || f == 3) ? 1 : 2);
  const bool hi = (f == 2 || f == 3 || f == 5);
  const R c23 = mu * R(2.0 / 3.0);
  R r0 = R(0), r1 = R(0), r2 = R(0), he = R(0);
#pragma unroll
  for (int d = 0; d < 3; ++d) {   // unrolled: all LDS loads in flight at once
    const int slo = d == 0 ? 4 : (d == 1 ? 1 : 0), shi = d == 0 ? 2 : (d == 1 ? 3 : 5);
    const int x = d == 0 ? i : (d == 1 ? j : k);
    const int t1 = d == 0 ? j : i, t2 = d == 2 ? j : k;
    const R klo = R(KE[x]), khi = R(KE[Q + x]);
    R a[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const R hl = Hn[((c * 6 + slo) * Q + t1) * QP + t2], hh = Hn[((c * 6 + shi) * Q + t1) * QP + t2];
      R val = klo * hl - khi * hh;                                // -r_d |grad xi_d|
      if (d == df) val += eta * (hi ? khi * hh : -(klo * hl));   // + eta * lifting of face f
      a[c] = val;
    }
    const R g0 = gs[3 * d], g1 = gs[3 * d + 1], g2 = gs[3 * d + 2];
    const R gn = g0 * n0 + g1 * n1 + g2 * n2;
    const R an = a[0] * n0 + a[1] * n1 + a[2] * n2;
    const R ga = g0 * a[0] + g1 * a[1] + g2 * a[2];
    r0 += mu * (a[0] * gn + g0 * an) - c23 * ga * n0;
    r1 += mu * (a[1] * gn + g1 * an) - c23 * ga * n1;
    r2 += mu * (a[2] * gn + g2 * an) - c23 * ga * n2;
    he += kap * a[3] * gn;
  }
  fd[0] = r0;
  fd[1] = r1;
  fd[2] = r2;
  fd[3] = (r0 * u + r1 * v + r2 * w) + he;
}

}  // namespace dgx
