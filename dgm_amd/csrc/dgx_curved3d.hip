// Curved hexes (Euler3d, p <= 8): the residual with metrics at the nodes and
// the projection through the element mass matrix.
//
//   volume term   Euler3d::convection with Hex::gradient on curved geometry:
//                 dF_x/dx = sum_d (dxi_d/dx)(node) D_d F_x at every node
//                 (src/Euler3d.cpp:468-575, src/Hex.cpp:2030-2071, 3992-4080)
//   faces         the Riemann flux with the master side's normal at each Gauss
//                 point (Euler3d::convective_flux evaluates a pair once, on its
//                 master side), lifted at the face nodes:
//                 G2GL((Fhat - F-.n) J_side/J_vol) / w_end (src/Hex.cpp:1786-1952)
//   project       b = B^T (wJ f) and M x = b with M = B^T diag(wJ) B, the curved
//                 element's mass matrix (src/Hex.cpp:289-318), solved inside
//                 the workgroup by corrections with a preconditioner, and by
//                 conjugate gradients where those converge slowly (MassSolve).
//                 The preconditioner is the exact inverse for a separable fit
//                 J ~ ja(xi) jb(eta) jc(zeta): the tensor product of three
//                 L x L inverses per element, built on the host.  On smoothly
//                 curved elements the fit leaves M's spectrum close to the
//                 preconditioner's, so a few corrections reach rounding.
#include <type_traits>
#include <vector>

#include "dgx_contract.hpp"
#include "dgx_kernels.hpp"

namespace dgx {

// Float copies of the basis tables for the mixed residual (FP32 contractions
// and derivatives; FP64 metrics, fluxes, state and the mass solve), filled
// beside c_tab at upload.  TE3<R, P> gives the even-odd tables of arithmetic
// type R.
static __constant__ float c_tabf3[kTabTotal];
struct EoBaseF3 {
  using R = float;
  __device__ static __forceinline__ const float *base() { return c_tabf3; }
};
template <typename R, int P> using TE3 = EOx<std::conditional_t<std::is_same<R, double>::value, EoBaseD, EoBaseF3>, P>;

template <int P> struct C3 {
  static constexpr int L = P + 1, Q = P + 2, QF = P + 1;
  static constexpr int L2 = L * L, L3 = L2 * L, Q2 = Q * Q, Q3 = Q2 * Q, QF2 = QF * QF;
  static constexpr int LP = odd(L), QP = odd(Q), FP = odd(QF);   // pitches of last dimensions
  // one thread per pencil of 5 fields (p = 4: also one per node)
  static constexpr int NT = P == 4 ? 256 : round64(5 * Q2);
  static constexpr int NPT = (Q3 + NT - 1) / NT;          // nodes per thread
  static constexpr int NML = (5 * L3 + NT - 1) / NT;      // modal entries per thread (5 fields)
  // LDS (doubles): W1, W2 [SZ], the largest tensor of any phase; G [GZ], the
  // face terms gF [5][6][QF][QF], then wJ and the mass solve's reductions
  static constexpr int SZ = cmax(5 * Q2 * QP, 30 * Q * cmax(QP, FP));
  static constexpr int GZ = cmax(30 * QF * FP, Q2 * QP + 2 * NT + 64);
  static constexpr int lds = (2 * SZ + GZ) * 8;
  static __device__ __forceinline__ int nidx(int n) { return (n / Q) * QP + n % Q; }   // padded node index
};

// Sums over each field's pencils of NV values per thread (thread f L2 + k holds
// pencil k of field f) into tot[v][f]: 8 partial sums per field in a fixed order.
template <int NF, int L2, int NT, int NV>
__device__ __forceinline__ void field_sums(const double (&v)[NV], double *red, double *tot, int tid) {
  if (tid < NF * L2) {
#pragma unroll
    for (int k = 0; k < NV; ++k) red[k * NT + tid] = v[k];
  }
  __syncthreads();
  for (int q = tid; q < NV * NF * 8; q += NT) {
    const int k = q / (NF * 8), f = (q >> 3) % NF;
    double s = 0.0;
    for (int i = q & 7; i < L2; i += 8) s += red[k * NT + f * L2 + i];
#pragma unroll
    for (int o = 4; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if ((q & 7) == 0) tot[k * NF + f] = s;
  }
  __syncthreads();
}

// The curved element's mass solve M x = b, M = B^T diag(wJ) B, for NF fields.
// One thread owns a pencil and keeps its vector entries in registers: r along
// a (thread f L2 + m L + n), x and z along c (thread f L2 + l L + m).  The
// preconditioner and M are each a chain of phases over W1, W2 whose
// neighbouring contractions along one direction run on the same pencil, so
// that an application of both takes seven LDS phases instead of twelve:
//   Pa | Pb | Pc, BT_c | BT_a | BT_b, wJ, BL_b | BL_c | BL_a
// The preconditioner's matrices are the same for the whole workgroup and come
// as scalar operands.
template <int P, int NF, int NT> struct MassSolve {
  static constexpr int L = P + 1, Q = P + 2, L2 = L * L, LP = odd(L), QP = odd(Q);
  static_assert(NF * L2 <= NT, "one pencil per thread");
  double *W1, *W2;
  const double *wJ;               // [Q][Q] rows of pitch QP
  const double *__restrict__ pre; // [3][L][L]
  int tid;

  static __device__ __forceinline__ void matvec(const double *__restrict__ M, const double (&x)[L], double (&y)[L]) {
#pragma unroll
    for (int o = 0; o < L; ++o) {
      double s = 0.0;
#pragma unroll
      for (int i = 0; i < L; ++i) s = fma(M[o * L + i], x[i], s);
      y[o] = s;
    }
  }
  // the thread's pencil: element k at base + k stride
  __device__ __forceinline__ int base_a() const {   // [NF][L][L][L], along a
    const int f = tid / L2, m = (tid / L) % L, n = tid % L;
    return (f * L2 + m) * LP + n;
  }
  __device__ __forceinline__ int base_c() const { return tid * LP; }   // along c
  __device__ __forceinline__ bool mine() const { return tid < NF * L2; }

  // the preconditioner's matrices as scalar loads (the pointer may come from
  // memory, in conjugate)
  __device__ __forceinline__ const double *pmat(int d) const {
    const uint64_t b = (uint64_t)(pre + d * L2);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)b),
                   hi = __builtin_amdgcn_readfirstlane((uint32_t)(b >> 32));
    return uniform_const((const double *)(((uint64_t)hi << 32) | lo));
  }

  // z = P r
  __device__ __forceinline__ void precondition(const double (&r)[L], double (&z)[L]) {
    if (mine()) {
      double y[L];
      matvec(pmat(0), r, y);
      const int b = base_a();
#pragma unroll
      for (int k = 0; k < L; ++k) W1[b + k * L * LP] = y[k];
    }
    __syncthreads();
    if (mine()) {   // along b, in place
      const int f = tid / L2, l = (tid / L) % L, n = tid % L, b = (f * L + l) * L * LP + n;
      double x[L], y[L];
#pragma unroll
      for (int k = 0; k < L; ++k) x[k] = W1[b + k * LP];
      matvec(pmat(1), x, y);
#pragma unroll
      for (int k = 0; k < L; ++k) W1[b + k * LP] = y[k];
    }
    __syncthreads();
    if (mine()) {
      double x[L];
      const int b = base_c();
#pragma unroll
      for (int k = 0; k < L; ++k) x[k] = W1[b + k];
      matvec(pmat(2), x, z);
    }
  }

  // y = M z (z along c, y along a)
  __device__ __forceinline__ void apply(const double (&z)[L], double (&y)[L]) {
    if (mine()) {
      double t[Q];
      eo_apply<EO_MN, L, Q>(fresh(EO<P>::BT()).h, z, t);
#pragma unroll
      for (int k = 0; k < Q; ++k) W2[tid * QP + k] = t[k];             // [NF][L][L][Q]
    }
    __syncthreads();
    con_mid<NF, L, L, Q, Q, QP, QP, NT>(fresh(EO<P>::BT()), W2, W1, tid);     // [NF][Q][L][Q]
    __syncthreads();
    for (int pc = tid; pc < NF * Q * Q; pc += NT) {                    // along b, in place
      const int fa = pc / Q, c = pc - fa * Q, b = fa * L * QP + c, w = (fa % Q) * Q * QP + c;
      double x[L], t[Q], u[L];
#pragma unroll
      for (int k = 0; k < L; ++k) x[k] = W1[b + k * QP];
      eo_apply<EO_MN, L, Q>(fresh(EO<P>::BT()).h, x, t);
#pragma unroll
      for (int k = 0; k < Q; ++k) t[k] *= wJ[w + k * QP];
      eo_apply<EO_NM, Q, L>(fresh(EO<P>::BL()).h, t, u);
#pragma unroll
      for (int k = 0; k < L; ++k) W1[b + k * QP] = u[k];
    }
    __syncthreads();
    con_last<NF * Q * L, Q, L, QP, LP, NT>(fresh(EO<P>::BL()), W1, W2, tid);  // [NF][Q][L][L]
    __syncthreads();
    if (mine()) {
      const int f = tid / L2, mn = tid % L2, m = mn / L, n = mn - m * L;
      double t[Q];
#pragma unroll
      for (int k = 0; k < Q; ++k) t[k] = W2[((f * Q + k) * L + m) * LP + n];
      eo_apply<EO_NM, Q, L>(fresh(EO<P>::BL()).h, t, y);
    }
  }

  // a vector along a -> the same along c, and back (through W1)
  __device__ __forceinline__ void turn(const double (&v)[L], double (&u)[L], bool to_c) {
    __syncthreads();
    if (mine()) {
      const int b = to_c ? base_a() : base_c(), s = to_c ? L * LP : 1;
#pragma unroll
      for (int k = 0; k < L; ++k) W1[b + k * s] = v[k];
    }
    __syncthreads();
    if (mine()) {
      const int b = to_c ? base_c() : base_a(), s = to_c ? 1 : L * LP;
#pragma unroll
      for (int k = 0; k < L; ++k) u[k] = W1[b + k * s];
    }
    __syncthreads();
  }

  static __device__ __forceinline__ double dot(const double (&u)[L], const double (&v)[L]) {
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < L; ++k) s = fma(u[k], v[k], s);
    return s;
  }

  // x = M^-1 r (r: the right-hand side, along a; overwritten).  Corrections
  // z = P r with the residual recomputed after each: on smoothly curved
  // elements P is close to M^-1, each correction leaves a small share of the
  // residual, and the last one needs no residual after it, once the observed
  // rate says that it falls to 1e-15 |b|.  (The slowest part of the residual
  // makes up more of it with each correction, so the rate can only grow and the
  // prediction errs low: at bump and twisted hexes of p = 2..7 what remains is
  // up to 1.15e-15 |b|.)  A bump of height 0.1 in a 3 x 3 x 1 channel takes at
  // most 6 applications of M at 4^3 and 6^3 hexes, 5 at 12^3 and 4 at 24^3
  // (p = 2..7), with one inner product each where conjugate gradients have
  // three.  A rate above 1/20 goes to conjugate gradients, on what is left.
  // red: 2 NT doubles, tot: 6 NF.  Returns the applications of M.
  __device__ __forceinline__ int solve(double (&r)[L], double *red, double *tot, double (&x)[L]) {
    constexpr double tol2 = 1e-30;   // (1e-15 relative)^2
    double z[L], y[L];
#pragma unroll
    for (int k = 0; k < L; ++k) x[k] = 0.0;
    double b2 = mine() ? dot(r, r) : 0.0;
    int it = 0, go = 1;   // go: 1 correct again, 2 correct once more and stop, 3 conjugate gradients, 0 done
    for (;;) {
      precondition(r, z);
      if (mine()) {
#pragma unroll
        for (int k = 0; k < L; ++k) x[k] += z[k];
      }
      if (go == 2) return it;
      apply(z, y);
      ++it;
      if (mine()) {
#pragma unroll
        for (int k = 0; k < L; ++k) r[k] -= y[k];
      }
      // |b|^2 in tot[0..NF), |r|^2 of the previous and this residual after it
      if (it == 1) {
        const double v[2] = {b2, mine() ? dot(r, r) : 0.0};
        field_sums<NF, L2, NT, 2>(v, red, tot, tid);
      } else {
        const double v[1] = {mine() ? dot(r, r) : 0.0};
        field_sums<NF, L2, NT, 1>(v, red, tot + (it & 1 ? NF : 2 * NF), tid);
      }
      const double *prev = it == 1 ? tot : tot + (it & 1 ? 2 * NF : NF), *cur = tot + (it & 1 ? NF : 2 * NF);
      bool done = true, last = true, slow = false;
#pragma unroll
      for (int f = 0; f < NF; ++f) {
        const double lim = tol2 * tot[f];
        // |b|^2 near 1, exactly: the squares below stay in range at any scale of the field
        const int ex = -__builtin_amdgcn_frexp_exp(tot[f]);
        const double c = ldexp(cur[f], ex);
        done = done && cur[f] <= lim;
        last = last && (cur[f] <= lim || c * c <= ldexp(lim, ex) * ldexp(prev[f], ex));
        slow = slow || (cur[f] > lim && cur[f] > 2.5e-3 * prev[f]);
      }
      if (done) return it;
      if (!last && (slow || it >= 8)) break;
      if (last) go = 2;
    }
    return it + conjugate(r, red, tot, x);
  }

  // conjugate gradients on M d = r added to x; tot[0..NF) holds |b|^2
  __device__ __forceinline__ int conjugate(double (&ra)[L], double *red, double *tot, double (&x)[L]) {
    double r[L], p[L], z[L], y[L], yc[L];
    double *rz = tot + 3 * NF;
    turn(ra, r, true);
    precondition(ra, p);
    {
      const double v[1] = {mine() ? dot(r, p) : 0.0};
      field_sums<NF, L2, NT, 1>(v, red, rz, tid);
    }
    int it = 0;
    for (; it < 60; ++it) {
      const int f = mine() ? tid / L2 : 0;
      apply(p, y);
      turn(y, yc, true);
      const double v[1] = {mine() ? dot(p, yc) : 0.0};
      field_sums<NF, L2, NT, 1>(v, red, tot + NF, tid);
      const double alpha = (rz[f] > 0.0 && tot[NF + f] > 0.0) ? rz[f] / tot[NF + f] : 0.0, old = rz[f];
      if (mine()) {
#pragma unroll
        for (int k = 0; k < L; ++k) { x[k] = fma(alpha, p[k], x[k]); r[k] = fma(-alpha, yc[k], r[k]); }
      }
      turn(r, y, false);
      precondition(y, z);
      const double w[2] = {mine() ? dot(r, r) : 0.0, mine() ? dot(r, z) : 0.0};
      double *t2 = tot + 4 * NF;
      field_sums<NF, L2, NT, 2>(w, red, t2, tid);
      bool conv = true;
#pragma unroll
      for (int g = 0; g < NF; ++g) conv = conv && t2[g] <= 1e-30 * tot[g];
      if (conv) { ++it; break; }
      const double beta = old > 0.0 ? t2[NF + f] / old : 0.0;
      if (mine()) {
#pragma unroll
        for (int k = 0; k < L; ++k) p[k] = fma(beta, p[k], z[k]);
      }
      __syncthreads();
      if (tid < NF) rz[tid] = t2[NF + tid];
      __syncthreads();
    }
    return it;
  }
};

// Weighted divergence at the nodes, Out[v] += sum_d gm[d][X] D_d F_X of NV
// fields for one Cartesian component X whose fluxes F holds ([NV][Q][Q][Q],
// pitch QP): one pencil of each reference direction in turn, its outputs
// scaled by the metric term at their nodes.  `first` writes Out.  The nine
// terms of a node cancel to a large part, so they are summed in FP64 also where
// the derivatives are FP32.
// `beside(d)` is other work of the phase of direction d, on other buffers.
template <int P, int NV, int NT, typename R, class F2>
__device__ __forceinline__ void metric_deriv(EoMat<EO_NNA, R> D, const R *F, double *Out, const double *ge, int X, bool first,
                                             int tid, F2 beside) {
  using S = C3<P>;
  constexpr int Q = S::Q, Q2 = S::Q2, Q3 = S::Q3, QP = S::QP;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    // strides of direction d among the metric's nodes and in the LDS tensors
    const int sn = d == 0 ? Q2 : (d == 1 ? Q : 1), sl = d == 0 ? Q * QP : (d == 1 ? QP : 1);
    for (int pc = tid; pc < NV * Q2; pc += NT) {
      const int v = pc / Q2, t = pc - v * Q2, t1 = t / Q, t2 = t - t1 * Q;
      const int node = d == 0 ? t : (d == 1 ? t1 * Q2 + t2 : t * Q);
      const int b = v * Q2 * QP + (d == 0 ? t1 * QP + t2 : (d == 1 ? t1 * Q * QP + t2 : t * QP));
      const double *g = ge + (3 * d + X) * Q3 + node;
      double m[Q];
#pragma unroll
      for (int k = 0; k < Q; ++k) m[k] = g[k * sn];
      R x[Q], y[Q];
#pragma unroll
      for (int k = 0; k < Q; ++k) x[k] = F[b + k * sl];
      eo_apply<EO_NNA, Q, Q>(fresh(D).h, x, y);
#pragma unroll
      for (int k = 0; k < Q; ++k) {
        const double val = m[k] * (double)y[k];
        if (first && d == 0) Out[b + k * sl] = val;
        else Out[b + k * sl] += val;
      }
    }
    beside(d);
    __syncthreads();
  }
}

// PROJ: project the nodal fields a.U [5][ne][Q^3] instead (the forward
// transform of a curved element: x = M^-1 B^T (wJ u)).
// Bound by the latency of its LDS phases: about 45 barriers per element, each
// contraction one pencil per thread.  Two LDS tensors and the face terms are
// 37 KB at p = 5, so four workgroups share a CU (four wavefronts per SIMD, at
// most 128 VGPRs).  On the bump channel's 24^3 hexes at p = 5 a stage went from
// 1.76 ms (this kernel with conjugate gradients and one thread per node's
// derivatives, and the traces' own kernel) to 0.65 ms.
// R: arithmetic of the residual before the mass solve (its element tensors,
// contractions and derivatives; the weighted divergence and the face terms are
// summed in FP64): double, or float on the mixed path, whose LDS views alias
// the same memory as the FP64 buffers of the mass solve.
// NS: Navier-Stokes (BR1), adding the viscous terms k_grad3c and k_visc3c
// wrote: the weighted nodal divergence V is subtracted before the projection,
// and each interior side's correction gains J_side/J_vol (1/2)(F_v.n- + F_v+.n+)
// (the BR1 face flux is the average of the two sides' own normal fluxes; a
// boundary side's ghost flux is -F_v, so its face flux is its own).
template <int P, bool PROJ, typename R = double, bool NS = false>
__global__ void __launch_bounds__(C3<P>::NT) __attribute__((amdgpu_waves_per_eu(lds_waves(C3<P>::lds, C3<P>::NT))))
k_rhs3c(CurvedArgs a, const double *__restrict__ gm, const double *__restrict__ pre) {
  using S = C3<P>;
  using TR = TE3<R, P>;
  constexpr int L = S::L, Q = S::Q, QF = S::QF, L2 = S::L2, L3 = S::L3, Q2 = S::Q2, Q3 = S::Q3, QF2 = S::QF2;
  constexpr int LP = S::LP, QP = S::QP, FP = S::FP, FS = Q2 * QP, NT = S::NT, NPT = S::NPT, NML = S::NML;
  extern __shared__ double sm[];
  double *W1 = sm, *W2 = W1 + S::SZ, *G = W2 + S::SZ;
  // the residual's views (type R) of the same buffers
  R *W1r = reinterpret_cast<R *>(W1), *W2r = reinterpret_cast<R *>(W2), *gF = reinterpret_cast<R *>(G);
  static_assert(S::lds <= 160 * 1024, "LDS");
  const int ne = a.ne, e = xcd_element(blockIdx.x, ne), tid = threadIdx.x;
  const Geo &geo = a.geo;
  const double *ge = gm + (size_t)e * 10 * Q3;   // wJ dxi_d/dx_x (9 rows), wJ
  const double gm1 = a.phys.gamma - 1.0;

  if (PROJ) {
    for (int i = tid; i < 5 * Q3; i += NT) {
      const int v = i / Q3, n = i - v * Q3;
      W1r[v * FS + S::nidx(n)] = (R)(ge[9 * Q3 + n] * a.U[((size_t)v * ne + e) * Q3 + n]);
    }
    for (int n = tid; n < Q3; n += NT) G[S::nidx(n)] = ge[9 * Q3 + n];
    __syncthreads();
  } else {
    // the modal state's loads are issued first; they land in LDS after the face
    // loop, whose dependent loads (links, orientation, neighbour traces) they overlap
    double um[NML];
#pragma unroll
    for (int k = 0; k < NML; ++k) {
      const int i = tid + k * NT, v = i / L3;
      um[k] = i < 5 * L3 ? a.U[((size_t)v * ne + e) * L3 + (i - v * L3)] : 0.0;
    }
    // face corrections g = (J_side/J_vol)(Fhat - F(U-).n) at the Gauss points,
    // before the nodal state is live (the Riemann solver's temporaries and it
    // would not fit in registers beside each other)
    bool bad = false;
    for (int i = tid; i < 6 * QF2; i += NT) {
      const int s = i / QF2, q = i - s * QF2;
      const int es = e * 6 + s;
      const double *fg = a.fgeo + ((size_t)es * QF2 + q) * 4;
      double nx = fg[0], ny = fg[1], nz = fg[2];
      const double jr = fg[3];
      const int nb = geo.nbr[es], ns = geo.nside[es];
      double UL[5], UR[5], FL[5], Fh[5];
      const double *tl = a.T + ((size_t)e * 6 + s) * 5 * QF2;
#pragma unroll
      for (int v = 0; v < 5; ++v) UL[v] = tl[v * QF2 + q];
      int qn = q;
      if (nb >= 0) {
        qn = geo.perm[geo.permid[es] * QF2 + q];
        if (!geo.master[es]) {   // the pair's flux uses the master side's normal (both sides' normals
                                 // come from their own interpolated metrics and differ slightly)
          const double *fm = a.fgeo + (((size_t)nb * 6 + ns) * QF2 + qn) * 4;
          nx = -fm[0]; ny = -fm[1]; nz = -fm[2];
        }
        const double *tr = a.T + ((size_t)nb * 6 + ns) * 5 * QF2;
#pragma unroll
        for (int v = 0; v < 5; ++v) UR[v] = tr[v * QF2 + qn];
      } else {
        ghost3(-1 - nb, UL, nx, ny, nz, a.phys.bcU, UR);
      }
      riemann3(UL, UR, nx, ny, nz, a.phys.gamma, a.phys.flux, FL, Fh, bad);
      const int qa = q / QF, qb = q - qa * QF;
#pragma unroll
      for (int v = 0; v < 5; ++v) {
        double g = jr * (Fh[v] - FL[v]);
        if (NS && v > 0 && nb >= 0) {
          const double *vl = a.TV + ((size_t)e * 6 + s) * 4 * QF2, *vr = a.TV + ((size_t)nb * 6 + ns) * 4 * QF2;
          g += 0.5 * jr * (vl[(v - 1) * QF2 + q] + vr[(v - 1) * QF2 + qn]);
        }
        gF[((v * 6 + s) * QF + qa) * FP + qb] = (R)g;
      }
    }
    if (bad) atomicOr(a.flag, 1);

    // modal state -> nodal (5 fields), each thread keeping its nodes in registers
#pragma unroll
    for (int k = 0; k < NML; ++k) {
      const int i = tid + k * NT, v = i / L3, m = i - v * L3;
      if (i < 5 * L3) W1r[(v * L2 + m / L) * LP + m % L] = (R)um[k];
    }
    __syncthreads();
    con_mid<5, L, L, L, Q, LP, LP, NT>(TR::BT(), W1r, W2r, tid);
    __syncthreads();
    con_mid<5 * Q, L, 1, L, Q, LP, LP, NT>(TR::BT(), W2r, W1r, tid);
    __syncthreads();
    con_last<5 * Q2, L, Q, LP, QP, NT>(TR::BT(), W1r, W2r, tid);
    __syncthreads();
    double un[NPT][5];
#pragma unroll
    for (int rr = 0; rr < NPT; ++rr) {
      const int n = tid + rr * NT, pn = S::nidx(n < Q3 ? n : 0);
#pragma unroll
      for (int v = 0; v < 5; ++v) un[rr][v] = n < Q3 ? (double)W2r[v * FS + pn] : 1.0;
    }
    // volume: wJ * sum_x sum_d (dxi_d/dx_x) D_d F_x at every node, one Cartesian
    // component of all 5 fluxes at a time
#pragma unroll 1
    for (int x = 0; x < 3; ++x) {
#pragma unroll
      for (int rr = 0; rr < NPT; ++rr) {
        const int n = tid + rr * NT;
        if (n >= Q3) continue;
        const int pn = S::nidx(n);
        const double ir = 1.0 / un[rr][0], mx = un[rr][1], my = un[rr][2], mz = un[rr][3], E = un[rr][4];
        const double p = gm1 * (E - 0.5 * (mx * (mx * ir) + my * (my * ir) + mz * (mz * ir)));
        const double m = x == 0 ? mx : (x == 1 ? my : mz), u = m * ir;
        W1r[pn] = (R)m;
        W1r[FS + pn] = (R)(x == 0 ? mx * u + p : mx * u);
        W1r[2 * FS + pn] = (R)(x == 1 ? my * u + p : my * u);
        W1r[3 * FS + pn] = (R)(x == 2 ? mz * u + p : mz * u);
        W1r[4 * FS + pn] = (R)((E + p) * u);
      }
      __syncthreads();
      metric_deriv<P, 5, NT, R>(TR::DN(), W1r, W2, ge, x, x == 0, tid, [](int) {});
    }
    double acc[NPT][5], wj[NPT];
#pragma unroll
    for (int rr = 0; rr < NPT; ++rr) {
      const int n = tid + rr * NT, pn = S::nidx(n < Q3 ? n : 0);
      wj[rr] = n < Q3 ? ge[9 * Q3 + n] : 0.0;
#pragma unroll
      for (int v = 0; v < 5; ++v) {
        acc[rr][v] = n < Q3 ? W2[v * FS + pn] : 0.0;
        if (NS && v > 0 && n < Q3) acc[rr][v] -= a.V[((size_t)e * 4 + v - 1) * Q3 + n];
      }
    }
    // faces: Gauss -> GLL face nodes for 30 blocks, then wJ / w_end at the face nodes
    con_mid<30, QF, 1, QF, Q, FP, FP, NT>(TR::GL(), gF, W1r, tid);     // [30][Q][QF]
    __syncthreads();
    con_last<30 * Q, QF, Q, FP, QP, NT>(TR::GL(), W1r, W2r, tid);      // [30][Q][Q]
    __syncthreads();
    const double iwend = CT<P>::BT()[0] / CT<P>::BW()[0];   // 1 / GLL end weight: phi_0 / (phi_0 w_0)
#pragma unroll
    for (int rr = 0; rr < NPT; ++rr) {
      const int n = tid + rr * NT;
      if (n < Q3) {
        const int i = n / Q2, j = (n / Q) % Q, k = n % Q, pn = S::nidx(n);
        const double c = wj[rr] * iwend;
        // the faces the node lies on, in a fixed order, each with a constant
        // face (no indexed arrays, which would live in scratch)
        auto add = [&](int f, int a1, int a2) {
#pragma unroll
          for (int v = 0; v < 5; ++v)
            acc[rr][v] = fma(c, (double)W2r[((v * 6 + f) * Q + a1) * QP + a2], acc[rr][v]);
        };
        if (k == 0) add(0, i, j);
        if (k == Q - 1) add(5, i, j);
        if (j == 0) add(1, i, k);
        if (j == Q - 1) add(3, i, k);
        if (i == 0) add(4, j, k);
        if (i == Q - 1) add(2, j, k);
#pragma unroll
        for (int v = 0; v < 5; ++v) W1r[v * FS + pn] = (R)acc[rr][v];
        G[pn] = wj[rr];
      }
    }
    __syncthreads();
  }   // !PROJ
  // b = B^T (wJ f), its last contraction into the registers of the mass solve
  con_last<5 * Q2, Q, L, QP, LP, NT>(TR::BL(), W1r, W2r, tid);
  __syncthreads();
  con_mid<5 * Q, Q, 1, L, L, LP, LP, NT>(TR::BL(), W2r, W1r, tid);     // [5][Q][L][L]
  __syncthreads();
  MassSolve<P, 5, NT> ms{W1, W2, G, pre + (size_t)e * 3 * L2, tid};
  double r[L], x[L];
  if (ms.mine()) {
    const int f = tid / L2, mn = tid % L2, m = mn / L, n = mn - m * L;
    R t[Q], y[L];
#pragma unroll
    for (int k = 0; k < Q; ++k) t[k] = W1r[((f * Q + k) * L + m) * LP + n];
    eo_apply<EO_NM, Q, L>(TR::BL().h, t, y);
#pragma unroll
    for (int k = 0; k < L; ++k) r[k] = y[k];
  }
  __syncthreads();
  double *red = G + FS, *tot = red + 2 * NT;
  const int it = ms.solve(r, red, tot, x);
  // the residual, or (update) the LSRK stage in place: this element's modes
  // were read at the start and no other workgroup reads them
  if (ms.mine()) {
    const int v = tid / L2;
    const size_t o = ((size_t)v * ne + e) * L3 + (tid - v * L2) * L;
    if (!PROJ && a.update) {
      const double mdt = -a.dt;
      double ut[L], u[L];
#pragma unroll
      for (int k = 0; k < L; ++k) { ut[k] = a.Ut[o + k]; u[k] = a.Us[o + k]; }
#pragma unroll
      for (int k = 0; k < L; ++k) {
        ut[k] = fma(mdt, x[k], a.ca * ut[k]);          // as the axpby Ut = ca Ut - dt R
        a.Ut[o + k] = ut[k];
        u[k] = fma(a.cb, ut[k], u[k]);                 // as the axpy U += cb Ut
        a.Us[o + k] = u[k];
        W2[tid * LP + k] = u[k];
      }
    } else {
#pragma unroll
      for (int k = 0; k < L; ++k) a.R[o + k] = x[k];
    }
  }
  if (tid == 0 && a.iters) atomicMax(a.iters, it);
  if (PROJ || !a.update || !a.Tn) return;
  // face traces of the updated state for the next stage
  static_assert(10 * QF * cmax(LP, 3 * L) + 15 * QF2 <= S::SZ && 20 * L * LP + 15 * L2 <= S::SZ, "trace buffers");
  __syncthreads();
  face_traces3<P, NT>(W2, W1, a.Tn + (size_t)e * 30 * QF2, tid);
}

// Navier-Stokes (BR1) on curved hexes, in the order of Navier_Stokes3d::diffusion
// (src/Navier_Stokes3d.cpp:113-258): k_grad3c lifts and projects the gradients
// of the primitives (u, v, w, e), k_visc3c forms the stresses and heat flux
// and writes their weighted divergence and each side's normal flux, and
// k_rhs3c<P, false, double, true> adds both to the Euler residual before its
// one projection.
template <int P> struct C3V {
  using B = C3<P>;
  static constexpr int L = P + 1, Q = P + 2, QF = P + 1;
  static constexpr int L2 = L * L, L3 = L2 * L, Q2 = Q * Q, Q3 = Q2 * Q, QF2 = QF * QF;
  static constexpr int LP = odd(L), QP = odd(Q), FP = odd(QF), FS = Q2 * QP;
  // k_grad3c: two primitives' gradients (6 components) per pass, one thread
  // per pencil of 6 fields
  static constexpr int NT = round64(6 * Q2), NPT = (Q3 + NT - 1) / NT;
  // LDS (doubles): Pq [4] the primitives at the nodes; Jq [4][6] the jumps;
  // W1, W2 [SZ]; wJ and the mass solve's reductions
  static constexpr int SZ = cmax(6 * FS, 36 * Q * cmax(QP, FP));
  static constexpr int grad = (4 * FS + 24 * QF * FP + 2 * SZ + FS + 2 * NT + 64) * 8;
  // k_visc3c: W1, W2 [6 FS] (transforms of 6 fields; one Cartesian component
  // of the 4 fluxes and their divergences); W3, W4 the 24 face blocks
  static constexpr int visc = (12 * FS + 24 * Q * QP + 24 * QF * QP) * 8;
};

bool curved3_ns_supported(int p) { return p >= 1 && p <= 7; }

// Lifted, projected gradients of (u, v, w, e) of a curved hex (the
// Euler3d::gradient_lift path, src/Euler3d.cpp:1144-1199): at the nodes
// wJ dq/dx_x = sum_d (wJ dxi_d/dx_x) D_d q, plus at the face nodes
// (wJ / w_end) G2GL(J_side/J_vol ({q} - q-) n_x) with the side's own normal,
// then M^-1 B^T of that.  G [ne][12][L3] in the order (u_x, u_y, u_z, v_x,
// ..., e_z).  A boundary side's ghost primitives are the isothermal wall's or
// the imposed state's (ghost_prim3).
// Bound, like k_rhs3c, by the latency of its LDS phases; the two mass solves
// of 6 fields are most of them (14^3 hexes at p = 4: 0.70 -> 0.19 ms).
template <int P>
__global__ void __launch_bounds__(C3V<P>::NT) __attribute__((amdgpu_waves_per_eu(lds_waves(C3V<P>::grad, C3V<P>::NT))))
k_grad3c(CurvedArgs a, const double *__restrict__ gm, const double *__restrict__ pre) {
  using S = C3V<P>;
  constexpr int L = S::L, Q = S::Q, QF = S::QF, L2 = S::L2, L3 = S::L3, Q2 = S::Q2, Q3 = S::Q3, QF2 = S::QF2;
  constexpr int LP = S::LP, QP = S::QP, FP = S::FP, FS = S::FS, NT = S::NT, NPT = S::NPT;
  extern __shared__ double sm[];
  double *Pq = sm, *Jq = Pq + 4 * FS, *W1 = Jq + 24 * QF * FP, *W2 = W1 + S::SZ, *wJ = W2 + S::SZ;
  double *red = wJ + FS, *tot = red + 2 * NT;
  static_assert(S::grad <= 160 * 1024, "LDS");
  const int ne = a.ne, e = xcd_element(blockIdx.x, ne), tid = threadIdx.x;
  const Geo &geo = a.geo;
  const double *ge = gm + (size_t)e * 10 * Q3;
  // modal state, landing in LDS after the jump loop
  constexpr int NML = (5 * L3 + NT - 1) / NT;
  double um[NML];
#pragma unroll
  for (int k = 0; k < NML; ++k) {
    const int i = tid + k * NT, v = i / L3;
    um[k] = i < 5 * L3 ? a.U[((size_t)v * ne + e) * L3 + (i - v * L3)] : 0.0;
  }
  // jumps J_side/J_vol ({q} - q-) of the primitives at the Gauss points
  for (int i = tid; i < 6 * QF2; i += NT) {
    const int s = i / QF2, q = i - s * QF2;
    const int es = e * 6 + s;
    const int nb = geo.nbr[es], ns = geo.nside[es];
    const double jr = a.fgeo[((size_t)es * QF2 + q) * 4 + 3];
    const double *tl = a.T + ((size_t)es) * 5 * QF2;
    double pl[4], pr[4];
    auto prim = [&](const double *t, int g, double (&o)[4]) {
      const double r = t[g], u = t[QF2 + g] / r, v = t[2 * QF2 + g] / r, w = t[3 * QF2 + g] / r;
      double en = t[4 * QF2 + g] / r;
      double wk = u * u; wk = v * v + wk; wk = w * w + wk;
      o[0] = u; o[1] = v; o[2] = w; o[3] = -0.5 * wk + en;
    };
    prim(tl, q, pl);
    if (nb < 0) ghost_prim3(-1 - nb, tl[q], a.phys, pr);
    else prim(a.T + ((size_t)nb * 6 + ns) * 5 * QF2, geo.perm[geo.permid[es] * QF2 + q], pr);
    const int qa = q / QF, qb = q - qa * QF;
#pragma unroll
    for (int c = 0; c < 4; ++c) Jq[((c * 6 + s) * QF + qa) * FP + qb] = jr * (0.5 * (pl[c] + pr[c]) - pl[c]);
  }
  // modal state -> nodal, then the primitives
#pragma unroll
  for (int k = 0; k < NML; ++k) {
    const int i = tid + k * NT, v = i / L3, m = i - v * L3;
    if (i < 5 * L3) W1[(v * L2 + m / L) * LP + m % L] = um[k];
  }
  __syncthreads();
  con_mid<5, L, L, L, Q, LP, LP, NT>(EO<P>::BT(), W1, W2, tid);
  __syncthreads();
  con_mid<5 * Q, L, 1, L, Q, LP, LP, NT>(EO<P>::BT(), W2, W1, tid);
  __syncthreads();
  con_last<5 * Q2, L, Q, LP, QP, NT>(EO<P>::BT(), W1, W2, tid);
  __syncthreads();
#pragma unroll
  for (int rr = 0; rr < NPT; ++rr) {
    const int n = tid + rr * NT;
    if (n < Q3) {
      const int pn = (n / Q) * QP + n % Q;
      const double r = W2[pn], u = W2[FS + pn] / r, v = W2[2 * FS + pn] / r, w = W2[3 * FS + pn] / r;
      double en = W2[4 * FS + pn] / r;
      double wk = u * u; wk = v * v + wk; wk = w * w + wk;
      Pq[pn] = u; Pq[FS + pn] = v; Pq[2 * FS + pn] = w; Pq[3 * FS + pn] = -0.5 * wk + en;
      wJ[pn] = ge[9 * Q3 + n];
    }
  }
  const double iwend = CT<P>::BT()[0] / CT<P>::BW()[0];   // 1 / GLL end weight
#pragma unroll 1
  for (int c0 = 0; c0 < 4; c0 += 2) {
    // a pass computes its own indices: hoisted out of the loop they fill the registers
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    __syncthreads();
    // D_d of primitives c0, c0 + 1 at the nodes, [2][3] blocks in W1
    const double *F = Pq + c0 * FS;
    for (int pc = tid; pc < 6 * Q2; pc += NT) {
      const int b = pc / Q2, t = pc - b * Q2, c = b / 3, d = b - 3 * c, t1 = t / Q, t2 = t - t1 * Q;
      const int o = d == 0 ? t1 * QP + t2 : (d == 1 ? t1 * Q * QP + t2 : t * QP);
      const int s = d == 0 ? Q * QP : (d == 1 ? QP : 1);
      double x[Q], y[Q];
#pragma unroll
      for (int k = 0; k < Q; ++k) x[k] = F[c * FS + o + k * s];
      eo_apply<EO_NNA, Q, Q>(fresh(EO<P>::DN()).h, x, y);
#pragma unroll
      for (int k = 0; k < Q; ++k) W1[b * FS + o + k * s] = y[k];
    }
    // face blocks n_x J_side/J_vol ({q} - q-) [6][6][QF][QF] in W2
    for (int i = tid; i < 36 * QF2; i += NT) {
      const int b = i / QF2, q = i - b * QF2, g = b / 6, s = b - g * 6, c = c0 + g / 3, x = g - (g / 3) * 3;
      const int qa = q / QF, qb = q - qa * QF;
      W2[(b * QF + qa) * FP + qb] =
          a.fgeo[(((size_t)e * 6 + s) * QF2 + q) * 4 + x] * Jq[((c * 6 + s) * QF + qa) * FP + qb];
    }
    __syncthreads();
    // the weighted nodal gradients, component 3 c + x
    double acc[NPT][6];
#pragma unroll
    for (int rr = 0; rr < NPT; ++rr) {
      const int n = tid + rr * NT, pn = n < Q3 ? (n / Q) * QP + n % Q : 0;
      double mg[9];
#pragma unroll
      for (int c = 0; c < 9; ++c) mg[c] = ge[c * Q3 + (n < Q3 ? n : 0)];
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const double dr = W1[(3 * c) * FS + pn], ds = W1[(3 * c + 1) * FS + pn], dt = W1[(3 * c + 2) * FS + pn];
#pragma unroll
        for (int x = 0; x < 3; ++x)
          acc[rr][3 * c + x] = fma(mg[6 + x], dt, fma(mg[3 + x], ds, mg[x] * dr));
      }
    }
    __syncthreads();
    con_mid<36, QF, 1, QF, Q, FP, FP, NT>(fresh(EO<P>::GL()), W2, W1, tid);   // [36][Q][QF]
    __syncthreads();
    con_last<36 * Q, QF, Q, FP, QP, NT>(fresh(EO<P>::GL()), W1, W2, tid);     // [36][Q][Q]
    __syncthreads();
#pragma unroll
    for (int rr = 0; rr < NPT; ++rr) {
      const int n = tid + rr * NT;
      if (n < Q3) {
        const int i = n / Q2, j = (n / Q) % Q, k = n % Q, pn = (n / Q) * QP + k;
        const double cw = wJ[pn] * iwend;
        auto add = [&](int f, int a1, int a2) {
#pragma unroll
          for (int g = 0; g < 6; ++g) acc[rr][g] = fma(cw, W2[((g * 6 + f) * Q + a1) * QP + a2], acc[rr][g]);
        };
        if (k == 0) add(0, i, j);
        if (k == Q - 1) add(5, i, j);
        if (j == 0) add(1, i, k);
        if (j == Q - 1) add(3, i, k);
        if (i == 0) add(4, j, k);
        if (i == Q - 1) add(2, j, k);
#pragma unroll
        for (int g = 0; g < 6; ++g) W1[g * FS + pn] = acc[rr][g];
      }
    }
    __syncthreads();
    // b = B^T (wJ g), then M x = b
    con_last<6 * Q2, Q, L, QP, LP, NT>(fresh(EO<P>::BL()), W1, W2, tid);
    __syncthreads();
    con_mid<6 * Q, Q, 1, L, L, LP, LP, NT>(fresh(EO<P>::BL()), W2, W1, tid);  // [6][Q][L][L]
    __syncthreads();
    MassSolve<P, 6, NT> ms{W1, W2, wJ, pre + (size_t)e * 3 * L2, tid};
    double r[L], x[L];
    if (ms.mine()) {
      const int f = tid / L2, mn = tid % L2, m = mn / L, n = mn - m * L;
      double t[Q];
#pragma unroll
      for (int k = 0; k < Q; ++k) t[k] = W1[((f * Q + k) * L + m) * LP + n];
      eo_apply<EO_NM, Q, L>(fresh(EO<P>::BL()).h, t, r);
    }
    __syncthreads();
    const int it = ms.solve(r, red, tot, x);
    if (ms.mine()) {
#pragma unroll
      for (int k = 0; k < L; ++k) a.G[((size_t)e * 12 + 3 * c0) * L3 + tid * L + k] = x[k];
    }
    if (tid == 0 && a.iters) atomicMax(a.iters, it);
  }
}

// Viscous terms of a curved hex from the state and the lifted gradients G
// (src/Navier_Stokes3d.cpp:113-258): the stresses and heat flux at the nodes;
// V [ne][4][Q3] = wJ div F_v for (rho u, rho v, rho w, rho E), and each side's
// normal flux F_v.n with its own normal at its Gauss points into TV
// [ne][6][4][QF2] (the three Cartesian components interpolated to the side
// first, then dotted, as the reference forms the side flux).
// One Cartesian component of all 4 fluxes at a time: its metric derivatives
// accumulate the divergence while its face values are interpolated to the
// Gauss points in the same LDS phases (14^3 hexes at p = 4: 77 -> 65 us).
template <int P>
__global__ void __launch_bounds__(C3V<P>::NT) __attribute__((amdgpu_waves_per_eu(lds_waves(C3V<P>::visc, C3V<P>::NT))))
k_visc3c(CurvedArgs a, const double *__restrict__ gm) {
  using S = C3V<P>;
  constexpr int L = S::L, Q = S::Q, QF = S::QF, L2 = S::L2, L3 = S::L3, Q2 = S::Q2, Q3 = S::Q3, QF2 = S::QF2;
  constexpr int LP = S::LP, QP = S::QP, FP = S::FP, FS = S::FS, NT = S::NT, NPT = S::NPT;
  extern __shared__ double sm[];
  double *W1 = sm, *W2 = W1 + 6 * FS, *W3 = W2 + 6 * FS, *W4 = W3 + 24 * Q * QP;
  static_assert(S::visc <= 160 * 1024 && 6 * QF2 <= NT, "LDS, one face point per thread");
  const int ne = a.ne, e = xcd_element(blockIdx.x, ne), tid = threadIdx.x;
  const double *ge = gm + (size_t)e * 10 * Q3;
  // velocity and the 12 gradient components at this thread's nodes
  double vel[NPT][3], gq[NPT][12];
  auto nodal = [&](const double *src, size_t stride, int nf) {   // nf fields, stride apart, into W2
    for (int i = tid; i < nf * L3; i += NT) {
      const int v = i / L3, m = i - v * L3;
      W1[(v * L2 + m / L) * LP + m % L] = src[v * stride + m];
    }
    __syncthreads();
    con_mid<6, L, L, L, Q, LP, LP, NT>(fresh(EO<P>::BT()), W1, W2, tid);
    __syncthreads();
    con_mid<6 * Q, L, 1, L, Q, LP, LP, NT>(fresh(EO<P>::BT()), W2, W1, tid);
    __syncthreads();
    con_last<6 * Q2, L, Q, LP, QP, NT>(fresh(EO<P>::BT()), W1, W2, tid);
    __syncthreads();
  };
  auto at = [&](int rr, int c) {
    const int n = tid + rr * NT;
    return W2[c * FS + (n < Q3 ? (n / Q) * QP + n % Q : 0)];
  };
  nodal(a.U + (size_t)e * L3, (size_t)ne * L3, 5);
#pragma unroll
  for (int rr = 0; rr < NPT; ++rr) {
    const double r = at(rr, 0);
#pragma unroll
    for (int x = 0; x < 3; ++x) vel[rr][x] = at(rr, 1 + x) / r;
  }
  nodal(a.G + (size_t)e * 12 * L3, L3, 6);
#pragma unroll
  for (int rr = 0; rr < NPT; ++rr)
#pragma unroll
    for (int c = 0; c < 6; ++c) gq[rr][c] = at(rr, c);
  nodal(a.G + ((size_t)e * 12 + 6) * L3, L3, 6);
#pragma unroll
  for (int rr = 0; rr < NPT; ++rr)
#pragma unroll
    for (int c = 0; c < 6; ++c) gq[rr][6 + c] = at(rr, c);
  const double mu = a.phys.vis, gp = a.phys.gamma / a.phys.Pr;
  // the thread's Gauss point q of side s
  const int s = tid / QF2 < 6 ? tid / QF2 : 0, q = tid - (tid / QF2) * QF2;
  const double *fg = a.fgeo + (((size_t)e * 6 + s) * QF2 + q) * 4;
  double tv[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 1
  for (int x = 0; x < 3; ++x) {
    // component x of the viscous fluxes of (rho u, rho v, rho w, rho E) at the nodes
#pragma unroll
    for (int rr = 0; rr < NPT; ++rr) {
      const int n = tid + rr * NT;
      if (n >= Q3) continue;
      const int pn = (n / Q) * QP + n % Q;
      const double *g = gq[rr];
      const double ux = g[0], uy = g[1], uz = g[2], vx = g[3], vy = g[4], vz = g[5];
      const double wx = g[6], wy = g[7], wz = g[8];
      const double t12 = mu * (uy + vx), t13 = mu * (uz + wx), t23 = mu * (vz + wy);
      const double t11 = mu * ((2.0 / 3.0) * ((2.0 * ux - vy) - wz));
      const double t22 = mu * ((2.0 / 3.0) * ((2.0 * vy - ux) - wz));
      const double t33 = mu * ((2.0 / 3.0) * ((2.0 * wz - ux) - vy));
      const double ex = g[9], ey = g[10], ez = g[11];
      double f0 = t11, f1 = t12, f2 = t13, ge3 = ex;
      if (x == 1) { f0 = t12; f1 = t22; f2 = t23; ge3 = ey; }
      if (x == 2) { f0 = t13; f1 = t23; f2 = t33; ge3 = ez; }
      W1[pn] = f0; W1[FS + pn] = f1; W1[2 * FS + pn] = f2;
      W1[3 * FS + pn] = fma(gp, mu * ge3, fma(f2, vel[rr][2], fma(f1, vel[rr][1], f0 * vel[rr][0])));
    }
    __syncthreads();
    metric_deriv<P, 4, NT, double>(EO<P>::DN(), W1, W2, ge, x, x == 0, tid, [&](int d) {
      if (d == 0) {   // the face nodes [6][4][Q][Q]
        for (int i = tid; i < 24 * Q2; i += NT) {
          const int b = i / Q2, t = i - b * Q2, f = b & 3, sd = b >> 2, t1 = t / Q, t2 = t - t1 * Q;
          int n;   // padded index of the side's node (t1, t2)
          switch (sd) {
            case 0: n = (t1 * Q + t2) * QP; break;
            case 5: n = (t1 * Q + t2) * QP + Q - 1; break;
            case 1: n = t1 * Q * QP + t2; break;
            case 3: n = (t1 * Q + Q - 1) * QP + t2; break;
            case 4: n = t1 * QP + t2; break;
            default: n = ((Q - 1) * Q + t1) * QP + t2; break;
          }
          W3[(b * Q + t1) * QP + t2] = W1[f * FS + n];
        }
      } else if (d == 1) {
        con_mid<24, Q, 1, Q, QF, QP, QP, NT>(fresh(EO<P>::Ig()), W3, W4, tid);    // [24][QF][Q]
      } else {
        con_last<24 * QF, Q, QF, QP, FP, NT>(fresh(EO<P>::Ig()), W4, W3, tid);    // [24][QF][QF]
      }
    });
    if (tid < 6 * QF2) {
      const double n = fg[x];
#pragma unroll
      for (int f = 0; f < 4; ++f) tv[f] = fma(n, W3[((s * 4 + f) * QF + q / QF) * FP + q % QF], tv[f]);
    }
  }
  if (tid < 6 * QF2) {
#pragma unroll
    for (int f = 0; f < 4; ++f) a.TV[(((size_t)e * 6 + s) * 4 + f) * QF2 + q] = tv[f];
  }
#pragma unroll
  for (int rr = 0; rr < NPT; ++rr) {
    const int n = tid + rr * NT;
    if (n < Q3) {
#pragma unroll
      for (int f = 0; f < 4; ++f) a.V[((size_t)e * 4 + f) * Q3 + n] = W2[f * FS + (n / Q) * QP + n % Q];
    }
  }
}

template <int P>
static hipError_t launch_c3(const CurvedArgs &a) {
  const int sh = C3<P>::lds;
  if (a.project) {   // the projection of given nodal data stays FP64 on both paths
    (void)hipFuncSetAttribute((const void *)k_rhs3c<P, true>, hipFuncAttributeMaxDynamicSharedMemorySize, sh);
    hipLaunchKernelGGL((k_rhs3c<P, true>), dim3(a.ne), dim3(C3<P>::NT), sh, a.stream, a, a.gm, a.pre);
  } else if (a.ns) {
    if constexpr (P <= 7) {
      if (a.op == 1) {
        (void)hipFuncSetAttribute((const void *)k_grad3c<P>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                  C3V<P>::grad);
        hipLaunchKernelGGL(k_grad3c<P>, dim3(a.ne), dim3(C3V<P>::NT), C3V<P>::grad, a.stream, a, a.gm, a.pre);
      } else if (a.op == 2) {
        (void)hipFuncSetAttribute((const void *)k_visc3c<P>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                  C3V<P>::visc);
        hipLaunchKernelGGL(k_visc3c<P>, dim3(a.ne), dim3(C3V<P>::NT), C3V<P>::visc, a.stream, a, a.gm);
      } else {
        (void)hipFuncSetAttribute((const void *)k_rhs3c<P, false, double, true>,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, sh);
        hipLaunchKernelGGL((k_rhs3c<P, false, double, true>), dim3(a.ne), dim3(C3<P>::NT), sh, a.stream, a, a.gm, a.pre);
      }
    } else {
      return hipErrorInvalidValue;
    }
  } else if (a.mixed) {
    (void)hipFuncSetAttribute((const void *)k_rhs3c<P, false, float>, hipFuncAttributeMaxDynamicSharedMemorySize,
                              sh);
    hipLaunchKernelGGL((k_rhs3c<P, false, float>), dim3(a.ne), dim3(C3<P>::NT), sh, a.stream, a, a.gm, a.pre);
  } else {
    (void)hipFuncSetAttribute((const void *)k_rhs3c<P, false>, hipFuncAttributeMaxDynamicSharedMemorySize, sh);
    hipLaunchKernelGGL((k_rhs3c<P, false>), dim3(a.ne), dim3(C3<P>::NT), sh, a.stream, a, a.gm, a.pre);
  }
  return hipGetLastError();
}

bool curved3_supported(int p) { return p >= 1 && p <= 8; }

hipError_t launch_curved3(const CurvedArgs &a) {
  switch (a.p) {
#define DGX_CASE(PP) case PP: return launch_c3<PP>(a);
    DGX_CASE(1) DGX_CASE(2) DGX_CASE(3) DGX_CASE(4) DGX_CASE(5) DGX_CASE(6) DGX_CASE(7) DGX_CASE(8)
#undef DGX_CASE
    default: return hipErrorInvalidValue;
  }
}

hipError_t upload_tables_c3d(const double *h) {
  hipError_t e = hipMemcpyToSymbol(HIP_SYMBOL(c_tab), h, sizeof(double) * kTabTotal);
  if (e != hipSuccess) return e;
  std::vector<float> f(h, h + kTabTotal);
  return hipMemcpyToSymbol(HIP_SYMBOL(c_tabf3), f.data(), sizeof(float) * kTabTotal);
}

}  // namespace dgx
