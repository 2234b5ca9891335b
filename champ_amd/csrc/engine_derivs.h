// engine_derivs.h -- parameter derivatives of ln Psi and of the local energy
// (the optimisation sample): Jastrow parameter derivatives, the
// pseudopotential pieces (psp_nonloc_orb over all orbitals, dpe), the
// orbital-resolved local energy and the CSF / Jastrow / orbital-rotation
// blocks.  All sums here are FP64; in the mixed engines the basis values and
// the points' Jastrow factors that they take are FP32.
#pragma once
#include "engine_kernels.h"

namespace qmcw {

// The slot pieces are sums: over the electrons and their pairs for the
// Jastrow's own derivatives (k_deriv_jas), over the quadrature points for the
// pseudopotential's (k_deriv_nlpp).  Both keep the sums of a slot group in
// registers over a lane's whole share and add the lanes up at the end; an
// update in memory per (pair, centre, slot) took 640 and 1,090 us of a
// derivative evaluation of 8,192 C2-like walkers (here 60 and 488), and 1,138
// and 2,589 of one of 601 walkers of a 25-electron molecule (the latter here
// 785), whose call went from 5.3 to 2.5 ms.

// number of e-e-n terms with power k of U (all of them: k = -1)
template <int ORD>
__host__ __device__ constexpr int een_count(int kk) {
  int n = 0;
  for (int k = 0; k <= ORD; k++)
    for (int m = 0; 2 * m <= ORD - k; m++)
      for (int l = 0; l <= ORD - k - 2 * m; l++)
        if (QMCW_EEN_TERM(k, l, m) && (kk < 0 || k == kk)) n++;
  return n;
}
// index of the first term with power k of U
template <int ORD>
__host__ __device__ constexpr int een_first(int kk) {
  int n = 0;
  for (int k = 0; k < kk; k++) n += een_count<ORD>(k);
  return n;
}

// Derivatives of an e-n (or e-e) Pade + polynomial term with respect to its
// coefficients, at scaled distance u, with their first two u derivatives, for
// coefficient iw = 1, 2, ... (1 and 2 the Pade form's; qmc/vmc/
// deriv_jastrow4.f90:95-220, 880-1090).  The powers advance with iw.
struct PadeSlots {
  double u, c0, c1, s, ar, bt, bta;     // coefficients of the form, spin factor, scaled distance at infinity
  double up, arp, um1, um2;
  __device__ __forceinline__ PadeSlots(double u_, double c0_, double c1_, double s_, double ar_)
      : u(u_), c0(c0_), c1(c1_), s(s_), ar(ar_), bt(1.0 / (1.0 + c1_ * u_)), bta(1.0 / (1.0 + c1_ * ar_)),
        up(u_), arp(ar_), um1(1.0), um2(0.0) {}
  __device__ __forceinline__ void get(int iw, double &g, double &g1, double &g2) {
    if (iw == 1) {
      g = s * (u * bt - ar * bta);
      g1 = s * bt * bt;
      g2 = -2.0 * c1 * g1 * bt;
    } else if (iw == 2) {
      g = s * c0 * (ar * ar * bta * bta - u * u * bt * bt);
      g1 = -2.0 * s * c0 * u * bt * bt * bt;
      g2 = -2.0 * s * c0 * (1.0 - 2.0 * c1 * u) * bt * bt * bt * bt;
    } else {
      const int io = iw - 1;
      um2 = um1;
      um1 = up;
      up *= u;
      arp *= ar;
      g = up - arp;
      g1 = io * um1;
      g2 = io * (io - 1) * um2;
    }
  }
};

// e-e coefficients and spin factor of a pair
__device__ __forceinline__ int b_spin(const DevSys &S, bool par, double &sspinn) {
  sspinn = 1.0;
  if (!par) return 0;
  if (S.nspin2b == 2) return 1;
  if (S.nocuspb == 0) sspinn = 0.5;
  return 0;
}

// One power K of U of the e-e-n slots of centre type it (k_deriv_jas): over
// this lane's electrons i, the type's centres and the other electrons j,
// with S_n = sum_j U^K B^n, X_n its part of i's laplacian plus twice its
// gradient along v_i and R_n its gradient along the vector to the centre
// (see k_deriv_jas), each term takes two entries of each.
template <int G, int ORD, int K>
__device__ __forceinline__ void deriv_een_power(const KArgs &A, const double *ws, const double *ss, int it,
                                                double *dj, int lane) {
  const DevSys &S = A.S;
  const int N = S.N, M = S.M;
  constexpr int NN = ORD - K + 1, NT = een_count<ORD>(K);
  if constexpr (NT > 0) {
    const double *x = ws + A.L.x, *ren = ws + A.L.r_en, *rven = ws + A.L.rvec_en;
    const double *vj = ss + A.SL.vj, *vd = ss + A.SL.vd;
    const double *tu = ss + A.DL.tu, *tb = ss + A.DL.tb;
    const int64_t NN2 = (int64_t)N * N;
    const double k = S.scalek, hb = S.hb;
    double av[NT], ae[NT];
#pragma unroll
    for (int q = 0; q < NT; q++) av[q] = ae[q] = 0.0;
    for (int i = lane; i < N; i += G) {
      const double vi[3] = {vj[3 * i] + vd[3 * i], vj[3 * i + 1] + vd[3 * i + 1], vj[3 * i + 2] + vd[3 * i + 2]};
      for (int c = cst(S.tc_off)[it]; c < cst(S.tc_off)[it + 1]; c++) {
        const int ic = ((cptr<TypeCent>)S.tcent)[c].ic;
        const double ri = ren[i * M + ic];
        const double rv[3] = {rven[(i * M + ic) * 3], rven[(i * M + ic) * 3 + 1], rven[(i * M + ic) * 3 + 2]};
        double s0[NN], x0[NN], r0[NN];
#pragma unroll
        for (int n = 0; n < NN; n++) s0[n] = x0[n] = r0[n] = 0.0;
        for (int j = 0; j < N; j++) {
          if (j == i) continue;
          const double U = tu[j * N + i], B = tb[ic * N + j];
          double uk2 = 1.0;                     // U^(K-2)
#pragma unroll
          for (int q = 0; q < K - 2; q++) uk2 *= U;
          const double uk1 = K >= 2 ? uk2 * U : 1.0, uk = K >= 1 ? uk1 * U : 1.0;
          double s = uk, xx = 0.0, r = 0.0;
          if (K >= 1) {
            // gu = Ud1 / rij, l1 = Ud2 + 2 Ud1 / rij, l2 = Ud1^2
            const double gu = tu[NN2 + j * N + i], l1 = tu[2 * NN2 + j * N + i], l2 = tu[3 * NN2 + j * N + i];
            const double d[3] = {x[3 * i] - x[3 * j], x[3 * i + 1] - x[3 * j + 1], x[3 * i + 2] - x[3 * j + 2]};
            const double fu = K * uk1, gd = fu * gu;
            xx = fu * l1 + (K >= 2 ? K * (K - 1) * uk2 * l2 : 0.0) +
                 2.0 * gd * (d[0] * vi[0] + d[1] * vi[1] + d[2] * vi[2]);
            r = gd * (d[0] * rv[0] + d[1] * rv[1] + d[2] * rv[2]);
          }
#pragma unroll
          for (int n = 0; n < NN; n++) {
            s0[n] += s;
            s *= B;
            if (K >= 1) {
              x0[n] += xx;
              r0[n] += r;
              xx *= B;
              r *= B;
            }
          }
        }
        double A0, Ad1, Ad2;
        scaled<double>(S.isc, k, ri, A0, Ad1, Ad2);
        A0 = 1.0 - k * A0; Ad1 = -k * Ad1; Ad2 = -k * Ad2;
        double ap[ORD + 1];
        ap[0] = 1.0;
#pragma unroll
        for (int q = 1; q <= ORD; q++) ap[q] = ap[q - 1] * A0;
        const double da = Ad1 / ri, l2 = Ad1 * Ad1;
        const double l1 = Ad2 + 2.0 * da * (1.0 + rv[0] * vi[0] + rv[1] * vi[1] + rv[2] * vi[2]);
        int idx = 0;
#pragma unroll
        for (int m = 0; 2 * m <= ORD - K; m++)
#pragma unroll
          for (int l = 0; l <= ORD - K - 2 * m; l++)
            if (QMCW_EEN_TERM(K, l, m)) {
              const int p = l + m;
              // every ordered pair is met from both sides: half the value each
              av[idx] += 0.5 * (ap[p] * s0[m] + ap[m] * s0[p]);
              double e = ap[p] * x0[m] + ap[m] * x0[p];
              if (p >= 1) e += p * ap[p >= 1 ? p - 1 : 0] * (l1 * s0[m] + 2.0 * da * r0[m]);
              if (m >= 1) e += m * ap[m >= 1 ? m - 1 : 0] * (l1 * s0[p] + 2.0 * da * r0[p]);
              if (p >= 2) e += p * (p - 1) * ap[p >= 2 ? p - 2 : 0] * l2 * s0[m];
              if (m >= 2) e += m * (m - 1) * ap[m >= 2 ? m - 2 : 0] * l2 * s0[p];
              ae[idx] += e;
              idx++;
            }
      }
    }
    const int s1 = S.slot_c0 + it * S.nterms + een_first<ORD>(K);
#pragma unroll
    for (int q = 0; q < NT; q++) {
      const double v = gsum<G>(av[q]), e = gsum<G>(ae[q]);
      if (lane == 0) { dj[2 * (s1 + q)] = v; dj[2 * (s1 + q) + 1] = -hb * e; }
    }
  }
}
template <int G, int ORD, int K>
__device__ __forceinline__ void deriv_een_powers(const KArgs &A, const double *ws, const double *ss, int it,
                                                 double *dj, int lane) {
  deriv_een_power<G, ORD, K>(A, ws, ss, it, dj, lane);
  if constexpr (K < ORD) deriv_een_powers<G, ORD, K + 1>(A, ws, ss, it, dj, lane);
}

// ---------------------------------------------------------------------------
// Jastrow parameter derivatives of the current configuration, per slot
// (qmc/vmc/deriv_jastrow4.f90): dj[slot] = {d ln J / dc,
// -hb (d lap ln J / dc + 2 sum_i v_i . d grad_i ln J / dc)} with v_i the
// electron's whole velocity (k_full_det has run): what d ln Psi/dp and
// dE_L/dp need of them, so no gradient per electron and slot is kept.  Each
// lane takes whole electrons i and every pair (i, j) from i's side.  For a
// power k of U and a centre, the sums over j of U^k B^n (and of its gradient
// and laplacian parts) serve all terms of that power.
template <int G, int ORD>
__global__ QMCW_HEAVY void k_deriv_jas(KArgs A) {
  QMCW_GROUP_SETUP
  const int N = S.N, M = S.M;
  const WLayout &L = A.L;
  const double *x = ws + L.x, *ren = ws + L.r_en, *rven = ws + L.rvec_en;
  const double *vj = ss + A.SL.vj, *vd = ss + A.SL.vd;
  double *tu = ss + A.DL.tu, *tb = ss + A.DL.tb, *dj = ss + A.DL.dj;
  const double k = S.scalek, ar = S.asymp_r, hb = S.hb;
  constexpr int MW = QMCW_MAX_ORD + 1;
  // ---- a-coefficients, a centre type at a time
  const int na = S.norda + 1;
  for (int it = 0; it < S.nctype; it++) {
    double av[MW], ae[MW];
#pragma unroll
    for (int q = 0; q < MW; q++) av[q] = ae[q] = 0.0;
    for (int i = lane; i < N; i += G) {
      const double vi[3] = {vj[3 * i] + vd[3 * i], vj[3 * i + 1] + vd[3 * i + 1], vj[3 * i + 2] + vd[3 * i + 2]};
      for (int c = cst(S.tc_off)[it]; c < cst(S.tc_off)[it + 1]; c++) {
        const int p = i * M + ((cptr<TypeCent>)S.tcent)[c].ic;
        const double ri = ren[p];
        double u, d7, d9;
        scaled<double>(S.isc, k, ri, u, d7, d9);
        const double gd = d7 / ri * (1.0 + rven[3 * p] * vi[0] + rven[3 * p + 1] * vi[1] + rven[3 * p + 2] * vi[2]);
        PadeSlots ps(u, cst(S.a4)[it * na], cst(S.a4)[it * na + 1], 1.0, ar);
#pragma unroll
        for (int iw = 1; iw <= MW; iw++) {
          if (iw > na) continue;
          double g, g1, g2;
          ps.get(iw, g, g1, g2);
          av[iw - 1] += g;
          ae[iw - 1] += g2 * d7 * d7 + g1 * (d9 + 2.0 * gd);
        }
      }
    }
#pragma unroll
    for (int q = 0; q < MW; q++) {
      if (q >= na) continue;
      const double v = gsum<G>(av[q]), e = gsum<G>(ae[q]);
      if (lane == 0) { dj[2 * (it * na + q)] = v; dj[2 * (it * na + q) + 1] = -hb * e; }
    }
  }
  // ---- b-coefficients, and the pair tables of the e-e-n terms: per (j, i)
  // U, Ud1 / rij, Ud2 + 2 Ud1 / rij and Ud1^2, per (centre, j) B
  const int nb = S.nordb + 1;
  const int64_t NN2 = (int64_t)N * N;
  for (int p = lane; p < N * M; p += G) {
    double b, t1, t2;
    scaled<double>(S.isc, k, ren[p], b, t1, t2);
    tb[(p % M) * N + p / M] = 1.0 - k * b;
  }
  for (int isb = 0; isb < (S.nspin2b == 2 ? 2 : 1); isb++) {
    double av[MW], ae[MW];
#pragma unroll
    for (int q = 0; q < MW; q++) av[q] = ae[q] = 0.0;
    for (int i = lane; i < N; i += G) {
      const double vi[3] = {vj[3 * i] + vd[3 * i], vj[3 * i + 1] + vd[3 * i + 1], vj[3 * i + 2] + vd[3 * i + 2]};
      for (int j = 0; j < N; j++) {
        if (j == i) continue;
        const double d[3] = {x[3 * i] - x[3 * j], x[3 * i + 1] - x[3 * j + 1], x[3 * i + 2] - x[3 * j + 2]};
        const double rij = sqrt(d[0] * d[0] + d[1] * d[1] + d[2] * d[2]);
        double u, d1, d2;
        scaled<double>(S.isc, k, rij, u, d1, d2);
        const double dr = d1 / rij;
        if (isb == 0) {
          tu[j * N + i] = 1.0 - k * u;
          tu[NN2 + j * N + i] = -k * dr;
          tu[2 * NN2 + j * N + i] = -k * (d2 + 2.0 * dr);
          tu[3 * NN2 + j * N + i] = k * k * d1 * d1;
        }
        double sp;
        if (b_spin(S, (i < S.nup) == (j < S.nup), sp) != isb) continue;
        const double gd = dr * (1.0 + d[0] * vi[0] + d[1] * vi[1] + d[2] * vi[2]);
        PadeSlots ps(u, cst(S.b)[isb * nb], cst(S.b)[isb * nb + 1], sp, ar);
#pragma unroll
        for (int iw = 1; iw <= MW; iw++) {
          if (iw > nb) continue;
          double g, g1, g2;
          ps.get(iw, g, g1, g2);
          av[iw - 1] += 0.5 * g;
          ae[iw - 1] += g2 * d1 * d1 + g1 * (d2 + 2.0 * gd);
        }
      }
    }
#pragma unroll
    for (int q = 0; q < MW; q++) {
      if (q >= nb) continue;
      const double v = gsum<G>(av[q]), e = gsum<G>(ae[q]);
      const int sl = S.slot_b0 + isb * nb + q;
      if (lane == 0) { dj[2 * sl] = v; dj[2 * sl + 1] = -hb * e; }
    }
  }
  if (S.nordc <= 1) return;
  __syncthreads();
  for (int it = 0; it < S.nctype; it++) deriv_een_powers<G, ORD, 0>(A, ws, ss, it, dj, lane);
}

// Quadrature point, or (t >= npt) pair taken at the electron's current
// position, that lane entry t of k_deriv_nlpp stands for: position,
// electron and the weight of its slot pieces
__device__ __forceinline__ void nlpp_entry(const KArgs &A, const double *ws, const double *pw, const int *plist,
                                           int npt, int t, double *xn, int &i, double &wt) {
  const DevSys &S = A.S;
  const int nq = S.nquad, M = S.M;
  const double *x = ws + A.L.x, *quad = ws + A.L.quad;
  if (t < npt) {
    const int iq = t % nq, p = plist[t / nq], ic = p % M;
    i = p / M;
    const double r = ws[A.L.r_en + p];
#pragma unroll
    for (int q = 0; q < 3; q++) xn[q] = r * quad[q * nq + iq] + cst(S.cent)[3 * ic + q];
    wt = pw[2 * t + 1];
  } else {
    const int kp = t - npt;
    i = plist[kp] / M;
    xn[0] = x[3 * i]; xn[1] = x[3 * i + 1]; xn[2] = x[3 * i + 2];
    wt = 0.0;
    for (int iq = 0; iq < nq; iq++) wt -= pw[2 * (kp * nq + iq) + 1];
  }
}

constexpr int kPhiCols = 32;       // basis functions per pass of k_deriv_nlpp's weighted sums
// LDS bytes of its tile: kPhiCols values (one column of padding) and the
// factor and electron of each of the block's 64 points
template <typename T>
__host__ __device__ constexpr size_t deriv_tile_bytes() {
  return 64 * ((kPhiCols + 1) * sizeof(T) + sizeof(double) + sizeof(int));
}

// ---------------------------------------------------------------------------
// Pseudopotential pieces of the derivatives (qmc/vmc/nonloc.f90:184-197,
// qmc/fit/deriv_nonloc_pot.f90:59-64).  k_full_nlpp has left, per quadrature
// point of the pairs in range, fac = w exp(dJ) v P_l and fac times the
// determinant ratio (DLayout::pw).  psp_nonloc_orb is linear in the orbitals,
// psp_nonloc_orb(i, q) = sum_b coef(b, q) sum_points fac phi_b(point): here the
// weighted basis sums pbc[i][b] (the contraction runs once per electron,
// k_pnl_mfma).  A lane evaluates the basis functions of its point into LDS, a
// group of shells at a time, then the lanes take a function each and add its
// values over the points.  dpe_slot[slot] = sum over points of fac ratio
// d(dJ)/dslot: a point's slot pieces, weighted, less the same pieces at the
// electron's current position; summed over the other electrons, the term
// values of a centre are A^(l+m) S(k, m) + A^m S(k, l+m) with
// S(k, n) = sum_j U_j^k B_j^n.
template <typename T, int G, int ORD>
__global__ QMCW_HEAVY void k_deriv_nlpp(KArgs A) {
  QMCW_GROUP_SETUP
  const int N = S.N, M = S.M, NO = S.NO, NB = S.NB, nq = S.nquad;
  const WLayout &L = A.L;
  const SLayout &SL = A.SL;
  const DLayout &DL = A.DL;
  const double *x = ws + L.x, *ren = ws + L.r_en;
  const double *pw = ss + DL.pw;
  double *pbc = ss + DL.pbc, *btd = ss + DL.tb, *dsl = ss + DL.dpe_slot;
  const int *plist = reinterpret_cast<const int *>(ss + SL.plist);
  const int npair = (int)ss[SL.phs + 57], npt = npair * nq;
  for (int p = lane; p < N * M; p += G) {
    double bu, t1, t2;
    scaled<double>(S.isc, S.scalek, ren[p], bu, t1, t2);
    btd[(p % M) * N + p / M] = 1.0 - S.scalek * bu;
  }
  for (int q = lane; q < N * NB; q += G) pbc[q] = 0.0;
  // ---- the weighted basis sums
  extern __shared__ double dyn_lds[];
  double *s_f = dyn_lds + grp * G;                                  // the group's points
  int *s_el = reinterpret_cast<int *>(dyn_lds + 64) + grp * G;
  T *s_phi = reinterpret_cast<T *>(dyn_lds + 96) + (int64_t)grp * G * (kPhiCols + 1);
  int maxpt = npt;                                                  // of the block's walkers
#pragma unroll
  for (int o = G; o < 64; o <<= 1) maxpt = max(maxpt, __shfl_xor(maxpt, o, 64));
  for (int t0 = 0; t0 < maxpt; t0 += G) {
    const int nin = max(0, min(G, npt - t0));
    double xn[3] = {0.0, 0.0, 0.0}, wt;
    int el = 0;
    if (lane < nin) nlpp_entry(A, ws, pw, plist, npt, t0 + lane, xn, el, wt);
    __syncthreads();
    s_f[lane] = lane < nin ? pw[2 * (t0 + lane)] : 0.0;
    s_el[lane] = el;
    // shells of one centre after another, up to kPhiCols functions a pass
    int ic = 0, sh = 0;
    while (ic < M) {
      const int ic_0 = ic, sh_0 = sh;
      int nf = 0;
      while (ic < M) {
        if (sh == cst(S.cent_sh_off)[ic + 1]) { ic++; continue; }
        const int nm = 2 * cst(S.sh_l)[sh] + 1;
        if (nf + nm > kPhiCols) break;
        nf += nm;
        sh++;
      }
      T *ph = s_phi + lane * (kPhiCols + 1);
      for (int q = sh_0, f = 0, c = ic_0; q < sh; q++) {
        while (q >= cst(S.cent_sh_off)[c + 1]) c++;
        const double dx = xn[0] - cst(S.cent)[3 * c], dy = xn[1] - cst(S.cent)[3 * c + 1],
                     dz = xn[2] - cst(S.cent)[3 * c + 2];
        shell_slots<T>(S, q, (T)dx, (T)dy, (T)dz, (T)sqrt(dx * dx + dy * dy + dz * dz), ph + f);
        f += 2 * cst(S.sh_l)[q] + 1;
      }
      __syncthreads();
      for (int f = lane; f < nf; f += G) {
        // the function of column f
        int q = sh_0, g = f;
        while (g > 2 * cst(S.sh_l)[q]) { g -= 2 * cst(S.sh_l)[q] + 1; q++; }
        const int b = S.sh_bas[q * kMaxShellM + g];
        if (b < 0) continue;
        double a = 0.0;
        int cur = s_el[0];
        for (int p = 0; p < nin; p++) {
          if (s_el[p] != cur) {
            pbc[cur * NB + b] += a;
            a = 0.0;
            cur = s_el[p];
          }
          a += s_f[p] * (double)s_phi[p * (kPhiCols + 1) + f];
        }
        if (nin > 0) pbc[cur * NB + b] += a;
      }
      __syncthreads();
    }
  }
  // ---- the slots: quadrature points and, after them, the pairs at the
  // electrons' current positions
  const int nent = npt + npair;
  const double k = S.scalek, ar = S.asymp_r;
  constexpr int MW = QMCW_MAX_ORD + 1;
  const int na = S.norda + 1, nb = S.nordb + 1;
  for (int isb = 0; isb < (S.nspin2b == 2 ? 2 : 1); isb++) {
    double av[MW];
#pragma unroll
    for (int q = 0; q < MW; q++) av[q] = 0.0;
    for (int t = lane; t < nent; t += G) {
      double xn[3], wt;
      int i;
      nlpp_entry(A, ws, pw, plist, npt, t, xn, i, wt);
      for (int j = 0; j < N; j++) {
        if (j == i) continue;
        double sp;
        if (b_spin(S, (i < S.nup) == (j < S.nup), sp) != isb) continue;
        const double dx = xn[0] - x[3 * j], dy = xn[1] - x[3 * j + 1], dz = xn[2] - x[3 * j + 2];
        double u, d1, d2;
        scaled<double>(S.isc, k, sqrt(dx * dx + dy * dy + dz * dz), u, d1, d2);
        PadeSlots ps(u, cst(S.b)[isb * nb], cst(S.b)[isb * nb + 1], sp, ar);
#pragma unroll
        for (int iw = 1; iw <= MW; iw++) {
          if (iw > nb) continue;
          double g, g1, g2;
          ps.get(iw, g, g1, g2);
          av[iw - 1] += wt * g;
        }
      }
    }
#pragma unroll
    for (int q = 0; q < MW; q++) {
      if (q >= nb) continue;
      const double v = gsum<G>(av[q]);
      if (lane == 0) dsl[S.slot_b0 + isb * nb + q] = v;
    }
  }
  constexpr int NG = een_gi<ORD>(ORD, 0) + 1, NT = een_count<ORD>(-1);
  const LaneArr<double> uq = A.lds_dnlpp
      ? LaneArr<double>{dyn_lds + deriv_tile_bytes<T>() / 8 + threadIdx.x, kWave}
      : LaneArr<double>{ss + DL.uqd + lane, G};
  for (int it = 0; it < S.nctype; it++) {
    double av[MW], ac[NT];
#pragma unroll
    for (int q = 0; q < MW; q++) av[q] = 0.0;
#pragma unroll
    for (int q = 0; q < NT; q++) ac[q] = 0.0;
    for (int t = lane; t < nent; t += G) {
      double xn[3], wt;
      int i;
      nlpp_entry(A, ws, pw, plist, npt, t, xn, i, wt);
      if (S.nordc > 1)
        for (int j = 0; j < N; j++) {
          const double dx = xn[0] - x[3 * j], dy = xn[1] - x[3 * j + 1], dz = xn[2] - x[3 * j + 2];
          double u, d1, d2;
          scaled<double>(S.isc, k, sqrt(dx * dx + dy * dy + dz * dz), u, d1, d2);
          uq[j] = 1.0 - k * u;
        }
      for (int c = cst(S.tc_off)[it]; c < cst(S.tc_off)[it + 1]; c++) {
        const cptr<TypeCent> tc = (cptr<TypeCent>)S.tcent + c;
        const double dx = xn[0] - tc->x, dy = xn[1] - tc->y, dz = xn[2] - tc->z;
        double u, d1, d2;
        scaled<double>(S.isc, k, sqrt(dx * dx + dy * dy + dz * dz), u, d1, d2);
        PadeSlots ps(u, cst(S.a4)[it * na], cst(S.a4)[it * na + 1], 1.0, ar);
#pragma unroll
        for (int iw = 1; iw <= MW; iw++) {
          if (iw > na) continue;
          double g, g1, g2;
          ps.get(iw, g, g1, g2);
          av[iw - 1] += wt * g;
        }
        if (S.nordc <= 1) continue;
        double sg[NG];
#pragma unroll
        for (int q = 0; q < NG; q++) sg[q] = 0.0;
        const double *bj = btd + tc->ic * N;
        for (int j = 0; j < N; j++) {
          if (j == i) continue;
          const double U = uq[j], B = bj[j];
          double uk = 1.0;
#pragma unroll
          for (int kk = 0; kk <= ORD; kk++) {
            double v = uk;
#pragma unroll
            for (int n = 0; n <= ORD - kk; n++) {
              sg[een_gi<ORD>(kk, n)] += v;
              v *= B;
            }
            uk *= U;
          }
        }
        double ap[ORD + 1];
        ap[0] = wt;
#pragma unroll
        for (int q = 1; q <= ORD; q++) ap[q] = ap[q - 1] * (1.0 - k * u);
        int idx = 0;
#pragma unroll
        for (int kk = 0; kk <= ORD; kk++)
#pragma unroll
          for (int m = 0; 2 * m <= ORD - kk; m++)
#pragma unroll
            for (int l = 0; l <= ORD - kk - 2 * m; l++)
              if (QMCW_EEN_TERM(kk, l, m)) {
                ac[idx] += ap[l + m] * sg[een_gi<ORD>(kk, m)] + ap[m] * sg[een_gi<ORD>(kk, l + m)];
                idx++;
              }
      }
    }
#pragma unroll
    for (int q = 0; q < MW; q++) {
      if (q >= na) continue;
      const double v = gsum<G>(av[q]);
      if (lane == 0) dsl[it * na + q] = v;
    }
    if (S.nordc > 1) {
#pragma unroll
      for (int q = 0; q < NT; q++) {
        const double v = gsum<G>(ac[q]);
        if (lane == 0) dsl[S.slot_c0 + it * S.nterms + q] = v;
      }
    }
  }
  // (k_pnl_mfma forms pnl after this kernel when A.pnl_mfma)
  if (A.pnl_mfma) return;
  double *pnl = ss + DL.pnl;
  for (int t = lane; t < N * NO; t += G) {
    const int i = t / NO, q = t % NO;
    double a = 0.0;
    for (int b = 0; b < NB; b++) a += cst(S.coefT)[(int64_t)b * NO + q] * pbc[i * NB + b];
    pnl[t] = a;
  }
}

// ---------------------------------------------------------------------------
// Assembly of d ln Psi / dp and d E_L / dp in the order CSF, Jastrow,
// orbitals (qmc/deriv_mod.f90:219-239): elocal_orb_bld, dt_bld,
// alpha_deloc_bld, dy_bld, dg_bld, csf_derivs_bld
// (qmc/deriv_fast_mod.f90:174-823), dpsi_orb_bld / deloc_orb_bld
// (qmc/deriv_orb_mod.f90:1486-1630) and the Jastrow denergy of
// qmc/vmc/hpsi.f90:366-374.  dpsi[w * P + p] and deloc[w * P + p].
// With LDS the intermediates (derivs_lds_doubles of them) stay in LDS, a
// wavefront per walker: each of the dozen dependent phases then waits for LDS
// instead of L2, which bounded the kernel (37 of 600 VALU instructions per
// SIMD and us): 469 -> 246 us for 8,192 C2-like walkers.
__host__ __device__ inline int derivs_lds_doubles(const DevSys &S) {
  const int nsm = S.ns[0] > S.ns[1] ? S.ns[0] : S.ns[1], nom = S.nocc[0] > S.nocc[1] ? S.nocc[0] : S.nocc[1];
  int n = (2 * S.N + nsm) * S.NO + nom * nsm;
  for (int s = 0; s < 2; s++)
    n += 2 * S.ns[s] * S.NO + S.ndetu[s] * (3 + S.kmax2) + 2 * S.nocc[s] * S.ns[s];
  return n;
}
template <int G, bool LDS>
__global__ QMCW_HEAVY void k_derivs(KArgs A, double *dpsi, double *deloc) {
  QMCW_GROUP_SETUP
  const int N = S.N, NO = S.NO, P = S.nparm;
  const WLayout &L = A.L;
  const SLayout &SL = A.SL;
  const DLayout &DL = A.DL;
  const double hb = S.hb;
  const double *orb = ss + SL.orb;
  const double *vj = ss + SL.vj, *vd = ss + SL.vd, *red = ss + SL.phs;
  const double *pnl = ss + DL.pnl;
  // the orbital values (component 0 of orb, or their copy in LDS)
  extern __shared__ double dyn_lds[];
  constexpr int OS = LDS ? 1 : 5;
  double *nxt = dyn_lds + (LDS ? N * NO : 0);
  auto part = [&](int64_t at, int n) {
    if (!LDS) return ss + at;
    double *p = nxt;
    nxt += n;
    return p;
  };
  const double *ob = LDS ? dyn_lds : orb;
  double *B = part(DL.B, N * NO), *tfs[2], *dts[2], *dels[2], *c0s[2], *c1s[2], *ids[2], *dys[2], *dgs[2];
  for (int s = 0; s < 2; s++) {
    tfs[s] = part(DL.tfull[s], S.ns[s] * NO);
    dts[s] = part(DL.dt[s], S.ns[s] * NO);
    dels[s] = part(DL.del[s], S.ndetu[s]);
    c0s[s] = part(DL.c0[s], S.ndetu[s]);
    c1s[s] = part(DL.c1[s], S.ndetu[s]);
    ids[s] = part(DL.idti[s], S.ndetu[s] * S.kmax2);
    dys[s] = part(DL.dy[s], S.nocc[s] * S.ns[s]);
    dgs[s] = part(DL.dg[s], S.nocc[s] * S.ns[s]);
  }
  double *aib = part(DL.aib, max(S.ns[0], S.ns[1]) * NO), *aux = part(DL.aux4, 0);
  const double vpsp = S.nloc > 0 ? red[56] : 0.0;
  const double epl = ws[L.epot] - vpsp;          // local part of the potential
  double vj2 = 0.0;
  for (int q = lane; q < 3 * N; q += G) vj2 += vj[q] * vj[q];
  vj2 = gsum<G>(vj2);
  const double ddjas = (red[53] + vj2) / N;
  // ---- elocal_orb_bld
  for (int t = lane; t < N * NO; t += G) {
    const int i = t / NO;
    const double *o = orb + (int64_t)t * 5;
    const double dv = vj[3 * i] * o[1] + vj[3 * i + 1] * o[2] + vj[3 * i + 2] * o[3];
    double b = -hb * (o[4] + 2.0 * dv + ddjas * o[0]) + epl * o[0] / N;
    if (S.nloc > 0) b += pnl[t];
    B[t] = b;
    if (LDS) dyn_lds[t] = o[0];
  }
  __syncthreads();
  // ---- full T, dt_bld, alpha_deloc_bld and the k x k inverse products
  for (int s = 0; s < 2; s++) {
    const int ns = S.ns[s], off = s ? S.nup : 0;
    if (ns == 0) continue;
    const double *ai = w_ai(L, ws, s);
    double *tf = tfs[s], *dt = dts[s];
    for (int e = lane; e < ns * NO; e += G) {
      const int k = e / NO, q = e % NO;
      double a1 = 0.0, a2 = 0.0;
      for (int i = 0; i < ns; i++) {
        const double aki = ai[k + ns * i];
        a1 += aki * ob[((int64_t)(off + i) * NO + q) * OS];
        a2 += aki * B[(off + i) * NO + q];
      }
      tf[e] = a1;
      aib[e] = a2;
    }
    __syncthreads();
    for (int e = lane; e < ns * NO; e += G) {
      const int k = e / NO, q = e % NO;
      double a = 0.0;
      for (int r = 0; r < ns; r++) a += aib[k * NO + cst(S.ref[s])[r]] * tf[r * NO + q];
      dt[e] = aib[e] - a;
    }
    __syncthreads();
    const double *inv = w_inv(L, ws, s);
    double *del = dels[s], *idti = ids[s];
    for (int u = lane; u < S.ndetu[s]; u += G) {
      const int k = cst(S.ord[s])[u];
      const double *iv = inv + u * S.kmax2;
      const int *rf = S.rf[s] + u * ns, *le = S.exl[s] + u * ns;
      double d = 0.0;
      for (int j = 0; j < k; j++)
        for (int i = 0; i < k; i++) d += iv[j + k * i] * dt[rf[i] * NO + le[j]];
      del[u] = d;
      // idti = inv (fdt inv), fdt(j, i) = dt(rf_j, le_i)
      double *id = idti + u * S.kmax2;
      for (int i = 0; i < k; i++)
        for (int j = 0; j < k; j++) {
          double a = 0.0;
          for (int kk = 0; kk < k; kk++) {
            double dti = 0.0;
            for (int k2 = 0; k2 < k; k2++) dti += dt[rf[kk] * NO + le[k2]] * iv[k2 + k * i];
            a += iv[j + k * kk] * dti;
          }
          id[j + k * i] = a;
        }
    }
    __syncthreads();
  }
  // ---- coefficient sums per unique det and esum
  const double chii = 1.0 / ws[L.chi];
  const double *dv0 = w_detv(L, ws, 0), *dv1 = w_detv(L, ws, 1);
  const double *del0 = dels[0], *del1 = dels[1];
  // over the dets that contain unique det u (the CSR lists of eval_y, in
  // ascending det order)
  for (int t = lane; t < S.ndetu[0] + S.ndetu[1]; t += G) {
    const int s = t < S.ndetu[0] ? 0 : 1, u = s ? t - S.ndetu[0] : t;
    const cptr<int> uiu = cst(S.uiu[s]), uid = cst(S.uid[s]);
    const cptr<double> ucf = cst(S.ucf[s]);
    double c0 = 0.0, c1 = 0.0;
    const int q1 = cst(S.udet_off[s])[u + 1];
#pragma unroll 4
    for (int q = cst(S.udet_off[s])[u]; q < q1; q++) {
      const int iu = uiu[q], id = uid[q];
      const double cf = ucf[q] * dv0[iu] * dv1[id];
      c0 += cf;
      c1 += cf * ((S.ns[0] ? del0[iu] : 0.0) + (S.ns[1] ? del1[id] : 0.0));
    }
    c0s[s][u] = c0;
    c1s[s][u] = c1;
  }
  double es = 0.0;
  for (int s = 0; s < 2; s++) {
    const int ns = S.ns[s], nocc = S.nocc[s];
    const double *y = w_y(L, ws, s), *dt = dts[s];
    for (int e = lane; e < nocc * ns; e += G) {
      const int j = e / ns, i = e % ns;
      es += y[e] * dt[i * NO + cst(S.occ[s])[j]];
    }
  }
  const double esum = gsum<G>(es);
  __syncthreads();
  // ---- dy_bld
  for (int s = 0; s < 2; s++) {
    const int ns = S.ns[s], nocc = S.nocc[s];
    const double *inv = w_inv(L, ws, s), *idti = ids[s], *y = w_y(L, ws, s);
    const double *c0 = c0s[s], *c1 = c1s[s];
    double *dy = dys[s];
    // contributions to entry e (the Y-entry CSR lists of eval_y, ascending u)
    const cptr<int> yoff = cst(S.yent_off[s]), yu = cst(S.yent_u[s]), yp = cst(S.yent_pos[s]);
    for (int e = lane; e < nocc * ns; e += G) {
      double a = 0.0;
      const int q1 = yoff[e + 1];
#pragma unroll 4
      for (int q = yoff[e]; q < q1; q++) {
        const int u = yu[q], o = yp[q];
        a += c1[u] * inv[o] - c0[u] * idti[o];
      }
      dy[e] = a * chii - esum * y[e];
    }
  }
  __syncthreads();
  // ---- dg_bld
  for (int s = 0; s < 2; s++) {
    const int ns = S.ns[s], nocc = S.nocc[s], off = s ? S.nup : 0;
    if (ns == 0) continue;
    const double *tf = tfs[s], *dt = dts[s], *dy = dys[s];
    const double *y = w_y(L, ws, s), *g = ss + SL.g[s], *ai = w_ai(L, ws, s);
    double *dg = dgs[s];
    for (int e = lane; e < nocc * ns; e += G) aux[e] = 0.0;
    __syncthreads();
    for (int e = lane; e < ns * ns; e += G) {
      const int k = e / ns, i = e % ns;
      double a = 0.0;
      for (int j = 0; j < nocc; j++) {
        const int oj = cst(S.occ[s])[j];
        a += tf[k * NO + oj] * dy[j * ns + i] + dt[k * NO + oj] * y[j * ns + i];
      }
      aux[cst(S.iref[s])[k] * ns + i] = a;
    }
    __syncthreads();
    for (int e = lane; e < nocc * ns; e += G) {
      const int j = e / ns, i = e % ns;
      double a3 = 0.0;
      for (int q = 0; q < ns; q++) a3 += g[j * ns + q] * B[(off + q) * NO + cst(S.ref[s])[i]];
      aux[e] = dy[e] - a3 - aux[e];
    }
    __syncthreads();
    for (int e = lane; e < nocc * ns; e += G) {
      const int j = e / ns, i = e % ns;
      double a = 0.0;
      for (int q = 0; q < ns; q++) a += aux[j * ns + q] * ai[q + ns * i];
      dg[e] = a;
    }
    __syncthreads();
  }
  // ---- outputs
  double *o1 = dpsi + (int64_t)w * P, *o2 = deloc + (int64_t)w * P;
  for (int ip = lane; ip < S.npcsf; ip += G) {
    const int icsf = cst(S.pcsf)[ip];
    double dd = 0.0, de = 0.0;
    for (int q = cst(S.csf_det_off)[icsf]; q < cst(S.csf_det_off)[icsf + 1]; q++) {
      const int d = cst(S.csf_det)[q];
      const int iu = cst(S.iwdet[0])[d], id = cst(S.iwdet[1])[d];
      const double cf = cst(S.dsgn[0])[iu] * cst(S.dsgn[1])[id] * cst(S.csf_det_coef)[q] * dv0[iu] * dv1[id] * chii;
      const double dl = (S.ns[0] ? del0[iu] : 0.0) + (S.ns[1] ? del1[id] : 0.0);
      dd += cf;
      de += cf * (dl - esum);
    }
    o1[ip] = dd;
    o2[ip] = de;
  }
  // the Jastrow's parameters from their slots (k_deriv_jas, and the
  // pseudopotential's part from k_deriv_nlpp)
  const double *dj = ss + DL.dj, *dsl = ss + DL.dpe_slot;
  for (int ip = lane; ip < S.npj; ip += G) {
    double dv = 0.0, de = 0.0;
    for (int q = cst(S.pj_off)[ip]; q < cst(S.pj_off)[ip + 1]; q++) {
      const int sl = S.pj_slot[q];
      const double w = S.pj_w[q];
      dv += w * dj[2 * sl];
      de += w * (dj[2 * sl + 1] + (S.nloc > 0 ? dsl[sl] : 0.0));
    }
    o1[S.npcsf + ip] = dv;
    o2[S.npcsf + ip] = de;
  }
  for (int ip = lane; ip < S.nporb; ip += G) {
    const int oi = cst(S.porb_i)[ip], oj = cst(S.porb_j)[ip];
    double dp = 0.0, de = 0.0;
    for (int pass = 0; pass < (cst(S.porb_rev)[ip] ? 2 : 1); pass++) {
      const int a = pass ? oj : oi, b = pass ? oi : oj;
      const double sg = pass ? -1.0 : 1.0;
      for (int s = 0; s < 2; s++) {
        const int ns = S.ns[s], off = s ? S.nup : 0;
        const int pa = cst(S.iocc_lab[s])[a];
        if (ns == 0 || pa < 0) continue;
        const double *g = ss + SL.g[s], *dg = dgs[s];
        for (int k = 0; k < ns; k++) {
          const double o = ob[((int64_t)(off + k) * NO + b) * OS];
          dp += sg * g[pa * ns + k] * o;
          de += sg * (g[pa * ns + k] * B[(off + k) * NO + b] + dg[pa * ns + k] * o);
        }
      }
    }
    o1[S.npcsf + S.npj + ip] = dp;
    o2[S.npcsf + S.npj + ip] = de;
  }
}

}  // namespace qmcw
