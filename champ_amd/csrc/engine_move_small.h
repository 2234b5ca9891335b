// engine_move_small.h -- the one-electron move of systems whose electrons
// fit a lane group, with everything pending in LDS and registers.
//
// k_ratio_1e keeps the pending move in global scratch: each of its phases
// stores what the next one loads, about a dozen trips to L2 and back per
// move, and the commit reads the record once more.  On the C2-like system the
// waves waited 62% of the time (16,384 walkers, 92 us mixed, 115 us FP64;
// here 73 and 78 us).
// Here a move that is decided in the same launch (VMC sweep, DMC, given
// moves to commit) reads what it needs of the walker's state in one batch,
// exchanges values between its phases through LDS, keeps the pair row in the
// registers of the lane that owns the other electron (N <= G), and stores the
// candidates and, when accepted, the rows once.  The operations are
// k_ratio_1e's, in its order but for the sums of the matrix product.
#pragma once
#include "engine_kernels.h"

namespace qmcw {

// The LDS record of a walker (doubles): ML's xn, ren, rven, misc and slat
// (A.ML holds their offsets for the launch), then A^-1 and T of the moved
// electron's spin (updated in place), its occupied-orbital row (old, then
// new), and the region that the old Y, the e-e-n tables, the basis values of a
// pass and eval_y's inputs with the new Y take in turn.  The region is as
// small as its users allow: eight blocks of the C2-like system's walkers fit
// a compute unit (18.9 KB each; with 26 KB the same kernel took 129 us).
struct SmallMove {
  int ai, t, orb, r, stride;
  int ynew;                    // the new Y's place in the region (eval_y's determinants, when they have room)
  int cols;                    // basis functions of a pass over the centres
};
__host__ __device__ inline int small_max(int a, int b) { return a > b ? a : b; }
// cols: basis functions a pass has room for; tab: T values of the tables; ts: sizeof(T)
__host__ __device__ inline void small_move_layout(const DevSys &S, int cols, int tab, int ts, MLayout &ML,
                                                  SmallMove &sm) {
  const int nsm = small_max(S.ns[0], S.ns[1]), nom = small_max(S.nocc[0], S.nocc[1]);
  int o = 0;
  ML.xn = o; o += 3;
  ML.ren = o; o += S.M;
  ML.rven = o; o += 3 * S.M;
  ML.misc = o; o += 14 + nsm + nom;
  ML.slat = o; o += 4;
  sm.ai = o; o += nsm * nsm;
  sm.t = o; o += S.single_det ? 0 : nsm * nom;     // (a single determinant needs neither T nor Y)
  sm.orb = o; o += 5 * nom;
  sm.r = o;
  const int y = S.single_det ? 0 : nsm * nom, nd = S.ndetu[0] + S.ndetu[1];
  int ev = S.single_det ? 0 : y_lds_doubles(S.ndetu[0], S.ndetu[1], S.kmax2);
  sm.ynew = nd >= y ? 0 : ev;
  if (nd < y) ev += y;
  o += small_max(small_max(small_max(y, ev), nsm), (small_max(5 * cols, tab) * ts + 7) / 8);
  sm.stride = o | 1;           // odd: the groups' records start in different banks
  sm.cols = cols;
}

typedef double sm_d4 __attribute__((ext_vector_type(4)));

// n values from src to dst by the group's lanes, four loads in flight per lane
template <int G>
__device__ __forceinline__ void stage(double *dst, const double *__restrict__ src, int n, int lane) {
  for (int b = 0; b < n; b += 4 * G) {
    double v[4];
#pragma unroll
    for (int u = 0; u < 4; u++) v[u] = b + lane + u * G < n ? src[b + lane + u * G] : 0.0;
#pragma unroll
    for (int u = 0; u < 4; u++)
      if (b + lane + u * G < n) dst[b + lane + u * G] = v[u];
  }
}

template <typename T, int G, int ORD>
__global__ QMCW_HEAVY void k_move_small(KArgs A, SmallMove sm, int ie, int mode, const double *xnew_in,
                                        double delta, double fbias, long long *nacc) {
  QMCW_GROUP_SETUP
  // the lanes of every group work on the wave's matrix products, so a wave
  // leaves as a whole (the moves not accepted then change nothing)
  const bool given = mode == 4 && A.acc_in[w] != 0;
  if (mode == 4 && !__any(given)) return;
  const int N = S.N, M = S.M, noccmax = S.noccmax;
  const WLayout &L = A.L;
  const MLayout &ML = A.ML;
  const int s = ie < S.nup ? 0 : 1, ns = S.ns[s], nocc = S.nocc[s], e = s ? ie - S.nup : ie;
  const bool single = S.single_det;
  extern __shared__ double dyn_lds[];
  double *mv = dyn_lds + (int64_t)grp * sm.stride;
  double *ai = mv + sm.ai, *t = mv + sm.t, *orb = mv + sm.orb, *R = mv + sm.r, *ynew = R + sm.ynew;
  double *xn = mv + ML.xn, *ren = mv + ML.ren, *rven = mv + ML.rven, *misc = mv + ML.misc;
  // ---- the walker's slots, then everything the move reads of its state
  const double pv = lane < 5 ? ws[L.par + lane] : 0.0;
  const int sl_a = __shfl(pv, s, G) != 0.0, sl_t = __shfl(pv, 2 + s, G) != 0.0,
            sl_o = __shfl(pv, 3 - s, G) != 0.0, sl_y = __shfl(pv, 4, G) != 0.0;
  const int j = lane;                          // the lane's electron
  const bool has = j < N, other = has && j != ie;
  const int jc = has ? j : 0, hi = jc < ie ? ie : jc, lo = jc < ie ? jc : ie;
  const double xj[3] = {ws[L.x + 3 * jc], ws[L.x + 3 * jc + 1], ws[L.x + 3 * jc + 2]};
  const double fj_old[3] = {ws[L.fjo + 3 * jc], ws[L.fjo + 3 * jc + 1], ws[L.fjo + 3 * jc + 2]};
  const double f_old = ws[L.fso + hi * N + lo];
  const double *gi_p = ws + L.fijo + 3 * (ie * N + jc), *gj_p = ws + L.fijo + 3 * (jc * N + ie);
  const double gi_old[3] = {gi_p[0], gi_p[1], gi_p[2]}, gj_old[3] = {gj_p[0], gj_p[1], gj_p[2]};
  const double fsumo = ws[L.fsumo], chio = ws[L.chi], deta_s = ws[L.deta[s]], deta_o = ws[L.deta[1 - s]];
  stage<G>(ai, ws + L.ai[s][sl_a], ns * ns, lane);
  stage<G>(orb, ws + L.oc + (int64_t)ie * noccmax * 5, 5 * nocc, lane);
  if (!single) {
    stage<G>(t, ws + L.tocc[s][sl_t], ns * nocc, lane);
    stage<G>(R, ws + L.y[s][sl_y], ns * nocc, lane);
  }
  __syncthreads();
  // ---- proposal (k_ratio_1e's modes: 2 VMC, 3 DMC; otherwise the position is given)
  if (mode == 2 || mode == 3) {
    const double fji[3] = {__shfl(fj_old[0], ie, G), __shfl(fj_old[1], ie, G), __shfl(fj_old[2], ie, G)};
    double vold[3];
    group_grad_1e<G>(A, ws, ie, orb, ai, t, R, fji, 0.0, vold, nullptr, lane);
    if (lane == 0) {
      if (mode == 3) dmc_propose_w(A, w, ie, vold, A.dm + (int64_t)w * kDmStride, A.dmp, xn);
      else vmc_propose_w(A, w, ie, ws, vold, delta, fbias, xn, mv);
    }
  } else if (lane < 3) {
    xn[lane] = xnew_in[3 * w + lane];
  }
  __syncthreads();
  // ---- distances
  for (int ic = lane; ic < M; ic += G) {
    double s2 = 0.0;
    for (int q = 0; q < 3; q++) {
      const double d = xn[q] - cst(S.cent)[3 * ic + q];
      rven[3 * ic + q] = d;
      s2 += d * d;
    }
    ren[ic] = sqrt(s2);
  }
  double rvee[3], ree = 0.0;
  {
    double s2 = 0.0;
#pragma unroll
    for (int q = 0; q < 3; q++) {
      rvee[q] = hi == ie ? xn[q] - xj[q] : xj[q] - xn[q];
      s2 += rvee[q] * rvee[q];
    }
    ree = sqrt(s2);
  }
  __syncthreads();
  // ---- Jastrow row: the lane's pair (ie, j), the e-n terms on lane ie
  T *Rt = reinterpret_cast<T *>(R);
  if (A.een_tab) {
    een_tables<T, ORD, G>(S, ren, rven, Rt, lane);
    __syncthreads();
  }
  double fn = 0.0, gin[3] = {0.0, 0.0, 0.0}, gjn[3] = {0.0, 0.0, 0.0}, lin = 0.0, ljn = 0.0;
  if (has && j == ie) {
    T f, g[3], lp;
    jas_en<T>(S, ren, rven, f, g, lp);
    fn = f; lin = lp;
    gin[0] = g[0]; gin[1] = g[1]; gin[2] = g[2];
  } else if (other) {
    PairOut<T> po;
    const bool par = (hi < S.nup) || (lo >= S.nup), mi = hi == ie;
    const T rvij[3] = {(T)rvee[0], (T)rvee[1], (T)rvee[2]};
    const EnFromX pJ{xj[0], xj[1], xj[2]};
    if (A.een_tab) {
      const T rvmo[3] = {mi ? rvij[0] : -rvij[0], mi ? rvij[1] : -rvij[1], mi ? rvij[2] : -rvij[2]};
      jas_pair_tab<T, ORD>(S, par, (T)ree, rvmo, Rt, pJ, mi, po);
    } else {
      const EnRows pI{ren, rven};
      if (mi) jas_pair_g<T, ORD>(S, par, (T)ree, rvij, pI, pJ, po);
      else jas_pair_g<T, ORD>(S, par, (T)ree, rvij, pJ, pI, po);
    }
    fn = po.f;
#pragma unroll
    for (int q = 0; q < 3; q++) {
      gin[q] = mi ? po.gi[q] : po.gj[q];
      gjn[q] = mi ? po.gj[q] : po.gi[q];
    }
    lin = mi ? po.li : po.lj;
    ljn = mi ? po.lj : po.li;
  }
  double fji[3], fjn[3];
#pragma unroll
  for (int q = 0; q < 3; q++) {
    fjn[q] = fj_old[q] + gjn[q] - gj_old[q];
    fji[q] = __shfl(fj_old[q], ie, G) + gsum<G>(has ? gin[q] - gi_old[q] : 0.0);
    if (j == ie) fjn[q] = fji[q];
  }
  const double fsumn = fsumo + gsum<G>(has ? fn - f_old : 0.0);
  const double lapjn = gsum<G>(lin) + fji[0] * fji[0] + fji[1] * fji[1] + fji[2] * fji[2];
  // ---- orbitals of the new position: the basis values of a few centres at a
  // time, contracted for all of the wave's walkers together on FP64 MFMA, rows
  // (walker, component) by columns of orbitals: the walkers share the
  // coefficients.  An orbital per lane took 1,400 of the move's 7,000 vector
  // instructions on the C2-like system (10 orbitals for 8 lanes).
  {
    constexpr int W = kWave / G, RT = (5 * W + 15) / 16, CT = RT == 2 ? 2 : 1;
    const int lid = threadIdx.x, r = lid & 15, kq = lid >> 4;
    const bool mfma = nocc <= 16 * CT;
    sm_d4 acc[RT][CT];
#pragma unroll
    for (int a = 0; a < RT; a++)
#pragma unroll
      for (int b = 0; b < CT; b++) acc[a][b] = sm_d4{0.0, 0.0, 0.0, 0.0};
    // the LDS address of this lane's rows (walker row / 5, component row % 5)
    const T *pa[RT];
    bool va[RT];
#pragma unroll
    for (int a = 0; a < RT; a++) {
      const int row = 16 * a + r;
      va[a] = row < 5 * W;
      pa[a] = reinterpret_cast<const T *>(dyn_lds + (int64_t)(va[a] ? row / 5 : 0) * sm.stride + sm.r) +
              (va[a] ? row % 5 : 0);
    }
    if (!mfma)
      for (int q = lane; q < 5 * nocc; q += G) orb[q] = 0.0;
    const cptr<double> co = cst(S.coef_occ[s]);
    for (int c0 = 0; c0 < M;) {
      const int b0 = cst(S.cent_bas)[c0];
      int c1 = c0 + 1;
      while (c1 < M && cst(S.cent_bas)[c1 + 1] - b0 <= sm.cols) c1++;
      const int nb = cst(S.cent_bas)[c1] - b0;
      __syncthreads();
      // shells of equal l on neighbouring lanes
      for (int q = cst(S.cent_sh_off)[c0] + lane; q < cst(S.cent_sh_off)[c1]; q += G) {
        const int sh = c1 - c0 == M ? cst(S.sh_by_l)[q] : q, ic = cst(S.sh_cent)[sh];
        eval_shell<T>(S, sh, (T)rven[3 * ic], (T)rven[3 * ic + 1], (T)rven[3 * ic + 2], (T)ren[ic], 1,
                      Rt - 5 * b0);
      }
      __syncthreads();
      if (mfma) {
        for (int k0 = 0; k0 < nb; k0 += 4) {
          const bool ok = k0 + kq < nb;
          double bv[CT];
#pragma unroll
          for (int b = 0; b < CT; b++)
            bv[b] = (ok && 16 * b + r < nocc) ? co[(int64_t)(b0 + k0 + kq) * nocc + 16 * b + r] : 0.0;
#pragma unroll
          for (int a = 0; a < RT; a++) {
            const double av = (ok && va[a]) ? (double)pa[a][5 * (k0 + kq)] : 0.0;
#pragma unroll
            for (int b = 0; b < CT; b++)
              if (16 * b < nocc) acc[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(av, bv[b], acc[a][b], 0, 0, 0);
          }
        }
      } else {
        for (int q = lane; q < nocc; q += G)
          contract5_add<T>(co + (int64_t)b0 * nocc, nocc, nb, q, Rt, orb + 5 * q);
      }
      c0 = c1;
    }
    if (mfma) {
#pragma unroll
      for (int a = 0; a < RT; a++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const int row = 16 * a + kq + 4 * q;
          if (row >= 5 * W) continue;
          double *o = dyn_lds + (int64_t)(row / 5) * sm.stride + sm.orb + row % 5;
#pragma unroll
          for (int b = 0; b < CT; b++)
            if (16 * b + r < nocc) o[5 * (16 * b + r)] = acc[a][b][q];
        }
    }
  }
  __syncthreads();
  // ---- dete_update (qmc/dete_mod.f90:114-214), in place; the candidates also
  // go to the state's other slots
  double rat = 0.0;
  for (int k = lane; k < ns; k += G) rat += orb[5 * cst(S.iref[s])[k]] * ai[k + ns * e];
  rat = gsum<G>(rat);
  double *vi1 = misc + 8, *vi2 = vi1 + ns, *u = R;
  sm_vectors<G>(vi1, vi2, orb, ai, t, S.iref[s], ns, nocc, e, lane, single);
  for (int k = lane; k < ns; k += G) u[k] = -ai[k + ns * e] / rat;
  __syncthreads();
  {
    double *g_ai = ws + L.ai[s][sl_a ^ 1], *g_t = ws + L.tocc[s][sl_t ^ 1];
    // (the division once, then the remainder carried along)
    for (int q = lane, c = lane / ns, k = lane - c * ns; q < ns * ns; q += G) {
      const double v = ai[q] + u[k] * vi1[c];
      ai[q] = v;
      g_ai[q] = v;
      for (k += G; k >= ns; k -= ns) c++;
    }
    if (!single)
      for (int q = lane, k = lane / nocc, c = lane - k * nocc; q < ns * nocc; q += G) {
        const double v = t[q] + u[k] * vi2[c];
        t[q] = v;
        g_t[q] = v;
        for (c += G; c >= nocc; c -= nocc) k++;
      }
  }
  __syncthreads();
  double chin;
  if (single) {
    chin = cst(S.cdd)[0] * ws[L.detv[0][(s ? sl_o : sl_t)]] * ws[L.detv[1][(s ? sl_t : sl_o)]];
  } else {
    // alpha blocks of the spin, the other spin's from the state, then chi and Y
    const int nu0 = S.ndetu[0], nu1 = S.ndetu[1], k2 = S.kmax2, nus = S.ndetu[s], nuo = S.ndetu[1 - s];
    double *dv0 = R, *dv1 = dv0 + nu0, *iv0 = dv1 + nu1, *iv1 = iv0 + nu0 * k2, *cup = iv1 + nu1 * k2;
    double *dvs = s ? dv1 : dv0, *ivs = s ? iv1 : iv0;
    stage<G>(s ? dv0 : dv1, ws + L.detv[1 - s][sl_o], nuo, lane);
    stage<G>(s ? iv0 : iv1, ws + L.inv[1 - s][sl_o], nuo * k2, lane);
    double *g_inv = ws + L.inv[s][sl_t ^ 1], *g_det = ws + L.detv[s][sl_t ^ 1];
    const cptr<int> ord = cst(S.ord[s]), rf = cst(S.rf[s]), exo = cst(S.exo[s]);
    for (int d = lane; d < nus; d += G) {
      const int k = ord[d];
      double *blk = ivs + d * k2;
      for (int ii = 0; ii < k; ii++)
        for (int jj = 0; jj < k; jj++) blk[jj + k * ii] = t[rf[d * ns + jj] * nocc + exo[d * ns + ii]];
      const double det = small_matinv(blk, k);
      dvs[d] = det;
      g_det[d] = det;
      for (int q = 0; q < k * k; q++) g_inv[d * k2 + q] = blk[q];
    }
    __syncthreads();
    chin = 0.0;
#pragma unroll 4
    for (int d = lane; d < S.ndet; d += G)
      chin += cst(S.cdd)[d] * dv0[cst(S.iwdet[0])[d]] * dv1[cst(S.iwdet[1])[d]];
    chin = gsum<G>(chin);
    const double chii = 1.0 / chin;
    for (int q = lane; q < nu0 + nu1; q += G) {
      const int sp = q < nu0 ? 0 : 1, d = sp ? q - nu0 : q;
      const cptr<int> iu = cst(S.uiu[sp]), id = cst(S.uid[sp]);
      const cptr<double> cf = cst(S.ucf[sp]);
      double cu = 0.0;
      const int q1 = cst(S.udet_off[sp])[d + 1];
#pragma unroll 4
      for (int p = cst(S.udet_off[sp])[d]; p < q1; p++) cu += cf[p] * dv0[iu[p]] * dv1[id[p]];
      cup[q] = cu;
    }
    __syncthreads();
    for (int sp = 0; sp < 2; sp++) {
      const cptr<int> off = cst(S.yent_off[sp]), yu = cst(S.yent_u[sp]), yp = cst(S.yent_pos[sp]);
      const double *cus = cup + (sp ? nu0 : 0), *iv = sp ? iv1 : iv0;
      double *g_y = ws + L.y[sp][sl_y ^ 1];
      for (int q = lane; q < S.nocc[sp] * S.ns[sp]; q += G) {
        double acc = 0.0;
        const int q1 = off[q + 1];
#pragma unroll 4
        for (int p = off[q]; p < q1; p++) acc += cus[yu[p]] * iv[yp[p]];
        acc *= chii;
        g_y[q] = acc;
        if (sp == s) ynew[q] = acc;
      }
    }
  }
  __syncthreads();
  // ---- new gradient, ratio, test
  const double deta_n = deta_s * rat;
  double gnew[3], lapn;
  group_grad_1e<G>(A, ws, ie, orb, ai, t, ynew, fji, lapjn, gnew, &lapn, lane);
  const double logn = log(fabs(chin)) + log(fabs(deta_n)) + log(fabs(deta_o));
  int acc = given;
  if (mode == 2 || mode == 3) {
    if (lane == 0) {
      misc[7] = fsumn;
      misc[8 + ns + nocc] = logn;
      misc[9 + ns + nocc] = (chin * deta_n * deta_o) / (chio * (s ? deta_o : deta_s) * (s ? deta_s : deta_o)) *
                            exp(fsumn - fsumo);
      for (int q = 0; q < 3; q++) misc[10 + ns + nocc + q] = gnew[q];
      acc = mode == 3 ? dmc_decide_w(A, w, ie, mv, A.dm + (int64_t)w * kDmStride, A.dmp)
                      : metrop_accept(A, ws, mv, w, ie, ns, nocc, delta, fbias);
      if (acc && nacc) nacc[w] += 1;
    }
    acc = __shfl(acc, 0, G);
  }
  if (!acc) return;
  // ---- commit (group_commit)
  for (int q = lane; q < 5 * nocc; q += G) ws[L.oc + (int64_t)ie * noccmax * 5 + q] = orb[q];
  for (int q = lane; q < M; q += G) ws[L.r_en + ie * M + q] = ren[q];
  for (int q = lane; q < 3 * M; q += G) ws[L.rvec_en + ie * M * 3 + q] = rven[q];
  if (lane < 3) ws[L.x + 3 * ie + lane] = xn[lane];
  if (has) {
#pragma unroll
    for (int q = 0; q < 3; q++) {
      ws[L.fjo + 3 * j + q] = fjn[q];
      ws[L.fijo + 3 * (ie * N + j) + q] = gin[q];
    }
    ws[L.fso + hi * N + lo] = fn;
    ws[L.lapj + ie * N + j] = lin;
    if (other) {
      ws[L.r_ee + hi * N + lo] = ree;
#pragma unroll
      for (int q = 0; q < 3; q++) {
        ws[L.rvec_ee + 3 * (hi * N + lo) + q] = rvee[q];
        ws[L.fijo + 3 * (j * N + ie) + q] = gjn[q];
      }
      ws[L.lapj + j * N + ie] = ljn;
    }
  }
  if (lane == 0) {
    ws[L.par + s] = sl_a ? 0.0 : 1.0;
    if (!single) {
      ws[L.par + 2 + s] = sl_t ? 0.0 : 1.0;
      ws[L.par + 4] = sl_y ? 0.0 : 1.0;
    }
    ws[L.chi] = chin;
    ws[L.deta[s]] = deta_n;
    ws[L.fsumo] = fsumn;
    ws[L.psij] = fsumn;
    ws[L.logpsid] = logn;
    ws[L.psi2o] = 2.0 * (logn + fsumn);
  }
}

}  // namespace qmcw
