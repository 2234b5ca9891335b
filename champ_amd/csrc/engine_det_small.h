// engine_det_small.h -- the determinant part of the full evaluation for
// small spins, with a walker's matrices in LDS.
//
// k_full_det inverts the Slater matrices, forms T, the alpha blocks, Y and G
// in the walker's record in global memory, about sixty dependent passes over
// matrices of a few dozen values: each pass waited for a store to reach L2
// and come back (85% of the 164 us of 16,384 C2-like walkers, mixed; 70 us
// here).  Now the orbital values are read once, both spins are worked on side
// by side (half of the walker's lanes each), every pass exchanges values
// through LDS, and the results go out once.  The operations and their order are
// k_full_det's.
#pragma once
#include "engine_kernels.h"

namespace qmcw {

constexpr int kDetSmallNs = 15;    // from 16 electrons of a spin on k_full_det stages them in LDS itself

// doubles of LDS per walker
__host__ __device__ inline int det_small_doubles(const DevSys &S) {
  int n = 0;
  for (int s = 0; s < 2; s++) {
    const int ns = S.ns[s], no = S.nocc[s];
    // orbital values, elimination, inverse, T, Y, Y A^-1, G; alpha inverses,
    // determinants and coefficient sums; two permutations of ns ints
    n += 2 * ns * ns + 5 * ns * no + S.ndetu[s] * (2 + S.kmax2) + ns + 1;
  }
  return n;
}

template <int G>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2, 8)))
void k_det_small(KArgs A) {
  QMCW_GROUP_SETUP
  constexpr int H = G / 2;                       // lanes of a spin
  const int N = S.N, noccmax = S.noccmax;
  const WLayout &L = A.L;
  const SLayout &SL = A.SL;
  double *oc = ws + L.oc;
  double *vd = ss + SL.vd, *divv = ss + SL.divv, *red = ss + SL.phs;
  const int s = lane / H, l = lane % H;
  const int ns = S.ns[s], nocc = S.nocc[s], off = s ? S.nup : 0, nu = S.ndetu[s], k2 = S.kmax2;
  const int nmax = max(S.ns[0], S.ns[1]);
  extern __shared__ double dyn_lds[];
  double *base = dyn_lds + (int64_t)grp * det_small_doubles(S);
  double *p_o[2], *p_a[2], *p_i[2], *p_t[2], *p_y[2], *p_m[2], *p_g[2], *p_iv[2], *p_dv[2], *p_cu[2];
  int *p_pv[2];
  for (int q = 0; q < 2; q++) {
    const int n = S.ns[q], no = S.nocc[q], u = S.ndetu[q];
    p_o[q] = base; base += n * no;
    p_a[q] = base; base += n * n;
    p_i[q] = base; base += n * n;
    p_t[q] = base; base += n * no;
    p_y[q] = base; base += n * no;
    p_m[q] = base; base += n * no;
    p_g[q] = base; base += n * no;
    p_iv[q] = base; base += u * k2;
    p_dv[q] = base; base += u;
    p_cu[q] = base; base += u;
    p_pv[q] = reinterpret_cast<int *>(base); base += n + 1;
  }
  double *o = s ? p_o[1] : p_o[0], *a = s ? p_a[1] : p_a[0], *ai = s ? p_i[1] : p_i[0];
  double *t = s ? p_t[1] : p_t[0], *y = s ? p_y[1] : p_y[0], *m = s ? p_m[1] : p_m[0];
  double *g = s ? p_g[1] : p_g[0], *iv = s ? p_iv[1] : p_iv[0], *dv = s ? p_dv[1] : p_dv[0];
  int *ipiv = s ? p_pv[1] : p_pv[0];
  const cptr<int> iref = cst(S.iref[s]);
  // orbital values o(i, j) of the spin's occupied orbitals at o[i + ns * j]
  for (int e = l; e < ns * nocc; e += H) {
    const int i = e % ns, j = e / ns;
    o[e] = oc[((int64_t)(off + i) * noccmax + j) * 5];
  }
  for (int i = l; i < ns; i += H) ipiv[i] = i;
  __syncthreads();
  for (int e = l; e < ns * ns; e += H) a[e] = o[e % ns + ns * iref[e / ns]];
  __syncthreads();
  // ---- group_matinv's elimination, both spins in step
  double det = 1.0;
  bool singular = false;
  for (int i = 0; i < nmax; i++) {
    const int col = i * ns;
    const bool on = i < ns;
    double am = -1.0, vm = __builtin_nan("");
    int km = i;
    if (on)
      for (int k = i + l; k < ns; k += H) {
        const double v = a[ipiv[k] + col];
        if (fabs(v) > am) { am = fabs(v); vm = v; km = k; }
      }
#pragma unroll
    for (int q = H / 2; q > 0; q >>= 1) {
      const double a2 = __shfl_xor(am, q, H), v2 = __shfl_xor(vm, q, H);
      const int kk = __shfl_xor(km, q, H);
      if (a2 > am || (a2 == am && kk < km)) { am = a2; km = kk; vm = v2; }
    }
    __syncthreads();
    if (on && !singular) {
      if (l == 0 && km != i) { const int q = ipiv[i]; ipiv[i] = ipiv[km]; ipiv[km] = q; }
      if (km != i) det = -det;
      det *= vm;
      if (vm == 0.0) singular = true;
    }
    __syncthreads();
    const bool go = on && !singular;
    const int p = on ? ipiv[i] : 0;
    const double inv = go ? 1.0 / vm : 0.0;
    if (go)
      for (int q = l; q < ns; q += H) a[p + q * ns] = (q == i ? 1.0 : a[p + q * ns]) * inv;
    __syncthreads();
    if (go)
      for (int j = l; j < ns; j += H) {
        if (j == p) continue;
        const double f = -a[j + col];
        a[j + col] = 0.0;
        for (int q = 0; q < ns; q++) a[j + q * ns] += f * a[p + q * ns];
      }
    __syncthreads();
  }
  if (singular) det = 0.0;
  // the inverse (r, ipiv[c]) = a(ipiv[r], c), to the record as well
  double *ai_g = w_ai(L, ws, s), *t_g = w_tocc(L, ws, s), *y_g = w_y(L, ws, s);
  double *iv_g = w_inv(L, ws, s), *dv_g = w_detv(L, ws, s), *g_g = ss + SL.g[s];
  if (l == 0) ws[L.deta[s]] = ns == 0 ? 1.0 : det;
  for (int q = l; q < ns * ns; q += H) {
    const int r = q % ns, c = q / ns, d = r + ipiv[c] * ns;
    const double v = singular ? 0.0 : a[ipiv[r] + c * ns];
    ai[d] = v;
    ai_g[d] = v;
  }
  __syncthreads();
  // ---- T(k, occ_j) = sum_i A^-1(k, i) orb(i, occ_j)
  for (int e = l; e < ns * nocc; e += H) {
    const int k = e / nocc, j = e % nocc;
    double acc = 0.0;
    for (int i = 0; i < ns; i++) acc += ai[k + ns * i] * o[i + ns * j];
    t[e] = acc;
    t_g[e] = acc;
  }
  __syncthreads();
  // ---- alpha blocks of the unique determinants
  if (ns == 0) {
    if (l == 0) { dv[0] = 1.0; dv_g[0] = 1.0; }
  } else {
    const cptr<int> ord = cst(S.ord[s]), rf = cst(S.rf[s]), exo = cst(S.exo[s]);
    for (int u = l; u < nu; u += H) {
      const int k = ord[u];
      double *blk = iv + u * k2;
      for (int ii = 0; ii < k; ii++)
        for (int jj = 0; jj < k; jj++) blk[jj + k * ii] = t[rf[u * ns + jj] * nocc + exo[u * ns + ii]];
      const double d = small_matinv(blk, k);
      dv[u] = d;
      dv_g[u] = d;
      for (int q = 0; q < k * k; q++) iv_g[u * k2 + q] = blk[q];
    }
  }
  __syncthreads();
  // ---- chi, coefficient sums and Y (group_eval_y_lds)
  double chi = 0.0;
  for (int d = lane; d < S.ndet; d += G)
    chi += cst(S.cdd)[d] * p_dv[0][cst(S.iwdet[0])[d]] * p_dv[1][cst(S.iwdet[1])[d]];
  chi = gsum<G>(chi);
  const double chii = 1.0 / chi;
  {
    const cptr<int> iu = cst(S.uiu[s]), id = cst(S.uid[s]), uo = cst(S.udet_off[s]);
    const cptr<double> cf = cst(S.ucf[s]);
    double *cu = s ? p_cu[1] : p_cu[0];
    for (int u = l; u < nu; u += H) {
      double v = 0.0;
      const int q1 = uo[u + 1];
#pragma unroll 4
      for (int q = uo[u]; q < q1; q++) v += cf[q] * p_dv[0][iu[q]] * p_dv[1][id[q]];
      cu[u] = v;
    }
    __syncthreads();
    const cptr<int> yo = cst(S.yent_off[s]), yu = cst(S.yent_u[s]), yp = cst(S.yent_pos[s]);
    for (int e = l; e < nocc * ns; e += H) {
      double v = 0.0;
      const int q1 = yo[e + 1];
#pragma unroll 4
      for (int q = yo[e]; q < q1; q++) v += cu[yu[q]] * iv[yp[q]];
      y[e] = v * chii;
      y_g[e] = v * chii;
    }
  }
  if (lane == 0) ws[L.chi] = chi;
  __syncthreads();
  // ---- G (group_g): A^-1 - T Y A^-1 on the reference rows, Y A^-1 on the others
  const bool plain = nu == 1;
  for (int e = l; e < nocc * ns; e += H) {
    const int j = e / ns, i = e % ns;
    double v = 0.0;
    if (!plain)
      for (int k = 0; k < ns; k++) v += y[j * ns + k] * ai[k + ns * i];
    m[e] = v;
    g[e] = v;
  }
  __syncthreads();
  for (int e = l; e < ns * ns; e += H) {
    const int k = e / ns, i = e % ns;
    double v = 0.0;
    if (!plain)
      for (int j = 0; j < nocc; j++) v += t[k * nocc + j] * m[j * ns + i];
    g[iref[k] * ns + i] = ai[k + ns * i] - v;
  }
  __syncthreads();
  for (int e = l; e < nocc * ns; e += H) g_g[e] = g[e];
  // ---- gradient and laplacian of ln D (qmc/vmc/determinant.f90:99-152)
  double d2d = 0.0;
  for (int i = lane; i < N; i += G) {
    const int sp = i < S.nup ? 0 : 1, ie = sp ? i - S.nup : i, n = S.ns[sp], no = S.nocc[sp];
    const double *gs = sp ? p_g[1] : p_g[0];
    double dx = 0, dy = 0, dz = 0, ek = 0;
#pragma unroll 4
    for (int j = 0; j < no; j++) {
      const double gj = gs[j * n + ie];
      const double *q = oc + ((int64_t)i * noccmax + j) * 5;
      dx += gj * q[1]; dy += gj * q[2]; dz += gj * q[3]; ek += gj * q[4];
    }
    vd[3 * i] = dx; vd[3 * i + 1] = dy; vd[3 * i + 2] = dz;
    const double dvd = ek - (dx * dx + dy * dy + dz * dz);
    divv[i] += dvd;
    d2d += dvd;
  }
  d2d = gsum<G>(d2d);
  if (lane == 0) red[54] = d2d;
  // the pseudopotential's projected coefficients, when k_gproj_mfma does not form them
  if (S.nloc > 0 && !A.gproj_mfma) {
    __syncthreads();
    group_gproj<G>(S, ss + SL.gproj, ss + SL.g[0], ss + SL.g[1], A.bf16, lane);
  }
}

}  // namespace qmcw
