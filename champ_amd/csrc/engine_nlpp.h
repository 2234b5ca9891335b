// engine_nlpp.h -- the pseudopotential of systems with many electrons and
// centres: the Jastrow of the quadrature points on the matrix cores.
//
// At a quadrature point the e-e-n terms are, for a fixed power k of U and
// with the moved electron's A at the point fixed, a sum over centres and
// powers of the other electron's B (een_gamma):
//   sum_j sum_k U_j^k W_kj,  W_kj = sum_c [gam_k0(A_c) + sum_n gam_kn(A_c) B_cj^n].
// W_k over (point, electron j) is a matrix product with inner index
// (centre, n): the powers of B are the walker's, shared by all of its points.
// Summed pair by pair (jas_point_val), each lane reads its U and each B for
// every (electron, centre) of its point, and the per-lane point scratch of a
// large system does not fit LDS: on the 98-electron chain (50 centres) the
// vector units issued 20% of the time.  Here a wavefront takes 64 points,
// forms their determinant ratios one point per lane, then takes them 16 at a
// time through 16x16x4 MFMA tiles (four centres per step; the lane that
// supplies a (point, centre) operand forms that centre's gammas), and the
// e-e terms and the powers of U in the layout of the result.
#pragma once
#include "engine_kernels.h"

namespace qmcw {

template <typename T>
struct MfmaTile;
template <>
struct MfmaTile<double> {
  typedef double v4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ v4 mac(double a, double b, v4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  // row of the lane's q-th result (column: lane % 16), kq = lane / 16
  static __device__ __forceinline__ int row(int kq, int q) { return kq + 4 * q; }
};
template <>
struct MfmaTile<float> {
  typedef float v4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ v4 mac(float a, float b, v4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int kq, int q) { return 4 * kq + q; }
};

constexpr int kNlppWaves = 4;      // most wavefronts of a walker's block
// 16-electron column tiles per pass over the centres: what two wavefronts
// per SIMD have registers for
template <typename T>
constexpr int nlpp_cols() { return sizeof(T) == 8 ? 3 : 4; }

// LDS of one wavefront: its 64 points and what the tiles return for them
template <typename T, int ORD>
struct NlppTile {
  double x[64][3], r[64];          // position, distance to the pair's centre
  double jas[64];                  // e-e and e-e-n sum
  T en[64], s0[16][ORD + 1];       // e-n sum; sum_c gam_k0 of a tile's rows
  int el[64], ic[64];              // moved electron, the pair's centre
};

// orders the LDS accesses of one wavefront (its lanes exchange data; LDS
// serves a wavefront's accesses in order)
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Jastrow sums (e-n into tl.en, e-e and e-e-n into tl.jas) of the 16 points
// sub, sub + 1, ... of the wavefront's tile.  c_t: the e-e-n coefficients,
// [nctype][nterms], in LDS; bt[ic * N + j] as jas_point_val.
template <typename T, int ORD>
__device__ __forceinline__ void nlpp_tile(const DevSys &S, NlppTile<T, ORD> &tl, int sub, const T *c_t,
                                          const double *x, const T *bt, int lane) {
  typedef MfmaTile<T> MT;
  typedef typename MT::v4 v4;
  constexpr int NG = een_gi<ORD>(ORD, 0) + 1, CT = nlpp_cols<T>();
  const int N = S.N, M = S.M, r = lane & 15, kq = lane >> 4;
  const int nct = (N + 15) / 16;
  const T k = T(S.scalek);
  const int er = sub + r;
  const double px = tl.x[er][0], py = tl.x[er][1], pz = tl.x[er][2], pr = tl.r[er];
  const int pic = tl.ic[er];
  double jsum[4] = {0.0, 0.0, 0.0, 0.0};
  for (int c0 = 0; c0 < nct; c0 += CT) {
    v4 acc[ORD][CT];
#pragma unroll
    for (int kk = 0; kk < ORD; kk++)
#pragma unroll
      for (int t = 0; t < CT; t++) acc[kk][t] = v4{T(0), T(0), T(0), T(0)};
    T en = T(0), s0[ORD + 1];
#pragma unroll
    for (int kk = 0; kk <= ORD; kk++) s0[kk] = T(0);
    for (int ic0 = 0; ic0 < M; ic0 += 4) {
      const bool ok = ic0 + kq < M;
      const int ic = ok ? ic0 + kq : M - 1, it = cst(S.iwctype)[ic];
      T bv[CT];
#pragma unroll
      for (int t = 0; t < CT; t++) {
        const int j = 16 * (c0 + t) + r;
        bv[t] = (ok && j < N) ? bt[ic * N + j] : T(0);
      }
      const double dx = px - cst(S.cent)[3 * ic], dy = py - cst(S.cent)[3 * ic + 1],
                   dz = pz - cst(S.cent)[3 * ic + 2];
      const T rc = (T)(ic == pic ? pr : sqrt(dx * dx + dy * dy + dz * dz));
      T u, t1, t2;
      scaled<T>(S.isc, k, rc, u, t1, t2);
      // een_gamma's table from the coefficients in LDS
      T gam[NG];
      {
        const T *c = c_t + it * S.nterms;
        const T A = T(1) - k * u;
        T ap[ORD + 1];
        ap[0] = T(1);
#pragma unroll
        for (int q = 1; q <= ORD; q++) ap[q] = ap[q - 1] * A;
#pragma unroll
        for (int q = 0; q < NG; q++) gam[q] = T(0);
        int idx = 0;
#pragma unroll
        for (int kk = 0; kk <= ORD; kk++)
#pragma unroll
          for (int m = 0; 2 * m <= ORD - kk; m++)
#pragma unroll
            for (int l = 0; l <= ORD - kk - 2 * m; l++)
              if (QMCW_EEN_TERM(kk, l, m)) {
                const T ct = c[idx];
                idx++;
                gam[een_gi<ORD>(kk, m)] += ct * ap[l + m];
                gam[een_gi<ORD>(kk, l + m)] += ct * ap[m];
              }
      }
      if (!ok) {
#pragma unroll
        for (int q = 0; q < NG; q++) gam[q] = T(0);
      }
      if (c0 == 0) {
#pragma unroll
        for (int kk = 0; kk <= ORD; kk++) s0[kk] += gam[een_gi<ORD>(kk, 0)];
        const cptr<double> a = cst(S.a4) + it * (S.norda + 1);
        T fe = T(a[0]) * u / (T(1) + T(a[1]) * u) - T(cst(S.asymp_jasa)[it]);
        T up = u;
        for (int iord = 2; iord <= S.norda; iord++) {
          up *= u;
          fe += T(a[iord]) * up;
        }
        if (ok) en += fe;
      }
      T bp[CT];
#pragma unroll
      for (int t = 0; t < CT; t++) bp[t] = bv[t];
#pragma unroll
      for (int n = 1; n <= ORD; n++) {
#pragma unroll
        for (int t = 0; t < CT; t++)
          if (c0 + t < nct) {
#pragma unroll
            for (int kk = 0; kk <= ORD - n; kk++)
              acc[kk][t] = MT::mac(gam[een_gi<ORD>(kk, n)], bp[t], acc[kk][t]);
            bp[t] *= bv[t];
          }
      }
    }
    if (c0 == 0) {
      en += __shfl_xor(en, 16, 64);
      en += __shfl_xor(en, 32, 64);
#pragma unroll
      for (int kk = 0; kk <= ORD; kk++) {
        s0[kk] += __shfl_xor(s0[kk], 16, 64);
        s0[kk] += __shfl_xor(s0[kk], 32, 64);
      }
      if (kq == 0) {
        tl.en[er] = en;
#pragma unroll
        for (int kk = 0; kk <= ORD; kk++) tl.s0[r][kk] = s0[kk];
      }
      wave_lds_fence();
    }
    // the e-e terms and the powers of U of the lane's four points and one
    // electron per column tile
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int row = MT::row(kq, q), e = sub + row, i = tl.el[e];
      const double ex = tl.x[e][0], ey = tl.x[e][1], ez = tl.x[e][2];
#pragma unroll
      for (int t = 0; t < CT; t++) {
        const int j = 16 * (c0 + t) + r;
        if (j >= N || j == i) continue;
        const double dx = ex - x[3 * j], dy = ey - x[3 * j + 1], dz = ez - x[3 * j + 2];
        const T rij = (T)sqrt(dx * dx + dy * dy + dz * dz);
        T u, d1, d2;
        scaled<T>(S.isc, k, rij, u, d1, d2);
        T f = jas_b_val<T>(S, (i < S.nup) == (j < S.nup), u);
        const T U = T(1) - k * u;
        T w = tl.s0[row][ORD];
#pragma unroll
        for (int kk = ORD - 1; kk >= 0; kk--) w = w * U + (acc[kk][t][q] + tl.s0[row][kk]);
        jsum[q] += (double)(f + w);
      }
    }
  }
#pragma unroll
  for (int q = 0; q < 4; q++) {
    double v = jsum[q];
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) v += __shfl_xor(v, o, 16);
    if (r == 0) tl.jas[sub + MT::row(kq, q)] = v;
  }
}

// doubles of dynamic LDS of a block: the flags of the (electron, centre)
// pairs in range, a bit each, and their running counts
__host__ __device__ inline int64_t nlpp_tiles_lds(int64_t npairs) { return (npairs + 63) / 64 * 3 / 2 + 1; }
// most bytes of its other LDS (the largest order in FP64)
constexpr size_t kNlppTilesStatic =
    kNlppWaves * sizeof(NlppTile<double, 7>) + sizeof(double) * (kMaxCtype * kMaxTerms + 2 * kNlppWaves);

// k_full_nlpp of one walker by a block of 64 to 64 kNlppWaves lanes
template <typename T, int ORD>
__device__ __forceinline__ void full_nlpp_tiles_b(const KArgs &A, int w) {
  const DevSys &S = A.S;
  const WLayout &L = A.L;
  const SLayout &SL = A.SL;
  const int N = S.N, M = S.M, nq = S.nquad;
  const int tid = threadIdx.x, nt = blockDim.x, lane = tid & 63, wave = tid >> 6;
  double *ws = A.st + (int64_t)w * L.stride, *ss = A.sc + (int64_t)w * SL.stride;
  const double *x = ws + L.x, *ren = ws + L.r_en, *rven = ws + L.rvec_en, *fso = ws + L.fso;
  __shared__ NlppTile<T, ORD> s_tile[kNlppWaves];
  __shared__ T s_c[kMaxCtype * kMaxTerms];
  __shared__ double s_red[2 * kNlppWaves];
  extern __shared__ double dyn_lds[];
  const int nwd = (N * M + 63) / 64;            // 64 pairs to a word
  unsigned long long *s_bits = reinterpret_cast<unsigned long long *>(dyn_lds);
  int *s_off = reinterpret_cast<int *>(dyn_lds + nwd);   // [nwd + 1] pairs in range before a word
  double *vnl = ss + SL.vnl, *foldv = ss + SL.fold;
  T *bt = reinterpret_cast<T *>(ss + SL.bt);
  int *plist = reinterpret_cast<int *>(ss + SL.plist);
  double ploc = 0.0, vpsp = 0.0;
  for (int q = tid; q < S.nctype * S.nterms; q += nt) s_c[q] = (T)cst(S.c)[q];
  // channel values of the pairs in range (nonlocal_pot's cutoff) and the
  // e-e-n variable of every pair
  for (int p = tid; p < 64 * nwd; p += nt) {
    bool inr = false;
    if (p < N * M) {
      const int ic = p % M, ict = cst(S.iwctype)[ic];
      const double r = fmax(1e-10, ren[p]);
      double *v = vnl + p * (QMCW_MAX_LPOT + 1);
      double vl[QMCW_MAX_LPOT];
#pragma unroll
      for (int l = 1; l <= QMCW_MAX_LPOT; l++) {
        vl[l - 1] = 0.0;
        if (l > cst(S.npotd)[ict]) continue;
        const double t = ecp_radial(S, r, l - 1, ict);
        if (l == cst(S.lpotp1)[ict]) ploc += t - cst(S.znuc)[ict] / r;
        else {
          vl[l - 1] = t;
          inr |= fabs(t) > 1e-4;
        }
      }
      if (inr) {
#pragma unroll
        for (int l = 0; l < QMCW_MAX_LPOT; l++) v[l] = vl[l];
      }
      T bu, t1, t2;
      scaled<T>(S.isc, (T)S.scalek, (T)ren[p], bu, t1, t2);
      bt[ic * N + p / M] = T(1) - (T)S.scalek * bu;
    }
    const unsigned long long b = __ballot(inr);
    if (lane == 0) s_bits[p >> 6] = b;
  }
  __syncthreads();
  if (wave == 0) {
    const int chunk = (nwd + 63) / 64, b0 = min(nwd, lane * chunk), b1 = min(nwd, b0 + chunk);
    int c = 0;
    for (int q = b0; q < b1; q++) c += __popcll(s_bits[q]);
    const int incl = gscan_incl<64>(c, lane);
    int o = incl - c;
    for (int q = b0; q < b1; q++) {
      s_off[q] = o;
      o += __popcll(s_bits[q]);
    }
    if (lane == 63) s_off[nwd] = incl;
  }
  __syncthreads();
  const int npair = s_off[nwd];
  for (int p = tid; p < 64 * nwd; p += nt) {
    const unsigned long long b = s_bits[p >> 6];
    if ((b >> lane) & 1) plist[s_off[p >> 6] + __popcll(b & ((1ull << lane) - 1))] = p;
  }
  __syncthreads();
  const bool mover = A.dmc_rot && (!A.dmove || A.dmove[(int64_t)w * A.dmove_stride] > 0.0);
  const int npt = (A.dmc_rot && !mover) ? 0 : npair * nq;
  // the pair sum of the Jastrow of each electron with points, at its current
  // position: an electron (its first pair) per wavefront, the lanes along its
  // row and column
  for (int q = wave; q < (npt > 0 ? npair : 0); q += nt / 64) {
    const int i = plist[q] / M;
    if (q > 0 && plist[q - 1] / M == i) continue;
    double f = 0.0;
    for (int j = lane; j < N; j += 64) f += fso[j <= i ? i * N + j : j * N + i];
    f = gsum<64>(f);
    if (lane == 0) foldv[i] = f;
  }
  // DMC: a rotation of the grid per pair in range, drawn in pair order (see
  // full_nlpp_b): one lane draws, then the lanes form the axes
  if (mover) {
    double *pax = ss + SL.prot;
    if (tid == 0) {
      int *rs = A.rng + 4 * w;
      int st4[4] = {rs[0], rs[1], rs[2], rs[3]};
      int prev = -1, j = 0;
      for (int q = 0; q < npair; q++) {
        rot_draws(st4, pax + 10 * q);
        const int i = plist[q] / M;
        j = (i == prev) ? j + 1 : 0;
        prev = i;
        if (j >= S.tm_kmax) A.flags[w] |= 4;
        pax[10 * q + 9] = j < S.tm_kmax ? (double)j : -1.0;
      }
      rs[0] = st4[0]; rs[1] = st4[1]; rs[2] = st4[2]; rs[3] = st4[3];
    }
    __syncthreads();
    for (int q = tid; q < npair; q += nt) {
      const double d[4] = {pax[10 * q], pax[10 * q + 1], pax[10 * q + 2], pax[10 * q + 3]};
      rot_from_draws(d, pax + 10 * q);
    }
  }
  __syncthreads();
  double *tqw = (mover && A.tq) ? A.tq + (int64_t)w * A.tq_stride : nullptr;
  NlppTile<T, ORD> &tl = s_tile[wave];
  const double *gp = ss + SL.gproj, *quad = ws + L.quad, *prot = ss + SL.prot;
  for (int t0 = 64 * wave; t0 < npt; t0 += nt) {
    // lanes past the last point repeat it and add nothing
    const bool on = t0 + lane < npt;
    const int t = on ? t0 + lane : npt - 1;
    const int iq = t % nq, p = plist[t / nq], ic = p % M, i = p / M;
    const double *v = vnl + p * (QMCW_MAX_LPOT + 1);
    const int ict = cst(S.iwctype)[ic];
    const double rei = ren[p];
    double qx, qy, qz;
    if (A.dmc_rot) {
      const double *ax = prot + 10 * (t / nq);
      const double a = cst(S.q0)[iq], b = cst(S.q0)[nq + iq], c = cst(S.q0)[2 * nq + iq];
      qx = a * ax[0] + b * ax[3] + c * ax[6];
      qy = a * ax[1] + b * ax[4] + c * ax[7];
      qz = a * ax[2] + b * ax[5] + c * ax[8];
    } else {
      qx = quad[iq]; qy = quad[nq + iq]; qz = quad[2 * nq + iq];
    }
    const double *rv0 = rven + 3 * p;
    const double costh = (rv0[0] * qx + rv0[1] * qy + rv0[2] * qz) / rei;
    const double xn[3] = {rei * qx + cst(S.cent)[3 * ic], rei * qy + cst(S.cent)[3 * ic + 1],
                          rei * qz + cst(S.cent)[3 * ic + 2]};
    wave_lds_fence();
    tl.x[lane][0] = xn[0]; tl.x[lane][1] = xn[1]; tl.x[lane][2] = xn[2];
    tl.r[lane] = rei;
    tl.el[lane] = i;
    tl.ic[lane] = ic;
    // determinant ratio of moving electron i to the point
    const double rd = point_ratio<T, double>(S, xn, gp + (int64_t)i * S.NB);
    wave_lds_fence();
    const int nsub = (min(64, npt - t0) + 15) / 16;
    for (int sub = 0; sub < nsub; sub++) nlpp_tile<T, ORD>(S, tl, 16 * sub, s_c, x, bt, lane);
    wave_lds_fence();
    if (on) {
      const double delta = (double)tl.en[lane] + tl.jas[lane] - foldv[i];
      double vpot = 0.0;
      for (int l = 1; l <= cst(S.npotd)[ict]; l++)
        if (l != cst(S.lpotp1)[ict]) vpot += v[l - 1] * legendre_w(l, costh);
      const double ej = exp(delta);
      const double fac = cst(S.q0)[3 * nq + iq] * ej * vpot;
      vpsp += fac * rd;
      if (A.full_orb) {      // for k_deriv_nlpp
        double *pw = ss + A.DL.pw + 2 * t;
        pw[0] = fac;
        pw[1] = fac * rd;
      }
      if (tqw) {
        const int j = (int)prot[10 * (t / nq) + 9];
        if (j >= 0) {
          tqw[tq_ratio(S, i, j, iq)] = rd * ej;
          double *qp = tqw + tq_point(S, i, j, iq);
          qp[0] = qx; qp[1] = qy; qp[2] = qz;
        }
      }
    }
  }
  ploc = gsum<64>(ploc);
  vpsp = gsum<64>(vpsp);
  if (lane == 0) { s_red[wave] = ploc; s_red[kNlppWaves + wave] = vpsp; }
  __syncthreads();
  if (tid == 0) {
    double a = 0.0, b = 0.0;
    for (int q = 0; q < nt / 64; q++) { a += s_red[q]; b += s_red[kNlppWaves + q]; }
    double *red = ss + SL.phs;
    red[55] = a;
    red[56] = b;
    red[57] = npair;
  }
}

template <typename T, int ORD>
__global__ __launch_bounds__(64 * kNlppWaves) __attribute__((amdgpu_waves_per_eu(2, 2)))
void k_full_nlpp_tiles(KArgs A) {
  full_nlpp_tiles_b<T, ORD>(A, blockIdx.x);
}

}  // namespace qmcw
