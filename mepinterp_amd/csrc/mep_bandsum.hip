// mep_bandsum.hip -- Fermi-Dirac weights and the Berry / Kubo / MEP band
// sums of one batch of k-points, accumulated into per-workgroup partial
// records (reduced once per run by reduce_parts_kernel).
//
// One k-point at a time per 256-thread workgroup (grid-stride over k; fixed
// k -> workgroup map and fixed-order reductions, so results are
// deterministic).  Rows of the reference it replaces:
//   d1_fd_stat, d1_fd_get_N_el          statistics.f90:65-124
//   kubo_ahc_tens, velo_ahc_tens,
//   kubo_ohc_tens                       kubo.f90:37-198
//   kubo_mep_CS / LC / IC               kubo_mep.f90:16-149
//   mep_niu_CS / LC / IC                mep_niu.f90:20-159
//
// Per k the workgroup stages in LDS the three velocity planes V_a (padded
// column-major) and the antisymmetric reciprocal table
// r(m, n) = 1 / (E_n - E_m) (0 on the diagonal), so no band sum divides.
//   pair phase    Hermitian V: each wave takes 8 bands n0, lane (n0, part)
//                 walks n = part, part + 8, ..., and the sums over the parts
//                 are scattered over the lanes; general V: wave 0 the Berry
//                 curvature, wave 1 the local (LC) MEP terms, wave 2 the
//                 velo/ohc pair sums (single (hw, E_F); several items:
//                 hwsum_kernel, launched after this one);
//   itinerant     C_j = V_k B_l - V_l B_k, (j,k,l) cyclic, with
//                 B_l(m, n0) = V_l(m, n0) r(m, n0): three complex n x n
//                 products on FP64 MFMA (three real products per complex
//                 one); the IC tensor of band n0 is the
//                 diagonal -Re[A_i C_j](n0, n0) with
//                 A_i(n0, n) = V_i(n0, n) r(n, n0)^2, contracted straight
//                 from the accumulator registers.  mep_niu's guard
//                 |(E0-En)^2 (E0-Em)| > kubo_tol excludes, for fixed (n0, n),
//                 one contiguous window of m around n0 (energies are
//                 sorted); those terms are subtracted from C (or the kept
//                 ones summed directly when the window covers most bands).
#include "mep_common.hpp"
#include "mep_kernels.hpp"
#include "mep_lane.hpp"
#include "../../include/mepinterp.h"

typedef double mep_v4d __attribute__((ext_vector_type(4)));

AccLayout acc_layout(const BandArgs& b) {
  AccLayout L;
  int64_t o = 0;
  L.Ne = o;   o += b.n_ef;
  L.ahc = o;  o += 9 * (int64_t)b.n_ef;
  L.velo = o; o += 2 * 9 * (int64_t)b.n_hw * b.n_ef;
  L.ohc = o;  o += 2 * 9 * (int64_t)b.n_hw * b.n_ef;
  L.kic = o;  o += 9 * (int64_t)b.n_ef;
  L.klc = o;  o += 9 * (int64_t)b.n_ef;
  L.kcs = o;  o += 9 * (int64_t)b.n_ef;
  L.nic = o;  o += 9 * (int64_t)(b.n_val > 0 ? b.n_val : 1);
  L.nlc = o;  o += 9 * (int64_t)(b.n_val > 0 ? b.n_val : 1);
  L.ncs = o;  o += 9 * (int64_t)(b.n_val > 0 ? b.n_val : 1);
  L.total = o;
  return L;
}

constexpr int BS_THREADS = 256;

// LDS plan: V planes (zd) 3*PL | E NMAX | r table PL | fd nef*NMAX | IC per
// band NT*9*NMAX, twice (all terms, Niu-kept terms) | pair sums or Chern-Simons
// terms 36 | per-band Berry and LC tensors (3 or 9 + 9)*NMAX | acc total
//                                           (doubles after the V planes)
// At 32 bands and one E_F this stays below half of the LDS, two workgroups a
// CU, for every number of valence bands.
template <int NMAX, bool HERM>
struct BsLds {
  static constexpr int LD = NMAX + 1;
  static constexpr int PL = NMAX * LD;
  static constexpr int NT = NMAX / 16;  // 16-row tiles per matrix
  static constexpr int OM = HERM ? 3 : 9;  // rows of the Berry curvature
  static size_t bytes(int nef, int64_t total) {
    return sizeof(zd) * 3 * (size_t)PL +
           sizeof(double) * ((size_t)PL + NMAX + (size_t)nef * NMAX + 2 * (size_t)NT * 9 * NMAX + 36 +
                             (OM + 9) * NMAX + (size_t)total);
  }
};
// what the number of Fermi levels is limited by, where it is more than the kernel
// takes (from a few levels on): V and r, E and the occupations, per-band tables
// of 27 (45 with two row tiles) rows and one more, sums of 9 per level and tile,
// 96, the record and two bytes per pair of bands.  A limit that callers know; the
// kernel's own tables would admit more levels.
static size_t bs_limit_bytes(int nmax, int nef, int64_t total) {
  const size_t pl = (size_t)nmax * (nmax + 1), nt = nmax / 16, m = nmax;
  return sizeof(zd) * 3 * pl + 2 * m * m +
         sizeof(double) * (pl + m + nef * m + nt * 9 * m + 9 * nt * nt * nef + m + 18 * m + 96 +
                           (size_t)total);
}


// FUSED: V is not read from HBM but formed in the V planes from the packed
// H(k) / dH_a(k) of the Fourier stage (Hk, per-k stride strideHk) and the
// eigenvectors U: V_a = U^H dH_a U on FP64 MFMA, with the same products and
// the same order as velo_mfma_kernel (so V, and every sum, is bit-identical
// to the two-kernel path).  n in 17..32, no position operator, Wannier
// convention.
//
// Bound by issue: at n = 32 the FP64 MFMA products take 0.52 of the SIMD-cycles and
// do not overlap with the VALU work of the other phases (0.27; LDS 0.2 of the
// CU-cycles), so what counts is the instructions: one sum instead of two where the Niu guards exclude nothing
// (decided per k-point), per-k reductions scattered over the lanes or kept in
// registers over all k-points, one weight per pair.
// n = 32, 262,144 k-points, all tensors: 15.2 ms (17.6 before these); n = 20,
// 24,273, five Fermi levels, V read: 0.85 ms (1.11).
template <int NMAX, bool FUSED, bool HERM>
__global__ __launch_bounds__(BS_THREADS, 2) void bandsum_kernel(BandArgs b, double Tsmear,
                                                                AccLayout L, int64_t gap,
                                                                int64_t nk,
                                                                const double* __restrict__ E,
                                                                const zd* __restrict__ V,
                                                                const zd* __restrict__ A,
                                                                const zd* __restrict__ Om,
                                                                const double* __restrict__ w,
                                                                double* __restrict__ part,
                                                                const zd* __restrict__ Hk,
                                                                int64_t strideHk,
                                                                const zd* __restrict__ U) {
  using S_ = BsLds<NMAX, HERM>;
  constexpr int LD = S_::LD, PL = S_::PL, NT = S_::NT;
  // U's plane (PL complex) lives over the per-k tables between the r table
  // and the accumulators while V is formed
  static_assert(!FUSED || (NMAX == 32 && HERM && PL + 2 * NT * 9 * NMAX >= 2 * PL),
                "fused velocities: U's plane must fit below the accumulators");
  extern __shared__ __attribute__((aligned(16))) double smem[];
  const int n = b.n, nef = b.n_ef, nhw = b.n_hw, nval = b.n_val;
  zd* Vs = reinterpret_cast<zd*>(smem);
  double* Es = reinterpret_cast<double*>(Vs + 3 * PL);
  double* Rs = Es + NMAX;
  double* fd = Rs + PL;
  double* QK = fd + (int64_t)nef * NMAX;        // [NT][9][NMAX] IC per band, row tile by row tile
  double* QF = QK + NT * 9 * NMAX;              // the same over the Niu-kept terms
  double* PW = QF + NT * 9 * NMAX;              // velo / ohc pair sums [36] (general V)
  double* red = PW;                             // Chern-Simons terms, once those are read
  double* OMA = PW + 36;                        // [OM][NMAX] Berry curvature per band
  double* F3A = OMA + S_::OM * NMAX;            // [9][NMAX] Kubo LC tensor per band
  double* acc = F3A + 9 * NMAX;
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  const int n2 = n * n;
  const bool finiteT = b.T_kelvin > 1e-2;
  const bool doAHC = (b.jobs & MEP_JOB_AHC) != 0;
  const bool doK = (b.jobs & MEP_JOB_KUBO) != 0;
  const bool doNjob = (b.jobs & MEP_JOB_MEP) != 0;
  const bool pmode = doAHC && (nhw * nef == 1);
  // HERM: V(n, m) = conj(V(m, n)), which holds for V built here without a
  // position operator (with one, the reference's connection is not Hermitian;
  // V from a caller is taken as it is)
  const double tol = b.kubo_tol;
  for (int64_t c = t; c < L.total; c += BS_THREADS) acc[c] = 0.0;
  // V planes, r, E and fd are staged for indices < n only: their padding
  // (up to NMAX) stays zero for every k, so loads need no bounds branch
  for (int c = t; c < 7 * PL + (1 + nef) * NMAX; c += BS_THREADS) smem[c] = 0.0;

  const zd wq = zd{b.hw[0], b.eta};
  const zd w2 = zmul(wq, wq);
  const double eta2 = b.eta * b.eta, B2 = 4.0 * wq.re * wq.re * eta2;
  double pacc[3] = {0.0, 0.0, 0.0};  // Hermitian V: this lane's velo / ohc pair sums, over all k

  // FUSED: U and the packed dH_a of a k-point, loaded into registers during
  // the last (light) phase of the previous k-point
  constexpr int NU = (NMAX * NMAX + BS_THREADS - 1) / BS_THREADS;
  constexpr int ND = (NMAX * (NMAX + 1) / 2 + BS_THREADS - 1) / BS_THREADS;
  const int np = n * (n + 1) / 2;
  zd ut[FUSED ? NU : 1], dt[3][FUSED ? ND : 1];
  double et = 0.0;
  auto fetch = [&](int64_t kk) {
    const int tt = threadIdx.x;
    const bool ok = kk < nk;
    const zd* Uk = U + (ok ? kk : 0) * (int64_t)n2;
    const zd* X = Hk + (ok ? kk : 0) * strideHk;
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      const int idx = tt + BS_THREADS * u;
      ut[u] = (ok && idx < n2) ? Uk[idx] : zd{0.0, 0.0};
    }
#pragma unroll
    for (int u = 0; u < ND; ++u) {
      const int p = tt + BS_THREADS * u;
#pragma unroll
      for (int a = 0; a < 3; ++a)
        dt[a][u] = (ok && p < np) ? X[(int64_t)(1 + a) * np + p] : zd{0.0, 0.0};
    }
    et = (ok && tt < n) ? E[kk * n + tt] : 0.0;
  };
  if constexpr (FUSED) fetch(blockIdx.x);
  // where those elements go in LDS, the same for every k-point: U(i, j) at
  // uo, dH's element p = i + j (j + 1) / 2 at (i, j) (low half) and (j, i)
  // (high half), out of range: all ones
  uint32_t uo[FUSED ? NU : 1], po[FUSED ? ND : 1];
  if constexpr (FUSED) {
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      const int idx = t + BS_THREADS * u;
      uo[u] = idx < n2 ? idx % n + LD * (idx / n) : ~0u;
    }
#pragma unroll
    for (int u = 0; u < ND; ++u) {
      const int p = t + BS_THREADS * u;
      int j = (int)((sqrtf(8.0f * (float)p + 1.0f) - 1.0f) * 0.5f);
      if ((j + 1) * (j + 2) / 2 <= p) ++j;
      if (j * (j + 1) / 2 > p) --j;
      const int i = p - j * (j + 1) / 2;
      po[u] = p < np ? (uint32_t)(i + LD * j) | (uint32_t)(j + LD * i) << 16 : ~0u;
    }
  }

  for (int64_t k = blockIdx.x; k < nk; k += gridDim.x) {
    // the thread index is made opaque per k-point: otherwise the compiler
    // hoists the lane-dependent indexes and masks of every unrolled loop out
    // of this one and spills them (the wave index stays scalar)
    int t = threadIdx.x;
    asm volatile("" : "+v"(t));
    const int lane = t & 63, wv = __builtin_amdgcn_readfirstlane(t >> 6);
    const double wk = w ? w[k] : 1.0;
    __syncthreads();
    // ---- stage V (planar [a][i + n j]) and E ------------------------------
    if constexpr (FUSED) {
      // V_a = U^H (dH_a U): U over the tables' region, dH_a (both halves of
      // the packed upper triangle) in the V planes, T_a = dH_a U written over
      // dH_a, then V_a from the accumulators into the V planes.  Rows and
      // columns >= n stay zero in every plane, so no operand load is guarded.
      zd* Us = reinterpret_cast<zd*>(Rs);
      if (n < NMAX) {
        for (int c = t; c < PL; c += BS_THREADS) stz(Us + c, zd{0.0, 0.0});
        __syncthreads();  // U's plane is zero
      }
      if (t < n) Es[t] = et;
#pragma unroll
      for (int u = 0; u < NU; ++u) {
        if (uo[u] != ~0u) stz(Us + uo[u], ut[u]);
      }
#pragma unroll
      for (int u = 0; u < ND; ++u) {
        if (po[u] == ~0u) continue;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          stz(Vs + a * PL + (po[u] >> 16), zconj(dt[a][u]));
          stz(Vs + a * PL + (po[u] & 0xffff), dt[a][u]);  // last: the diagonal keeps the value as stored
        }
      }
      __syncthreads();
      // the 4 waves own the 2 x 2 output tiles of 16 x 16 (n > 16: all busy)
      const int r0 = 16 * (wv & 1), c0 = 16 * (wv >> 1);
      const int ar = r0 + (lane & 15), bc = c0 + (lane & 15), kq = lane >> 4;
      mep_v4d q1[3], q2[3], q3[3];
#pragma unroll
      for (int a = 0; a < 3; ++a) q1[a] = q2[a] = q3[a] = mep_v4d{0, 0, 0, 0};
#pragma unroll
      for (int k0 = 0; k0 < NMAX; k0 += 4) {
        if (k0 >= n) break;
        const int m = k0 + kq;
        const zd bu = ldz(Us + m + LD * bc);
        const double bsum = bu.re + bu.im;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          const zd x = ldz(Vs + a * PL + ar + LD * m);
          q1[a] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.re, bu.re, q1[a], 0, 0, 0);
          q2[a] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.im, bu.im, q2[a], 0, 0, 0);
          q3[a] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.re + x.im, bsum, q3[a], 0, 0, 0);
        }
      }
      __syncthreads();  // every wave has read dH
#pragma unroll
      for (int a = 0; a < 3; ++a)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int row = r0 + kq + 4 * v;
          stz(Vs + a * PL + row + LD * bc, zd{q1[a][v] - q2[a][v], q3[a][v] - q1[a][v] - q2[a][v]});
        }
      __syncthreads();
#pragma unroll
      for (int a = 0; a < 3; ++a) q1[a] = q2[a] = q3[a] = mep_v4d{0, 0, 0, 0};
#pragma unroll
      for (int k0 = 0; k0 < NMAX; k0 += 4) {
        if (k0 >= n) break;
        const int m = k0 + kq;
        const zd uu = ldz(Us + m + LD * ar);  // A(row, m) = conj(U(m, row))
        const double us = uu.re - uu.im;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          const zd y = ldz(Vs + a * PL + m + LD * bc);
          q1[a] = __builtin_amdgcn_mfma_f64_16x16x4f64(uu.re, y.re, q1[a], 0, 0, 0);
          q2[a] = __builtin_amdgcn_mfma_f64_16x16x4f64(-uu.im, y.im, q2[a], 0, 0, 0);
          q3[a] = __builtin_amdgcn_mfma_f64_16x16x4f64(us, y.re + y.im, q3[a], 0, 0, 0);
        }
      }
      __syncthreads();  // every wave has read T and U
      // V (zero in rows and columns >= n, as T and U are) into the planes
#pragma unroll
      for (int a = 0; a < 3; ++a)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int row = r0 + kq + 4 * v;
          stz(Vs + a * PL + row + LD * bc, zd{q1[a][v] - q2[a][v], q3[a][v] - q1[a][v] - q2[a][v]});
        }
      // the r table's diagonal and padding are zero again
      if (n < NMAX) {
        for (int c = t; c < PL; c += BS_THREADS) {
          const int i = c % LD, j = c / LD;
          if (i >= n || j >= n || i == j) Rs[c] = 0.0;
        }
      } else if (t < NMAX) {
        Rs[t + LD * t] = 0.0;
      }
    } else {
    const zd* Vk = V + k * 3 * (int64_t)n2;
    {
      // every load of the k-point is issued before the first LDS store
      constexpr int JS = BS_THREADS / NMAX, NJ = NMAX / JS;
      const int i = t % NMAX, jb = t / NMAX;
      zd vt[3][NJ];
#pragma unroll
      for (int a = 0; a < 3; ++a)
#pragma unroll
        for (int jj = 0; jj < NJ; ++jj) {
          const int j = jb + JS * jj;
          vt[a][jj] = (i < n && j < n) ? Vk[a * n2 + i + n * j] : zd{0.0, 0.0};
        }
      et = (t < n) ? E[k * n + t] : 0.0;
#pragma unroll
      for (int a = 0; a < 3; ++a)
#pragma unroll
        for (int jj = 0; jj < NJ; ++jj) {
          const int j = jb + JS * jj;
          if (i < n && j < n) stz(Vs + a * PL + i + LD * j, vt[a][jj]);
        }
      if (t < n) Es[t] = et;
    }
    __syncthreads();
    }
    // mep_niu's guards exclude nothing where, with g the gap to the nearest
    // band, g^3 > kubo_tol for every valence band (the energies are sorted and
    // rounding is monotone, so every |(E0-En)^2 (E0-Em)| and |E0-En|^3 is at
    // least that): such a k-point needs no windows and no second sums.  The
    // same in every wavefront.  (n = 32, 16 valence bands over 4 Ha: 95 of 100
    // k-points at the default kubo_tol.)  General V: the energies may be a
    // caller's, in any order, so that the neighbouring index need not be the
    // nearest band; a k-point out of order is not clean.
    bool clean = true;
    if (doNjob && lane < n && (!HERM || lane < nval)) {
      const double g0 = lane > 0 ? Es[lane] - Es[lane - 1] : HUGE_VAL;
      const double g1 = lane < n - 1 ? Es[lane + 1] - Es[lane] : HUGE_VAL;
      clean = lane < nval ? g0 * g0 * g0 > tol && g1 * g1 * g1 > tol : g0 >= 0.0;
    }
    clean = __ballot(!clean) == 0;
    // ---- r(m, c) = 1 / (E_c - E_m); occupations ---------------------------
    {
      // one division per pair m < c: r(c, m) = -r(m, c) exactly in IEEE
      // arithmetic; the diagonal stays 0 (zeroed once with the padding)
      const int npair = n * (n - 1) / 2;
      for (int pi = t; pi < npair; pi += BS_THREADS) {
        int c = (int)((1.0f + sqrtf(1.0f + 8.0f * (float)pi)) * 0.5f);  // p = c(c-1)/2 + m
        if (c * (c - 1) / 2 > pi) --c;
        if ((c + 1) * c / 2 <= pi) ++c;
        const int m = pi - c * (c - 1) / 2;
        const double v = 1.0 / (Es[c] - Es[m]);
        Rs[m + LD * c] = v;
        Rs[c + LD * m] = -v;
      }
    }
    for (int idx = t; idx < nef * n; idx += BS_THREADS) {
      if (b.fd_in) {
        fd[idx] = b.fd_in[k * (int64_t)nef * n + idx];
      } else {
        const int ef = (nef == 1) ? 0 : idx % nef, nb = (nef == 1) ? idx : idx / nef;
        const double e = Es[nb], f = b.ef[ef];
        fd[idx] = finiteT ? 1.0 / (1.0 + exp((e - f) / Tsmear)) : ((e < f) ? 1.0 : 0.0);
      }
    }
    __syncthreads();

    if constexpr (!HERM) {
      // ==== pair phase, general V (position operator: the reference's
      // connection makes V non-Hermitian, so V(n, n0) is read as stored).
      // Lane (p0, pp) of each wave walks n = pp, pp + P, ...: wave 0 the
      // Berry curvature of p0, wave 1 its local (LC) terms, waves 2-3 the
      // velo / ohc pair sums at the single (hw, E_F).
      constexpr int PARTS = 64 / NMAX;
      const int p0 = lane % NMAX, pp = lane / NMAX;
      if (wv == 0) {
        double om[9];
#pragma unroll
        for (int q = 0; q < 9; ++q) om[q] = 0.0;
        if (doAHC)
          for (int nn = pp; nn < n; nn += PARTS) {
            zd x[3], y[3];
#pragma unroll
            for (int a = 0; a < 3; ++a) {
              x[a] = ldz(Vs + a * PL + p0 + LD * nn);  // V_a(n0, n)
              y[a] = ldz(Vs + a * PL + nn + LD * p0);  // V_a(n, n0)
            }
            const double r = Rs[nn + LD * p0];  // 1 / (E0 - En)
            const double r2 = r * r;
            // Omega_n0,ij = -2 Im(V_i(n0,n) V_j(n,n0)) / (En - E0)^2
#pragma unroll
            for (int j = 0; j < 3; ++j)
#pragma unroll
              for (int i = 0; i < 3; ++i) om[i + 3 * j] -= 2.0 * zmul(x[i], y[j]).im * r2;
          }
#pragma unroll
        for (int q = 0; q < 9; ++q) om[q] = (NMAX == 32) ? swap32_sum(om[q], om[q]) : rows4_sum(om[q]);
        if (pp == 0)
#pragma unroll
          for (int q = 0; q < 9; ++q) OMA[q * NMAX + p0] = om[q];
      } else if (wv == 1) {
        double f3[9], f3m[9];
#pragma unroll
        for (int q = 0; q < 9; ++q) f3[q] = f3m[q] = 0.0;
        const bool doN = doNjob && p0 < n && p0 < nval;
        if (doK || doNjob) {
          const double E0 = Es[p0];
          zd z0[3];
#pragma unroll
          for (int l = 0; l < 3; ++l) z0[l] = ldz(Vs + l * PL + p0 + LD * p0);
          for (int nn = pp; nn < n; nn += PARTS) {
            zd x[3], y[3];
#pragma unroll
            for (int a = 0; a < 3; ++a) {
              x[a] = ldz(Vs + a * PL + p0 + LD * nn);
              y[a] = ldz(Vs + a * PL + nn + LD * p0);
            }
            const double r = Rs[nn + LD * p0];  // 0 for nn == n0: adds nothing
            const double r3 = r * r * r;
            // F3_ij = eps_jkl Re(V_i(n0,n) V_k(n,n0) V_l(n0,n0)) / (E0-En)^3
            zd cr[3];
            cr[0] = zsub(zmul(y[1], z0[2]), zmul(y[2], z0[1]));
            cr[1] = zsub(zmul(y[2], z0[0]), zmul(y[0], z0[2]));
            cr[2] = zsub(zmul(y[0], z0[1]), zmul(y[1], z0[0]));
            const double dn = E0 - Es[nn];
            const bool keep3 = doN && (fabs(dn * dn * dn) > tol);
#pragma unroll
            for (int j = 0; j < 3; ++j)
#pragma unroll
              for (int i = 0; i < 3; ++i) {
                const double v = zmul(x[i], cr[j]).re * r3;
                f3[i + 3 * j] += v;
                if (keep3) f3m[i + 3 * j] += v;
              }
          }
        }
#pragma unroll
        for (int q = 0; q < 9; ++q) {
          f3[q] = (NMAX == 32) ? swap32_sum(f3[q], f3[q]) : rows4_sum(f3[q]);
          f3m[q] = (NMAX == 32) ? swap32_sum(f3m[q], f3m[q]) : rows4_sum(f3m[q]);
        }
        if (pp == 0) {
#pragma unroll
          for (int q = 0; q < 9; ++q) F3A[q * NMAX + p0] = f3[q];
          if (doN)
#pragma unroll
            for (int q = 0; q < 9; ++q) acc[L.nlc + q + 9 * p0] += wk * f3m[q];
        }
      } else if (pmode && wv == 2) {
        // components q = i + 3j:
        //   velo_q += (f0 - fn) Im(V_i(n0,n) V_j(n,n0)) / ((E0-En)^2 - (hw + i eta)^2)
        //   ohc_q  += i (f0 - fn) V_i(n,n0) V_j(n0,n) / ((E0-En)(E0-En - hw - i eta))
        double pv[36];
#pragma unroll
        for (int u = 0; u < 36; ++u) pv[u] = 0.0;
        const double E0 = Es[p0];
        for (int nn = pp; nn < n; nn += PARTS) {
          zd x[3], y[3];
#pragma unroll
          for (int a = 0; a < 3; ++a) {
            x[a] = ldz(Vs + a * PL + p0 + LD * nn);
            y[a] = ldz(Vs + a * PL + nn + LD * p0);
          }
          const double dE = E0 - Es[nn];
          const double dfv = fd[p0] - fd[nn];
          const zd denv = zd{dE * dE - w2.re, -w2.im};
          const zd deno = zmul(zd{dE, 0.0}, zd{dE - wq.re, -wq.im});
          const double iv = 1.0 / zabs2(denv), io = 1.0 / zabs2(deno);
          // (the padding's energy, 0, may be a band's)
          const bool off = nn != p0 && p0 < n;
          const zd rv = off ? zd{denv.re * iv * dfv, -denv.im * iv * dfv} : zd{0.0, 0.0};
          const zd ro = off ? zd{deno.re * io * dfv, -deno.im * io * dfv} : zd{0.0, 0.0};
#pragma unroll
          for (int q = 0; q < 9; ++q) {
            const int i = q % 3, j = q / 3;
            const double vim = zmul(x[i], y[j]).im;
            pv[2 * q] += vim * rv.re;
            pv[2 * q + 1] += vim * rv.im;
            const zd o = zmuli(zmul(zmul(y[i], x[j]), ro));
            pv[18 + 2 * q] += o.re;
            pv[19 + 2 * q] += o.im;
          }
        }
#pragma unroll
        for (int u = 0; u < 36; ++u) pv[u] = rows4_sum(row16_sum(pv[u]));
        if (lane == 0)
#pragma unroll
          for (int u = 0; u < 36; ++u) PW[u] = pv[u];
      }
    } else {
    // ==== pair phase: wave w owns the bands n0 = 8w .. 8w + 7; lane
    // (n0 = 8w + lane % 8, part = lane / 8) walks n = part, part + 8, ...
    // V is Hermitian, so V_a(n, n0) = conj(x_a) with x_a = V_a(n0, n), and
    // every pair sum is built from P_ij = x_i conj(x_j) (i < j) and |x_i|^2.
    // r = 1 / (E0 - En) is 0 for n = n0 and in the padding.
    if (wv * 8 < n) {
      const int n0 = wv * 8 + (lane & 7), part = lane >> 3;
      const bool doN = doNjob && n0 < nval && n0 < n;
      const double E0 = Es[n0];
      double om[3] = {0.0, 0.0, 0.0};        // sum r^2 Im P_ij
      double gd[3] = {0.0, 0.0, 0.0};        // sum r^3 |x_i|^2
      zd go[3];                              // sum r^3 P_ij (i < j)
      double ps[24];                         // velo / ohc pair sums
#pragma unroll
      for (int c = 0; c < 3; ++c) go[c] = zd{0.0, 0.0};
#pragma unroll
      for (int c = 0; c < 24; ++c) ps[c] = 0.0;
      const double f0 = pmode ? fd[n0] : 0.0;
      auto pair = [&](int nn, zd* P, double* d) {
        zd x[3];
#pragma unroll
        for (int a = 0; a < 3; ++a) x[a] = ldz(Vs + a * PL + n0 + LD * nn);
#pragma unroll
        for (int a = 0; a < 3; ++a) d[a] = x[a].re * x[a].re + x[a].im * x[a].im;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          const zd xi = x[c == 2 ? 1 : 0], xj = x[c == 0 ? 1 : 2];
          P[c] = zd{xi.re * xj.re + xi.im * xj.im, xi.im * xj.re - xi.re * xj.im};
        }
      };
      for (int nn = part; nn < n; nn += 8) {
        zd P[3];
        double d[3];
        pair(nn, P, d);
        const double r = Rs[nn + LD * n0];
        const double r2 = r * r, r3 = r2 * r;
        if (doAHC)
#pragma unroll
          for (int c = 0; c < 3; ++c) om[c] += r2 * P[c].im;
        if (doK || doNjob) {
#pragma unroll
          for (int a = 0; a < 3; ++a) gd[a] += r3 * d[a];
#pragma unroll
          for (int c = 0; c < 3; ++c) go[c] = zd{go[c].re + r3 * P[c].re, go[c].im + r3 * P[c].im};
        }
        if (pmode) {
          // both orders of a pair weigh g = f / (dE^2 - w^2) = (D + i B) q and
          // w g / dE (see hwsum_kernel): the sums of D q v and q v, v = Im P,
          // Re P / dE, |x|^2 / dE.  Selects, not a branch, drop pairs of equal
          // occupation, n = n0 among them
          const double dE = E0 - Es[nn], f = f0 - fd[nn];
          const bool on = f != 0.0 && nn != n0 && n0 < n;
          const double D = (dE - wq.re) * (dE + wq.re) + eta2;
          const double q = on ? f * rcp_nr(D * D + B2) : 0.0, Dq = D * q;
          const double rs = on ? r : 0.0, qr = q * rs, Dqr = Dq * rs;
#pragma unroll
          for (int c = 0; c < 3; ++c) {
            ps[c] += Dq * P[c].im;
            ps[3 + c] += q * P[c].im;
            ps[6 + c] += Dqr * P[c].re;
            ps[9 + c] += qr * P[c].re;
            ps[12 + c] += Dqr * d[c];
            ps[15 + c] += qr * d[c];
          }
        }
      }
      // local terms of n0: F3_ij = Re(z_l G_ik - z_k G_il), (j, k, l) cyclic,
      // z = V(n0, n0), G_ik = sum_n r^3 x_i conj(x_k) (Hermitian in i, k)
      zd z[3];
#pragma unroll
      for (int a = 0; a < 3; ++a) z[a] = ldz(Vs + a * PL + n0 + LD * n0);
      auto local = [&](const double* gd_, const zd* go_, double* o) {
        auto G = [&](int i, int k) {
          if (i == k) return zd{gd_[i], 0.0};
          const zd g = go_[i + k - 1];
          return i < k ? g : zd{g.re, -g.im};
        };
#pragma unroll
        for (int j = 0; j < 3; ++j) {
          const int k = (j + 1) % 3, l = (j + 2) % 3;
#pragma unroll
          for (int i = 0; i < 3; ++i) {
            const zd a = G(i, k), bb = G(i, l);
            o[i + 3 * j] = (z[l].re * a.re - z[l].im * a.im) - (z[k].re * bb.re - z[k].im * bb.im);
          }
        }
      };
      // sums over the 8 parts (lane bits 3-5), scattered: lane (n0, g) ends
      // with the slots 8 g5 + 4 g4 + 2 g3 + s, s < 2, of its n0
      double v16[16], v2[2];
      local(gd, go, v16);
#pragma unroll
      for (int c = 0; c < 3; ++c) v16[9 + c] = om[c];
#pragma unroll
      for (int c = 12; c < 16; ++c) v16[c] = 0.0;
      scatter_sum<16>(v16, v2, lane);
      const int base2 = 8 * ((lane >> 5) & 1) + 4 * ((lane >> 4) & 1) + 2 * ((lane >> 3) & 1);
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const int slot = base2 + s;
        if (slot < 9) {
          F3A[slot * NMAX + n0] = v2[s];
          if (clean && doN) acc[L.nlc + slot + 9 * n0] += wk * v2[s];
        } else if (slot < 12) {  // Omega_ij = -2 v, Omega_ji = 2 v, Omega_ii = 0
          OMA[(slot - 9) * NMAX + n0] = v2[s];
        }
      }
      if (!clean) {  // the local terms over the Niu-kept n
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          gd[c] = 0.0;
          go[c] = zd{0.0, 0.0};
        }
#pragma unroll 1
        for (int nn = part; nn < n; nn += 8) {
          zd P[3];
          double d[3];
          pair(nn, P, d);
          const double r = Rs[nn + LD * n0], dn = E0 - Es[nn];
          const double r3 = (doN && fabs(dn * dn * dn) > tol) ? r * r * r : 0.0;
#pragma unroll
          for (int a = 0; a < 3; ++a) gd[a] += r3 * d[a];
#pragma unroll
          for (int c = 0; c < 3; ++c) go[c] = zd{go[c].re + r3 * P[c].re, go[c].im + r3 * P[c].im};
        }
        local(gd, go, v16);
#pragma unroll
        for (int c = 9; c < 16; ++c) v16[c] = 0.0;
        scatter_sum<16>(v16, v2, lane);
#pragma unroll
        for (int s = 0; s < 2; ++s)
          if (doN && base2 + s < 9) acc[L.nlc + base2 + s + 9 * n0] += wk * v2[s];
      }
      if (pmode) {
        double v3[3];
        scatter_sum<24>(ps, v3, lane);
#pragma unroll
        for (int s = 0; s < 3; ++s) pacc[s] += wk * v3[s];
      }
    }
    }
    // (the Hall and optical conductivities of several (hw, E_F) items run in
    // hwsum_kernel after this kernel)

    // ==== itinerant (IC) terms on MFMA ======================================
    // Wave item: one 16 x 16 block (tr, tc) of all three C_j when the
    // matrices hold several blocks (NT = 2), one C_j when they hold one.
    // The three products share their operands, V_c(row, m) and
    // B_c(m, col) = V_c(m, col) r(m, col), and give nine independent MFMA
    // chains.  Loads are unconditional: LDS rows and columns >= n are zero
    // and r is zero on the diagonal, so padded entries add nothing.
    if (doK || doNjob) {
      constexpr int NB = NT * NT;               // 16 x 16 blocks per matrix
      constexpr int JN = (NB >= 4) ? 3 : 1;     // components per wave item
      constexpr int NITEM = NB * (3 / JN);
      constexpr int NP = (JN == 3) ? 3 : 2;      // velocity planes an item reads
      for (int item = wv; item < NITEM; item += 4) {
        const int blk = item % NB, jsel = item / NB;  // jsel: the component when JN == 1
        const int tr = blk / NT, tc = blk % NT;
        const int r0 = 16 * tr, c0 = 16 * tc;
        const int ar = r0 + (lane & 15), bc = c0 + (lane & 15), kq = lane >> 4;
        // plane of operand slot c; component jj pairs slot ks(jj) (its k)
        // with slot ls(jj) (its l)
        int pl[NP];
#pragma unroll
        for (int c = 0; c < NP; ++c) pl[c] = (JN == 3) ? c : (jsel + 1 + c) % 3;
        auto ks = [](int jj) { return (JN == 3) ? (jj + 1) % 3 : 0; };
        auto ls = [](int jj) { return (JN == 3) ? (jj + 2) % 3 : 1; };
        // C = sum_m A(., m) B(m, .) with three real products per complex
        // one: P1 = Ar Br, P2 = Ai Bi, P3 = (Ar + Ai)(Br + Bi);
        // Re C = P1 - P2, Im C = P3 - P1 - P2
        mep_v4d p1[JN], p2[JN], p3[JN];
#pragma unroll
        for (int jj = 0; jj < JN; ++jj) p1[jj] = p2[jj] = p3[jj] = mep_v4d{0, 0, 0, 0};
        auto step = [&](int k0) {
          const int m = k0 + kq;
          const double rr = Rs[m + LD * bc];
          zd a[NP], s[NP];
          double as[NP], ss[NP];
#pragma unroll
          for (int c = 0; c < NP; ++c) {
            a[c] = ldz(Vs + pl[c] * PL + ar + LD * m);
            s[c] = zscale(ldz(Vs + pl[c] * PL + m + LD * bc), rr);
            as[c] = a[c].re + a[c].im;
            ss[c] = s[c].re + s[c].im;
          }
          // C_j += V_k B_l, then C_j -= V_l B_k   ((j, k, l) cyclic)
#pragma unroll
          for (int jj = 0; jj < JN; ++jj) {
            const int kk = ks(jj), ll = ls(jj);
            p1[jj] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[kk].re, s[ll].re, p1[jj], 0, 0, 0);
            p2[jj] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[kk].im, s[ll].im, p2[jj], 0, 0, 0);
            p3[jj] = __builtin_amdgcn_mfma_f64_16x16x4f64(as[kk], ss[ll], p3[jj], 0, 0, 0);
          }
#pragma unroll
          for (int jj = 0; jj < JN; ++jj) {
            const int kk = ks(jj), ll = ls(jj);
            p1[jj] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[ll].re, -s[kk].re, p1[jj], 0, 0, 0);
            p2[jj] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[ll].im, -s[kk].im, p2[jj], 0, 0, 0);
            p3[jj] = __builtin_amdgcn_mfma_f64_16x16x4f64(as[ll], -ss[kk], p3[jj], 0, 0, 0);
          }
        };
        constexpr int K1 = NMAX == 32 ? 24 : NMAX;  // one branch for the last quarter
#pragma unroll
        for (int k0 = 0; k0 < K1; k0 += 4) step(k0);
        if (n > K1)
#pragma unroll
          for (int k0 = K1; k0 < NMAX; k0 += 4) step(k0);
        // contraction with A_i(n0, n) = V_i(n0, n) r(n, n0)^2, n0 = column;
        // r(n, n0) = 0 for n = n0 and outside n, so those rows add nothing.
        // f2[i + 3 jj]: component (i, j) with j = jj (JN == 3) or jsel
        const int n0 = bc;
        const bool colok = n0 < n;
        const bool doN = doNjob && colok && n0 < nval;
        double f2[3 * JN], f2m[3 * JN];
#pragma unroll
        for (int q = 0; q < 3 * JN; ++q) f2[q] = f2m[q] = 0.0;
        // mep_niu keeps, for (n0, n), the m outside one window [lo, hi]:
        // narrow windows take -Re[A C] here and add back the excluded terms
        // below; wide windows sum the kept terms directly below
        auto wide = [&](int lo, int hi) { return 2 * (hi - lo + 1) > n; };
        // rows whose window holds more than n0 itself (the others need no
        // second pass) and is not the whole band range
        bool wterm[4];
        unsigned win[4];  // lo, hi << 8
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int row = r0 + kq + 4 * v;
          const double rr = Rs[row + LD * n0];
          const double rr2 = rr * rr;
          bool narrow = false;
          wterm[v] = false;
          win[v] = 0;
          if (!clean && doN && row < n && row != n0) {
            // mep_niu's guard |(E0-En)^2 (E0-Em)| > kubo_tol: energies are
            // sorted, so the excluded m of (n0, n) form one range around n0
            const double E0 = Es[n0], dn = E0 - Es[row], dn2 = dn * dn;
            int lo = n0, hi = n0;
            while (lo > 0 && !(fabs(dn2 * (E0 - Es[lo - 1])) > tol)) --lo;
            while (hi < n - 1 && !(fabs(dn2 * (E0 - Es[hi + 1])) > tol)) ++hi;
            win[v] = (unsigned)lo | (unsigned)hi << 8;
            const bool all = lo == 0 && hi == n - 1;
            narrow = !all && !wide(lo, hi);
            wterm[v] = !all && !(lo == n0 && hi == n0);
          }
          zd ai[3];
#pragma unroll
          for (int i = 0; i < 3; ++i) ai[i] = zscale(ldz(Vs + i * PL + n0 + LD * row), rr2);
#pragma unroll
          for (int jj = 0; jj < JN; ++jj) {
            const zd cv = zd{p1[jj][v] - p2[jj][v], p3[jj][v] - p1[jj][v] - p2[jj][v]};
#pragma unroll
            for (int i = 0; i < 3; ++i) {
              const double c = ai[i].re * cv.re - ai[i].im * cv.im;
              f2[i + 3 * jj] -= c;
              if (!clean) f2m[i + 3 * jj] -= narrow ? c : 0.0;
            }
          }
        }
        // window terms, after the accumulators are dead
        if (!clean && doN)
#pragma unroll 1
          for (int v = 0; v < 4; ++v) {
            const unsigned wv_ = v == 0 ? win[0] : v == 1 ? win[1] : v == 2 ? win[2] : win[3];
            if (!(v == 0 ? wterm[0] : v == 1 ? wterm[1] : v == 2 ? wterm[2] : wterm[3])) continue;
            const int row = r0 + kq + 4 * v;
            const int lo = (int)(wv_ & 255), hi = (int)(wv_ >> 8);
            const bool wd = wide(lo, hi);
            const double rr = Rs[row + LD * n0];
            const double rr2 = rr * rr;
            zd ai[3];
#pragma unroll
            for (int i = 0; i < 3; ++i) ai[i] = zscale(ldz(Vs + i * PL + n0 + LD * row), rr2);
#pragma unroll
            for (int jj = 0; jj < JN; ++jj) {
              const zd* Vk_ = Vs + pl[ks(jj)] * PL;
              const zd* Vl_ = Vs + pl[ls(jj)] * PL;
              auto term = [&](int mm) {
                const double rm = Rs[mm + LD * n0];
                const zd bl = zscale(Vl_[mm + LD * n0], rm), bk = zscale(Vk_[mm + LD * n0], rm);
                return zsub(zmul(Vk_[row + LD * mm], bl), zmul(Vl_[row + LD * mm], bk));
              };
              zd x = zd{0.0, 0.0};
              if (wd) {  // kept terms: f2m -= Re(A x)
#pragma unroll 1
                for (int mm = 0; mm < lo; ++mm) x = zadd(x, term(mm));
#pragma unroll 1
                for (int mm = hi + 1; mm < n; ++mm) x = zadd(x, term(mm));
                x = zd{-x.re, -x.im};
              } else {   // excluded terms: f2m += Re(A x)
#pragma unroll 1
                for (int mm = lo; mm <= hi; ++mm)
                  if (mm != n0) x = zadd(x, term(mm));
              }
#pragma unroll
              for (int i = 0; i < 3; ++i) f2m[i + 3 * jj] += ai[i].re * x.re - ai[i].im * x.im;
            }
          }
        // sums over the 4 row groups of the block (lane bits 4, 5), scattered:
        // group g holds the slots NS g .. NS g + NS - 1
        constexpr int NS = (JN == 3) ? 3 : 1;
        const int jb = (JN == 3) ? 0 : 3 * jsel;  // component of f2[0]
        auto put = [&](const double* f, double* Q) {
          double h[2 * NS], o[NS];
          auto at = [&](int q) { return q < 3 * JN ? f[q < 3 * JN ? q : 0] : 0.0; };
#pragma unroll
          for (int q = 0; q < 2 * NS; ++q) h[q] = swap32_sum(at(q), at(q + 2 * NS));
#pragma unroll
          for (int q = 0; q < NS; ++q) o[q] = swap16_sum(h[q], h[q + NS]);
#pragma unroll
          for (int q = 0; q < NS; ++q)
            if (colok && NS * kq + q < 3 * JN) Q[(tr * 9 + jb + NS * kq + q) * NMAX + n0] = o[q];
        };
        put(f2, QK);
        if (!clean) put(f2m, QF);
      }
    }
    __syncthreads();
    if constexpr (FUSED) fetch(k + gridDim.x);  // in flight during the sums below
    // ---- sums over the bands n0 and over the waves' partial records --------
    // Ne, kubo_ahc_tens (-sum f Omega), kubo_mep_LC and kubo_mep_IC for every E_F;
    // item (c, ef) is summed by 8 lanes, lane g taking the
    // bands m0 = g, g + 8, ...
    // (Hermitian V: the three Berry sums are each two entries)
    constexpr int NO = S_::OM, NI = 1 + NO + 18;
    for (int base = 0; base < 8 * NI * nef; base += BS_THREADS) {
      const int it = base + t, item = it >> 3, g = it & 7;
      const int c = item % NI, ef = item / NI;
      const bool valid = item < NI * nef &&
                         (c == 0 || (c <= NO && doAHC) || (c > NO && doK));
      double s = 0.0;
      if (valid) {
        const double* src = (c == 0)        ? nullptr
                            : (c <= NO)     ? OMA + (c - 1) * NMAX
                            : (c <= NO + 9) ? F3A + (c - 1 - NO) * NMAX
                                            : QK + (c - 10 - NO) * NMAX;
        const double* src2 = (NT == 2 && c > NO + 9) ? src + 9 * NMAX : nullptr;
        for (int m0 = g; m0 < n; m0 += 8)
          s += fd[ef + nef * m0] * (src2 ? src[m0] + src2[m0] : src ? src[m0] : 1.0);
      }
      s = group8_sum(s);  // the loop bounds are uniform over the wave
      if (valid && g == 0) {
        if (c == 0) {
          acc[L.Ne + ef] += wk * s;
        } else if (c <= NO) {
          if constexpr (HERM) {
            const int i = (c == 3) ? 1 : 0, j = (c == 1) ? 1 : 2;
            acc[L.ahc + i + 3 * j + 9 * ef] += wk * (2.0 * s);
            acc[L.ahc + j + 3 * i + 9 * ef] -= wk * (2.0 * s);
          } else {
            acc[L.ahc + (c - 1) + 9 * ef] -= wk * s;
          }
        } else if (c <= NO + 9) {
          acc[L.klc + (c - 1 - NO) + 9 * ef] += wk * s;
        } else {
          acc[L.kic + (c - 10 - NO) + 9 * ef] += wk * s;
        }
      }
    }
    // general V: velo_ahc_tens / kubo_ohc_tens at the single (hw, E_F), the
    // last 18 threads, o = q (velo) and 9 + q (ohc)
    if (!HERM && pmode && t >= BS_THREADS - 18) {
      const int o = t - (BS_THREADS - 18);
      double* dst = acc + (o < 9 ? L.velo : L.ohc) + 2 * (o % 9);
      dst[0] += wk * PW[2 * o];
      dst[1] += wk * PW[2 * o + 1];
    }
    if (doNjob)
      for (int it = t; it < 9 * nval; it += BS_THREADS) {
        const int q = it % 9, n0 = it / 9;
        double s = 0.0;
        const double* Q = clean ? QK : QF;
        for (int tr = 0; tr < NT; ++tr) s += Q[(tr * 9 + q) * NMAX + n0];
        acc[L.nic + q + 9 * n0] += wk * s;
      }
    // ---- Chern-Simons term (needs A and Omega) ------------------------------
    if ((doK || doNjob) && b.pos_op && A && Om) {
      __syncthreads();
      if (t < n) {
        const int64_t NN = (int64_t)n2;
        const zd* Ak = A + k * 3 * NN + 3 * ((int64_t)t + (int64_t)n * t);
        const zd* Ok = Om + k * 9 * NN + 9 * ((int64_t)t + (int64_t)n * t);
        zd omc[3];
        omc[0] = zsub(Ok[1 + 3 * 2], Ok[2 + 3 * 1]);
        omc[1] = zsub(Ok[2 + 3 * 0], Ok[0 + 3 * 2]);
        omc[2] = zsub(Ok[0 + 3 * 1], Ok[1 + 3 * 0]);
        zd dp = zd{0.0, 0.0};
#pragma unroll
        for (int a = 0; a < 3; ++a) dp = zadd(dp, zcmul(Ak[a], omc[a]));
        red[t] = dp.re;
      }
      __syncthreads();
      if (doK)
        for (int ef = t; ef < nef; ef += BS_THREADS) {
          double s = 0.0;
          for (int m0 = 0; m0 < n; ++m0) s += 0.5 * fd[ef + nef * m0] * red[m0];
          for (int i = 0; i < 3; ++i) acc[L.kcs + i + 3 * i + 9 * ef] += wk * s;
        }
      if (doNjob)
        for (int n0 = t; n0 < nval && n0 < n; n0 += BS_THREADS)
          for (int i = 0; i < 3; ++i) acc[L.ncs + i + 3 * i + 9 * n0] += wk * (0.5 * red[n0]);
    }
  }
  __syncthreads();
  if (HERM && pmode) {
    // the pair sums of the 8 bands of a group, then of the wavefronts that had
    // bands (8 to a wavefront); every pair was summed in both orders
    const int base = 12 * ((lane >> 5) & 1) + 6 * ((lane >> 4) & 1) + 3 * ((lane >> 3) & 1);
#pragma unroll
    for (int s = 0; s < 3; ++s) {
      const double v = group8_sum(pacc[s]);
      if ((lane & 7) == 0) QK[wv * 24 + base + s] = v;
    }
    __syncthreads();
    if (t < 9) {
      const int i = t % 3, j = t / 3, c = i + j - 1;
      const double B = 2.0 * wq.re * wq.im;
      auto u = [&](int e) { return ((QK[e] + QK[24 + e]) + QK[48 + e]) + QK[72 + e]; };
      auto g = [&](int e) { return zd{u(e), B * u(e + 3)}; };  // sum of g v
      zd av = zd{0.0, 0.0}, ao;
      if (i == j) {      // ohc_ii = i w sum g |x_i|^2 / dE
        ao = zmuli(zmul(wq, g(12 + i)));
      } else {           // velo_ij = M, ohc_ij = M + i w N (i < j); -M for j > i
        const zd M = g(c), iwN = zmuli(zmul(wq, g(6 + c)));
        av = i < j ? M : zd{-M.re, -M.im};
        ao = zadd(av, iwN);
      }
      acc[L.velo + 2 * t] += av.re;
      acc[L.velo + 2 * t + 1] += av.im;
      acc[L.ohc + 2 * t] += ao.re;
      acc[L.ohc + 2 * t + 1] += ao.im;
    }
    __syncthreads();
  }
  // the record in HBM holds the velo / ohc block (gap entries from L.velo)
  // that this layout leaves out
  double* out = part + (int64_t)blockIdx.x * (L.total + gap);
  for (int64_t c = t; c < L.total; c += BS_THREADS) out[c < L.velo ? c : c + gap] += acc[c];
}

// ===========================================================================
// 32 < n <= 128.  Same sums and the same record layout; V and E are read from
// HBM / L2 instead of LDS, the workgroup's accumulator record lives in `part`
// (one writer per entry, fixed order).
//   pair phase       thread (n0, part) over n = part, part + P, ...; parts
//                    combined through LDS.  HERM (V built here without a
//                    position operator): V_a(n, n0) = conj V_a(n0, n), so one
//                    coalesced read of V serves the Berry, local and, for a
//                    single (hw, E_F), the velo / ohc sums; otherwise V(n, n0)
//                    is read as stored
//   hw-resolved sums a kernel of their own (hwsum_kernel below)
//   itinerant terms  all three C_j on FP64 MFMA by wave item (16 x 16 tile);
//                    the items' sums pass through the workgroup's slot
// LDS: E n | fd nef*n | S 21*256 | F2, F2m 2*9*n | red 4*36 | windows
// ===========================================================================
static __device__ inline double rinv(const double* Es, int m, int c) {
  return (m == c) ? 0.0 : 1.0 / (Es[c] - Es[m]);  // 1 / (E_c - E_m)
}

// complex elements of a workgroup's slot: three scaled planes (general V only) and
// 18 sums of 16 columns for each 16 x 16 tile (at most the eigensolver record of a
// k-point)
__host__ __device__ inline int64_t wide_planes(int n, bool herm) {
  return herm ? 0 : 3 * (int64_t)n * n;
}
__host__ __device__ inline int64_t wide_slot(int n, bool herm) {
  const int64_t nt = (n + 15) / 16;
  return wide_planes(n, herm) + nt * nt * (18 * 16 / 2);
}
size_t bandsum_wide_scratch(const BandArgs& b, int nblocks) {
  return b.n > 32 ? sizeof(zd) * (size_t)wide_slot(b.n, b.v_herm) * nblocks : 0;
}

constexpr int BW_SLOTS = 21;  // per-band partial sums a thread leaves in LDS
// lane group of 8 sums f over the bands and adds it to *dst (all 8 lanes call)
static __device__ inline void band_item(int n, int nef, int ef, int g, bool valid, const double* fd,
                                        const double* src, double w, double* dst) {
  double s = 0.0;
  if (valid)
    for (int m0 = g; m0 < n; m0 += 8) s += fd[ef + nef * m0] * (src ? src[m0] : 1.0);
  s = group8_sum(s);
  if (valid && g == 0) *dst += w * s;
}
template <bool HERM>
__global__ __launch_bounds__(256, 2) void bandsum_wide_kernel(BandArgs b, double Tsmear, AccLayout L,
                                                           int64_t nk, const double* __restrict__ E,
                                                           const zd* __restrict__ V,
                                                           const double* __restrict__ w,
                                                           double* __restrict__ part,
                                                           zd* __restrict__ Bscr,
                                                           const zd* __restrict__ A,
                                                           const zd* __restrict__ Om) {
  extern __shared__ double smem[];
  __shared__ uint8_t ord[2 * 64];  // the wave items' row and column tiles
  const int n = b.n, nef = b.n_ef, nhw = b.n_hw, nval = b.n_val;
  double* Es = smem;
  double* fd = Es + n;
  double* S = fd + (int64_t)nef * n;  // [BW_SLOTS][256]
  double* S2 = S + 9 * 256;
  double* F2 = S + BW_SLOTS * 256;    // [9][n]
  double* F2m = F2 + 9 * n;           // [9][n]
  double* red = F2m + 9 * n;          // [4][36]
  uint8_t* win = reinterpret_cast<uint8_t*>(red + 4 * 36);  // [nval][n] lo, hi
  const int t = threadIdx.x, lane = t & 63, wv = __builtin_amdgcn_readfirstlane(t >> 6);
  const int n2 = n * n;
  const bool finiteT = b.T_kelvin > 1e-2;
  const bool doAHC = (b.jobs & MEP_JOB_AHC) != 0;
  const bool doK = (b.jobs & MEP_JOB_KUBO) != 0;
  const bool doNjob = (b.jobs & MEP_JOB_MEP) != 0;
  const bool pmode = HERM && doAHC && (nhw * nef == 1);
  const zd wq = zd{b.hw[0], b.eta};
  const double eta2 = b.eta * b.eta, B2 = 4.0 * wq.re * wq.re * eta2;
  const double tol = b.kubo_tol;
  double* acc = part + (int64_t)blockIdx.x * L.total;
  const int npad = n <= 64 ? 64 : 128, P = 256 / npad;
  const int p0 = t % npad, pp = t / npad;
  const bool pact = p0 < n;

  if (t == 0) {
    // 2 x 2 tiles at a time, (a, b) and then (b, a): the four wavefronts share
    // their operands in L1
    const int nt = (n + 15) / 16, nq = (nt + 1) / 2;
    int c = 0;
    auto quad = [&](int a, int b_) {
      for (int u = 0; u < 4; ++u) {
        const int tr = 2 * a + (u & 1), tc = 2 * b_ + (u >> 1);
        if (tr < nt && tc < nt) {
          ord[2 * c] = (uint8_t)tr;
          ord[2 * c + 1] = (uint8_t)tc;
          ++c;
        }
      }
    };
    for (int a = 0; a < nq; ++a)
      for (int b_ = a; b_ < nq; ++b_) {
        quad(a, b_);
        if (a != b_) quad(b_, a);
      }
  }

  for (int64_t k = blockIdx.x; k < nk; k += gridDim.x) {
    const double wk = w ? w[k] : 1.0;
    const zd* Vk = V + k * 3 * (int64_t)n2;
    __syncthreads();
    if (t < n) Es[t] = E[k * n + t];
    __syncthreads();
    // the valence bands whose Niu guards exclude something: not those with g^3 >
    // kubo_tol, g the gap to the nearest band (see bandsum_kernel), nor, at a
    // k-point out of order, any.  Bit n0 of dirty, the same in every wavefront;
    // only these have windows
    uint64_t dirty[2] = {0, 0};
    if (doNjob) {
      bool up = true;  // ascending
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int n0 = 64 * q + lane;
        bool d = false;
        if (n0 < n && (!HERM || n0 < nval)) {
          const double g0 = n0 > 0 ? Es[n0] - Es[n0 - 1] : HUGE_VAL;
          const double g1 = n0 < n - 1 ? Es[n0 + 1] - Es[n0] : HUGE_VAL;
          d = n0 < nval && !(g0 * g0 * g0 > tol && g1 * g1 * g1 > tol);
          up = up && (HERM || g0 >= 0.0);
        }
        dirty[q] = __ballot(d);
      }
      if (!HERM && __ballot(!up)) {
        auto low = [](int c) { return c >= 64 ? ~0ull : c > 0 ? (1ull << c) - 1 : 0ull; };
        const int nv = nval < n ? nval : n;
        dirty[0] = low(nv);
        dirty[1] = low(nv - 64);
      }
    }
#pragma unroll
    for (int q = 0; q < 2; ++q)
      for (uint64_t m = dirty[q]; m; m &= m - 1) {
        const int n0 = 64 * q + __builtin_ctzll(m), nn = t;
        if (nn >= n || nn == n0) continue;
        const double E0 = Es[n0], dn = E0 - Es[nn];
        const double dn2 = dn * dn;
        int lo = n0, hi = n0;
        while (lo > 0 && !(fabs(dn2 * (E0 - Es[lo - 1])) > tol)) --lo;
        while (hi < n - 1 && !(fabs(dn2 * (E0 - Es[hi + 1])) > tol)) ++hi;
        win[2 * (n0 * n + nn)] = (uint8_t)lo;
        win[2 * (n0 * n + nn) + 1] = (uint8_t)hi;
      }
    for (int idx = t; idx < nef * n; idx += 256) {
      if (b.fd_in) {
        fd[idx] = b.fd_in[k * (int64_t)nef * n + idx];
      } else {
        const int ef = (nef == 1) ? 0 : idx % nef, nb = (nef == 1) ? idx : idx / nef;
        const double e = Es[nb], f = b.ef[ef];
        fd[idx] = finiteT ? 1.0 / (1.0 + exp((e - f) / Tsmear)) : ((e < f) ? 1.0 : 0.0);
      }
    }
    __syncthreads();
    if constexpr (HERM) {
      // x_a = V_a(n0, n), P_ij = x_i conj(x_j) (i < j), r = 1 / (E0 - En), as
      // the pair phase of bandsum_kernel
      // gd, go: over the n that mep_niu keeps, gx, gy: over those it excludes
      // (few), which the Kubo sums add
      const bool guard = pact && ((dirty[p0 >> 6] >> (p0 & 63)) & 1);
      const double E0 = pact ? Es[p0] : 0.0, f0 = (pmode && pact) ? fd[p0] : 0.0;
      double om[3] = {0.0, 0.0, 0.0}, gd[3] = {0.0, 0.0, 0.0}, gx[3] = {0.0, 0.0, 0.0}, ps[24];
      zd go[3], gy[3];
#pragma unroll
      for (int c = 0; c < 3; ++c) go[c] = gy[c] = zd{0.0, 0.0};
#pragma unroll
      for (int c = 0; c < 24; ++c) ps[c] = 0.0;
      if (pact)
#pragma unroll 2
        for (int nn = pp; nn < n; nn += P) {
          zd x[3], Pc[3];
          double d[3];
#pragma unroll
          for (int a = 0; a < 3; ++a) {
            x[a] = Vk[a * (int64_t)n2 + p0 + (int64_t)n * nn];
            d[a] = zabs2(x[a]);
          }
#pragma unroll
          for (int c = 0; c < 3; ++c) {
            const zd xi = x[c == 2 ? 1 : 0], xj = x[c == 0 ? 1 : 2];
            Pc[c] = zd{xi.re * xj.re + xi.im * xj.im, xi.im * xj.re - xi.re * xj.im};
          }
          const bool off = nn != p0;
          const double dE = E0 - Es[nn];
          const double r = off ? rcp_nr(dE) : 0.0, r2 = r * r, r3 = r2 * r;
          const bool ex = guard && !(fabs(dE * dE * dE) > tol);
          const double r3k = ex ? 0.0 : r3;
#pragma unroll
          for (int c = 0; c < 3; ++c) {
            om[c] += r2 * Pc[c].im;
            gd[c] += r3k * d[c];
            go[c] = zd{go[c].re + r3k * Pc[c].re, go[c].im + r3k * Pc[c].im};
          }
          if (ex)
#pragma unroll
            for (int c = 0; c < 3; ++c) {
              gx[c] += r3 * d[c];
              gy[c] = zd{gy[c].re + r3 * Pc[c].re, gy[c].im + r3 * Pc[c].im};
            }
          if (pmode) {  // the weights of bandsum_kernel's pair phase
            const double f = f0 - fd[nn];
            const bool on = f != 0.0 && off;
            const double D = (dE - wq.re) * (dE + wq.re) + eta2;
            const double q = on ? f * rcp_nr(D * D + B2) : 0.0, Dq = D * q;
            const double rs = on ? r : 0.0, qr = q * rs, Dqr = Dq * rs;
#pragma unroll
            for (int c = 0; c < 3; ++c) {
              ps[c] += Dq * Pc[c].im;
              ps[3 + c] += q * Pc[c].im;
              ps[6 + c] += Dqr * Pc[c].re;
              ps[9 + c] += qr * Pc[c].re;
              ps[12 + c] += Dqr * d[c];
              ps[15 + c] += qr * d[c];
            }
          }
        }
      // local terms: F3_ij = Re(z_l G_ik - z_k G_il), (j, k, l) cyclic, z =
      // V(n0, n0), G_ik = sum_n r^3 x_i conj(x_k)
      zd z[3];
#pragma unroll
      for (int a = 0; a < 3; ++a)
        z[a] = pact ? Vk[a * (int64_t)n2 + p0 + (int64_t)n * p0] : zd{0.0, 0.0};
      auto local = [&](const double* gd_, const zd* go_, double* o) {
        auto G = [&](int i, int k_) {
          if (i == k_) return zd{gd_[i], 0.0};
          const zd g = go_[i + k_ - 1];
          return i < k_ ? g : zd{g.re, -g.im};
        };
#pragma unroll
        for (int j = 0; j < 3; ++j) {
          const int k_ = (j + 1) % 3, l = (j + 2) % 3;
#pragma unroll
          for (int i = 0; i < 3; ++i) {
            const zd a = G(i, k_), bb = G(i, l);
            o[i + 3 * j] = (z[l].re * a.re - z[l].im * a.im) - (z[k_].re * bb.re - z[k_].im * bb.im);
          }
        }
      };
      {
        double f3[9];
        local(gd, go, f3);
#pragma unroll
        for (int q = 0; q < 9; ++q) S[(9 + q) * 256 + t] = f3[q];
        if (__ballot(guard)) {
          double fx[9];
          local(gx, gy, fx);
#pragma unroll
          for (int q = 0; q < 9; ++q) f3[q] += fx[q];
        }
#pragma unroll
        for (int q = 0; q < 9; ++q) S[q * 256 + t] = f3[q];
      }
#pragma unroll
      for (int c = 0; c < 3; ++c) S[(18 + c) * 256 + t] = om[c];
      if (pmode) {
        double v3[3];
        scatter_sum<24>(ps, v3, lane);
        const int base = 12 * ((lane >> 5) & 1) + 6 * ((lane >> 4) & 1) + 3 * ((lane >> 3) & 1);
#pragma unroll
        for (int q = 0; q < 3; ++q) v3[q] = group8_sum(v3[q]);
        if ((lane & 7) == 0)
#pragma unroll
          for (int q = 0; q < 3; ++q) red[wv * 24 + base + q] = v3[q];
      }
      __syncthreads();
      // the parts of a band into part 0's place
      for (int e = t; e < BW_SLOTS * npad; e += 256) {
        const int q = e / npad, m0 = e % npad;
        double o = 0.0;
        for (int u = 0; u < P; ++u) o += S[q * 256 + u * npad + m0];
        S[q * 256 + m0] = o;
      }
      __syncthreads();
      // Ne, kubo_ahc_tens (Omega_ij = -2 om, antisymmetric) and kubo_mep_LC
      for (int base = 0; base < 8 * 13 * nef; base += 256) {
        const int it = base + t, item = it >> 3, g = it & 7, c = item % 13, ef = item / 13;
        const bool in = item < 13 * nef;
        if (c >= 1 && c < 4) {
          const int i = (c == 3) ? 1 : 0, j = (c == 1) ? 1 : 2;
          double s = 0.0;
          if (in && doAHC)
            for (int m0 = g; m0 < n; m0 += 8) s += fd[ef + nef * m0] * S[(17 + c) * 256 + m0];
          s = group8_sum(s);
          if (in && doAHC && g == 0) {
            acc[L.ahc + i + 3 * j + 9 * ef] += wk * (2.0 * s);
            acc[L.ahc + j + 3 * i + 9 * ef] -= wk * (2.0 * s);
          }
        } else {
          band_item(n, nef, ef, g, in && (c == 0 || doK), fd, c == 0 ? nullptr : S + (c - 4) * 256, wk,
                    acc + (c == 0 ? L.Ne + ef : L.klc + (c - 4) + 9 * ef));
        }
      }
      if (doNjob)
        for (int it = t; it < 9 * nval; it += 256)
          acc[L.nlc + it] += wk * S[(9 + it % 9) * 256 + it / 9];
      // velo_ahc_tens / kubo_ohc_tens at the single (hw, E_F)
      if (pmode && t < 9) {
        const int i = t % 3, j = t / 3, c = i + j - 1;
        const double B = 2.0 * wq.re * wq.im;
        auto u = [&](int e) { return ((red[e] + red[24 + e]) + red[48 + e]) + red[72 + e]; };
        auto g = [&](int e) { return zd{u(e), B * u(e + 3)}; };  // sum of g v
        zd av = zd{0.0, 0.0}, ao;
        if (i == j) {
          ao = zmuli(zmul(wq, g(12 + i)));
        } else {
          const zd M = g(c), iwN = zmuli(zmul(wq, g(6 + c)));
          av = i < j ? M : zd{-M.re, -M.im};
          ao = zadd(av, iwN);
        }
        acc[L.velo + 2 * t] += wk * av.re;
        acc[L.velo + 2 * t + 1] += wk * av.im;
        acc[L.ohc + 2 * t] += wk * ao.re;
        acc[L.ohc + 2 * t + 1] += wk * ao.im;
      }
    } else {
    for (int ef = t; ef < nef; ef += 256) {
      double sN = 0.0;
      for (int m0 = 0; m0 < n; ++m0) sN += fd[ef + nef * m0];
      acc[L.Ne + ef] += wk * sN;
    }
    // ---- Berry curvature per band -> kubo_ahc_tens --------------------------
    if (doAHC) {
      double om[9];
#pragma unroll
      for (int q = 0; q < 9; ++q) om[q] = 0.0;
      if (pact)
        for (int nn = pp; nn < n; nn += P) {
          if (nn == p0) continue;
          zd x[3], y[3];
#pragma unroll
          for (int a = 0; a < 3; ++a) {
            x[a] = Vk[a * (int64_t)n2 + p0 + (int64_t)n * nn];
            y[a] = Vk[a * (int64_t)n2 + nn + (int64_t)n * p0];
          }
          const double r = rinv(Es, nn, p0);  // 1 / (E_0 - E_n)
          const double r2 = r * r;
#pragma unroll
          for (int j = 0; j < 3; ++j)
#pragma unroll
            for (int i = 0; i < 3; ++i) om[i + 3 * j] -= 2.0 * zmul(x[i], y[j]).im * r2;
        }
#pragma unroll
      for (int q = 0; q < 9; ++q) S[q * 256 + t] = om[q];
      __syncthreads();
      for (int it = t; it < 9 * nef; it += 256) {
        const int q = it % 9, ef = it / 9;
        double sA = 0.0;
        for (int m0 = 0; m0 < n; ++m0) {
          double o = 0.0;
          for (int u = 0; u < P; ++u) o += S[q * 256 + u * npad + m0];
          sA += fd[ef + nef * m0] * o;
        }
        acc[L.ahc + q + 9 * ef] -= wk * sA;
      }
      __syncthreads();
    }
    // ---- local (LC) MEP terms ----------------------------------------------
    if (doK || doNjob) {
      double f3[9], f3m[9];
#pragma unroll
      for (int q = 0; q < 9; ++q) f3[q] = f3m[q] = 0.0;
      const bool doN = doNjob && pact && p0 < nval;
      if (pact) {
        const double E0 = Es[p0];
        zd z0[3];
#pragma unroll
        for (int l = 0; l < 3; ++l) z0[l] = Vk[l * (int64_t)n2 + p0 + (int64_t)n * p0];
        for (int nn = pp; nn < n; nn += P) {
          if (nn == p0) continue;
          zd x[3], y[3];
#pragma unroll
          for (int a = 0; a < 3; ++a) {
            x[a] = Vk[a * (int64_t)n2 + p0 + (int64_t)n * nn];
            y[a] = Vk[a * (int64_t)n2 + nn + (int64_t)n * p0];
          }
          const double r = rinv(Es, nn, p0);  // 1 / (E_0 - E_n)
          const double r3 = r * r * r;
          zd cr[3];
          cr[0] = zsub(zmul(y[1], z0[2]), zmul(y[2], z0[1]));
          cr[1] = zsub(zmul(y[2], z0[0]), zmul(y[0], z0[2]));
          cr[2] = zsub(zmul(y[0], z0[1]), zmul(y[1], z0[0]));
          const double dn = E0 - Es[nn];
          const bool keep3 = doN && (fabs(dn * dn * dn) > tol);
#pragma unroll
          for (int j = 0; j < 3; ++j)
#pragma unroll
            for (int i = 0; i < 3; ++i) {
              const double v = zmul(x[i], cr[j]).re * r3;
              f3[i + 3 * j] += v;
              if (keep3) f3m[i + 3 * j] += v;
            }
        }
      }
#pragma unroll
      for (int q = 0; q < 9; ++q) {
        S[q * 256 + t] = f3[q];
        S2[q * 256 + t] = f3m[q];
      }
      __syncthreads();
      if (doK)
        for (int it = t; it < 9 * nef; it += 256) {
          const int q = it % 9, ef = it / 9;
          double sL = 0.0;
          for (int m0 = 0; m0 < n; ++m0) {
            double o = 0.0;
            for (int u = 0; u < P; ++u) o += S[q * 256 + u * npad + m0];
            sL += fd[ef + nef * m0] * o;
          }
          acc[L.klc + q + 9 * ef] += wk * sL;
        }
      if (doNjob)
        for (int it = t; it < 9 * nval; it += 256) {
          const int q = it % 9, m0 = it / 9;
          double o = 0.0;
          for (int u = 0; u < P; ++u) o += S2[q * 256 + u * npad + m0];
          acc[L.nlc + q + 9 * m0] += wk * o;
        }
      __syncthreads();
    }
    }
    // ---- itinerant (IC) terms on MFMA ----------------------------------------
    // B_a(m, n0) = V_a(m, n0) r(m, n0), r(m, n0) = 1 / (E_n0 - E_m), 0 for m = n0
    // and for an m of exactly n0's energy, in the product and in the windows'
    // terms alike: the Niu guards exclude such an m whatever n is, and the Kubo
    // sum is not finite all the same, through its row m of the contraction.
    // Hermitian V: formed in the step from conj V_a(n0, m), which
    // loads as one run of the 16 columns n0, so V is all that is read (a scaled
    // copy per workgroup doubled a working set that the caches miss as it is);
    // general V: scaled planes in the workgroup's slot of Bscr, transposed.
    // A wave item is one 16 x 16 tile of all three C_j = V_k B_l - V_l B_k: six
    // operands a step feed 18 products, and the next step's operands are in
    // flight during a step's products; the four wavefronts take 2 x 2 tiles, whose
    // operands they share in L1.  Two row tiles an item (9 operands for 36
    // products) spill, three wavefronts a SIMD too.  The contraction with
    // A_i(n0, n) = V_i(n0, n) r(n, n0)^2 comes straight from the accumulators;
    // the items' sums go through the slot.  Bound by the operands' way from beyond
    // L2 (n = 96: 9.9 GB at 4.0 TB/s; n = 44: 1.5 TB/s) and by issue (MFMA 0.45 and
    // VALU 0.20 of the SIMD-cycles; 0.33 and 0.24), at two wavefronts a SIMD.
    // n = 96, 2,744 k-points: 2.5 ms (one C_j an item, V read three times: 5.6;
    // with scaled planes and tiles in row order 3.0); n = 44, 9,261: 1.48 ms
    // (3.0 with its velo / ohc kernel; 1.72).
    if (doK || doNjob) {
      const int nt = (n + 15) / 16;
      const int lr = lane & 15, kq = lane >> 4;
      zd* Bw = Bscr + (int64_t)blockIdx.x * wide_slot(n, HERM);
      double* Pw = reinterpret_cast<double*>(Bw + wide_planes(n, HERM));  // [item][18][16]
      if constexpr (!HERM) {
        for (int idx = t; idx < n2; idx += 256) {
          const int n0 = idx % n, m = idx / n;
          const double dE = Es[n0] - Es[m], rr = dE != 0.0 ? rcp_nr(dE) : 0.0;
#pragma unroll
          for (int a = 0; a < 3; ++a)
            Bw[a * (int64_t)n2 + idx] = zscale(Vk[a * (int64_t)n2 + m + (int64_t)n * n0], rr);
        }
        __syncthreads();
      }
      for (int item = wv; item < nt * nt; item += 4) {
        const int tr = ord[2 * item], tc = ord[2 * item + 1];
        const int r0 = 16 * tr, n0 = 16 * tc + lr;
        const bool colok = n0 < n;
        // this column has windows; without any in the tile, the kept sums are all
        const bool doN = colok && ((dirty[n0 >> 6] >> (n0 & 63)) & 1);
        const bool anyN = __ballot(doN) != 0;
        const int nc = colok ? n0 : n - 1;  // padded rows and columns repeat the last: not used
        const int ar = r0 + lr < n ? r0 + lr : n - 1;
        mep_v4d p1[3] = {}, p2[3] = {}, p3[3] = {};
        const double E0 = Es[nc];
        struct Step {
          zd a[3], b[3];
          double r;
        };
        auto load = [&](int m0, Step& s) {  // past the end: the last row, weight 0
          const bool mok = m0 + kq < n;
          const int64_t mo = (int64_t)n * (mok ? m0 + kq : n - 1);
#pragma unroll
          for (int c = 0; c < 3; ++c) {
            s.b[c] = HERM ? Vk[c * (int64_t)n2 + mo + nc] : Bw[c * (int64_t)n2 + mo + nc];
            s.a[c] = Vk[c * (int64_t)n2 + mo + ar];
          }
          s.r = HERM ? E0 - Es[mok ? m0 + kq : n - 1] : 1.0;
          if (!mok || (HERM && m0 + kq == nc)) s.r = 0.0;  // no such m; r(n0, n0) = 0
        };
        auto mac = [&](Step& s) {
          double as[3], bs[3];
          const double r = HERM ? (s.r != 0.0 ? rcp_nr(s.r) : 0.0) : s.r;
#pragma unroll
          for (int c = 0; c < 3; ++c) {
            s.b[c] = zd{s.b[c].re * r, s.b[c].im * (HERM ? -r : r)};
            as[c] = s.a[c].re + s.a[c].im;
            bs[c] = s.b[c].re + s.b[c].im;
          }
#pragma unroll
          for (int j = 0; j < 3; ++j) {
            const int kk = (j + 1) % 3, ll = (j + 2) % 3;
            p1[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(s.a[kk].re, s.b[ll].re, p1[j], 0, 0, 0);
            p2[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(s.a[kk].im, s.b[ll].im, p2[j], 0, 0, 0);
            p3[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(as[kk], bs[ll], p3[j], 0, 0, 0);
          }
#pragma unroll
          for (int j = 0; j < 3; ++j) {
            const int kk = (j + 1) % 3, ll = (j + 2) % 3;
            p1[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(s.a[ll].re, -s.b[kk].re, p1[j], 0, 0, 0);
            p2[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(s.a[ll].im, -s.b[kk].im, p2[j], 0, 0, 0);
            p3[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(as[ll], -bs[kk], p3[j], 0, 0, 0);
          }
        };
        Step s0, s1;  // the next step's operands are in flight during this one's products
        load(0, s0);
        for (int m0 = 0; m0 < n; m0 += 8) {
          load(m0 + 4, s1);
          mac(s0);
          load(m0 + 8, s0);
          mac(s1);
        }
        double f2[9], f2m[9];
#pragma unroll
        for (int q = 0; q < 9; ++q) f2[q] = f2m[q] = 0.0;
        // mep_niu keeps, for (n0, n), the m outside one window [lo, hi]: narrow
        // windows take -Re[A C] here and add back the excluded terms below; wide
        // windows sum the kept terms directly below; a window of n0 itself or of
        // every m needs no second pass
        auto wide = [&](int lo, int hi) { return 2 * (hi - lo + 1) > n; };
        unsigned wterm = 0;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int row = r0 + kq + 4 * v;
          if (!colok || row >= n || row == n0) continue;
          const double rr = rcp_nr(Es[n0] - Es[row]), rr2 = rr * rr;
          bool narrow = !doN;
          if (doN) {
            const int lo = win[2 * (n0 * n + row)], hi = win[2 * (n0 * n + row) + 1];
            const bool all = lo == 0 && hi == n - 1;
            narrow = !all && !wide(lo, hi);
            if (!all && !(lo == n0 && hi == n0)) wterm |= 1u << v;
          }
          zd ai[3];
#pragma unroll
          for (int i = 0; i < 3; ++i) ai[i] = zscale(Vk[i * (int64_t)n2 + n0 + (int64_t)n * row], rr2);
#pragma unroll
          for (int j = 0; j < 3; ++j) {
            const zd cv = zd{p1[j][v] - p2[j][v], p3[j][v] - p1[j][v] - p2[j][v]};
#pragma unroll
            for (int i = 0; i < 3; ++i) {
              const double c = ai[i].re * cv.re - ai[i].im * cv.im;
              f2[i + 3 * j] -= c;
              if (anyN) f2m[i + 3 * j] -= narrow ? c : 0.0;
            }
          }
        }
        for (int v = 0; v < 4 && wterm >> v; ++v) {  // after the accumulators are dead
          if (!((wterm >> v) & 1)) continue;
          const int row = r0 + kq + 4 * v;
          const int lo = win[2 * (n0 * n + row)], hi = win[2 * (n0 * n + row) + 1];
          const bool wd = wide(lo, hi);
          const double rr = rcp_nr(Es[n0] - Es[row]), rr2 = rr * rr;
          zd ai[3], x[3];
#pragma unroll
          for (int i = 0; i < 3; ++i) {
            ai[i] = zscale(Vk[i * (int64_t)n2 + n0 + (int64_t)n * row], rr2);
            x[i] = zd{0.0, 0.0};
          }
          auto terms = [&](int from, int to) {
            for (int mm = from; mm < to; ++mm) {
              zd vm[3], bm[3];
              const double dm = Es[n0] - Es[mm];
              const double rm = HERM ? (dm != 0.0 ? rcp_nr(dm) : 0.0) : 1.0;
#pragma unroll
              for (int c = 0; c < 3; ++c) {
                vm[c] = Vk[c * (int64_t)n2 + row + (int64_t)n * mm];
                bm[c] = HERM ? zscale(zconj(Vk[c * (int64_t)n2 + n0 + (int64_t)n * mm]), rm)
                             : Bw[c * (int64_t)n2 + n0 + (int64_t)n * mm];
              }
#pragma unroll
              for (int j = 0; j < 3; ++j) {
                const int kk = (j + 1) % 3, ll = (j + 2) % 3;
                x[j] = zadd(x[j], zsub(zmul(vm[kk], bm[ll]), zmul(vm[ll], bm[kk])));
              }
            }
          };
          if (wd) {  // kept terms: f2m -= Re(A x)
            terms(0, lo);
            terms(hi + 1, n);
          } else {   // excluded terms: f2m += Re(A x)
            terms(lo, hi + 1);
          }
#pragma unroll
          for (int j = 0; j < 3; ++j)
#pragma unroll
            for (int i = 0; i < 3; ++i) {
              const double c = ai[i].re * x[j].re - ai[i].im * x[j].im;
              f2m[i + 3 * j] += wd ? -c : c;
            }
        }
#pragma unroll
        for (int q = 0; q < 9; ++q) {
          const double s0 = rows4_sum(f2[q]), s1 = anyN ? rows4_sum(f2m[q]) : s0;
          if (kq == 0) {
            Pw[((tr * nt + tc) * 18 + q) * 16 + lr] = s0;
            Pw[((tr * nt + tc) * 18 + 9 + q) * 16 + lr] = s1;
          }
        }
      }
      __syncthreads();
      for (int e = t; e < 18 * n; e += 256) {  // F2 and F2m are neighbours
        const int q = e / n, m0 = e % n;
        double o = 0.0;
        for (int tr = 0; tr < nt; ++tr) o += Pw[((tr * nt + m0 / 16) * 18 + q) * 16 + m0 % 16];
        F2[e] = o;
      }
      __syncthreads();
      if (doK)
        for (int base = 0; base < 8 * 9 * nef; base += 256) {
          const int it = base + t, item = it >> 3, q = item % 9, ef = item / 9;
          band_item(n, nef, ef, it & 7, item < 9 * nef, fd, F2 + q * n, wk, acc + L.kic + q + 9 * ef);
        }
      if (doNjob)
        for (int it = t; it < 9 * nval; it += 256)
          acc[L.nic + it] += wk * F2m[(it % 9) * n + it / 9];
    }
    // ---- Chern-Simons terms (position operator: A and Omega) ---------------
    // kubo_mep_CS / mep_niu_CS (kubo_mep.f90:16-47, mep_niu.f90:20-45):
    // red[n0] = Re sum_a conj(A_a(n0,n0)) omega_a(n0,n0), omega_c from Omega_ab
    if ((doK || doNjob) && b.pos_op && A && Om) {
      __syncthreads();
      for (int n0 = t; n0 < n; n0 += 256) {
        const int64_t NN = (int64_t)n2;
        const zd* Ak = A + k * 3 * NN + 3 * ((int64_t)n0 + (int64_t)n * n0);
        const zd* Ok = Om + k * 9 * NN + 9 * ((int64_t)n0 + (int64_t)n * n0);
        zd omc[3];
        omc[0] = zsub(Ok[1 + 3 * 2], Ok[2 + 3 * 1]);
        omc[1] = zsub(Ok[2 + 3 * 0], Ok[0 + 3 * 2]);
        omc[2] = zsub(Ok[0 + 3 * 1], Ok[1 + 3 * 0]);
        zd dp = zd{0.0, 0.0};
#pragma unroll
        for (int a = 0; a < 3; ++a) dp = zadd(dp, zcmul(Ak[a], omc[a]));
        red[n0] = dp.re;
      }
      __syncthreads();
      if (doK)
        for (int ef = t; ef < nef; ef += 256) {
          double s_ = 0.0;
          for (int m0 = 0; m0 < n; ++m0) s_ += 0.5 * fd[ef + nef * m0] * red[m0];
          for (int i = 0; i < 3; ++i) acc[L.kcs + i + 3 * i + 9 * ef] += wk * s_;
        }
      if (doNjob)
        for (int n0 = t; n0 < nval && n0 < n; n0 += 256)
          for (int i = 0; i < 3; ++i) acc[L.ncs + i + 3 * i + 9 * n0] += wk * (0.5 * red[n0]);
    }
  }
}

size_t bandsum_wide_lds_bytes(const BandArgs& b) {
  const size_t n = b.n;
  return sizeof(double) * (n + (size_t)b.n_ef * n + BW_SLOTS * 256 + 2 * 9 * n + 4 * 36) +
         2 * (size_t)(b.n_val > 0 ? b.n_val : 1) * n;
}

// ===========================================================================
// velo_ahc_tens / kubo_ohc_tens over a list of items (hw, E_F): per k, the
// pairs x < y whose occupations differ at some E_F are compacted, in pair
// order, into LDS chunks of up to 256 records; thread (slot, split) walks
// every split-th record for its IPT items, accumulating in registers over all
// k; the splits are combined once at the end.  Items beyond 256 IPT are taken
// in further passes over the k-points.
//
// A record stands for (x, y) and (y, x).  With dE = E_x - E_y, f = f_x - f_y,
// w = hw + i eta and P_ij = V_i(y, x) V_j(x, y), the two orders' weights are
//   velo  g Im(P_ji - P_ij),  g = f / (dE^2 - w^2)
//   ohc   f / (dE (dE - w)) P_ij - f / (dE (dE + w)) P_ji
//         = g (P_ij - P_ji) + w g (P_ij + P_ji) / dE
// so with Hermitian V one complex g serves all of them: the sums of g A, A_c =
// P_ij - P_ji, and of g S, S_ij = (P_ij + P_ji) / dE, are what the items keep,
// and w enters once at the end.  With D = (dE - hw)(dE + hw) + eta^2 (no
// cancellation at resonance) and B = 2 hw eta, g = (D + i B) r, r = f / (D^2 +
// B^2): the items sum D r v and r v over the real values v of A and S, and B
// waits as well: Im A (3), Re S (3) and S_ii (3), the others being zero.
//
// General V: P_ij and P_ji are of different sizes.  The weight of the order
// that is not in resonance would be the difference of two terms larger by dE /
// eta, so the off-diagonal ohc sums (6, complex) take each order's own weight,
//   f / (dE - w) = (dE - hw + i eta) f m2 / (m1 m2),  m1 = |dE - w|^2
//   f / (dE + w) = (dE + hw - i eta) f m1 / (m1 m2),  m2 = |dE + w|^2
// (1 / dE is in the record), which share g's one reciprocal, m1 m2 = D^2 + B^2;
// S_ii (3, complex), where both orders weigh the same value, and Im A (3) as
// above.
//
// Bound by FP64 VALU issue (n = 96: 0.69 of the SIMD-cycles, n = 20: 0.61; general
// V, with its few items, by latency): 2 x 9 fma and about 13 more a record and item
// (Hermitian V); four items a thread take the reads of a record from LDS off
// the LDS return path.
// n = 96, 256 frequencies, 2,744 k-points: 2.6 ms (three denominators for the
// two orders, 24 sums an item: 4.2); n = 20, 80 items, 24,273: 0.50 ms (0.88);
// general V, n = 14, 16 items, 2,730: 45 us (59 with a reciprocal for each
// weight and ordered pair; 40 with g alone, at the loss above: 7e-9 of an element
// at eta = 1e-8, now 3e-16).
// ===========================================================================
constexpr int HW_CH = 256;  // pair candidates per chunk (one per thread)

// values of a record; real sums of an item, in three parts of at most hw_part
template <bool HERM>
__host__ __device__ constexpr int hw_vals() { return HERM ? 9 : 21; }
template <bool HERM>
__host__ __device__ constexpr int hw_part() { return HERM ? 6 : 12; }

template <bool HERM, int IPT>
__global__ __launch_bounds__(256, HERM ? 2 : 3) void hwsum_kernel(BandArgs b, double Tsmear, AccLayout L,
                                                       int64_t nk, const double* __restrict__ E,
                                                       const zd* __restrict__ V,
                                                       const double* __restrict__ w,
                                                       double* __restrict__ part) {
  constexpr int NV = hw_vals<HERM>(), NP = hw_part<HERM>();
  extern __shared__ double smem[];
  const int n = b.n, nef = b.n_ef, nhw = b.n_hw;
  const int PS = 1 + nef + NV;  // doubles per record: dE, f[nef], v[NV]
  double* Es = smem;
  double* fd = Es + n;
  int* cnt_w = reinterpret_cast<int*>(fd + (int64_t)nef * n);  // [4] per-wave counts
  double* st = fd + (int64_t)nef * n + 4;  // [HW_CH][PS]; reused for the split reduction
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  const int n2 = n * n, npair = n * (n - 1) / 2;
  const bool finiteT = b.T_kelvin > 1e-2;
  const int items = nhw * nef;
  double* accp = part + (int64_t)blockIdx.x * L.total;
  for (int g0 = 0; g0 < items; g0 += 256 * IPT) {
    // this pass: IW items, IWT thread slots per split, each slot holding the
    // items slot + IWT u (u < IPT), S splits over the records
    const int IW = (items - g0 < 256 * IPT) ? items - g0 : 256 * IPT;
    const int IWT = (IW + IPT - 1) / IPT;
    const int S = 256 / IWT;
    const int slot = t % IWT, split = t / IWT;
    const bool act = split < S;
    bool iok[IPT];
    int ef[IPT];
    double wr[IPT], B2[IPT];
    const double eta2 = b.eta * b.eta;
#pragma unroll
    for (int u = 0; u < IPT; ++u) {
      iok[u] = act && slot + IWT * u < IW;
      const int it = g0 + (iok[u] ? slot + IWT * u : 0);
      ef[u] = it / nhw;
      wr[u] = b.hw[it % nhw];
      B2[u] = 4.0 * wr[u] * wr[u] * eta2;
    }
    // HERM: sums of D r v and of r v of A, S, S_ii; general V: the ohc sums, then
    // those of S_ii and of Im A
    double acc[IPT][3][NP];
#pragma unroll
    for (int u = 0; u < IPT; ++u)
#pragma unroll
      for (int q = 0; q < 3 * NP; ++q) acc[u][q / NP][q % NP] = 0.0;
    for (int64_t k = blockIdx.x; k < nk; k += gridDim.x) {
      const double wk = w ? w[k] : 1.0;
      const zd* Vk = V + k * 3 * (int64_t)n2;
      __syncthreads();
      if (t < n) Es[t] = E[k * n + t];
      __syncthreads();
      for (int idx = t; idx < nef * n; idx += 256) {
        if (b.fd_in) {
          fd[idx] = b.fd_in[k * (int64_t)nef * n + idx];
        } else {
          const int e_ = (nef == 1) ? 0 : idx % nef, nb = (nef == 1) ? idx : idx / nef;
          const double e = Es[nb], f = b.ef[e_];
          fd[idx] = finiteT ? 1.0 / (1.0 + exp((e - f) / Tsmear)) : ((e < f) ? 1.0 : 0.0);
        }
      }
      for (int c0 = 0; c0 < npair; c0 += HW_CH) {
        __syncthreads();  // fd ready; the previous chunk consumed
        // pair x < y, p = x + y (y - 1) / 2
        const int p = c0 + t;
        int y = (int)((sqrtf(8.0f * (float)p + 1.0f) + 1.0f) * 0.5f);
        if (y * (y + 1) / 2 <= p) ++y;
        if (y * (y - 1) / 2 > p) --y;
        const int x = p - y * (y - 1) / 2;
        bool keep = p < npair;
        if (keep) {
          bool any = false;
          for (int e_ = 0; e_ < nef; ++e_) any |= fd[e_ + nef * x] != fd[e_ + nef * y];
          keep = any;  // pairs of equal occupation contribute exactly zero
        }
        const uint64_t ball = __ballot(keep);
        const int below = __popcll(ball & ((1ull << lane) - 1ull));
        if (lane == 0) cnt_w[wv] = __popcll(ball);
        __syncthreads();
        int base = 0;
        for (int u = 0; u < wv; ++u) base += cnt_w[u];
        const int cnt = cnt_w[0] + cnt_w[1] + cnt_w[2] + cnt_w[3];
        if (keep) {
          double* sp = st + (int64_t)(base + below) * PS;
          const double dE = Es[x] - Es[y], iE = 1.0 / dE;
          sp[0] = dE;
          for (int e_ = 0; e_ < nef; ++e_) sp[1 + e_] = wk * (fd[e_ + nef * x] - fd[e_ + nef * y]);
          double* v = sp + 1 + nef;
          zd vxy[3];
#pragma unroll
          for (int a = 0; a < 3; ++a) vxy[a] = Vk[a * (int64_t)n2 + x + (int64_t)n * y];
          // v: A_c, S_c (c = (0,1), (0,2), (1,2)), S_ii; general V: P_ij / dE and
          // P_ji / dE of each c, S_ii, Im A_c
          if constexpr (HERM) {  // V(y, x) = conj V(x, y): Im A, Re S, S_ii
#pragma unroll
            for (int c = 0; c < 3; ++c) {
              const zd xi = vxy[c == 2 ? 1 : 0], xj = vxy[c == 0 ? 1 : 2];
              v[c] = 2.0 * (xi.re * xj.im - xi.im * xj.re);
              v[3 + c] = 2.0 * (xi.re * xj.re + xi.im * xj.im) * iE;
              v[6 + c] = 2.0 * zabs2(vxy[c]) * iE;
            }
          } else {
            zd vyx[3];
#pragma unroll
            for (int a = 0; a < 3; ++a) vyx[a] = Vk[a * (int64_t)n2 + y + (int64_t)n * x];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
              const int i = c == 2 ? 1 : 0, j = c == 0 ? 1 : 2;
              const zd pij = zmul(vyx[i], vxy[j]), pji = zmul(vyx[j], vxy[i]);
              const zd Sd = zscale(zmul(vyx[c], vxy[c]), 2.0 * iE);
              v[4 * c] = pij.re * iE;
              v[4 * c + 1] = pij.im * iE;
              v[4 * c + 2] = pji.re * iE;
              v[4 * c + 3] = pji.im * iE;
              v[12 + 2 * c] = Sd.re;
              v[13 + 2 * c] = Sd.im;
              v[18 + c] = pij.im - pji.im;
            }
          }
        }
        __syncthreads();
        if (act)
          for (int j = split; j < cnt; j += S) {
            const double* sp = st + (int64_t)j * PS;
            const double dE = sp[0];
            double v[NV];
#pragma unroll
            for (int q = 0; q < NV; ++q) v[q] = sp[1 + nef + q];
#pragma unroll
            for (int u = 0; u < IPT; ++u) {
              // f = 0 records (another E_F differs) contribute exactly zero
              const double D1 = dE - wr[u], D2 = dE + wr[u];
              const double D = D1 * D2 + eta2;
              if constexpr (HERM) {
                const double r = sp[1 + ef[u]] * rcp_nr(D * D + B2[u]), Dr = D * r;
#pragma unroll
                for (int q = 0; q < NV; ++q) {
                  acc[u][q / 3][q % 3] += Dr * v[q];
                  acc[u][q / 3][3 + q % 3] += r * v[q];
                }
              } else {
                const double m1 = D1 * D1 + eta2, m2 = D2 * D2 + eta2;
                const double r = sp[1 + ef[u]] * rcp_nr(m1 * m2), Dr = D * r;
                const double t1 = r * m2, t2 = r * m1;
                const zd w1 = zd{D1 * t1, b.eta * t1}, w2 = zd{D2 * t2, -b.eta * t2};
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                  const zd pij = zd{v[4 * c], v[4 * c + 1]}, pji = zd{v[4 * c + 2], v[4 * c + 3]};
                  const zd xij = zsub(zmul(w1, pij), zmul(w2, pji));
                  const zd xji = zsub(zmul(w1, pji), zmul(w2, pij));
                  acc[u][0][4 * c] += xij.re;
                  acc[u][0][4 * c + 1] += xij.im;
                  acc[u][0][4 * c + 2] += xji.re;
                  acc[u][0][4 * c + 3] += xji.im;
                  acc[u][2][c] += Dr * v[18 + c];
                  acc[u][2][3 + c] += r * v[18 + c];
                }
#pragma unroll
                for (int q = 0; q < 6; ++q) {
                  acc[u][1][q] += Dr * v[12 + q];
                  acc[u][1][6 + q] += r * v[12 + q];
                }
              }
            }
          }
      }
    }
    // combine the splits of each item, part by part, in red[split][item][NP] over
    // the staging area, and add what each gives.  With G = sum g v (g = (D + i B)
    // r): velo_ij = -G(Im A) (+ for ji), ohc_ij = i (G(A) + w G(S)), ohc_ji = i (w
    // G(S) - G(A)), ohc_ii = i w G(S_ii); general V: ohc_ij is i times its own sum
#pragma unroll
    for (int third = 0; third < 3; ++third) {
      __syncthreads();
      if (act)
#pragma unroll
        for (int u = 0; u < IPT; ++u)
          if (iok[u])
#pragma unroll
            for (int q = 0; q < NP; ++q) st[(split * IW + slot + IWT * u) * NP + q] = acc[u][third][q];
      __syncthreads();
      for (int o = t; o < IW * 3; o += 256) {
        const int i2 = o / 3, c = o % 3;
        const int item = g0 + i2, hh = item % nhw, e2 = item / nhw;
        const zd wq = zd{b.hw[hh], b.eta};
        const double B = 2.0 * wq.re * wq.im;
        auto sum = [&](int q) {  // over the splits
          double s_ = 0.0;
          for (int u = 0; u < S; ++u) s_ += st[(u * IW + i2) * NP + q];
          return s_;
        };
        double* av = accp + L.velo + 2 * 9 * (hh + (int64_t)nhw * e2);
        double* ao = accp + L.ohc + 2 * 9 * (hh + (int64_t)nhw * e2);
        const int i = c == 2 ? 1 : 0, j = c == 0 ? 1 : 2;
        auto add = [](double* p, const zd& z, double sgn) {
          p[0] += sgn * z.re;
          p[1] += sgn * z.im;
        };
        if constexpr (HERM) {
          const zd x = zd{sum(c), B * sum(3 + c)};  // sum of g v
          if (third == 0) {                         // v = Im A
            add(av + 2 * (i + 3 * j), x, -1.0);
            add(av + 2 * (j + 3 * i), x, 1.0);
            add(ao + 2 * (i + 3 * j), x, -1.0);
            add(ao + 2 * (j + 3 * i), x, 1.0);
          } else {
            const zd iwZ = zmuli(zmul(wq, x));
            if (third == 1) {
              add(ao + 2 * (i + 3 * j), iwZ, 1.0);
              add(ao + 2 * (j + 3 * i), iwZ, 1.0);
            } else {
              add(ao + 2 * 4 * c, iwZ, 1.0);
            }
          }
        } else if (third == 0) {
          add(ao + 2 * (i + 3 * j), zmuli(zd{sum(4 * c), sum(4 * c + 1)}), 1.0);
          add(ao + 2 * (j + 3 * i), zmuli(zd{sum(4 * c + 2), sum(4 * c + 3)}), 1.0);
        } else if (third == 1) {
          const zd gr = zd{sum(2 * c), B * sum(6 + 2 * c)}, gi = zd{sum(2 * c + 1), B * sum(7 + 2 * c)};
          add(ao + 2 * 4 * c, zmuli(zmul(wq, zadd(gr, zmuli(gi)))), 1.0);
        } else {
          const zd x = zd{sum(c), B * sum(3 + c)};
          add(av + 2 * (i + 3 * j), x, -1.0);
          add(av + 2 * (j + 3 * i), x, 1.0);
        }
      }
    }
  }
}

// items per thread: four from eight items on (n = 96, 256 items: 2.8 ms, one
// 3.1; n = 20, 80 items: 0.50, 0.51); general V's 30 sums an item leave no
// registers for four, and two were slower (with 36 sums, n = 14, 16 items: 52
// us, one 40); one leaves room for three workgroups a CU
static int hwsum_ipt(const BandArgs& b) {
  return b.v_herm && (int64_t)b.n_hw * b.n_ef >= 8 ? 4 : 1;
}

// LDS of a record of `beside` doubles beside its Fermi levels
static size_t hwsum_lds(const BandArgs& b, int beside) {
  const size_t red = 256 * 24;  // the split reduction: 24 doubles a thread at most
  const size_t st = (size_t)HW_CH * (b.n_ef + beside);
  return sizeof(double) * ((size_t)b.n + (size_t)b.n_ef * b.n + 4 + (st > red ? st : red));
}
// (13 and 28 doubles are what the number of Fermi levels is limited by.  General V
// is launched with its own 22: 51 KB at three levels, three workgroups a CU.)
size_t hwsum_lds_bytes(const BandArgs& b) { return hwsum_lds(b, b.v_herm ? 13 : 28); }

// ===========================================================================
// Per-k Berry curvature at one Fermi level: out[k][i + 3j] = the k-point's
// term of kubo_ahc_tens (kubo.f90:37-78),
//   sum_n0 f(n0) sum_{n != n0} 2 Im(V_i(n0,n) V_j(n,n0)) / (E_n - E_n0)^2,
// one k-point per wavefront, the pairs spread over the lanes (any n).
// ===========================================================================
__global__ __launch_bounds__(64) void curv_kernel(int n, int64_t nk, const double* __restrict__ E,
                                                  const zd* __restrict__ V, double ef,
                                                  double Tsmear, int finiteT,
                                                  double* __restrict__ out) {
  const int lane = threadIdx.x;
  const int n2 = n * n;
  for (int64_t k = blockIdx.x; k < nk; k += gridDim.x) {
    const double* Ek = E + k * n;
    const zd* Vk = V + k * 3 * (int64_t)n2;
    double om[9];
#pragma unroll
    for (int q = 0; q < 9; ++q) om[q] = 0.0;
    for (int idx = lane; idx < n2; idx += 64) {
      const int n0 = idx % n, nn = idx / n;
      if (n0 == nn) continue;
      const double e0 = Ek[n0];
      const double f = finiteT ? 1.0 / (1.0 + exp((e0 - ef) / Tsmear)) : ((e0 < ef) ? 1.0 : 0.0);
      if (f == 0.0) continue;
      const double r = 1.0 / (e0 - Ek[nn]);
      const double w2 = 2.0 * f * r * r;
      zd x[3], y[3];
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        x[a] = Vk[a * (int64_t)n2 + n0 + (int64_t)n * nn];
        y[a] = Vk[a * (int64_t)n2 + nn + (int64_t)n * n0];
      }
#pragma unroll
      for (int j = 0; j < 3; ++j)
#pragma unroll
        for (int i = 0; i < 3; ++i) om[i + 3 * j] += w2 * zmul(x[i], y[j]).im;
    }
#pragma unroll
    for (int q = 0; q < 9; ++q) {
      const double v = wave_sum(om[q]);
      if (lane == 0) out[k * 9 + q] = v;
    }
  }
}

void launch_curv(hipStream_t s, int n, int64_t nk, const double* E, const zd* V, double ef,
                 double T_kelvin, double* out) {
  const double kB = 8.6173303 * 1e-5 / 27.211385;  // constants.f90:22
  unsigned grid = (unsigned)(nk < 65536 ? nk : 65536);
  hipLaunchKernelGGL(curv_kernel, dim3(grid), dim3(64), 0, s, n, nk, E, V, ef, kB * T_kelvin,
                     T_kelvin > 1e-2 ? 1 : 0, out);
}

// acc[c] = sum over the nblocks partial records of part[g][c], for one or two
// sets of records (len2 = 0: one).  A workgroup takes 16 consecutive c (128
// bytes of a record); thread (r, c) sums the records r, r + 64, ... with up to
// 16 loads in flight, and the 64 row sums are added in two steps of fixed
// order, so the result is deterministic.  Latency-bound at the usual record of
// a few hundred sums, which is why the columns are spread over many
// workgroups: 505 sums of 1,024 records 9 us (64 columns a workgroup, one
// load in flight: 21 to 33).
constexpr int RP_COLS = 16, RP_ROWS = 64;
__global__ __launch_bounds__(RP_COLS * RP_ROWS) void reduce_parts_kernel(
    int nblocks, int64_t len, const double* __restrict__ part, double* __restrict__ acc,
    int64_t len2, const double* __restrict__ part2, double* __restrict__ acc2) {
  __shared__ double ws[RP_ROWS][RP_COLS + 1];
  const int col = threadIdx.x % RP_COLS, row = threadIdx.x / RP_COLS;
  const int64_t nb1 = (len + RP_COLS - 1) / RP_COLS;
  int64_t blk = blockIdx.x;
  if (blk >= nb1) {
    blk -= nb1;
    len = len2;
    part = part2;
    acc = acc2;
  }
  const int64_t c = blk * RP_COLS + col;
  double s = 0.0;
  if (c < len) {
    double v[16];
    for (int g0 = row; g0 < nblocks; g0 += 16 * RP_ROWS) {
#pragma unroll
      for (int u = 0; u < 16; ++u) {
        const int g = g0 + u * RP_ROWS;
        v[u] = g < nblocks ? part[(int64_t)g * len + c] : 0.0;
      }
#pragma unroll
      for (int u = 0; u < 16; ++u) s += v[u];
    }
  }
  ws[row][col] = s;
  __syncthreads();
  double t = 0.0;
  if (row < 8) {
#pragma unroll
    for (int v = 0; v < 8; ++v) t += ws[row * 8 + v][col];
  }
  __syncthreads();
  if (row < 8) ws[row][col] = t;
  __syncthreads();
  if (row == 0 && c < len) {
    double r = 0.0;
#pragma unroll
    for (int v = 0; v < 8; ++v) r += ws[v][col];
    acc[c] = r;
  }
}

// ===========================================================================
// n <= 32, no magnetoelectric sums, up to HALL_EF Fermi levels, V in memory:
// N_el, kubo_ahc_tens and, for a single (hw, E_F), velo_ahc_tens and
// kubo_ohc_tens, over the pairs x < y of as many k-points at a time as fill the
// workgroup, one pair a thread.  Every sum is over pairs, so it stays in the
// thread's registers over all k-points and is reduced once: no per-band tables,
// and only the occupations go through LDS.  With P_ij = V_i(y, x) V_j(x, y),
// A_c = P_ij - P_ji and S_ij = P_ij + P_ji, the curvatures of x and y give
//   ahc_ij = sum ((f_x + f_y) Im S_ij - (f_x - f_y) Im A_c) / dE^2   (ji: + A)
// and the velo / ohc sums are hwsum_kernel's.  General V: nothing is assumed of
// V(y, x).
// Bound by the reads of V and by VALU issue (at 8 bands, 32,768 k-points: 31 us for
// 100 MB, VALU 0.59 of the SIMD-cycles; the band-sum kernel, with three of its
// wavefronts waiting on the fourth's shuffles, 411).
// Several Fermi levels cost 9 sums each: from HALL_EF on, the band-sum kernel.
// ===========================================================================
constexpr int HALL_EF = 4, HALL_KB = 32;

template <int NEF, bool PMODE>
__global__ __launch_bounds__(256, 2) void hall_kernel(BandArgs b, double Tsmear, AccLayout L,
                                                      int64_t nk, const double* __restrict__ E,
                                                      const zd* __restrict__ V,
                                                      const double* __restrict__ w,
                                                      double* __restrict__ part) {
  static_assert(!PMODE || NEF == 1, "");
  constexpr int NA = 9 * NEF, NQ = PMODE ? 30 : 0;
  __shared__ double Es[128], fd[NEF * 128], wks[HALL_KB], red[4 * (NA + NQ + NEF)];
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  const int n = b.n, n2 = n * n, npair = n * (n - 1) / 2;
  const bool finiteT = b.T_kelvin > 1e-2, doAHC = (b.jobs & MEP_JOB_AHC) != 0;
  // k-points at a time: KB n <= 128
  int KB = npair ? 256 / npair : HALL_KB;
  KB = KB < 1 ? 1 : KB > HALL_KB ? HALL_KB : KB;
  const double wr = b.hw[0], eta2 = b.eta * b.eta;
  // per level: S (3), A (3), S_ii (3); the ohc sums (6, complex), then D q v and
  // q v of S_ii and of Im A
  double ah[NA], pv[NQ + 1], ne[NEF];
#pragma unroll
  for (int q = 0; q < NA; ++q) ah[q] = 0.0;
#pragma unroll
  for (int q = 0; q < NQ; ++q) pv[q] = 0.0;
#pragma unroll
  for (int e = 0; e < NEF; ++e) ne[e] = 0.0;
  for (int64_t k0 = (int64_t)blockIdx.x * KB; k0 < nk; k0 += (int64_t)gridDim.x * KB) {
    const int kb = nk - k0 < KB ? (int)(nk - k0) : KB;
    __syncthreads();
    for (int c = t; c < kb * n; c += 256) {
      const double e = E[k0 * n + c], wk = w ? w[k0 + c / n] : 1.0;
      Es[c] = e;
#pragma unroll
      for (int ef = 0; ef < NEF; ++ef) {
        double f;
        if (b.fd_in) f = b.fd_in[(k0 * n + c) * NEF + ef];
        else f = finiteT ? 1.0 / (1.0 + exp((e - b.ef[ef]) / Tsmear)) : ((e < b.ef[ef]) ? 1.0 : 0.0);
        fd[c * NEF + ef] = f;
        ne[ef] += wk * f;
      }
      if (c % n == 0) wks[c / n] = wk;
    }
    __syncthreads();
    if (!doAHC) continue;
    for (int c = t; c < kb * npair; c += 256) {
      const int kk = c / npair, p = c - kk * npair;
      // pair x < y, p = x + y (y - 1) / 2
      int y = (int)((sqrtf(8.0f * (float)p + 1.0f) + 1.0f) * 0.5f);
      if (y * (y + 1) / 2 <= p) ++y;
      if (y * (y - 1) / 2 > p) --y;
      const int x = p - y * (y - 1) / 2;
      const zd* Vk = V + (k0 + kk) * 3 * (int64_t)n2;
      zd vxy[3], vyx[3];
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        vxy[a] = Vk[a * n2 + x + n * y];
        vyx[a] = Vk[a * n2 + y + n * x];
      }
      const double wk = wks[kk], dE = Es[kk * n + x] - Es[kk * n + y], r = 1.0 / dE;
      const double* fx = fd + (kk * n + x) * NEF;
      const double* fy = fd + (kk * n + y) * NEF;
      zd A[3], S[3], Sd[3];
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        const int i = q == 2 ? 1 : 0, j = q == 0 ? 1 : 2;
        const zd pij = zmul(vyx[i], vxy[j]), pji = zmul(vyx[j], vxy[i]);
        A[q] = zsub(pij, pji);
        S[q] = zadd(pij, pji);
        Sd[q] = zscale(zmul(vyx[q], vxy[q]), 2.0);
      }
      const double wr2 = wk * (r * r);
#pragma unroll
      for (int ef = 0; ef < NEF; ++ef) {
        const double s = wr2 * (fx[ef] + fy[ef]), d = wr2 * (fx[ef] - fy[ef]);
#pragma unroll
        for (int q = 0; q < 3; ++q) {
          ah[9 * ef + q] += s * S[q].im;
          ah[9 * ef + 3 + q] += d * A[q].im;
          ah[9 * ef + 6 + q] += s * Sd[q].im;
        }
      }
      if constexpr (PMODE) {
        // selects drop pairs of equal occupation
        const double f = fx[0] - fy[0];
        const bool on = f != 0.0;
        const double D1 = dE - wr, D2 = dE + wr, D = D1 * D2 + eta2;
        const double m1 = D1 * D1 + eta2, m2 = D2 * D2 + eta2;
        const double g = on ? wk * f * rcp_nr(m1 * m2) : 0.0, Dg = D * g;
        const double rs = on ? r : 0.0, gr = g * rs, Dgr = Dg * rs;
        const double t1 = gr * m2, t2 = gr * m1;
        const zd w1 = zd{D1 * t1, b.eta * t1}, w2 = zd{D2 * t2, -b.eta * t2};
#pragma unroll
        for (int q = 0; q < 3; ++q) {
          const int i = q == 2 ? 1 : 0, j = q == 0 ? 1 : 2;
          const zd pij = zmul(vyx[i], vxy[j]), pji = zmul(vyx[j], vxy[i]);
          const zd xij = zsub(zmul(w1, pij), zmul(w2, pji));
          const zd xji = zsub(zmul(w1, pji), zmul(w2, pij));
          pv[4 * q] += xij.re;
          pv[4 * q + 1] += xij.im;
          pv[4 * q + 2] += xji.re;
          pv[4 * q + 3] += xji.im;
          pv[12 + 2 * q] += Dgr * Sd[q].re;
          pv[13 + 2 * q] += Dgr * Sd[q].im;
          pv[18 + 2 * q] += gr * Sd[q].re;
          pv[19 + 2 * q] += gr * Sd[q].im;
          pv[24 + q] += Dg * A[q].im;
          pv[27 + q] += g * A[q].im;
        }
      }
    }
  }
  // the workgroup's sums, wavefront by wavefront
  constexpr int NR = NA + NQ + NEF;
  auto put = [&](int q, double v) {
    v = rows4_sum(row16_sum(v));
    if (lane == 0) red[wv * NR + q] = v;
  };
#pragma unroll
  for (int q = 0; q < NA; ++q) put(q, ah[q]);
#pragma unroll
  for (int q = 0; q < NQ; ++q) put(NA + q, pv[q]);
#pragma unroll
  for (int q = 0; q < NEF; ++q) put(NA + NQ + q, ne[q]);
  __syncthreads();
  auto R = [&](int q) { return ((red[q] + red[NR + q]) + red[2 * NR + q]) + red[3 * NR + q]; };
  double* out = part + (int64_t)blockIdx.x * L.total;
  if (t < NEF) out[L.Ne + t] += R(NA + NQ + t);
  if (doAHC && t < 9 * NEF) {
    const int ef = t / 9, i = t % 3, j = t / 3 % 3, c = i + j - 1;
    double v;
    if (i == j) v = R(9 * ef + 6 + i);
    else v = i < j ? R(9 * ef + c) - R(9 * ef + 3 + c) : R(9 * ef + c) + R(9 * ef + 3 + c);
    out[L.ahc + t] += v;
  }
  if (PMODE && doAHC && t >= 64 && t < 73) {
    const int o = t - 64, i = o % 3, j = o / 3, c = i + j - 1;
    const zd wq = zd{wr, b.eta};
    const double B = 2.0 * wr * b.eta;
    zd av = zd{0.0, 0.0}, ao;
    if (i == j) {  // i w sum g S_ii / dE
      const zd gr = zd{R(NA + 12 + 2 * i), B * R(NA + 18 + 2 * i)};
      const zd gi = zd{R(NA + 13 + 2 * i), B * R(NA + 19 + 2 * i)};
      ao = zmuli(zmul(wq, zadd(gr, zmuli(gi))));
    } else {
      const zd gi = zd{R(NA + 24 + c), B * R(NA + 27 + c)};  // sum g Im A
      const int q = NA + 4 * c + (i < j ? 0 : 2);
      av = i < j ? zd{-gi.re, -gi.im} : gi;
      ao = zmuli(zd{R(q), R(q + 1)});
    }
    out[L.velo + 2 * o] += av.re;
    out[L.velo + 2 * o + 1] += av.im;
    out[L.ohc + 2 * o] += ao.re;
    out[L.ohc + 2 * o + 1] += ao.im;
  }
}

static bool hall_only(const BandArgs& b) {
  return b.n <= 32 && b.n_ef <= HALL_EF && !(b.jobs & (MEP_JOB_KUBO | MEP_JOB_MEP));
}

// n <= 32: the Hall and optical conductivities of several (hw, E_F) items
// (velo_ahc_tens / kubo_ohc_tens over a frequency list or several Fermi
// levels) run in hwsum_kernel, every item on its own threads, reading V
// from HBM; the single-item sums stay in the band-sum kernel's pair phase
static bool hw_many(const BandArgs& b) {
  return (b.jobs & MEP_JOB_AHC) && (int64_t)b.n_hw * b.n_ef > 1;
}

// The n <= 32 kernel's accumulators in LDS: the record's layout, with drop
// without the velo / ohc block (which hwsum_kernel fills, or nobody); *gap is
// the length of the block left out
static AccLayout lds_layout(const AccLayout& L, bool drop, int64_t* gap) {
  AccLayout S = L;
  *gap = 0;
  if (drop) {
    *gap = L.kic - L.velo;
    S.ohc = L.velo;
    S.kic -= *gap; S.klc -= *gap; S.kcs -= *gap;
    S.nic -= *gap; S.nlc -= *gap; S.ncs -= *gap;
    S.total -= *gap;
  }
  return S;
}

// the velo / ohc block is not the band-sum kernel's to fill
static bool bs_drop(const BandArgs& b) { return hw_many(b) || !(b.jobs & MEP_JOB_AHC); }

template <int NMAX, bool FUSED, bool HERM>
static void launch_bs(hipStream_t s, const BandArgs& b, double Tsmear, const AccLayout& L,
                      int64_t nk, const double* E, const zd* V, const zd* A, const zd* Om,
                      const double* w, int nblocks, double* part, const VeloFuse* f) {
  int64_t gap;
  const AccLayout S = lds_layout(L, bs_drop(b), &gap);
  size_t lds = BsLds<NMAX, HERM>::bytes(b.n_ef, S.total);
  (void)hipFuncSetAttribute((const void*)bandsum_kernel<NMAX, FUSED, HERM>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  hipLaunchKernelGGL((bandsum_kernel<NMAX, FUSED, HERM>), dim3(nblocks), dim3(BS_THREADS), lds, s,
                     b, Tsmear, S, gap, nk, E, V, A, Om, w, part, f ? f->Hk : nullptr,
                     f ? f->strideHk : (int64_t)0, f ? f->U : nullptr);
}

size_t bandsum_lds_bytes(const BandArgs& b) {
  AccLayout L = acc_layout(b);
  if (b.n > 32) {
    const size_t a = bandsum_wide_lds_bytes(b), h = hwsum_lds_bytes(b);
    return a > h ? a : h;
  }
  int64_t gap;
  const AccLayout S = lds_layout(L, hw_many(b), &gap);
  size_t a = bs_limit_bytes(b.n <= 16 ? 16 : 32, b.n_ef, S.total);
  // never less than launch_bs asks for
  const AccLayout K = lds_layout(L, bs_drop(b), &gap);
  const size_t k = b.n <= 16 ? (b.v_herm ? BsLds<16, true>::bytes(b.n_ef, K.total)
                                         : BsLds<16, false>::bytes(b.n_ef, K.total))
                             : (b.v_herm ? BsLds<32, true>::bytes(b.n_ef, K.total)
                                         : BsLds<32, false>::bytes(b.n_ef, K.total));
  if (k > a) a = k;
  const size_t h = hw_many(b) ? hwsum_lds_bytes(b) : 0;
  return a > h ? a : h;
}

// the velocities formed inside the band-sum kernel never reach HBM, which
// hwsum_kernel reads
bool bandsum_can_fuse(const BandArgs& b) {
  return b.n > 16 && b.n <= 32 && b.v_herm && !b.pos_op && !hw_many(b);
}

static void launch_hwsum(hipStream_t s, const BandArgs& b, double Tsmear, const AccLayout& L,
                         int64_t nk, const double* E, const zd* V, const double* w, int nblocks,
                         double* part) {
  const size_t lh = b.v_herm ? hwsum_lds_bytes(b) : hwsum_lds(b, 1 + hw_vals<false>());
  auto go = [&](auto kernel) {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lh);
    hipLaunchKernelGGL(kernel, dim3(nblocks), dim3(256), lh, s, b, Tsmear, L, nk, E, V, w, part);
  };
  if (!b.v_herm) go(hwsum_kernel<false, 1>);
  else if (hwsum_ipt(b) == 4) go(hwsum_kernel<true, 4>);
  else go(hwsum_kernel<true, 1>);
}

void launch_bandsum(hipStream_t s, const BandArgs& b, int64_t nk, const double* E, const zd* V,
                    const zd* A, const zd* Om, const double* w, int nblocks, double* part,
                    const VeloFuse* fuse, zd* wide_scr) {
  AccLayout L = acc_layout(b);
  // kBoltz_Eh_K * T  (constants.f90:22, statistics.f90:77)
  const double kB = 8.6173303 * 1e-5 / 27.211385;
  double Tsmear = kB * b.T_kelvin;
  if (b.n > 32) {
    const size_t lds = bandsum_wide_lds_bytes(b);
    auto go = [&](auto kernel) {
      (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
      hipLaunchKernelGGL(kernel, dim3(nblocks), dim3(256), lds, s, b, Tsmear, L, nk, E, V, w, part,
                         wide_scr, A, Om);
    };
    if (b.v_herm) go(bandsum_wide_kernel<true>);
    else go(bandsum_wide_kernel<false>);
    // the single (hw, E_F) of a Hermitian V is summed in the pair phase
    if (hw_many(b) || ((b.jobs & MEP_JOB_AHC) && !b.v_herm))
      launch_hwsum(s, b, Tsmear, L, nk, E, V, w, nblocks, part);
  } else {
    if (!fuse && hall_only(b)) {
      auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(nblocks), dim3(256), 0, s, b, Tsmear, L, nk, E, V, w, part);
      };
      if (b.n_ef == 1 && !hw_many(b)) go(hall_kernel<1, true>);
      else if (b.n_ef == 1) go(hall_kernel<1, false>);
      else if (b.n_ef == 2) go(hall_kernel<2, false>);
      else if (b.n_ef == 3) go(hall_kernel<3, false>);
      else go(hall_kernel<4, false>);
    } else if (b.n <= 16) {
      if (b.v_herm) launch_bs<16, false, true>(s, b, Tsmear, L, nk, E, V, A, Om, w, nblocks, part, nullptr);
      else launch_bs<16, false, false>(s, b, Tsmear, L, nk, E, V, A, Om, w, nblocks, part, nullptr);
    } else if (fuse) {
      launch_bs<32, true, true>(s, b, Tsmear, L, nk, E, V, A, Om, w, nblocks, part, fuse);
    } else {
      if (b.v_herm) launch_bs<32, false, true>(s, b, Tsmear, L, nk, E, V, A, Om, w, nblocks, part, nullptr);
      else launch_bs<32, false, false>(s, b, Tsmear, L, nk, E, V, A, Om, w, nblocks, part, nullptr);
    }
    if (hw_many(b)) launch_hwsum(s, b, Tsmear, L, nk, E, V, w, nblocks, part);
  }
}

void launch_reduce_parts(hipStream_t s, int nblocks, int64_t len, const double* part, double* acc,
                         int64_t len2, const double* part2, double* acc2) {
  const int64_t nb = (len + RP_COLS - 1) / RP_COLS + (len2 + RP_COLS - 1) / RP_COLS;
  hipLaunchKernelGGL(reduce_parts_kernel, dim3((unsigned)nb), dim3(RP_COLS * RP_ROWS), 0, s, nblocks,
                     len, part, acc, len2, part2, acc2);
}

__global__ void fill_zero_kernel(double* __restrict__ p, int64_t n) {
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0.0;
}

void launch_fill_zero(hipStream_t s, double* p, int64_t n) {
  int64_t nb = (n + 255) / 256;
  hipLaunchKernelGGL(fill_zero_kernel, dim3((unsigned)nb), dim3(256), 0, s, p, n);
}
