// mep_velo.hip -- velocity (and connection / curvature) in the Hamiltonian
// gauge.
//
// Replaces W_to_H_gaugeTRAFO + get_velo (wann_interp.f90:100-101, 406-658).
// Inputs per k: the Fourier GEMM output in the Wannier gauge, stacked as
//   mat 0: H, 1-3: dH_a, [4-6: A_a, 7-9: Omega_yz, Omega_zx, Omega_xy]
// plus U (eigenvectors) and E.  The tight-binding phase of the reference's
// convention (wann_interp.f90:192-241) is applied on load:
//   X'_nm = e^{2 pi i k.(tau_m - tau_n)} X_nm,
//   dH'_a = ph (dH_a + i c_a(tau_m - tau_n) H),
//   Om'_ab = ph (Om_ab + i c_a(dtau) A_b - i c_b(dtau) A_a).
// Output: V per k planar, V[k][a][i + n j]; with a position operator also
// A^(H) (3,n,n) and Omega^(H) (3,3,n,n) in the reference layout.
#include "mep_common.hpp"
#include "mep_kernels.hpp"
#include "mep_mfma.hpp"
#include "mep_lane.hpp"

struct TBPhase {
  double kx, ky, kz;
  const double* kpts;
  const double* tau;
  double cm[9];
  __device__ inline TBPhase at(int64_t k) const {
    TBPhase r = *this;
    r.kx = kpts[3 * k];
    r.ky = kpts[3 * k + 1];
    r.kz = kpts[3 * k + 2];
    return r;
  }
  __device__ inline zd phase(int n, int m, double dtau[3]) const {
    dtau[0] = tau[3 * m] - tau[3 * n];
    dtau[1] = tau[3 * m + 1] - tau[3 * n + 1];
    dtau[2] = tau[3 * m + 2] - tau[3 * n + 2];
    const double two_pi = 2.0 * 3.14159265358979323846;
    double ang = two_pi * (kx * dtau[0] + ky * dtau[1] + kz * dtau[2]);
    double sn, cs;
    sincos(ang, &sn, &cs);
    return zd{cs, sn};
  }
  // c_a(dt) = sum_b cm[a][b] dt_b, with a selected without indexing cm
  __device__ inline double c(int a, const double dt[3]) const {
    double c0 = cm[0] * dt[0] + cm[1] * dt[1] + cm[2] * dt[2];
    double c1 = cm[3] * dt[0] + cm[4] * dt[1] + cm[5] * dt[2];
    double c2 = cm[6] * dt[0] + cm[7] * dt[1] + cm[8] * dt[2];
    return a == 0 ? c0 : (a == 1 ? c1 : c2);
  }
};

// f_m and the centres of a workgroup's k-point into LDS (threads t < n)
__device__ inline void pos_phases(const TBPhase& tb, int n, int t, zd* f, double* tau) {
  if (!tb.tau || t >= n) return;
  const double* tm = tb.tau + 3 * t;
  double sn, cs;
  sincos(2.0 * 3.14159265358979323846 * (tb.kx * tm[0] + tb.ky * tm[1] + tb.kz * tm[2]), &sn, &cs);
  f[t] = zd{cs, sn};
#pragma unroll
  for (int a = 0; a < 3; ++a) tau[3 * t + a] = tm[a];
}
// Wannier-gauge element (row, col) of matrix `mat`: full column-major
// matrices of N x N, or (packed) the upper triangles of Hermitian matrices
// with (i <= j) at i + j(j+1)/2 and the lower half as conjugates.  HT is the
// stored complex type (FP64, or FP32 from the mixed-precision GEMM).
__device__ inline zd up64(zd x) { return x; }
__device__ inline zd up64(zf x) { return zd{(double)x.re, (double)x.im}; }
template <class HT>
__device__ inline zd load_w(const HT* X, int N, int packed, int row, int col, int mat) {
  if (!packed) return up64(X[(int64_t)mat * N * N + row + (int64_t)N * col]);
  const int64_t NP = ((int64_t)N * (N + 1)) / 2;
  if (row <= col) return up64(X[mat * NP + row + ((int64_t)col * (col + 1)) / 2]);
  return zconj(up64(X[mat * NP + col + ((int64_t)row * (row + 1)) / 2]));
}

// element (row, col) of mat `mat` after the TB epilogue (mats 0..9 as above)
template <class HT>
__device__ inline zd load_tb(const HT* X, int packed, int N, int row, int col, int mat,
                             const TBPhase& tb) {
  zd x = load_w(X, N, packed, row, col, mat);
  if (!tb.tau) return x;
  double dt[3];
  zd ph = tb.phase(row, col, dt);
  if (mat >= 1 && mat <= 3) {
    zd h = load_w(X, N, packed, row, col, 0);
    x = zadd(x, zmuli(zscale(h, tb.c(mat - 1, dt))));
  } else if (mat >= 7) {
    // Omega_ab with (a,b) = (1,2), (2,0), (0,1)
    int a = (mat == 7) ? 1 : (mat == 8) ? 2 : 0;
    int b = (mat == 7) ? 2 : (mat == 8) ? 0 : 1;
    zd Ab = load_w(X, N, packed, row, col, 4 + b), Aa = load_w(X, N, packed, row, col, 4 + a);
    x = zadd(x, zmuli(zsub(zscale(Ab, tb.c(a, dt)), zscale(Aa, tb.c(b, dt)))));
  }
  return zmul(ph, x);
}

// --------------------------------------------------------------------------
// no position operator: V_a = U^H dH_a U for the three directions, or
// V_a = dH_a without the gauge transformation.  V is written planar:
// V[k][a][i + n*j].
//
// One k-point per 256-thread workgroup; the waves own the 2 x 2 output
// tiles of 16 x 16.  U and the three dH_a are staged in LDS (dH_a is
// Hermitian: its packed upper triangle is read once, coalesced, and both
// halves are written).  T_a = dH_a U is formed in registers for all three a
// (nine MFMA chains: three real products per complex one), written over
// dH_a, and V_a = U^H T_a goes from the accumulators straight to HBM.
// LDS rows and columns >= n stay zero, so no operand load is guarded.
// --------------------------------------------------------------------------
template <class HT>
__global__ __launch_bounds__(256, 2) void velo_mfma_kernel(int n, int64_t nk,
                                                           const HT* __restrict__ Hk,
                                                           int64_t strideHk, int packed,
                                                           TBPhase tb0, int gauge_trafo,
                                                           const zd* __restrict__ U,
                                                           zd* __restrict__ V) {
  constexpr int NM = 32, LD = NM + 1, PL = NM * LD;
  __shared__ zd Us[PL], Ds[3 * PL];
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  const int n2 = n * n;
  const int np = packed ? n * (n + 1) / 2 : n2;
  for (int c = t; c < PL; c += 256) Us[c] = zd{0.0, 0.0};
  for (int c = t; c < 3 * PL; c += 256) Ds[c] = zd{0.0, 0.0};
  const int r0 = 16 * (w & 1), c0 = 16 * (w >> 1);
  const int ar = r0 + (lane & 15), bc = c0 + (lane & 15), kq = lane >> 4;
  const bool tile = r0 < n && c0 < n;  // wave-uniform
  for (int64_t k = blockIdx.x; k < nk; k += gridDim.x) {
    const TBPhase tb = tb0.at(k);
    const HT* X = Hk + k * strideHk;
    zd* Vk = V + k * 3 * (int64_t)n2;
    __syncthreads();  // the previous k-point's readers are done
    // ---- stage: every global load of the k-point before the LDS stores
    {
      constexpr int NU = (NM * NM + 255) / 256, ND = (NM * (NM + 1) / 2 + 255) / 256;
      zd ut[NU], dt[3][ND], ht[ND];
#pragma unroll
      for (int u = 0; u < NU; ++u) {
        const int idx = t + 256 * u;
        ut[u] = (gauge_trafo && idx < n2) ? U[k * (int64_t)n2 + idx] : zd{0.0, 0.0};
      }
      // element p of the packed upper triangle: (i, j), i <= j, p = i + j(j+1)/2
      int pi[ND], pj[ND];
#pragma unroll
      for (int u = 0; u < ND; ++u) {
        const int p = t + 256 * u;
        int j = (int)((sqrtf(8.0f * (float)p + 1.0f) - 1.0f) * 0.5f);
        if ((j + 1) * (j + 2) / 2 <= p) ++j;
        if (j * (j + 1) / 2 > p) --j;
        pj[u] = j;
        pi[u] = p - j * (j + 1) / 2;
      }
      if (packed) {
        const int64_t NPk = np;
#pragma unroll
        for (int u = 0; u < ND; ++u) {
          const int p = t + 256 * u;
          const bool ok = p < np;
#pragma unroll
          for (int a = 0; a < 3; ++a) dt[a][u] = ok ? up64(X[(1 + a) * NPk + p]) : zd{0.0, 0.0};
          ht[u] = (ok && tb.tau) ? up64(X[p]) : zd{0.0, 0.0};
        }
      }
#pragma unroll
      for (int u = 0; u < NU; ++u) {
        const int idx = t + 256 * u;
        if (idx < n2) Us[idx % n + LD * (idx / n)] = ut[u];
      }
      if (packed) {
#pragma unroll
        for (int u = 0; u < ND; ++u) {
          const int p = t + 256 * u;
          if (p >= np) continue;
          const int i = pi[u], j = pj[u];
          zd ph = zd{1.0, 0.0};
          double dtau[3] = {0.0, 0.0, 0.0};
          if (tb.tau) ph = tb.phase(i, j, dtau);
#pragma unroll
          for (int a = 0; a < 3; ++a) {
            // dH'_a(i, j) = e^{2 pi i k.(tau_j - tau_i)} (dH_a + i c_a(tau_j - tau_i) H)
            zd x = dt[a][u];
            if (tb.tau) x = zmul(ph, zadd(x, zmuli(zscale(ht[u], tb.c(a, dtau)))));
            Ds[a * PL + j + LD * i] = zconj(x);
            Ds[a * PL + i + LD * j] = x;  // last: the diagonal keeps x as stored
          }
        }
      } else {
        for (int a = 0; a < 3; ++a)
          for (int idx = t; idx < n2; idx += 256) {
            const int i = idx % n, j = idx / n;
            Ds[a * PL + i + LD * j] = load_tb(X, 0, n, i, j, 1 + a, tb);
          }
      }
    }
    __syncthreads();
    if (!gauge_trafo) {
      for (int a = 0; a < 3; ++a)
        for (int idx = t; idx < n2; idx += 256)
          Vk[a * (int64_t)n2 + idx] = Ds[a * PL + idx % n + LD * (idx / n)];
      continue;
    }
    // ---- T_a = dH_a U (C = sum_m A(., m) B(m, .): P1 = Ar Br, P2 = Ai Bi,
    // P3 = (Ar + Ai)(Br + Bi); Re C = P1 - P2, Im C = P3 - P1 - P2)
    mep_v4d p1[3], p2[3], p3[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) p1[a] = p2[a] = p3[a] = mep_v4d{0, 0, 0, 0};
    if (tile)
#pragma unroll
      for (int k0 = 0; k0 < NM; k0 += 4) {
        if (k0 >= n) break;
        const int m = k0 + kq;
        const zd b = Us[m + LD * bc];
        const double bs = b.re + b.im;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          const zd x = Ds[a * PL + ar + LD * m];
          p1[a] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.re, b.re, p1[a], 0, 0, 0);
          p2[a] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.im, b.im, p2[a], 0, 0, 0);
          p3[a] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.re + x.im, bs, p3[a], 0, 0, 0);
        }
      }
    __syncthreads();  // every wave has read dH
    if (tile)
#pragma unroll
      for (int a = 0; a < 3; ++a)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int row = r0 + kq + 4 * v;
          Ds[a * PL + row + LD * bc] = zd{p1[a][v] - p2[a][v], p3[a][v] - p1[a][v] - p2[a][v]};
        }
    __syncthreads();
    // ---- V_a = U^H T_a, A(row, m) = conj(U(m, row))
#pragma unroll
    for (int a = 0; a < 3; ++a) p1[a] = p2[a] = p3[a] = mep_v4d{0, 0, 0, 0};
    if (tile) {
#pragma unroll
      for (int k0 = 0; k0 < NM; k0 += 4) {
        if (k0 >= n) break;
        const int m = k0 + kq;
        const zd u = Us[m + LD * ar];
        const double us = u.re - u.im;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          const zd y = Ds[a * PL + m + LD * bc];
          p1[a] = __builtin_amdgcn_mfma_f64_16x16x4f64(u.re, y.re, p1[a], 0, 0, 0);
          p2[a] = __builtin_amdgcn_mfma_f64_16x16x4f64(-u.im, y.im, p2[a], 0, 0, 0);
          p3[a] = __builtin_amdgcn_mfma_f64_16x16x4f64(us, y.re + y.im, p3[a], 0, 0, 0);
        }
      }
      if (bc < n)
#pragma unroll
        for (int a = 0; a < 3; ++a)
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const int row = r0 + kq + 4 * v;
            if (row < n)
              Vk[a * (int64_t)n2 + row + (int64_t)n * bc] =
                  zd{p1[a][v] - p2[a][v], p3[a][v] - p1[a][v] - p2[a][v]};
          }
    }
  }
}

// --------------------------------------------------------------------------
// 32 < n <= 128, no position operator: V_a = U^H dH_a U on FP64 MFMA, three
// real products per complex one, operands from L2.
// --------------------------------------------------------------------------
typedef double velo_v4d __attribute__((ext_vector_type(4)));

// The tight-binding epilogue of the packed dH_a, in place, with one sincos a
// band: dH'_a(i, j) = conj(f_i) f_j (dH_a + i c_a(tau_j - tau_i) H), f_m =
// e^{2 pi i k.tau_m}.  One k-point per workgroup.
__global__ __launch_bounds__(256) void velo_tb_kernel(int n, int64_t nk, zd* __restrict__ Hk,
                                                      int64_t strideHk, TBPhase tb0) {
  __shared__ zd f[128];
  __shared__ double tau[3 * 128];
  const int t = threadIdx.x;
  const int np = n * (n + 1) / 2;
  for (int64_t k = blockIdx.x; k < nk; k += gridDim.x) {
    const TBPhase tb = tb0.at(k);
    zd* X = Hk + k * strideHk;
    __syncthreads();
    pos_phases(tb, n, t, f, tau);
    __syncthreads();
    for (int p = t; p < np; p += 256) {
      // p = i + j (j + 1) / 2
      int j = (int)((sqrtf(8.0f * (float)p + 1.0f) - 1.0f) * 0.5f);
      if ((j + 1) * (j + 2) / 2 <= p) ++j;
      if (j * (j + 1) / 2 > p) --j;
      const int i = p - j * (j + 1) / 2;
      const double dt[3] = {tau[3 * j] - tau[3 * i], tau[3 * j + 1] - tau[3 * i + 1],
                            tau[3 * j + 2] - tau[3 * i + 2]};
      const zd ph = zcmul(f[i], f[j]), h = X[p];
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        zd* x = X + (int64_t)(1 + a) * np + p;
        *x = zmul(ph, zadd(*x, zmuli(zscale(h, tb.c(a, dt)))));
      }
    }
  }
}

// A wavefront forms 16 columns of V (one of NT column tiles, 16 (NT - 1) < n <=
// 16 NT).  T_a = dH_a U of its columns stays in its registers: the accumulator
// of a tile (row lane / 16 + 4 v, column lane % 16) is the B operand of the
// second product's steps as it stands, so T_a goes through neither LDS nor
// memory and there is no barrier.  V_a = U^H T_a is Hermitian: the wavefront of
// column tile c forms the row tiles c, c + 1, ... c + NT / 2 (mod NT), every
// pair of tiles once and as many for each wavefront, and writes each
// off-diagonal one twice.  dH_a is read from its packed upper triangle: below
// the diagonal as conj dH_a(m, row), known per step outside the diagonal tile.
// REG: the columns of U as well in registers, which takes half of the first
// product's loads away (up to 64 bands; above, they would spill: n = 96 took
// 2.4 ms so against 1.9).
// The wavefronts of one k-point follow each other on one XCD (workgroup index
// mod 8), so that dH_a and U come from its L2 after the first.  Bound by the
// operand loads: MFMA 0.57 (n = 44) and 0.46 (n = 96, where 12 GB come from beyond
// L2 at 6.3 TB/s) of the SIMD-cycles at two wavefronts a SIMD; three with spills took 1.2 and 2.6 ms, two columns a
// wavefront at one wavefront a SIMD 1.1 and 2.0.
// n = 44, 9,261 k-points: 0.70 ms (U and one component at a time in LDS, T_a
// through memory: 1.42); n = 96, 2,744: 1.92 ms (T_a through memory: 4.07).
template <int NT, bool REG>
__global__ __launch_bounds__(64, 2) void velo_wide_kernel(
    int n, int64_t nk, const zd* __restrict__ Hk, int64_t strideHk, int gauge_trafo,
    const zd* __restrict__ U, zd* __restrict__ V) {
  const int lane = threadIdx.x, lr = lane & 15, kq = lane >> 4;
  const int n2 = n * n, np = n * (n + 1) / 2;
  const int64_t slots = (nk + 7) / 8 * NT;
  constexpr int NS = 4 * NT;                      // steps of four
  constexpr int GS = NT >= 7 ? 2 : 4, NQ = NS / GS;  // a group's loads are one group ahead
  for (int64_t slot = blockIdx.x >> 3; slot < slots; slot += gridDim.x >> 3) {
    const int64_t k = slot / NT * 8 + (blockIdx.x & 7);
    const int c = (int)(slot % NT), bc = 16 * c + lr;
    if (k >= nk) break;
    const zd* X0 = Hk + k * strideHk + np;
    const zd* Uk = U + k * (int64_t)n2;
    zd* Vk = V + k * 3 * (int64_t)n2;
    if (!gauge_trafo) {
      for (int idx = 64 * c + lane; idx < n2; idx += 64 * NT) {
        const int i = idx % n, j = idx / n, lo = i < j ? i : j, hi = i < j ? j : i;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          const zd x = X0[a * (int64_t)np + lo + hi * (hi + 1) / 2];
          Vk[a * (int64_t)n2 + idx] = i > j ? zconj(x) : x;
        }
      }
      continue;
    }
    // row 4 s + kk; past the end (the last tile only): the last one, zero in U
    auto row4 = [&](int s, int kk) {
      const int m = 4 * s + kk;
      return s < NS - 4 || m < n ? m : n - 1;
    };
    auto uload = [&](const zd* Uc, int s, int kk) {
      zd u = Uc[row4(s, kk)];
      if (s >= NS - 4) {
        const bool ok = 4 * s + kk < n;
        u.re = ok ? u.re : 0.0;
        u.im = ok ? u.im : 0.0;
      }
      return u;
    };
    const zd* Ub = Uk + (int64_t)n * (bc < n ? bc : n - 1);
    zd ur[REG ? NS : 1];
    if constexpr (REG)
#pragma unroll
      for (int s = 0; s < NS; ++s) ur[s] = uload(Ub, s, kq);
#pragma unroll 1
    for (int a = 0; a < 3; ++a) {
      const zd* X = X0 + a * (int64_t)np;
      zd T[NS];
      {  // T(16 r ..) = sum over m of dH(row, m) U(m, col), GS steps a group
        struct Group {
          zd x[GS], u[REG ? 1 : GS];
        } g[2];
        auto load = [&](int q, Group& o) {
          const int r = q / NQ, s0 = q % NQ * GS;
          int kk = kq;
          asm volatile("" : "+v"(kk));  // offsets are formed here, not kept across a
          const int ar0 = 16 * r + lr, ar = r < NT - 1 || ar0 < n ? ar0 : n - 1;
          const int low = ar * (ar + 1) / 2;
#pragma unroll
          for (int j = 0; j < GS; ++j) {
            const int s = s0 + j, m = row4(s, kk);
            const bool cj = s / 4 < r || (s / 4 == r && ar > m);
            o.x[j] = X[cj ? m + low : ar + m * (m + 1) / 2];
            o.x[j].im = cj ? -o.x[j].im : o.x[j].im;
            if (!REG) o.u[REG ? 0 : j] = uload(Ub, s, kk);
          }
        };
        load(0, g[0]);
#pragma unroll
        for (int r = 0; r < NT; ++r) {
          velo_v4d p1 = {}, p2 = {}, p3 = {};
#pragma unroll
          for (int sq = 0; sq < NQ; ++sq) {
            const int q = r * NQ + sq;
            if (q + 1 < NT * NQ) load(q + 1, g[(q + 1) & 1]);
#pragma unroll
            for (int j = 0; j < GS; ++j) {
              const zd x = g[q & 1].x[j];
              const zd u = REG ? ur[REG ? GS * sq + j : 0] : g[q & 1].u[REG ? 0 : j];
              p1 = __builtin_amdgcn_mfma_f64_16x16x4f64(x.re, u.re, p1, 0, 0, 0);
              p2 = __builtin_amdgcn_mfma_f64_16x16x4f64(x.im, u.im, p2, 0, 0, 0);
              p3 = __builtin_amdgcn_mfma_f64_16x16x4f64(x.re + x.im, u.re + u.im, p3, 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
          }
#pragma unroll
          for (int v = 0; v < 4; ++v) T[4 * r + v] = zd{p1[v] - p2[v], p3[v] - p1[v] - p2[v]};
        }
      }
      zd* Va = Vk + a * (int64_t)n2;
      const int cnt = NT / 2 + ((NT & 1) || c < NT / 2 ? 1 : 0);
#pragma unroll 1
      for (int q = 0; q < cnt; ++q) {  // V(16 r ..) = sum over m of conj U(m, row) T(m, col)
        const int r = c + q < NT ? c + q : c + q - NT;
        const int ar = 16 * r + lr;
        const zd* Ua = Uk + (int64_t)n * (ar < n ? ar : n - 1);
        zd g[2][GS];
        auto load = [&](int q4, zd* o) {
          int kk = kq;
          asm volatile("" : "+v"(kk));
#pragma unroll
          for (int j = 0; j < GS; ++j) o[j] = uload(Ua, GS * q4 + j, kk);
        };
        load(0, g[0]);
        velo_v4d p1 = {}, p2 = {}, p3 = {};
#pragma unroll
        for (int q4 = 0; q4 < NQ; ++q4) {
          if (q4 + 1 < NQ) load(q4 + 1, g[(q4 + 1) & 1]);
#pragma unroll
          for (int j = 0; j < GS; ++j) {
            const zd u = g[q4 & 1][j], x = T[GS * q4 + j];
            p1 = __builtin_amdgcn_mfma_f64_16x16x4f64(u.re, x.re, p1, 0, 0, 0);
            p2 = __builtin_amdgcn_mfma_f64_16x16x4f64(-u.im, x.im, p2, 0, 0, 0);
            p3 = __builtin_amdgcn_mfma_f64_16x16x4f64(u.re - u.im, x.re + x.im, p3, 0, 0, 0);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int row = 16 * r + kq + 4 * v;
          if (row < n && bc < n) {
            const zd z = zd{p1[v] - p2[v], p3[v] - p1[v] - p2[v]};
            Va[row + (int64_t)n * bc] = z;
            if (r != c) Va[bc + (int64_t)n * row] = zconj(z);
          }
        }
      }
    }
  }
}

// V (3,n,n) per k: planar [a][i + n j]  <->  reference (a fastest)
__global__ void v_planar_to_ref(int n, int64_t nk, const zd* __restrict__ Vp, zd* __restrict__ Vr) {
  int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  const int64_t per = 3 * (int64_t)n * n;
  if (t >= nk * per) return;
  int64_t k = t / per, r = t % per;
  int a = (int)(r % 3);
  int64_t ij = r / 3;
  Vr[t] = Vp[k * per + a * (int64_t)n * n + ij];
}
__global__ void v_ref_to_planar(int n, int64_t nk, const zd* __restrict__ Vr, zd* __restrict__ Vp) {
  int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  const int64_t per = 3 * (int64_t)n * n, n2 = (int64_t)n * n;
  if (t >= nk * per) return;
  int64_t k = t / per, r = t % per;
  int a = (int)(r / n2);
  int64_t ij = r % n2;
  Vp[t] = Vr[k * per + a + 3 * ij];
}

void launch_v_layout(hipStream_t s, int n, int64_t nk, const zd* src, zd* dst, bool to_ref) {
  int64_t tot = nk * 3 * (int64_t)n * n;
  unsigned nb = (unsigned)((tot + 255) / 256);
  if (to_ref)
    hipLaunchKernelGGL(v_planar_to_ref, dim3(nb), dim3(256), 0, s, n, nk, src, dst);
  else
    hipLaunchKernelGGL(v_ref_to_planar, dim3(nb), dim3(256), 0, s, n, nk, src, dst);
}

// --------------------------------------------------------------------------
// Position operator: PRB 74 195118 Eqs. 21-31 with the reference's evaluation
// order (rotate_gauge :502-550, get_gauge_covar_deriv :565-617,
// conn_gaugeTrafo :620-633, curv_gaugeTrafo :636-658, get_velo :406-444);
// textbook != 0 selects the printed equations instead.
//   Hb_a = U^H dH_a U,  Ab_a = Hb_a U (reference) or U^H A_a U (textbook)
//   D_a(i,j) = Hb_a(i,j) / (E_j - E_i) where |E_j - E_i| > kubo_tol, i != j
//   A^(H)_a = Ab_a + i D_a,  V_a = Hb_a - i (E_j - E_i) X_a off the diagonal
//   Om^(H)_c = U^H Om_c U - [D_a, X_b] + [D_b, X_a] - i [D_a, D_b]
// with X = A^(H) (reference) or Ab (textbook) and c = (a, b) cyclic.  With
// Y = X + i D the commutators are four products,
//   X_b D_a - X_a D_b + D_b Y_a - D_a Y_b.
// What is formed is what the caller reads (VeloArgs::want).  The band sums
// read Omega on the diagonal only, which costs no product but Om_c U: the
// rest of it are row and column sums of elementwise products,
//   Om^(H)_c(i,i) = sum_m conj(U(m,i)) (Om_c U)(m,i)
//     + sum_l [X_b(i,l) D_a(l,i) - X_a(i,l) D_b(l,i)]
//     + sum_l [D_b(i,l) Y_a(l,i) - D_a(i,l) Y_b(l,i)].
// --------------------------------------------------------------------------

// The Wannier-gauge matrices of one k-point, unpacked (n^2 each), with the
// tight-binding epilogue from per-band phases f_m = e^{2 pi i k.tau_m} and
// centres in LDS: n sincos a k-point instead of one an element and matrix.
struct PosLoad {
  const zd* X;
  const zd* f;        // null: Wannier convention
  const double* tau;  // (3, n)
  int n;
  const TBPhase* tb;
  __device__ inline zd operator()(int mat, int i, int j) const {
    const int64_t n2 = (int64_t)n * n, o = i + (int64_t)n * j;
    zd x = X[mat * n2 + o];
    if (!f) return x;
    const double dt[3] = {tau[3 * j] - tau[3 * i], tau[3 * j + 1] - tau[3 * i + 1],
                          tau[3 * j + 2] - tau[3 * i + 2]};
    if (mat >= 1 && mat <= 3) {
      x = zadd(x, zmuli(zscale(X[o], tb->c(mat - 1, dt))));
    } else if (mat >= 7) {
      // Omega_ab with (a,b) = (1,2), (2,0), (0,1)
      const int a = (mat - 6) % 3, b = (mat - 5) % 3;
      x = zadd(x, zmuli(zsub(zscale(X[(4 + b) * n2 + o], tb->c(a, dt)),
                             zscale(X[(4 + a) * n2 + o], tb->c(b, dt)))));
    }
    return zmul(zcmul(f[i], f[j]), x);
  }
};
// Omega(3,3) of one element: antisymmetric, zero diagonal in (a, b)
__device__ inline void pos_store_om(zd* O, zd oyz, zd ozx, zd oxy) {
  O[0] = O[1 + 3 * 1] = O[2 + 3 * 2] = zd{0, 0};
  O[1 + 3 * 2] = oyz;
  O[2 + 3 * 1] = zsub(zd{0, 0}, oyz);
  O[2 + 3 * 0] = ozx;
  O[0 + 3 * 2] = zsub(zd{0, 0}, ozx);
  O[0 + 3 * 1] = oxy;
  O[1 + 3 * 0] = zsub(zd{0, 0}, oxy);
}

// n <= 32: one k-point per workgroup of NM / 16 x NM / 16 wavefronts (one for
// n <= 16), each owning one 16 x 16 tile of every product, as
// velo_mfma_kernel: U and three planes in LDS, three components at a time on
// FP64 MFMA, every result kept in the accumulators' layout so that D, A^(H),
// V and the curvature's diagonal are formed in registers.  FULL: the whole
// Omega (three more planes, for the commutators' operands).
// 9 products for V alone, 12 with the diagonal of Omega, 27 in all.
// n = 24, 4,096 k-points, V and the diagonals: 400 us (VALU products on
// global-memory operands, every output: 3,277 us); n = 8, 32,768 k-points, V
// alone: 222 us (LDS VALU products, every output: 1,490 us).
template <int NM, bool FULL>
__global__ __launch_bounds__(NM == 32 ? 256 : 64, 2) void velo_pos_kernel(
    int n, int64_t nk, const zd* __restrict__ Hk, int64_t strideHk, TBPhase tb0, int gauge_trafo,
    int textbook, double kubo_tol, int want, const zd* __restrict__ U, const double* __restrict__ E,
    zd* __restrict__ V, zd* __restrict__ Aout, zd* __restrict__ Omout) {
  constexpr int LD = NM + 1, PL = NM * LD, NT = NM == 32 ? 256 : 64, TD = NM / 16;
  __shared__ zd Us[PL], Ds[3 * PL], Xs[FULL ? 3 * PL : 1];
  __shared__ zd fph[NM], rsum[TD][3][NM], csum[TD][3][NM];
  __shared__ double Es[NM], taus[3 * NM];
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  const int n2 = n * n;
  const int64_t NN = n2;
  for (int c = t; c < PL; c += NT) {
    Us[c] = Ds[c] = Ds[PL + c] = Ds[2 * PL + c] = zd{0.0, 0.0};
    if (FULL) Xs[c] = Xs[PL + c] = Xs[2 * PL + c] = zd{0.0, 0.0};
  }
  const int rt = w % TD, ct = w / TD, r0 = 16 * rt, c0 = 16 * ct;
  const int ar = r0 + (lane & 15), bc = c0 + (lane & 15), kq = lane >> 4;
  const bool tile = r0 < n && c0 < n;  // wave-uniform
  typedef zd Frag[3][4];  // three components, rows r0 + kq + 4 v of column bc
  // R_a = P_a U (P in the planes) / R_a = U^H P_a
  auto right = [&](const zd* P, Frag R) {
    mep_v4d p1[3] = {}, p2[3] = {}, p3[3] = {};
    if (tile)
#pragma unroll
      for (int k0 = 0; k0 < NM; k0 += 4) {
        if (k0 >= n) break;
        const int m = k0 + kq;
        const zd b = ldz(Us + m + LD * bc);
        const double bs = b.re + b.im;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          const zd x = ldz(P + a * PL + ar + LD * m);
          p1[a] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.re, b.re, p1[a], 0, 0, 0);
          p2[a] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.im, b.im, p2[a], 0, 0, 0);
          p3[a] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.re + x.im, bs, p3[a], 0, 0, 0);
        }
      }
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int v = 0; v < 4; ++v) R[a][v] = zd{p1[a][v] - p2[a][v], p3[a][v] - p1[a][v] - p2[a][v]};
  };
  auto left = [&](const zd* P, Frag R) {
    mep_v4d p1[3] = {}, p2[3] = {}, p3[3] = {};
    if (tile)
#pragma unroll
      for (int k0 = 0; k0 < NM; k0 += 4) {
        if (k0 >= n) break;
        const int m = k0 + kq;
        const zd u = ldz(Us + m + LD * ar);
        const double us = u.re - u.im;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          const zd y = ldz(P + a * PL + m + LD * bc);
          p1[a] = __builtin_amdgcn_mfma_f64_16x16x4f64(u.re, y.re, p1[a], 0, 0, 0);
          p2[a] = __builtin_amdgcn_mfma_f64_16x16x4f64(-u.im, y.im, p2[a], 0, 0, 0);
          p3[a] = __builtin_amdgcn_mfma_f64_16x16x4f64(us, y.re + y.im, p3[a], 0, 0, 0);
        }
      }
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int v = 0; v < 4; ++v) R[a][v] = zd{p1[a][v] - p2[a][v], p3[a][v] - p1[a][v] - p2[a][v]};
  };
  auto store = [&](const Frag R, zd* P) {  // every reader of P has passed a barrier
    if (tile)
#pragma unroll
      for (int a = 0; a < 3; ++a)
#pragma unroll
        for (int v = 0; v < 4; ++v) stz(P + a * PL + r0 + kq + 4 * v + LD * bc, R[a][v]);
  };
  for (int64_t k = blockIdx.x; k < nk; k += gridDim.x) {
    const TBPhase tb = tb0.at(k);
    const PosLoad ld{Hk + k * strideHk, tb.tau ? fph : nullptr, taus, n, &tb};
    zd* Vk = V + k * 3 * NN;
    zd* Ak = Aout + k * 3 * NN;
    zd* Ok = Omout + k * 9 * NN;
    __syncthreads();  // the previous k-point's readers are done
    pos_phases(tb, n, t, fph, taus);
    if (t < n) Es[t] = E[k * n + t];
    for (int idx = t; idx < n2; idx += NT) stz(Us + idx % n + LD * (idx / n), U[k * NN + idx]);
    __syncthreads();
    // three matrices mat0 .. mat0 + 2 into the planes
    auto stage = [&](int mat0) {
      for (int idx = t; idx < n2; idx += NT) {
        const int i = idx % n, j = idx / n;
#pragma unroll
        for (int a = 0; a < 3; ++a) stz(Ds + a * PL + i + LD * j, ld(mat0 + a, i, j));
      }
    };
    if (!gauge_trafo) {
      for (int idx = t; idx < n2; idx += NT) {
        const int i = idx % n, j = idx / n;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          const zd x = ld(4 + a, i, j);
          zd v = ld(1 + a, i, j);
          if (i != j) v = zsub(v, zmul(zd{0.0, Es[j] - Es[i]}, x));
          Vk[a * NN + idx] = v;
          Ak[a + 3 * (int64_t)idx] = x;
        }
        pos_store_om(Ok + 9 * (int64_t)idx, ld(7, i, j), ld(8, i, j), ld(9, i, j));
      }
      continue;
    }
    Frag hb, ab, tmp;
    stage(1);
    __syncthreads();
    right(Ds, tmp);  // dH U
    __syncthreads();
    store(tmp, Ds);
    __syncthreads();
    left(Ds, hb);    // Hb
    __syncthreads();
    if (textbook) {
      stage(4);
      __syncthreads();
      right(Ds, tmp);
      __syncthreads();
      store(tmp, Ds);
      __syncthreads();
      left(Ds, ab);
      __syncthreads();
      store(hb, Ds);
      __syncthreads();
    } else {
      store(hb, Ds);
      __syncthreads();
      right(Ds, ab);
    }
    // D, A^(H) (over ab's place in X for the reference) and V, elementwise
    Frag dm;
    double de[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int row = r0 + kq + 4 * v;
      const bool in = row < n && bc < n;
      de[v] = in ? Es[bc] - Es[row] : 0.0;
      const bool far = in && row != bc && fabs(de[v]) > kubo_tol;
      const double rd = far ? 1.0 / de[v] : 0.0;
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        dm[a][v] = zscale(hb[a][v], rd);
        const zd ah = zadd(ab[a][v], zmuli(dm[a][v]));
        if (!textbook) ab[a][v] = ah;  // ab = X from here on
        if (in) {
          zd vv = hb[a][v];
          if (row != bc) vv = zsub(vv, zmul(zd{0.0, de[v]}, ab[a][v]));
          Vk[a * NN + row + (int64_t)n * bc] = vv;
          if ((want & VELO_A) || ((want & VELO_DIAG) && row == bc))
            Ak[a + 3 * ((int64_t)row + (int64_t)n * bc)] = ah;
        }
      }
    }
    if (FULL) {
      __syncthreads();  // Hb's readers are done
      store(dm, Ds);
      store(ab, Xs);
      __syncthreads();
      Frag cm;
      {
        mep_v4d p1[3] = {}, p2[3] = {}, p3[3] = {};
        auto mac = [&](int c, zd x, zd y) {
          p1[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.re, y.re, p1[c], 0, 0, 0);
          p2[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.im, y.im, p2[c], 0, 0, 0);
          p3[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.re + x.im, y.re + y.im, p3[c], 0, 0, 0);
        };
        if (tile)
          for (int k0 = 0; k0 < n; k0 += 4) {
            const int m = k0 + kq;
            zd xr[3], dr[3], dc[3], yc[3];
#pragma unroll
            for (int a = 0; a < 3; ++a) {
              xr[a] = ldz(Xs + a * PL + ar + LD * m);
              dr[a] = ldz(Ds + a * PL + ar + LD * m);
              dc[a] = ldz(Ds + a * PL + m + LD * bc);
              yc[a] = zadd(ldz(Xs + a * PL + m + LD * bc), zmuli(dc[a]));
            }
#pragma unroll
            for (int c = 0; c < 3; ++c) {
              const int a = (c + 1) % 3, b = (c + 2) % 3;
              mac(c, xr[b], dc[a]);
              mac(c, zscale(xr[a], -1.0), dc[b]);
              mac(c, dr[b], yc[a]);
              mac(c, zscale(dr[a], -1.0), yc[b]);
            }
          }
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
          for (int v = 0; v < 4; ++v) cm[c][v] = zd{p1[c][v] - p2[c][v], p3[c][v] - p1[c][v] - p2[c][v]};
      }
      __syncthreads();
      stage(7);
      __syncthreads();
      right(Ds, tmp);
      __syncthreads();
      store(tmp, Ds);
      __syncthreads();
      left(Ds, tmp);  // U^H Om U
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int row = r0 + kq + 4 * v;
        if (row < n && bc < n)
          pos_store_om(Ok + 9 * ((int64_t)row + (int64_t)n * bc), zadd(tmp[0][v], cm[0][v]),
                       zadd(tmp[1][v], cm[1][v]), zadd(tmp[2][v], cm[2][v]));
      }
    } else if (want & VELO_DIAG) {
      // D(l, i) of this thread's (i, l) from Hb's planes (no symmetry assumed)
      zd cs[3] = {};
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int row = r0 + kq + 4 * v;
        const bool far = row < n && bc < n && row != bc && fabs(de[v]) > kubo_tol;
        const double rd = far ? -1.0 / de[v] : 0.0;
        zd dt[3], y[3];
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          dt[a] = zscale(ldz(Ds + a * PL + bc + LD * row), rd);
          y[a] = zadd(ab[a][v], zmuli(dm[a][v]));
        }
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          const int a = (c + 1) % 3, b = (c + 2) % 3;
          const zd f = zsub(zmul(ab[b][v], dt[a]), zmul(ab[a][v], dt[b]));
          cs[c] = zadd(cs[c], zsub(zmul(dt[b], y[a]), zmul(dt[a], y[b])));
          const zd rs = zd{row16_sum(f.re), row16_sum(f.im)};
          if ((lane & 15) == 0) rsum[ct][c][row] = rs;  // zero beyond n
        }
      }
      __syncthreads();  // Hb's readers are done
      stage(7);
      __syncthreads();
      right(Ds, tmp);  // Om U
#pragma unroll
      for (int c = 0; c < 3; ++c) {
#pragma unroll
        for (int v = 0; v < 4; ++v)
          cs[c] = zadd(cs[c], zcmul(ldz(Us + r0 + kq + 4 * v + LD * bc), tmp[c][v]));
        const zd s = zd{rows4_sum(cs[c].re), rows4_sum(cs[c].im)};
        if (kq == 0) csum[rt][c][bc] = s;
      }
      __syncthreads();
      if (t < n) {
        zd o[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          o[c] = zadd(rsum[0][c][t], csum[0][c][t]);
          if (TD == 2 && n > 16) o[c] = zadd(o[c], zadd(rsum[TD - 1][c][t], csum[TD - 1][c][t]));
        }
        pos_store_om(Ok + 9 * ((int64_t)t + (int64_t)n * t), o[0], o[1], o[2]);
      }
    }
  }
}

// C = sum over the terms of op(A) B for n x n matrices of pitch n in global
// memory (the workgroup's slot): FP64 MFMA, the 16 x 16 tiles over four waves,
// operands loaded in chunks of four steps ahead of their products.  aload(i, m)
// and bload(m, j) return the elements; terms are run one after the other into
// the same accumulators.
template <class ALoad, class BLoad>
__device__ inline void gmm_acc(int n, int ar, int bc, int kq, const ALoad& aload, const BLoad& bload,
                               velo_v4d& p1, velo_v4d& p2, velo_v4d& p3) {
  constexpr int CH = 4;
  for (int m0 = 0; m0 < n; m0 += 4 * CH) {
    zd av[CH], bv[CH];
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      const int m = m0 + 4 * i + kq;
      av[i] = (m < n && ar < n) ? aload(ar, m) : zd{0.0, 0.0};
      bv[i] = (m < n && bc < n) ? bload(m, bc) : zd{0.0, 0.0};
    }
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      p1 = __builtin_amdgcn_mfma_f64_16x16x4f64(av[i].re, bv[i].re, p1, 0, 0, 0);
      p2 = __builtin_amdgcn_mfma_f64_16x16x4f64(av[i].im, bv[i].im, p2, 0, 0, 0);
      p3 = __builtin_amdgcn_mfma_f64_16x16x4f64(av[i].re + av[i].im, bv[i].re + bv[i].im, p3, 0, 0, 0);
    }
  }
}
// every tile of C: acc(ar, bc, kq, p1, p2, p3) forms it, out(row, col, value)
// takes the elements
template <class Acc, class Out>
__device__ inline void gmm_tiles(int n, const Acc& acc, const Out& out) {
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lr = lane & 15, kq = lane >> 4, nt = (n + 15) / 16;
  for (int it = wv; it < nt * nt; it += 4) {
    const int r0 = 16 * (it % nt), bc = 16 * (it / nt) + lr;
    velo_v4d p1 = {0, 0, 0, 0}, p2 = {0, 0, 0, 0}, p3 = {0, 0, 0, 0};
    acc(r0 + lr, bc, kq, p1, p2, p3);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int row = r0 + kq + 4 * v;
      if (row < n && bc < n) out(row, bc, zd{p1[v] - p2[v], p3[v] - p1[v] - p2[v]});
    }
  }
}
__device__ inline void gmm(int n, const zd* A, bool adjA, const zd* B, zd* C) {
  gmm_tiles(
      n,
      [&](int ar, int bc, int kq, velo_v4d& p1, velo_v4d& p2, velo_v4d& p3) {
        auto b = [&](int m, int j) { return B[m + (int64_t)n * j]; };
        if (adjA)
          gmm_acc(n, ar, bc, kq, [&](int i, int m) { return zconj(A[m + (int64_t)n * i]); }, b, p1,
                  p2, p3);
        else
          gmm_acc(n, ar, bc, kq, [&](int i, int m) { return A[i + (int64_t)n * m]; }, b, p1, p2, p3);
      },
      [&](int i, int j, zd x) { C[i + (int64_t)n * j] = x; });
}

// 32 < n <= 128: the same steps with the matrices in the workgroup's slot of
// `slots` (18 n^2 complex each; the slots lie in the consumed eigensolver
// records) instead of LDS, products on MFMA from L2.
__global__ __launch_bounds__(256) void velo_pos_global_kernel(int n, int64_t nk,
                                                              const zd* __restrict__ Hk,
                                                              int64_t strideHk, TBPhase tb0,
                                                              int gauge_trafo, int textbook,
                                                              double kubo_tol, int want,
                                                              const zd* __restrict__ U,
                                                              const double* __restrict__ E,
                                                              zd* __restrict__ V, zd* __restrict__ Aout,
                                                              zd* __restrict__ Omout,
                                                              zd* __restrict__ slots) {
  __shared__ double Es[128], taus[3 * 128];
  __shared__ zd fph[128];
  const int t = threadIdx.x;
  const int64_t NN = (int64_t)n * n;
  zd* base = slots + (int64_t)blockIdx.x * 18 * NN;
  zd *Us = base, *T1 = base + NN, *T2 = base + 2 * NN;
  zd *Hb[3], *Ab[3], *Dm[3], *Om[3], *Abar[3];
  for (int a = 0; a < 3; ++a) {
    Hb[a] = base + (3 + a) * NN;
    Ab[a] = base + (6 + a) * NN;
    Dm[a] = base + (9 + a) * NN;
    Om[a] = base + (12 + a) * NN;
    Abar[a] = base + (15 + a) * NN;
  }
  const bool full = (want & VELO_OM) != 0, om = full || (want & VELO_DIAG);
  for (int64_t k = blockIdx.x; k < nk; k += gridDim.x) {
    const TBPhase tb = tb0.at(k);
    const PosLoad ld{Hk + k * strideHk, tb.tau ? fph : nullptr, taus, n, &tb};
    __syncthreads();  // the previous k-point's reads of the slot are done
    pos_phases(tb, n, t, fph, taus);
    if (t < n) Es[t] = E[k * n + t];
    __syncthreads();
    for (int idx = t; idx < n * n; idx += 256) {
      const int i = idx % n, j = idx / n;
      Us[idx] = U[k * NN + idx];
      for (int a = 0; a < 3; ++a) {
        Hb[a][idx] = ld(1 + a, i, j);
        if (textbook || !gauge_trafo) Ab[a][idx] = ld(4 + a, i, j);
        if (om || !gauge_trafo) Om[a][idx] = ld(7 + a, i, j);
      }
    }
    __syncthreads();
    if (gauge_trafo) {
      for (int a = 0; a < 3; ++a) {
        gmm(n, Hb[a], false, Us, T1);  // dH U
        if (textbook) gmm(n, Ab[a], false, Us, T2);
        __syncthreads();
        gmm(n, Us, true, T1, Hb[a]);   // Hb = U^H dH U
        if (textbook) gmm(n, Us, true, T2, Ab[a]);
        __syncthreads();
        if (!textbook) gmm(n, Hb[a], false, Us, Ab[a]);  // A = (U^H (dH U)) U
        if (om) gmm(n, Om[a], false, Us, T2);
        __syncthreads();
        if (full) {
          gmm(n, Us, true, T2, Om[a]);  // U^H Om U
        } else if (om) {                // its diagonal
          for (int i = t; i < n; i += 256) {
            zd s = zd{0.0, 0.0};
#pragma unroll 8
            for (int m = 0; m < n; ++m)
              s = zadd(s, zcmul(Us[m + (int64_t)n * i], T2[m + (int64_t)n * i]));
            Om[a][i + (int64_t)n * i] = s;
          }
        }
        __syncthreads();
      }
      // D, Abar and A^(H) = Abar + i D
      for (int idx = t; idx < n * n; idx += 256) {
        const int i = idx % n, j = idx / n;
        const double de = Es[j] - Es[i];
        const double rd = (i != j && fabs(de) > kubo_tol) ? 1.0 / de : 0.0;
        for (int a = 0; a < 3; ++a) {
          const zd dv = zscale(Hb[a][idx], rd), ab = Ab[a][idx];
          Dm[a][idx] = dv;
          Abar[a][idx] = ab;
          Ab[a][idx] = zadd(ab, zmuli(dv));
        }
      }
      __syncthreads();
      zd* const* X = textbook ? Abar : Ab;
      auto Y = [&](int a, int64_t o) { return zadd(X[a][o], zmuli(Dm[a][o])); };
      for (int c = 0; c < 3 && om; ++c) {
        const int a = (c + 1) % 3, b = (c + 2) % 3;
        if (full) {
          gmm_tiles(
              n,
              [&](int ar, int bc, int kq, velo_v4d& p1, velo_v4d& p2, velo_v4d& p3) {
                auto at = [&](const zd* M, double sg) {
                  return [=](int i, int m) { return zscale(M[i + (int64_t)n * m], sg); };
                };
                auto bt = [&](const zd* M) {
                  return [=](int m, int j) { return M[m + (int64_t)n * j]; };
                };
                gmm_acc(n, ar, bc, kq, at(X[b], 1.0), bt(Dm[a]), p1, p2, p3);
                gmm_acc(n, ar, bc, kq, at(X[a], -1.0), bt(Dm[b]), p1, p2, p3);
                gmm_acc(n, ar, bc, kq, at(Dm[b], 1.0),
                        [&](int m, int j) { return Y(a, m + (int64_t)n * j); }, p1, p2, p3);
                gmm_acc(n, ar, bc, kq, at(Dm[a], -1.0),
                        [&](int m, int j) { return Y(b, m + (int64_t)n * j); }, p1, p2, p3);
              },
              // each element of Om_c is read and written by its own thread
              [&](int i, int j, zd x) {
                zd* o = Om[c] + i + (int64_t)n * j;
                *o = zadd(*o, x);
              });
        } else {
          for (int i = t; i < n; i += 256) {
            zd s = Om[c][i + (int64_t)n * i];
            for (int l = 0; l < n; ++l) {
              const int64_t il = i + (int64_t)n * l, li = l + (int64_t)n * i;
              s = zadd(s, zsub(zmul(X[b][il], Dm[a][li]), zmul(X[a][il], Dm[b][li])));
              s = zadd(s, zsub(zmul(Dm[b][il], Y(a, li)), zmul(Dm[a][il], Y(b, li))));
            }
            Om[c][i + (int64_t)n * i] = s;
          }
        }
      }
      __syncthreads();
    }
    // velocity, connection and curvature in the reference's layouts
    const bool all = full || !gauge_trafo;
    for (int idx = t; idx < n * n; idx += 256) {
      const int i = idx % n, j = idx / n;
      for (int a = 0; a < 3; ++a) {
        zd v = Hb[a][idx];
        if (i != j) {
          // V_nm = H_nm - i (E_m - E_n) A_nm
          const zd* Asel = (gauge_trafo && textbook) ? Abar[a] : Ab[a];
          const zd ce = zd{0.0, Es[j] - Es[i]};
          v = zsub(v, zmul(ce, Asel[idx]));
        }
        V[k * 3 * NN + a * NN + idx] = v;
        if (all || (want & VELO_A) || i == j) Aout[k * 3 * NN + a + 3 * (int64_t)idx] = Ab[a][idx];
      }
      if (all || (om && i == j))
        pos_store_om(Omout + k * 9 * NN + 9 * (int64_t)idx, Om[0][idx], Om[1][idx], Om[2][idx]);
    }
  }
}

bool velo_pos_scratch_ok(int n, size_t scratch_bytes) {
  return n <= 32 || scratch_bytes >= 18 * (size_t)n * n * sizeof(zd);
}

void launch_velo(hipStream_t s, const VeloArgs& va, int64_t nk, zd* Hk, int64_t strideHk,
                 const KGeom& g, const zd* U, const double* E, zd* V, zd* A, zd* Om) {
  unsigned grid = (unsigned)(nk < 65536 ? nk : 65536);
  TBPhase tb;
  tb.kx = tb.ky = tb.kz = 0.0;
  tb.kpts = g.kpts;
  tb.tau = g.tau;
  for (int i = 0; i < 9; ++i) tb.cm[i] = g.cmat[i];
  if (va.pos_op && va.n <= 32) {
    const bool full = (va.want & VELO_OM) != 0;
#define MEP_POS_LAUNCH(NM, FULL)                                                                   \
  hipLaunchKernelGGL((velo_pos_kernel<NM, FULL>), dim3(grid), dim3(NM == 32 ? 256 : 64), 0, s,    \
                     va.n, nk, Hk, strideHk, tb, va.gauge_trafo, va.textbook, va.kubo_tol,        \
                     va.want, U, E, V, A, Om)
    if (va.n <= 16) {
      if (full) MEP_POS_LAUNCH(16, true);
      else MEP_POS_LAUNCH(16, false);
    } else {
      if (full) MEP_POS_LAUNCH(32, true);
      else MEP_POS_LAUNCH(32, false);
    }
#undef MEP_POS_LAUNCH
    return;
  }
  if (va.pos_op) {
    // one workgroup per slot of 18 n^2 complex in the scratch
    const int64_t slot = 18 * (int64_t)va.n * va.n * (int64_t)sizeof(zd);
    int64_t pg = (int64_t)(va.scratch_bytes / (size_t)slot);
    if (pg > nk) pg = nk;
    if (pg > 2048) pg = 2048;
    if (pg < 1) pg = 1;  // the caller guarantees one slot (velo_pos_scratch_ok)
    hipLaunchKernelGGL(velo_pos_global_kernel, dim3((unsigned)pg), dim3(256), 0, s, va.n, nk, Hk,
                       strideHk, tb, va.gauge_trafo, va.textbook, va.kubo_tol, va.want, U, E, V, A,
                       Om, va.scratch);
    return;
  }
  if (va.n > 32) {
    if (tb.tau)
      hipLaunchKernelGGL(velo_tb_kernel, dim3(grid), dim3(256), 0, s, va.n, nk, Hk, strideHk, tb);
    const int nt = (va.n + 15) / 16;
    // 8 slots of a column each, at most 65536 times 8 workgroups
    const int64_t slots = (nk + 7) / 8 * nt;
    const unsigned wgrid = 8 * (unsigned)(slots < 65536 ? slots : 65536);
#define MEP_VELO_WIDE(NT)                                                                    \
  case NT:                                                                                   \
    hipLaunchKernelGGL((velo_wide_kernel<NT, (NT <= 4)>), dim3(wgrid), dim3(64), 0, s, va.n,      \
                       nk, Hk, strideHk, va.gauge_trafo, U, V);                              \
    break;
    switch (nt) {
      MEP_VELO_WIDE(3)
      MEP_VELO_WIDE(4)
      MEP_VELO_WIDE(5)
      MEP_VELO_WIDE(6)
      MEP_VELO_WIDE(7)
      MEP_VELO_WIDE(8)
    }
#undef MEP_VELO_WIDE
    return;
  }
  hipLaunchKernelGGL(velo_mfma_kernel<zd>, dim3(grid), dim3(256), 0, s, va.n, nk, Hk, strideHk,
                     va.packed, tb, va.gauge_trafo, U, V);
}

void launch_velo_h32(hipStream_t s, const VeloArgs& va, int64_t nk, const zf* Hk,
                     int64_t strideHk, const KGeom& g, const zd* U, zd* V) {
  unsigned grid = (unsigned)(nk < 65536 ? nk : 65536);
  TBPhase tb;
  tb.kx = tb.ky = tb.kz = 0.0;
  tb.kpts = g.kpts;
  tb.tau = g.tau;
  for (int i = 0; i < 9; ++i) tb.cm[i] = g.cmat[i];
  hipLaunchKernelGGL(velo_mfma_kernel<zf>, dim3(grid), dim3(256), 0, s, va.n, nk, Hk, strideHk,
                     va.packed, tb, va.gauge_trafo, U, V);
}
