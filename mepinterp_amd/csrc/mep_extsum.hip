// mep_extsum.hip -- the optical, photogalvanic and gyrotropic band sums of
// the k-loop (core.f90:235-253), accumulated into per-workgroup partial
// records like the main band sums.
//   kubo_opt_tens        kubo.f90:204-405   (wann guide 12.10-12.15; needs A)
//   photo_2nd_cond       photo.f90:16-86    (Yang et al. PRB 97 241118 Eq. 1)
//   get_gyro_C / D / Dw  gyro.f90:153-300   (Souza et al. PRB 97 035158)
//   d1_fd_stat_deriv     statistics.f90:160-196 (1/(2 + 2 cosh) of the
//                        occupation itself, as the reference evaluates it)
// One k-point at a time per 256-thread workgroup, into the workgroup's record
// (fixed order, deterministic).  photo_2nd_cond of up to 32 bands has a kernel
// of its own (photo_kernel).  A and Omega are read in the reference layout
// (position operator only).  The occupations, their derivative and the
// per-band curvature sit in dynamic LDS, sized by n and n_eF (ext_lds_bytes).
#include "mep_common.hpp"
#include "mep_kernels.hpp"
#include "mep_lane.hpp"
#include "../../include/mepinterp.h"

ExtLayout ext_layout(const BandArgs& b) {
  ExtLayout X;
  const int64_t hf = (int64_t)b.n_hw * b.n_ef;
  int64_t o = 0;
  X.opt_s = o;   o += 18 * hf;
  X.opt_a = o;   o += 18 * hf;
  X.photo = o;   o += 54 * hf;
  X.gyro_C = o;  o += 18 * (int64_t)b.n_ef;
  X.gyro_D = o;  o += 18 * (int64_t)b.n_ef;
  X.gyro_Dw = o; o += 18 * hf;
  X.total = o;
  return X;
}

typedef double mep_v4d __attribute__((ext_vector_type(4)));

constexpr int XS_THREADS = 256;
constexpr int XS_NMAX = 32;
constexpr int XS_LD = XS_NMAX + 1;
constexpr int XS_PL = XS_NMAX * XS_LD;

__device__ inline int levi3(int a, int b, int c) {
  return (a == b || b == c || a == c) ? 0 : (((b - a + 3) % 3 == 1) ? 1 : -1);
}

constexpr size_t XS_LDS = 160 * 1024;

// ---------------------------------------------------------------------------
// photo_2nd_cond, n <= 32:
//   sum_{n, m, l != n} (f_l - f_n) / hw^2 V_a(n,l) V_b(l,m) V_c(m,n)
//     / (E_n - E_m - i eta) sum_{+-} 1 / (E_n - E_l +- hw - 2 i eta)
// The m sum is a matrix product per (b, c), P = V_b W_c with W_c(m,n) =
// V_c(m,n) / (E_n - E_m - i eta), on FP64 MFMA: a wavefront forms one 16 x 16
// tile of P for the three b of one c (n <= 16: wave c, else wave = tile and a
// round per c).  64 pairs (l, n) of a tile at a time then become records
// G_ab = V_a(n,l) P_b(l,n) in LDS, and thread (item, split), item = (hw, E_F),
// walks the records of its split, adding record times weight to its 27 sums,
// which stay in registers over every k-point.  So a pair's weight (two
// reciprocals) is formed once an item (n <= 16) or once an item and c, not
// for each of the 27 components, and P once.  Blocks of 256 items run side by
// side (blockIdx.y).
// n = 14, 2,730 k-points, 8 frequencies x 2 Fermi levels: 145 us (one thread a
// component and item, walking all pairs: about 1,500 us).
// ---------------------------------------------------------------------------
template <int NM>
struct PhLds {
  static constexpr int LD = NM + 1, PL = NM * LD;
  static constexpr int SLOTS = NM == 16 ? 192 : 256;  // records in LDS
  static constexpr int RL = 9;                        // complex per record
  static size_t bytes(int n, int nef) {
    return sizeof(zd) * (4 * (size_t)PL + (size_t)SLOTS * RL) +
           sizeof(double) * (NM + (size_t)nef * n);
  }
};

template <int NM>
__global__ __launch_bounds__(XS_THREADS, NM == 16 ? 2 : 1) void photo_kernel(
    BandArgs b, double Tsmear, ExtLayout X, int64_t nk, const double* __restrict__ E,
    const zd* __restrict__ V, const double* __restrict__ w, double* __restrict__ part) {
  using S_ = PhLds<NM>;
  constexpr int LD = S_::LD, PL = S_::PL, RL = S_::RL, TD = NM / 16, ROUNDS = NM == 16 ? 1 : 3;
  extern __shared__ __attribute__((aligned(16))) double xs_smem[];
  zd* Vs = reinterpret_cast<zd*>(xs_smem);  // three planes, zero beyond n
  zd* Gt = Vs + 3 * PL;                     // 1 / (E_n - E_m - i eta) at [m + LD n]
  zd* rec = Gt + PL;                        // [SLOTS][9]
  double* Es = reinterpret_cast<double*>(rec + S_::SLOTS * RL);
  double* fd = Es + NM;                     // (n_ef, band)
  const int n = b.n, nef = b.n_ef, n2 = n * n;
  const int t = threadIdx.x, lane = t & 63, wv = __builtin_amdgcn_readfirstlane(t >> 6);
  const int lr = lane & 15, kq = lane >> 4;
  const int NI = b.n_hw * nef, g0 = blockIdx.y * XS_THREADS;
  const int IW = (NI - g0 < XS_THREADS) ? NI - g0 : XS_THREADS;
  const int S = XS_THREADS / IW, slot = t % IW, split = t / IW;
  const int h = (g0 + slot) % b.n_hw, ef = (g0 + slot) / b.n_hw;
  const double hwv = b.hw[h], e2 = 4.0 * b.eta * b.eta;
  const bool finiteT = b.T_kelvin > 1e-2;
  for (int c = t; c < 4 * PL; c += XS_THREADS) stz(Vs + c, zd{0.0, 0.0});
  zd acc[3][9];
#pragma unroll
  for (int c = 0; c < 3; ++c)
#pragma unroll
    for (int q = 0; q < 9; ++q) acc[c][q] = zd{0.0, 0.0};
  for (int64_t k = blockIdx.x; k < nk; k += gridDim.x) {
    const double wk = w ? w[k] : 1.0;
    const zd* Vk = V + k * 3 * (int64_t)n2;
    __syncthreads();
    for (int idx = t; idx < n2; idx += XS_THREADS) {
      const int o = idx % n + LD * (idx / n);
#pragma unroll
      for (int a = 0; a < 3; ++a) stz(Vs + a * PL + o, Vk[a * (int64_t)n2 + idx]);
    }
    if (t < n) Es[t] = E[k * n + t];
    __syncthreads();
    for (int idx = t; idx < n2; idx += XS_THREADS) {
      const int m = idx % n, nn = idx / n;
      const double x = Es[nn] - Es[m], iv = 1.0 / (x * x + b.eta * b.eta);
      stz(Gt + m + LD * nn, zd{x * iv, b.eta * iv});
    }
    for (int idx = t; idx < nef * n; idx += XS_THREADS) {
      if (b.fd_in) {
        fd[idx] = b.fd_in[k * (int64_t)nef * n + idx];
      } else {
        const double e = Es[idx / nef], ff = b.ef[idx % nef];
        fd[idx] = finiteT ? 1.0 / (1.0 + exp((e - ff) / Tsmear)) : ((e < ff) ? 1.0 : 0.0);
      }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r) {
      const int c = NM == 16 ? wv : r;  // this wave's component c and tile
      const int r0 = NM == 16 ? 0 : 16 * (wv % TD), c0 = NM == 16 ? 0 : 16 * (wv / TD);
      const bool work = NM != 16 || wv < 3;
      const int ar = r0 + lr, bc = c0 + lr;
      mep_v4d p1[3] = {}, p2[3] = {}, p3[3] = {};
      if (work)
        for (int k0 = 0; k0 < n; k0 += 4) {
          const int m = k0 + kq;
          const zd wc = zmul(ldz(Vs + c * PL + m + LD * bc), ldz(Gt + m + LD * bc));
          const double ws = wc.re + wc.im;
#pragma unroll
          for (int bb = 0; bb < 3; ++bb) {
            const zd x = ldz(Vs + bb * PL + ar + LD * m);
            p1[bb] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.re, wc.re, p1[bb], 0, 0, 0);
            p2[bb] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.im, wc.im, p2[bb], 0, 0, 0);
            p3[bb] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.re + x.im, ws, p3[bb], 0, 0, 0);
          }
        }
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        if (NM == 16 && 4 * v >= n) break;  // uniform: no rows left
        __syncthreads();  // the previous records' readers are done
        if (work) {
          const int l = r0 + kq + 4 * v, nn = bc;
          zd* rc = rec + (wv * 64 + lane) * RL;
#pragma unroll
          for (int a = 0; a < 3; ++a) {
            const zd va = ldz(Vs + a * PL + nn + LD * l);
#pragma unroll
            for (int bb = 0; bb < 3; ++bb)
              stz(rc + a + 3 * bb, zmul(va, zd{p1[bb][v] - p2[bb][v],
                                               p3[bb][v] - p1[bb][v] - p2[bb][v]}));
          }
        }
        __syncthreads();
        if (split < S)
          for (int p = split; p < (NM == 16 ? 64 : 256); p += S) {
            const int tile = p >> 6, pl = p & 63;
            const int l = 16 * (tile % TD) + (pl >> 4) + 4 * v, nn = 16 * (tile / TD) + (pl & 15);
            if (l >= n || nn >= n || l == nn) continue;
            const double df = wk * (fd[ef + nef * l] - fd[ef + nef * nn]);
            const double x = Es[nn] - Es[l], xp = x + hwv, xm = x - hwv;
            const double ip = rcp_nr(xp * xp + e2), im = rcp_nr(xm * xm + e2);
            const zd sh = zd{(xp * ip + xm * im) * df, 2.0 * b.eta * (ip + im) * df};
#pragma unroll
            for (int cc = 0; cc < (NM == 16 ? 3 : 1); ++cc)
#pragma unroll
              for (int q = 0; q < 9; ++q) {
                const zd g = ldz(rec + ((NM == 16 ? 64 * cc : 0) + p) * RL + q);
                zd& s = acc[NM == 16 ? cc : r][q];
                s.re = fma(g.re, sh.re, fma(-g.im, sh.im, s.re));
                s.im = fma(g.re, sh.im, fma(g.im, sh.re, s.im));
              }
          }
      }
    }
  }
  // splits in a fixed order
  double* out = part + (int64_t)blockIdx.x * X.total + X.photo + 54 * ((int64_t)h + (int64_t)b.n_hw * ef);
#pragma unroll
  for (int c = 0; c < 3; ++c)
#pragma unroll
    for (int q = 0; q < 9; ++q) {
      __syncthreads();
      stz(rec + t, acc[c][q]);
      __syncthreads();
      if (split == 0) {
        zd sum = rec[slot];
        for (int u = 1; u < S; ++u) sum = zadd(sum, rec[slot + IW * u]);
        out[2 * (q + 9 * c)] += sum.re / (hwv * hwv);
        out[2 * (q + 9 * c) + 1] += sum.im / (hwv * hwv);
      }
    }
}

static size_t photo_lds(const BandArgs& b) {
  return b.n <= 16 ? PhLds<16>::bytes(b.n, b.n_ef) : PhLds<32>::bytes(b.n, b.n_ef);
}
// photo_kernel serves the run (otherwise extsum_kernel's own loops)
static bool photo_fast(const BandArgs& b) {
  return (b.jobs & MEP_JOB_OPT) && b.n <= XS_NMAX && photo_lds(b) <= XS_LDS;
}

// dynamic LDS of extsum_kernel: [V planes if LDSV] | E (128) | omega
// (3 x 128 complex) | fd (n_ef x n) | fd_stat_deriv (n_ef x n) | work area:
// photo_2nd_cond here (n > 32): P (n^2 complex) where it fits, split sums
// (XS_THREADS complex); kubo_opt_tens: pair records and split sums; get_gyro_Dw:
// frequency-resolved curvatures, one frequency at the least.  The last two take
// what is left, up to XS_WORK doubles.
constexpr size_t XS_WORK = 18 * XS_THREADS;
__host__ __device__ inline size_t ext_base_doubles(int n, int nef, bool ldsv) {
  return (ldsv ? 2 * 3 * (size_t)XS_PL : 0) + 128 + 2 * 3 * 128 + 2 * (size_t)nef * n;
}
// V from L2: photo_2nd_cond's per-(b, c) product P (n^2 complex) in LDS
// where it fits beside the occupation tables (n <= 64)
constexpr int XS_PMAX = 64;
__host__ __device__ inline bool ext_photo_p(int n, int nef) {
  return n <= XS_PMAX && sizeof(double) * (ext_base_doubles(n, nef, false) + 2 * (size_t)n * n +
                                           2 * XS_THREADS) <= 160 * 1024;
}
// doubles of the work area
static size_t ext_work(const BandArgs& b, bool ldsv) {
  const bool opt = (b.jobs & MEP_JOB_OPT) != 0;
  const size_t base = ext_base_doubles(b.n, b.n_ef, ldsv);
  size_t least = opt ? 2 * XS_THREADS : 0;
  if (opt && !photo_fast(b) && ext_photo_p(b.n, b.n_ef)) least += 2 * (size_t)b.n * b.n;
  if ((b.jobs & MEP_JOB_GYRO) && b.pos_op && least < 3 * (size_t)b.n) least = 3 * (size_t)b.n;
  const size_t left = XS_LDS / sizeof(double) > base ? XS_LDS / sizeof(double) - base : 0;
  const size_t most = left < XS_WORK ? left : XS_WORK;
  return least > most ? least : most;
}

template <bool LDSV>
__global__ __launch_bounds__(XS_THREADS) void extsum_kernel(BandArgs b, double Tsmear, ExtLayout X,
                                                           int64_t nk, const double* __restrict__ E,
                                                           const zd* __restrict__ V,
                                                           const zd* __restrict__ A,
                                                           const zd* __restrict__ Om,
                                                           const double* __restrict__ w,
                                                           double* __restrict__ part,
                                                           zd* __restrict__ scr, bool photo,
                                                           int nwork) {
  extern __shared__ __attribute__((aligned(16))) double xs_smem[];
  zd* Vs = reinterpret_cast<zd*>(xs_smem);                         // LDSV only
  double* Es = xs_smem + (LDSV ? 2 * 3 * XS_PL : 0);
  zd* omg = reinterpret_cast<zd*>(Es + 128);                         // omega_c(n) of get_gyro_D
  double* fd = reinterpret_cast<double*>(omg + 3 * 128);             // (n_ef, band)
  const int n = b.n, nef = b.n_ef, nhw = b.n_hw, n2 = n * n;
  double* fdd = fd + (int64_t)nef * n;                               // fd_stat_deriv
  const int t = threadIdx.x;
  const bool finiteT = b.T_kelvin > 1e-2;
  const bool doOpt = (b.jobs & MEP_JOB_OPT) != 0, doGyro = (b.jobs & MEP_JOB_GYRO) != 0;
  const bool pos = b.pos_op && A && Om;
  const double eta = b.eta;
  double* rec = part + (int64_t)blockIdx.x * X.total;
  double* work = fdd + (int64_t)nef * n;  // nwork doubles, 16-byte aligned (every part is even)
  // kubo_opt_tens: thread (item, split), item = (hw, E_F); its 18 sums stay in
  // registers over every k-point (over one k-point where the items need
  // several passes)
  const int NI = nhw * nef;
  const int npass = (NI + XS_THREADS - 1) / XS_THREADS;
  zd ox[9], oy[9];  // sum amn eta df / ((dE - hw)^2 + eta^2), sum amn df / (dE - hw)
#pragma unroll
  for (int q = 0; q < 9; ++q) ox[q] = oy[q] = zd{0.0, 0.0};
  auto opt_flush = [&](int g0) {
    const int IW = (NI - g0 < XS_THREADS) ? NI - g0 : XS_THREADS;
    const int S = XS_THREADS / IW, slot = t % IW, split = t / IW;
    zd* red = reinterpret_cast<zd*>(work);
#pragma unroll
    for (int q = 0; q < 9; ++q) {
      zd sx = zd{0.0, 0.0}, sy = zd{0.0, 0.0};
      __syncthreads();
      red[t] = ox[q];
      __syncthreads();
      if (split == 0)
        for (int u = 0; u < S; ++u) sx = zadd(sx, red[slot + IW * u]);
      __syncthreads();
      red[t] = oy[q];
      __syncthreads();
      if (split == 0) {
        for (int u = 0; u < S; ++u) sy = zadd(sy, red[slot + IW * u]);
        // herm = -sum amn pi delta df, aherm = i sum amn df / (dE - hw)
        const zd herm = zd{-sx.re, -sx.im}, aherm = zmuli(sy);
        const int64_t o = 2 * (q + 9 * (int64_t)(g0 + slot));
        rec[X.opt_s + o] += herm.re;       // (12.14) Re herm + i Im aherm
        rec[X.opt_s + o + 1] += aherm.im;
        rec[X.opt_a + o] += aherm.re;      // (12.15) Re aherm + i Im herm
        rec[X.opt_a + o + 1] += herm.im;
      }
      ox[q] = oy[q] = zd{0.0, 0.0};
    }
    __syncthreads();
  };
  auto Aat = [&](int64_t k, int a, int i, int j) {  // A_a(i, j) of k, reference layout
    return A[k * 3 * (int64_t)n2 + a + 3 * ((int64_t)i + (int64_t)n * j)];
  };
  for (int64_t k = blockIdx.x; k < nk; k += gridDim.x) {
    const double wk = w ? w[k] : 1.0;
    __syncthreads();
    const zd* Vk = V + k * 3 * (int64_t)n2;
    // V_a(i, j): the LDS planes or the k-point's planar V
    auto Vat = [&](int a, int i, int j) {
      return LDSV ? Vs[a * XS_PL + i + XS_LD * j] : Vk[a * (int64_t)n2 + i + (int64_t)n * j];
    };
    if (LDSV)
      for (int idx = t; idx < 3 * n2; idx += XS_THREADS) {
        const int a = idx / n2, r = idx - a * n2;
        Vs[a * XS_PL + r % n + XS_LD * (r / n)] = Vk[idx];
      }
    for (int i = t; i < n; i += XS_THREADS) Es[i] = E[k * n + i];
    __syncthreads();
    for (int idx = t; idx < nef * n; idx += XS_THREADS) {
      double f;
      if (b.fd_in) {
        f = b.fd_in[k * (int64_t)nef * n + idx];
      } else {
        const int ef = idx % nef, nb = idx / nef;
        const double e = Es[nb], ff = b.ef[ef];
        f = finiteT ? 1.0 / (1.0 + exp((e - ff) / Tsmear)) : ((e < ff) ? 1.0 : 0.0);
      }
      fd[idx] = f;
      fdd[idx] = 1.0 / (2.0 + 2.0 * cosh(f));
    }
    // omega_c(n) = sum_ab eps_abc curv_ab(n): Omega_ab(n,n) with a position
    // operator, else get_kubo_curv (wann_interp.f90:113-146)
    for (int t0 = t; doGyro && t0 < n; t0 += XS_THREADS) {
      const int t = t0;  // the band of this pass
      zd curv[9];
      if (pos) {
        const zd* On = Om + k * 9 * (int64_t)n2 + 9 * ((int64_t)t + (int64_t)n * t);
        for (int q = 0; q < 9; ++q) curv[q] = On[q];
      } else {
        for (int q = 0; q < 9; ++q) curv[q] = zd{0.0, 0.0};
        for (int np = 0; np < n; ++np) {
          if (np == t) continue;
          const double dEE = (Es[np] - Es[t]) * (Es[np] - Es[t]);
          if (fabs(dEE) < b.kubo_tol) continue;
          for (int j = 0; j < 3; ++j)
            for (int a = 0; a < 3; ++a)
              curv[a + 3 * j].re +=
                  zmul(Vat(a, t, np), Vat(j, np, t)).im / dEE;
        }
        for (int q = 0; q < 9; ++q) curv[q] = zscale(curv[q], -2.0);
      }
      for (int c = 0; c < 3; ++c) {
        zd s = zd{0.0, 0.0};
        for (int bb = 0; bb < 3; ++bb)
          for (int a = 0; a < 3; ++a) {
            const int l = levi3(a, bb, c);
            if (l) s = zadd(s, zscale(curv[a + 3 * bb], (double)l));
          }
        omg[c + 3 * t] = s;
      }
    }
    __syncthreads();
    // ---- kubo_opt_tens -------------------------------------------------------
    // pairs (nn, m) in chunks of records amn_ab = (E_m - E_nn) A_a(nn,m) A_b(m,nn)
    // in the work area; a record's weights are formed once an item for all nine
    // components (n = 14, 2,730 k-points, 16 items: 211 us with the gyrotropic
    // sums; one thread a component and item, with A from L2: about 500 us)
    if (doOpt && pos)
      for (int pass = 0; pass < npass; ++pass) {
        const int g0 = pass * XS_THREADS;
        const int IW = (NI - g0 < XS_THREADS) ? NI - g0 : XS_THREADS;
        const int S = XS_THREADS / IW, slot = t % IW, split = t / IW;
        const int h = (g0 + slot) % nhw, ef = (g0 + slot) / nhw;
        const double hwv = b.hw[h];
        zd* rc = reinterpret_cast<zd*>(work);
        const int chunk = nwork / 18 < XS_THREADS ? nwork / 18 : XS_THREADS;
        for (int p0 = 0; p0 < n2; p0 += chunk) {
          const int np = n2 - p0 < chunk ? n2 - p0 : chunk;
          __syncthreads();
          for (int e = t; e < np; e += XS_THREADS) {
            const int nn = (p0 + e) % n, m = (p0 + e) / n;
            const double dE = Es[m] - Es[nn];
            zd x[3], y[3];
#pragma unroll
            for (int a = 0; a < 3; ++a) {
              x[a] = Aat(k, a, nn, m);
              y[a] = Aat(k, a, m, nn);
            }
#pragma unroll
            for (int q = 0; q < 9; ++q) rc[9 * e + q] = zscale(zmul(x[q % 3], y[q / 3]), dE);
          }
          __syncthreads();
          if (split < S)
            for (int e = split; e < np; e += S) {
              const int nn = (p0 + e) % n, m = (p0 + e) / n;
              if (nn == m) continue;
              const double dE = Es[m] - Es[nn], x = dE - hwv;
              const double df = wk * (fd[ef + nef * m] - fd[ef + nef * nn]);
              // pi times delta_broad: Im 1 / (dE - hw - i eta)
              const double u = df * (eta / (x * x + eta * eta)), v = df / x;
#pragma unroll
              for (int q = 0; q < 9; ++q) {
                const zd g = rc[9 * e + q];
                ox[q].re = fma(g.re, u, ox[q].re);
                ox[q].im = fma(g.im, u, ox[q].im);
                oy[q].re = fma(g.re, v, oy[q].re);
                oy[q].im = fma(g.im, v, oy[q].im);
              }
            }
        }
        if (npass > 1) opt_flush(g0);
      }
    // ---- photo_2nd_cond above 32 bands (photo_kernel's sums): item
    // (a, b, c, hw, ef) -------------------------------------------------------
    if (photo) {
      // P in LDS (n <= 64), else in the workgroup's slot of scr
      const bool pl = ext_photo_p(n, nef);
      // the m sum does not depend on a, hw or E_F: per (b, c) the product
      // P(l, n) = sum_m V_b(l, m) V_c(m, n) / (E_n - E_m - i eta); then each
      // item (a, hw, E_F) is the O(n^2) contraction with V_a(n, l) (n^3 per
      // (b, c) instead of per item).  Items are split over the threads:
      // thread (slot, split), splits combined in a fixed order.
      zd* Pm = pl ? reinterpret_cast<zd*>(work) : scr + (int64_t)blockIdx.x * n2;
      zd* red = pl ? Pm + n2 : reinterpret_cast<zd*>(work);  // [XS_THREADS]
      const int NI = 3 * nhw * nef;
      for (int c = 0; c < 3; ++c) {
        for (int bb = 0; bb < 3; ++bb) {
          __syncthreads();  // the previous P's readers are done
          for (int e = t; e < n2; e += XS_THREADS) {
            const int l = e % n, nn = e / n;
            zd sp = zd{0.0, 0.0};
            for (int m = 0; m < n; ++m) {
              const double x = Es[nn] - Es[m], iv = 1.0 / (x * x + eta * eta);
              sp = zadd(sp, zmul(Vat(bb, l, m), zmul(Vat(c, m, nn), zd{x * iv, eta * iv})));
            }
            Pm[e] = sp;
          }
          __syncthreads();
          for (int g0 = 0; g0 < NI; g0 += XS_THREADS) {
            const int IW = (NI - g0 < XS_THREADS) ? NI - g0 : XS_THREADS;
            const int S = XS_THREADS / IW, slot = t % IW, split = t / IW;
            const int it = g0 + slot, a = it % 3, h = (it / 3) % nhw, ef = it / (3 * nhw);
            const double hwv = b.hw[h];
            zd acc = zd{0.0, 0.0};
            if (split < S)
              for (int pp = split; pp < n2; pp += S) {
                const int l = pp % n, nn = pp / n;
                if (l == nn) continue;
                const double df = fd[ef + nef * l] - fd[ef + nef * nn];
                const double x = Es[nn] - Es[l];
                const double xp = x + hwv, xm = x - hwv, e2 = 4.0 * eta * eta;
                const double ip = 1.0 / (xp * xp + e2), im = 1.0 / (xm * xm + e2);
                const zd sh = zd{xp * ip + xm * im, 2.0 * eta * (ip + im)};
                acc = zadd(acc, zscale(zmul(zmul(Vat(a, nn, l), Pm[pp]), sh), df));
              }
            red[t] = acc;
            __syncthreads();
            if (split == 0) {
              zd sum = red[slot];
              for (int u = 1; u < S; ++u) sum = zadd(sum, red[slot + IW * u]);
              const int q = a + 3 * bb + 9 * c;
              const int64_t o = 2 * (q + 27 * (h + (int64_t)nhw * ef));
              rec[X.photo + o] += wk * (sum.re / (hwv * hwv));
              rec[X.photo + o + 1] += wk * (sum.im / (hwv * hwv));
            }
            __syncthreads();  // red is free again
          }
        }
      }
    }
    // ---- gyrotropic C, D: item (a, b, ef); Dw: item (a, b, hw, ef) -----------
    if (doGyro) {
      for (int it = t; it < 9 * nef; it += XS_THREADS) {
        const int q = it % 9, ef = it / 9, a = q % 3, bb = q / 3;
        zd c = zd{0.0, 0.0}, d = zd{0.0, 0.0};
        for (int nn = 0; nn < n; ++nn) {
          const zd va = Vat(a, nn, nn), vb = Vat(bb, nn, nn);
          const double f = fdd[ef + nef * nn];
          c = zadd(c, zscale(zmul(va, vb), f));
          d = zsub(d, zscale(zmul(va, omg[bb + 3 * nn]), f));
        }
        rec[X.gyro_C + 2 * it] += wk * c.re;
        rec[X.gyro_C + 2 * it + 1] += wk * c.im;
        rec[X.gyro_D + 2 * it] += wk * d.re;
        rec[X.gyro_D + 2 * it + 1] += wk * d.im;
      }
      // get_curvTilde_hw (gyro.f90:271-300) of (band, hw), three components,
      // for as many frequencies as the work area holds, then the items
      const int hc = nwork / (3 * n);  // at least 1 (ext_work)
      if (pos)
        for (int h0 = 0; h0 < nhw; h0 += hc) {
          const int nh = nhw - h0 < hc ? nhw - h0 : hc;
          __syncthreads();
          for (int e = t; e < n * nh; e += XS_THREADS) {
            const int nn = e % n, hh = e / n;
            const double hwv = b.hw[h0 + hh];
            double om[3] = {0.0, 0.0, 0.0};
            for (int m = 0; m < n; ++m) {
              if (m == nn) continue;
              const double ww = (Es[m] - Es[nn]) * (Es[m] - Es[nn]), g = ww / (ww - hwv);
              zd x[3], y[3];
#pragma unroll
              for (int a = 0; a < 3; ++a) {
                x[a] = Aat(k, a, nn, m);
                y[a] = Aat(k, a, m, nn);
              }
#pragma unroll
              for (int c = 0; c < 3; ++c) {
                const int b1 = (c + 1) % 3, b2 = (c + 2) % 3;
                om[c] -= zsub(zmul(x[b1], y[b2]), zmul(x[b2], y[b1])).im * g;
              }
            }
#pragma unroll
            for (int c = 0; c < 3; ++c) work[c + 3 * e] = om[c];
          }
          __syncthreads();
          for (int it = t; it < 9 * nh * nef; it += XS_THREADS) {
            const int q = it % 9, hh = (it / 9) % nh, ef = it / (9 * nh), a = q % 3, bb = q / 3;
            zd dw = zd{0.0, 0.0};
            for (int nn = 0; nn < n; ++nn)
              dw = zsub(dw, zscale(Vat(a, nn, nn), work[bb + 3 * (nn + n * hh)] * fdd[ef + nef * nn]));
            const int64_t o = 2 * (q + 9 * (h0 + hh + (int64_t)nhw * ef));
            rec[X.gyro_Dw + o] += wk * dw.re;
            rec[X.gyro_Dw + o + 1] += wk * dw.im;
          }
        }
    }
  }
  if (doOpt && pos && npass == 1) opt_flush(0);
}

// V in LDS for n <= 32 where it fits beside the tables; otherwise it is read
// from L2 / HBM
static bool ext_ldsv(const BandArgs& b) {
  return b.n <= XS_NMAX &&
         sizeof(double) * (ext_base_doubles(b.n, b.n_ef, true) + ext_work(b, true)) <= XS_LDS;
}

size_t ext_lds_bytes(const BandArgs& b) {
  const bool ldsv = ext_ldsv(b);
  return sizeof(double) * (ext_base_doubles(b.n, b.n_ef, ldsv) + ext_work(b, ldsv));
}

size_t extsum_scratch(const BandArgs& b, int nblocks) {
  const bool slots = (b.jobs & MEP_JOB_OPT) && !photo_fast(b) && !ext_photo_p(b.n, b.n_ef);
  return slots ? sizeof(zd) * (size_t)b.n * b.n * nblocks : 0;
}

void launch_extsum(hipStream_t s, const BandArgs& b, int64_t nk, const double* E, const zd* V,
                   const zd* A, const zd* Om, const double* w, int nblocks, double* part,
                   zd* scr) {
  ExtLayout X = ext_layout(b);
  const double kB = 8.6173303 * 1e-5 / 27.211385;  // kBoltz_Eh_K (constants.f90:22)
  const size_t lds = ext_lds_bytes(b);
  const bool fast = photo_fast(b), photo = (b.jobs & MEP_JOB_OPT) && !fast;
  if (fast) {
    const size_t pl = photo_lds(b);
    const dim3 grid(nblocks, (unsigned)(((int64_t)b.n_hw * b.n_ef + XS_THREADS - 1) / XS_THREADS));
    auto go = [&](auto kernel) {
      (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)pl);
      hipLaunchKernelGGL(kernel, grid, dim3(XS_THREADS), pl, s, b, kB * b.T_kelvin, X, nk, E, V, w,
                         part);
    };
    if (b.n <= 16) go(photo_kernel<16>);
    else go(photo_kernel<32>);
  }
  const bool ldsv = ext_ldsv(b);
  const int nwork = (int)ext_work(b, ldsv);
  auto go = [&](auto kernel) {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    hipLaunchKernelGGL(kernel, dim3(nblocks), dim3(XS_THREADS), lds, s, b, kB * b.T_kelvin, X, nk, E,
                       V, A, Om, w, part, scr, photo, nwork);
  };
  if (ldsv) go(extsum_kernel<true>);
  else go(extsum_kernel<false>);
}
