// mep_mlp.hip -- the learned part of adaptive k refinement.
//
// A small MLP predicts log|Omega(k)| from sin/cos Fourier features of k:
//   features  x = [sin(2 pi m k_a), cos(2 pi m k_a)], m = 1..n_freq, a = x,y,z
//             (6 n_freq values, zero-padded to FP, a multiple of 16)
//   layers    h1 = tanh(x W1 + b1), h2 = tanh(h1 W2 + b2), h3 = tanh(h2 W3 + b3),
//             y = h3 W4 + b4 (W4 padded to 16 output columns; column 0 is y)
// FP32 weights.  One training step is three launches, whatever the batch:
//   mlp_rows_kernel    a tile of rows through features, the three layers, the
//                      output, the error and back to dZ3, dZ2, dZ1
//   mlp_wgrad_kernel   the weight gradients H^T dZ, the batch split over waves
//   mlp_update_kernel  the splits' sum in a fixed order, and the Adam update
// (inference is mlp_rows_kernel alone, without its backward half).
// A step of 4,096 rows at H = 128 takes 40 us (20 + 14 + 6); as separate
// products, activations and one-thread-a-column sums over the batch it took
// 2.8 ms, of which the four column sums 1.4 ms and the unsplit weight-gradient
// products most of the rest.
// Parameter layout (floats): W1[FP][H] b1[H] W2[H][H] b2[H] W3[H][H] b3[H]
// W4[H][16] b4[16], matrices row-major (input index slow).  Column 0 of W4
// and b4[0] are the output; the other columns are padding.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <numeric>
#include <random>
#include <string>
#include <vector>

#include "../../include/mepinterp.h"

typedef float mlp_v4f __attribute__((ext_vector_type(4)));

extern void mep_set_error(const std::string& msg);  // mep_capi.hip

namespace {

constexpr int OUTP = 16;  // padded output width

constexpr int OUTP_SHIFT = 4;
constexpr int ROWS_THREADS = 512;  // mlp_rows_kernel: 8 wavefronts

// offsets of the parameter blocks
struct MlpDims {
  int nfreq, F, FP, H;
  int64_t P, oW1, ob1, oW2, ob2, oW3, ob3, oW4, ob4;
};

// activations of one batch, row-major: X [B][FP], h[l] and z[l] [B][H], dy [B]
struct MlpActs {
  float* X;
  float* h[3];
  float* z[3];
  float* dy;
  double* loss;  // one partial sum per row tile
};

// B fragments of one 16-column tile for K (a multiple of 16) values of k, from
// the weights: BT = false: B(k, c) = W[k ldw + c], BT = true: B(k, c) =
// W[c ldw + k].  Lane l holds the k-values k0 + 4 (l / 16) .. + 3 of column c.
template <bool BT>
__device__ inline mlp_v4f rows_wfrag(int k0, const float* __restrict__ W, int ldw, int c) {
  const int kk = k0 + 4 * ((threadIdx.x & 63) >> 4);
  if (BT) return *reinterpret_cast<const mlp_v4f*>(W + (int64_t)c * ldw + kk);
  mlp_v4f b;
#pragma unroll
  for (int j = 0; j < 4; ++j) b[j] = W[(int64_t)(kk + j) * ldw + c];
  return b;
}
// acc[t] += in(16 t .. 16 t + 15, k0 .. k0 + 15) B: in is a row tile in LDS
// (leading dimension ld).  A lane's four k-values are one 16-byte LDS access
// and feed four MFMA steps; the order of the sum over k is permuted the same
// way in B.
template <int RT>
__device__ inline void rows_mfma(int k0, const float* in, int ld, mlp_v4f b, mlp_v4f* acc) {
  const int lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    const mlp_v4f a = *reinterpret_cast<const mlp_v4f*>(in + (16 * t + lr) * ld + k0 + 4 * lk);
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], b[j], acc[t], 0, 0, 0);
  }
}
template <int RT, bool BT>
__device__ inline void rows_gemm(int K, const float* in, int ld, const float* __restrict__ W,
                                 int ldw, int c, mlp_v4f* acc) {
#pragma unroll 8
  for (int k0 = 0; k0 < K; k0 += 16) rows_mfma<RT>(k0, in, ld, rows_wfrag<BT>(k0, W, ldw, c), acc);
}

constexpr int REG_H = 16 * (ROWS_THREADS / 64);  // one column tile per wavefront
constexpr int REG_K = REG_H / 16;

// the fragments of a whole layer (K <= REG_H) in registers
template <bool BT>
__device__ inline void rows_wload(int K, const float* __restrict__ W, int ldw, int c, mlp_v4f* b) {
#pragma unroll
  for (int i = 0; i < REG_K; ++i)
    if (16 * i < K) b[i] = rows_wfrag<BT>(16 * i, W, ldw, c);
}
template <int RT>
__device__ inline void rows_gemm_reg(int K, const float* in, int ld, const mlp_v4f* b, mlp_v4f* acc) {
#pragma unroll
  for (int i = 0; i < REG_K; ++i)
    if (16 * i < K) rows_mfma<RT>(16 * i, in, ld, b[i], acc);
}

// The batch's row tiles in the order of the launch: workgroups b, b + 8, ...
// share an XCD, and the four 16-row (two 32-row) tiles of one 64-row split of
// mlp_wgrad_kernel go to the XCD that sums that split.
template <int RT>
__device__ inline int64_t rows_tile(int64_t b, int64_t nb) {
  constexpr int S = 4 / RT;  // tiles per split
  if (nb % (8 * S)) return b;
  const int64_t j = b >> 3;
  return ((j / S) * 8 + (b & 7)) * S + j % S;
}

// One tile of 16 RT rows per workgroup.  The tile's activations pass from
// layer to layer through two LDS buffers [16 RT][ld]; the weights come from
// L2 (every workgroup reads all of them once, twice in training).  TRAIN also
// writes X, h and z for the weight gradients.  Rows >= rows (padding of the
// batch) carry zero features and a zero error.
// Bound by the latency of the weight loads.  REG (H <= 128 and FP <= 128: a
// wavefront owns one column tile) therefore keeps a layer's weights in
// registers, loaded one or two layers ahead, and the thread's own h values
// for the way back (4,096 rows, H = 128: 36 -> 20 us in training, 17 -> 13 us
// in inference); otherwise the weights are loaded in the loops and each thread
// reads back h values that it wrote itself.
template <int RT, bool TRAIN, bool REG>
__global__ __launch_bounds__(ROWS_THREADS) void mlp_rows_kernel(
    MlpDims d, int64_t rows, const double* __restrict__ kpts, const int64_t* __restrict__ idx,
    const float* __restrict__ t, const float* __restrict__ p, MlpActs g, float* __restrict__ out) {
  extern __shared__ float4 mlp_lds[];
  constexpr int R = 16 * RT;
  const int H = d.H, FP = d.FP, ld = (H > FP ? H : FP) + 4;
  float* cur = reinterpret_cast<float*>(mlp_lds);
  float* nxt = cur + R * ld;
  float* sdy = nxt + R * ld;                           // [R]
  double* se = reinterpret_cast<double*>(sdy + R);     // [R] squared errors
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, lr = lane & 15, lk = lane >> 4;
  const int64_t r0 = (TRAIN ? rows_tile<RT>(blockIdx.x, gridDim.x) : (int64_t)blockIdx.x) * R;
  const int64_t oW[3] = {d.oW1, d.oW2, d.oW3}, ob[3] = {d.ob1, d.ob2, d.ob3};
  const int cw = 16 * w + lr;         // the wavefront's (first) column
  const bool own = 16 * w < H;        // wave-uniform
  mlp_v4f wa[REG_K] = {}, wb[REG_K] = {}, wc[REG_K] = {};
  float hr[3][RT][4] = {};
  if (REG && own) {
    rows_wload<false>(FP, p + oW[0], H, cw, wa);
    rows_wload<false>(H, p + oW[1], H, cw, wb);
    rows_wload<false>(H, p + oW[2], H, cw, wc);
  }

  // features of row r: sin, cos of 2 pi m k_a at a 2 nfreq + 2 (m - 1)
  const int nsc = 3 * d.nfreq;
  for (int i = tid; i < R * nsc; i += ROWS_THREADS) {
    const int r = i / nsc, q = i - r * nsc, a = q / d.nfreq, m = q - a * d.nfreq;
    double sn = 0.0, cs = 0.0;
    if (r0 + r < rows) {
      const int64_t s = idx ? idx[r0 + r] : r0 + r;
      sincos(6.283185307179586476925 * (m + 1) * kpts[3 * s + a], &sn, &cs);
    }
    cur[r * ld + 2 * q] = (float)sn;
    cur[r * ld + 2 * q + 1] = (float)cs;
  }
  const int npad = FP - d.F;
  for (int i = tid; i < R * npad; i += ROWS_THREADS)
    cur[(i / npad) * ld + d.F + i % npad] = 0.f;
  __syncthreads();
  if (TRAIN)
    for (int i = tid; i < R * FP; i += ROWS_THREADS)
      g.X[(r0 + i / FP) * FP + i % FP] = cur[(i / FP) * ld + i % FP];

#pragma unroll
  for (int l = 0; l < 3; ++l) {
    for (int c0 = 16 * w; c0 < H; c0 += REG_H) {
      const int c = c0 + lr;
      const float bias = p[ob[l] + c];
      mlp_v4f acc[RT] = {};
      if (REG)
        rows_gemm_reg<RT>(l == 0 ? FP : H, cur, ld, l == 0 ? wa : (l == 1 ? wb : wc), acc);
      else
        rows_gemm<RT, false>(l == 0 ? FP : H, cur, ld, p + oW[l], H, c, acc);
      // the weights of the way back: W3^T into wa, then W2^T into wb
      if (REG && TRAIN && l == 0) rows_wload<true>(H, p + oW[2], H, cw, wa);
      if (REG && TRAIN && l == 1) rows_wload<true>(H, p + oW[1], H, cw, wb);
#pragma unroll
      for (int q = 0; q < RT; ++q)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int r = 16 * q + 4 * lk + v;
          const float h = tanhf(acc[q][v] + bias);
          nxt[r * ld + c] = h;
          if (REG) hr[l][q][v] = h;
          if (TRAIN) g.h[l][(r0 + r) * H + c] = h;
        }
    }
    __syncthreads();
    float* x = cur;
    cur = nxt;
    nxt = x;
  }

  const float* W4 = p + d.oW4;
  for (int r = w; r < R; r += ROWS_THREADS / 64) {
    float y = 0.f;
    for (int c = lane; c < H; c += 64) y += cur[r * ld + c] * W4[c << OUTP_SHIFT];
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) y += __shfl_xor(y, o, 64);
    y += p[d.ob4];
    if (lane == 0) {
      if (!TRAIN) {
        if (r0 + r < rows) out[r0 + r] = y;
      } else {
        float e = 0.f;
        if (r0 + r < rows) e = y - t[idx ? idx[r0 + r] : r0 + r];
        sdy[r] = 2.f * e * (1.f / (float)rows);
        se[r] = (double)e * (double)e;
        g.dy[r0 + r] = sdy[r];
      }
    }
  }
  if (!TRAIN) return;
  __syncthreads();
  if (tid == 0) {
    double s = 0.0;
    for (int r = 0; r < R; ++r) s += se[r];
    g.loss[r0 / R] = s;
  }
  // dZ3 = dy W4^T (1 - h3^2) in place, then dZ2 and dZ1 through the layers
  for (int c0 = 16 * w; c0 < H; c0 += REG_H) {
    const int c = c0 + lr;
    const float w4 = W4[c << OUTP_SHIFT];
#pragma unroll
    for (int q = 0; q < RT; ++q)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int r = 16 * q + 4 * lk + v;
        const float h = REG ? hr[2][q][v] : cur[r * ld + c];
        const float z = sdy[r] * w4 * (1.f - h * h);
        cur[r * ld + c] = z;
        g.z[2][(r0 + r) * H + c] = z;
      }
  }
  __syncthreads();
#pragma unroll
  for (int l = 1; l >= 0; --l) {
    for (int c0 = 16 * w; c0 < H; c0 += REG_H) {
      const int c = c0 + lr;
      float h[RT][4];
#pragma unroll
      for (int q = 0; q < RT; ++q)
#pragma unroll
        for (int v = 0; v < 4; ++v)
          h[q][v] = REG ? hr[l][q][v] : g.h[l][(r0 + 16 * q + 4 * lk + v) * H + c];
      mlp_v4f acc[RT] = {};
      if (REG)
        rows_gemm_reg<RT>(H, cur, ld, l ? wa : wb, acc);
      else
        rows_gemm<RT, true>(H, cur, ld, p + oW[l + 1], H, c, acc);
#pragma unroll
      for (int q = 0; q < RT; ++q)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int r = 16 * q + 4 * lk + v;
          const float z = acc[q][v] * (1.f - h[q][v] * h[q][v]);
          if (l) nxt[r * ld + c] = z;
          g.z[l][(r0 + r) * H + c] = z;
        }
    }
    __syncthreads();
    float* x = cur;
    cur = nxt;
    nxt = x;
  }
}

// Partial gradients of one split of the batch (rows [s RS, min(B, (s + 1) RS)),
// RS and B multiples of 4): one wavefront per 32 x 32 block of W1, W2 or W3
// (two A and two B values per lane feed four MFMA steps, so a block reads a
// quarter of what single tiles would), and one per 64 rows of W4.  The blocks
// of the first row also sum the columns of dZ for the bias.  part[s] has the
// parameter layout; the padding columns of W4 and b4 are not written.
// Without the split the 144 tiles of H = 128 would be 144 waves of 4096
// serial rows; with 64 rows a split they are 2,304 waves of 36 blocks.
__global__ __launch_bounds__(256) void mlp_wgrad_kernel(MlpDims d, int B, int RS, int nsplit,
                                                        MlpActs g, float* __restrict__ part) {
  const int lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
  const int H = d.H;
  const int nn = (H + 31) / 32, m1 = (d.FP + 31) / 32;
  const int per = (m1 + 2 * nn) * nn + (H + 63) / 64;
  // workgroups b, b + 8, ... share an XCD: one split's blocks stay on one, so
  // that its rows are read into one L2 only
  const int wgs = (per + 3) / 4, j = blockIdx.x >> 3;
  const int s = (j / wgs) * 8 + (blockIdx.x & 7);
  int it = (j % wgs) * 4 + (threadIdx.x >> 6);
  if (s >= nsplit || it >= per) return;
  const int k_lo = s * RS, k_hi = (B < k_lo + RS) ? B : k_lo + RS;
  float* ps = part + (int64_t)s * d.P;
  if (it >= (m1 + 2 * nn) * nn) {  // W4 and b4: H3^T dy
    const int c = 64 * (it - (m1 + 2 * nn) * nn) + lane;
    float a = 0.f, sb = 0.f;
    const int cc = c < H ? c : H - 1;
#pragma unroll 8
    for (int k = k_lo; k < k_hi; ++k) {
      const float e = g.dy[k];
      a += g.h[2][(int64_t)k * H + cc] * e;
      sb += e;
    }
    if (c < H) ps[d.oW4 + ((int64_t)c << OUTP_SHIFT)] = a;
    if (c == 0) ps[d.ob4] = sb;
    return;
  }
  const int l = it < m1 * nn ? 0 : (it < (m1 + nn) * nn ? 1 : 2);
  if (l == 1) it -= m1 * nn;
  if (l == 2) it -= (m1 + nn) * nn;
  const int M = l == 0 ? d.FP : H;
  const float* __restrict__ Am = l == 0 ? g.X : (l == 1 ? g.h[0] : g.h[1]);
  const float* __restrict__ Bm = l == 0 ? g.z[0] : (l == 1 ? g.z[1] : g.z[2]);
  const int64_t oW = l == 0 ? d.oW1 : (l == 1 ? d.oW2 : d.oW3);
  const int64_t ob = l == 0 ? d.ob1 : (l == 1 ? d.ob2 : d.ob3);
  const int mi = it / nn, m0 = 32 * mi, n0 = 32 * (it % nn);
  // M and H are multiples of 16: the second half block may be absent; its
  // loads then repeat the first half and its products are not stored
  const int m1off = m0 + 16 < M ? 16 : 0, n1off = n0 + 16 < H ? 16 : 0;
  const float* pa = Am + (int64_t)(k_lo + lk) * M + m0 + lr;
  const float* pb = Bm + (int64_t)(k_lo + lk) * H + n0 + lr;
  mlp_v4f acc[2][2] = {};
  float sb0 = 0.f, sb1 = 0.f;
#pragma unroll 16
  for (int k = k_lo; k < k_hi; k += 4) {
    const float a0 = pa[0], a1 = pa[m1off], b0 = pb[0], b1 = pb[n1off];
    pa += 4 * (int64_t)M;
    pb += 4 * (int64_t)H;
    acc[0][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a0, b0, acc[0][0], 0, 0, 0);
    acc[0][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a0, b1, acc[0][1], 0, 0, 0);
    acc[1][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a1, b0, acc[1][0], 0, 0, 0);
    acc[1][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a1, b1, acc[1][1], 0, 0, 0);
    sb0 += b0;
    sb1 += b1;
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      if ((i && !m1off) || (j && !n1off)) continue;
#pragma unroll
      for (int v = 0; v < 4; ++v)
        ps[oW + (int64_t)(m0 + 16 * i + 4 * lk + v) * H + n0 + 16 * j + lr] = acc[i][j][v];
    }
  if (mi == 0) {
    sb0 += __shfl_xor(sb0, 16, 64);
    sb1 += __shfl_xor(sb1, 16, 64);
    sb0 += __shfl_xor(sb0, 32, 64);
    sb1 += __shfl_xor(sb1, 32, 64);
    if (lk == 0) {
      ps[ob + n0 + lr] = sb0;
      if (n1off) ps[ob + n0 + 16 + lr] = sb1;
    }
  }
}

// Sum of the splits in order, then the gradient is stored (grad != null) or
// applied (Adam).  The last block sums the tiles' losses, in a fixed order.
__global__ __launch_bounds__(256) void mlp_update_kernel(
    MlpDims d, int nsplit, const float* __restrict__ part, int ntile, int64_t rows,
    const double* __restrict__ tloss, double* __restrict__ loss_out, float* __restrict__ grad,
    float* __restrict__ p, float* __restrict__ m, float* __restrict__ v, float lr, float b1,
    float b2, float eps, float c1, float c2) {
  if (blockIdx.x == gridDim.x - 1) {
    __shared__ double red[256];
    double s = 0.0;
    for (int i = threadIdx.x; i < ntile; i += 256) s += tloss[i];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
      if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
      __syncthreads();
    }
    if (threadIdx.x == 0) *loss_out = red[0] / (double)rows;
    return;
  }
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= d.P) return;
  const bool pad = (i >= d.oW4 && i < d.ob4 && ((i - d.oW4) & (OUTP - 1))) || i > d.ob4;
  float gi = 0.f;
  if (!pad) {
#pragma unroll 8
    for (int s = 0; s < nsplit; ++s) gi += part[(int64_t)s * d.P + i];
  }
  if (grad) {
    grad[i] = gi;
    return;
  }
  const float mi = b1 * m[i] + (1.f - b1) * gi;
  const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

inline unsigned nblk(int64_t n, int b) { return (unsigned)((n + b - 1) / b); }

}  // namespace

struct mep_mlp {
  MlpDims d;
  float* dp = nullptr;    // parameters, Adam moments m and v, gradient: 4 P floats
  int64_t bcap = 0;
  float* dact = nullptr;  // activations, errors and losses of one batch
  int64_t pcap = 0;
  float* dpart = nullptr; // partial gradients, one per split
  double* dloss = nullptr;
  int64_t lcap = 0;
  int64_t dcap = 0;  // training / prediction data capacity (k-points)
  double* dk = nullptr;
  float* dt = nullptr;
  int64_t* didx = nullptr;
  float* dout = nullptr;
  hipStream_t st = nullptr;
  int64_t step = 0;
};

namespace {

#define MLP_HIP(x)                                                          \
  do {                                                                      \
    hipError_t e_ = (x);                                                    \
    if (e_ != hipSuccess) {                                                 \
      mep_set_error(std::string(#x) + ": " + hipGetErrorString(e_));        \
      return MEP_ERR_HIP;                                                   \
    }                                                                       \
  } while (0)

// rows of one split of the weight gradients: a multiple of 64, and at most 64
// splits
int split_rows(int64_t B) { return (int)((((B + 63) / 64 + 63) / 64) * 64); }

int ensure_batch(mep_mlp* q, int64_t B) {
  const int64_t nsplit = (B + split_rows(B) - 1) / split_rows(B);
  if (nsplit > q->pcap) {
    hipFree(q->dpart);
    q->dpart = nullptr;
    q->pcap = 0;
    MLP_HIP(hipMalloc(&q->dpart, sizeof(float) * nsplit * q->d.P));
    q->pcap = nsplit;
  }
  if (B <= q->bcap) return MEP_OK;
  hipFree(q->dact);
  q->dact = nullptr;
  q->bcap = 0;
  // X, h, z, dy and (double) one loss per 16 rows
  MLP_HIP(hipMalloc(&q->dact, sizeof(float) * B * (q->d.FP + 6 * q->d.H + 1) + sizeof(double) * (B / 16)));
  q->bcap = B;
  return MEP_OK;
}

MlpActs acts(const mep_mlp* q) {
  const int64_t B = q->bcap, H = q->d.H;
  MlpActs g;
  g.loss = reinterpret_cast<double*>(q->dact);  // first: 8-byte aligned
  g.X = reinterpret_cast<float*>(g.loss + B / 16);
  float* f = g.X + B * q->d.FP;
  for (int l = 0; l < 3; ++l) {
    g.h[l] = f + l * B * H;
    g.z[l] = f + (3 + l) * B * H;
  }
  g.dy = f + 6 * B * H;
  return g;
}

// epochs whose permutations of n points fit 1 MB (at least one)
constexpr int64_t PERM_MIN = 1 << 17;
int64_t perm_epochs(int64_t n) { return std::max<int64_t>(1, PERM_MIN / n); }
// one of the two device buffers for them, for data of any size up to n
int64_t perm_half(int64_t n) { return std::max<int64_t>(n, PERM_MIN); }

int ensure_data(mep_mlp* q, int64_t n) {
  if (n <= q->dcap) return MEP_OK;
  hipFree(q->dk); hipFree(q->dt); hipFree(q->didx); hipFree(q->dout);
  MLP_HIP(hipMalloc(&q->dk, sizeof(double) * 3 * n));
  MLP_HIP(hipMalloc(&q->dt, sizeof(float) * n));
  MLP_HIP(hipMalloc(&q->didx, sizeof(int64_t) * 2 * perm_half(n)));
  MLP_HIP(hipMalloc(&q->dout, sizeof(float) * n));
  q->dcap = n;
  return MEP_OK;
}

// Two events of a training run; destroyed once the stream is done with the
// host buffers, also when the run returns early.
struct EventPair {
  hipEvent_t e[2] = {nullptr, nullptr};
  ~EventPair() {
    for (hipEvent_t x : e)
      if (x) {
        hipEventSynchronize(x);
        hipEventDestroy(x);
      }
  }
};

size_t rows_lds(const MlpDims& d, int rt) {
  const int ld = std::max(d.H, d.FP) + 4;
  return sizeof(float) * (size_t)(2 * 16 * rt * ld + 16 * rt) + sizeof(double) * 16 * rt;
}

// Row tiles of 32 halve the weight reads from 8,192 rows on (a tile for every
// CU either way) where two of their buffers fit in LDS; tiles of 16 below.
bool wide_tiles(const MlpDims& d, int64_t B) { return B >= 8192 && rows_lds(d, 2) <= 160 * 1024; }

template <bool TRAIN>
int launch_rows(mep_mlp* q, int64_t B, int64_t rows, const double* kpts, const int64_t* idx,
                const float* t, const MlpActs& g, float* out, int* ntile) {
  const int rt = wide_tiles(q->d, B) ? 2 : 1;
  const bool reg = q->d.H <= REG_H && q->d.FP <= REG_H;
  const size_t lds = rows_lds(q->d, rt);
  const unsigned nb = nblk(B, 16 * rt);
  auto go = [&](auto kernel) -> int {
    if (lds > 64 * 1024)
      MLP_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(kernel, dim3(nb), dim3(ROWS_THREADS), lds, q->st, q->d, rows, kpts, idx, t,
                       q->dp, g, out);
    return MEP_OK;
  };
  if (ntile) *ntile = (int)nb;
  if (reg) return rt == 2 ? go(mlp_rows_kernel<2, TRAIN, true>) : go(mlp_rows_kernel<1, TRAIN, true>);
  return rt == 2 ? go(mlp_rows_kernel<2, TRAIN, false>) : go(mlp_rows_kernel<1, TRAIN, false>);
}

// loss and gradient of one batch of B rows (`rows` of them real), stored in
// grad or applied as the Adam step q->step
int batch_step(mep_mlp* q, int64_t B, int64_t rows, const int64_t* idx, double* loss, float* grad,
               float lr) {
  const MlpDims& d = q->d;
  const MlpActs g = acts(q);
  int ntile = 0;
  if (int rc = launch_rows<true>(q, B, rows, q->dk, idx, q->dt, g, nullptr, &ntile)) return rc;
  const int RS = split_rows(B), nsplit = (int)((B + RS - 1) / RS);
  const int nn = (d.H + 31) / 32, m1 = (d.FP + 31) / 32;
  const int wgs = ((m1 + 2 * nn) * nn + (d.H + 63) / 64 + 3) / 4;
  hipLaunchKernelGGL(mlp_wgrad_kernel, dim3(8 * ((nsplit + 7) / 8) * wgs), dim3(256), 0, q->st, d, (int)B, RS,
                     nsplit, g, q->dpart);
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  const float c1 = 1.f - std::pow(b1, (float)q->step), c2 = 1.f - std::pow(b2, (float)q->step);
  hipLaunchKernelGGL(mlp_update_kernel, dim3(nblk(d.P, 256) + 1), dim3(256), 0, q->st, d, nsplit,
                     q->dpart, ntile, rows, g.loss, loss, grad, q->dp, q->dp + d.P,
                     q->dp + 2 * d.P, lr, b1, b2, eps, c1, c2);
  return MEP_OK;
}

int64_t round_batch(int64_t b) { return ((std::max<int64_t>(b, 16) + 63) / 64) * 64; }

}  // namespace

extern "C" int mep_mlp_create(int32_t n_freq, int32_t hidden, uint64_t seed, mep_mlp** out) {
  if (!out || n_freq < 1 || n_freq > 64 || hidden < 16 || hidden > 1024 || hidden % 16) {
    mep_set_error("mep_mlp_create: n_freq in [1, 64], hidden a multiple of 16 in [16, 1024]");
    return MEP_ERR_ARG;
  }
  mep_mlp* q = new mep_mlp();
  MlpDims& d = q->d;
  d.nfreq = n_freq;
  d.F = 6 * n_freq;
  d.FP = ((d.F + 15) / 16) * 16;
  d.H = hidden;
  const int64_t H = hidden, FP = d.FP;
  int64_t o = 0;
  d.oW1 = o; o += FP * H;
  d.ob1 = o; o += H;
  d.oW2 = o; o += H * H;
  d.ob2 = o; o += H;
  d.oW3 = o; o += H * H;
  d.ob3 = o; o += H;
  d.oW4 = o; o += H * OUTP;
  d.ob4 = o; o += OUTP;
  d.P = o;
  // seeded uniform +-sqrt(6 / (fan_in + fan_out)) weights, zero biases;
  // padded feature rows and output columns stay zero
  std::vector<float> p((size_t)d.P, 0.f);
  std::mt19937_64 rng(seed);
  auto fill = [&](int64_t off, int64_t fin, int64_t fout, int64_t cols, int64_t rows_used,
                  int64_t cols_used) {
    std::uniform_real_distribution<double> U(-std::sqrt(6.0 / (fin + fout)), std::sqrt(6.0 / (fin + fout)));
    for (int64_t r = 0; r < rows_used; ++r)
      for (int64_t c = 0; c < cols_used; ++c) p[(size_t)(off + r * cols + c)] = (float)U(rng);
  };
  fill(d.oW1, d.F, H, H, d.F, H);
  fill(d.oW2, H, H, H, H, H);
  fill(d.oW3, H, H, H, H, H);
  fill(d.oW4, H, 1, OUTP, H, 1);
  hipError_t e = hipStreamCreate(&q->st);
  if (e == hipSuccess) e = hipMalloc(&q->dp, sizeof(float) * 4 * d.P);
  if (e == hipSuccess) e = hipMemcpy(q->dp, p.data(), sizeof(float) * d.P, hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemset(q->dp + d.P, 0, sizeof(float) * 2 * d.P);
  if (e != hipSuccess) {
    mep_set_error(std::string("mep_mlp_create: ") + hipGetErrorString(e));
    mep_mlp_destroy(q);
    return MEP_ERR_HIP;
  }
  *out = q;
  return MEP_OK;
}

extern "C" int mep_mlp_destroy(mep_mlp* q) {
  if (!q) return MEP_OK;
  hipFree(q->dp); hipFree(q->dact); hipFree(q->dpart); hipFree(q->dloss);
  hipFree(q->dk); hipFree(q->dt); hipFree(q->didx); hipFree(q->dout);
  if (q->st) hipStreamDestroy(q->st);
  delete q;
  return MEP_OK;
}

extern "C" int mep_mlp_num_params(const mep_mlp* q, int64_t* n) {
  if (!q || !n) {
    mep_set_error("mep_mlp_num_params: bad argument");
    return MEP_ERR_ARG;
  }
  *n = q->d.P;
  return MEP_OK;
}

extern "C" int mep_mlp_get_params(mep_mlp* q, float* params) {
  if (!q || !params) {
    mep_set_error("mep_mlp_get_params: bad argument");
    return MEP_ERR_ARG;
  }
  MLP_HIP(hipMemcpyAsync(params, q->dp, sizeof(float) * q->d.P, hipMemcpyDeviceToHost, q->st));
  MLP_HIP(hipStreamSynchronize(q->st));
  return MEP_OK;
}

extern "C" int mep_mlp_set_params(mep_mlp* q, const float* params) {
  if (!q || !params) {
    mep_set_error("mep_mlp_set_params: bad argument");
    return MEP_ERR_ARG;
  }
  MLP_HIP(hipMemcpyAsync(q->dp, params, sizeof(float) * q->d.P, hipMemcpyHostToDevice, q->st));
  MLP_HIP(hipStreamSynchronize(q->st));
  return MEP_OK;
}

extern "C" int mep_mlp_predict(mep_mlp* q, int64_t n, const double* kpts, float* out) {
  if (!q || n < 0 || (n > 0 && (!kpts || !out))) {
    mep_set_error("mep_mlp_predict: bad argument");
    return MEP_ERR_ARG;
  }
  if (n == 0) return MEP_OK;
  if (int rc = ensure_data(q, n)) return rc;
  MLP_HIP(hipMemcpyAsync(q->dk, kpts, sizeof(double) * 3 * n, hipMemcpyHostToDevice, q->st));
  if (int rc = launch_rows<false>(q, n, n, q->dk, nullptr, nullptr, MlpActs{}, q->dout, nullptr))
    return rc;
  MLP_HIP(hipGetLastError());
  MLP_HIP(hipMemcpyAsync(out, q->dout, sizeof(float) * n, hipMemcpyDeviceToHost, q->st));
  MLP_HIP(hipStreamSynchronize(q->st));
  return MEP_OK;
}

extern "C" int mep_mlp_grad(mep_mlp* q, int64_t n, const double* kpts, const float* target,
                            float* grad, float* loss) {
  if (!q || n < 1 || !kpts || !target || !grad) {
    mep_set_error("mep_mlp_grad: bad argument");
    return MEP_ERR_ARG;
  }
  const int64_t B = round_batch(n);
  if (int rc = ensure_batch(q, B)) return rc;
  if (int rc = ensure_data(q, n)) return rc;
  if (!q->dloss) MLP_HIP(hipMalloc(&q->dloss, sizeof(double) * 64));
  q->lcap = std::max<int64_t>(q->lcap, 64);
  MLP_HIP(hipMemcpyAsync(q->dk, kpts, sizeof(double) * 3 * n, hipMemcpyHostToDevice, q->st));
  MLP_HIP(hipMemcpyAsync(q->dt, target, sizeof(float) * n, hipMemcpyHostToDevice, q->st));
  if (int rc = batch_step(q, B, n, nullptr, q->dloss, q->dp + 3 * q->d.P, 0.f)) return rc;
  MLP_HIP(hipGetLastError());
  double l = 0.0;
  MLP_HIP(hipMemcpyAsync(grad, q->dp + 3 * q->d.P, sizeof(float) * q->d.P, hipMemcpyDeviceToHost, q->st));
  MLP_HIP(hipMemcpyAsync(&l, q->dloss, sizeof(double), hipMemcpyDeviceToHost, q->st));
  MLP_HIP(hipStreamSynchronize(q->st));
  if (loss) *loss = (float)l;
  return MEP_OK;
}

extern "C" int mep_mlp_train(mep_mlp* q, int64_t n, const double* kpts, const float* target,
                             int32_t epochs, int32_t batch, float lr, uint64_t seed,
                             float* final_loss) {
  if (!q || n < 1 || !kpts || !target || epochs < 1 || batch < 1 || !(lr > 0.f)) {
    mep_set_error("mep_mlp_train: bad argument");
    return MEP_ERR_ARG;
  }
  const int64_t B = round_batch(std::min<int64_t>(batch, n));
  const int64_t nb = (n + B - 1) / B;
  if (int rc = ensure_batch(q, B)) return rc;
  if (int rc = ensure_data(q, n)) return rc;
  if (nb > q->lcap) {
    hipFree(q->dloss);
    q->dloss = nullptr;
    MLP_HIP(hipMalloc(&q->dloss, sizeof(double) * nb));
    q->lcap = nb;
  }
  MLP_HIP(hipMemcpyAsync(q->dk, kpts, sizeof(double) * 3 * n, hipMemcpyHostToDevice, q->st));
  MLP_HIP(hipMemcpyAsync(q->dt, target, sizeof(float) * n, hipMemcpyHostToDevice, q->st));
  // The permutations go up in chunks of 1, 2, 4, ... epochs (up to 1 MB): the
  // host shuffles the next chunk while the GPU works through this one, and few
  // uploads interrupt the stream.  Two buffers: a host buffer is reused when
  // the copy out of it has ended, a device buffer in stream order.
  const int max_chunk = (int)std::max<int64_t>(1, std::min<int64_t>(epochs, perm_epochs(n)));
  std::vector<int64_t> perm[2];
  EventPair ev;
  int ep = 0;
  for (int c = 0, chunk = 1; ep < epochs; ++c, chunk = std::min(2 * chunk, max_chunk)) {
    const int ne = std::min(chunk, epochs - ep);
    std::vector<int64_t>& pe = perm[c & 1];
    hipEvent_t& e = ev.e[c & 1];
    if (e) MLP_HIP(hipEventSynchronize(e));
    else MLP_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    pe.resize((size_t)(n * ne));
    for (int i = 0; i < ne; ++i) {
      const auto lo = pe.begin() + i * n, hi = lo + n;
      std::iota(lo, hi, (int64_t)0);
      std::mt19937_64 rng(seed + 0x9e3779b97f4a7c15ull * (uint64_t)(ep + i + 1));
      std::shuffle(lo, hi, rng);
    }
    int64_t* di = q->didx + (int64_t)(c & 1) * perm_half(q->dcap);
    MLP_HIP(hipMemcpyAsync(di, pe.data(), sizeof(int64_t) * n * ne, hipMemcpyHostToDevice, q->st));
    MLP_HIP(hipEventRecord(e, q->st));
    for (int i = 0; i < ne; ++i)
      for (int64_t bi = 0; bi < nb; ++bi) {
        const int64_t rows = std::min<int64_t>(B, n - bi * B);
        q->step += 1;
        if (int rc = batch_step(q, B, rows, di + i * n + bi * B, q->dloss + bi, nullptr, lr)) return rc;
      }
    MLP_HIP(hipGetLastError());
    ep += ne;
  }
  MLP_HIP(hipStreamSynchronize(q->st));
  std::vector<double> lb((size_t)nb);
  MLP_HIP(hipMemcpy(lb.data(), q->dloss, sizeof(double) * nb, hipMemcpyDeviceToHost));
  if (final_loss) {
    double s = 0.0, w = 0.0;
    for (int64_t bi = 0; bi < nb; ++bi) {
      const double rows = (double)std::min<int64_t>(B, n - bi * B);
      s += lb[(size_t)bi] * rows;
      w += rows;
    }
    *final_loss = (float)(s / w);
  }
  return MEP_OK;
}
