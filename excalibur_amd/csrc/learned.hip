// Learned bisection brackets: the data the network learns from (Golub-Kahan bidiagonals of
// matrices with prescribed spectra, their singular values by the reference's bisection), the
// network itself (a 3-layer MLP trained in FP32 and run in BF16), and the bisection that starts
// from a proposed bracket once exact Sturm counts have verified it.
//
// Bisection from a bracket keeps the reference's tree (bbtsvd.cpp:19-52: root [0, ||a||^2 +
// ||b||^2], midpoints (lo + hi) / 2, leaf when the width is <= tol or the midpoint equals an
// endpoint). A verified bracket [blo, bhi) holding the target (nc(blo) <= t < nc(bhi) for the
// t-th smallest value) decides every tree node whose midpoint lies outside it without a count: a
// midpoint at or below blo sends the target right, one at or above bhi sends it left, as the
// reference's counts do when they are monotone. Inside the bracket the counts are evaluated as in
// the reference. The leaf, and so the value, is the reference's. A bracket that fails its two
// counts is dropped and the target is bisected from the root.
#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>

#include <algorithm>
#include <cmath>

#include "exc_common.hpp"
#include "gemm.hpp"
#include "sturm.hpp"

#pragma clang fp contract(off)

namespace {

constexpr int kLzThreads = 1024;
constexpr int kLzPerThread = 16;  // n <= 16384

__device__ double block_sum(double v, double* red) {
  v = wave_sum(v);
  const int w = threadIdx.x >> 6, nw = blockDim.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[w] = v;
  __syncthreads();
  double s = 0.0;
  for (int q = 0; q < nw; q++) s += red[q];
  return s;
}

// Golub-Kahan (Lanczos) bidiagonalization of diag(sig) from the start vector v1 = start/||start||:
// alpha_j u_j = D v_j - beta_{j-1} u_{j-1}, beta_j v_{j+1} = D u_j - alpha_j v_j. The upper
// bidiagonal (alpha, beta) is that of A = Q1 diag(sig) Q2^T run from Q2 v1. One workgroup per
// bidiagonal; each thread holds its elements of u, v and sig in registers.
__global__ __launch_bounds__(kLzThreads) void k_gk_lanczos(const int* __restrict__ ns, const long* __restrict__ off,
                                                           const double* __restrict__ sig,
                                                           const double* __restrict__ start, double* __restrict__ d,
                                                           double* __restrict__ e) {
  __shared__ double red[16];
  const int b = blockIdx.x;
  const int n = ns[b];
  const long o = off[b];
  double s[kLzPerThread], u[kLzPerThread], v[kLzPerThread];
  double ss = 0.0;
#pragma unroll
  for (int q = 0; q < kLzPerThread; q++) {
    const int i = threadIdx.x + q * kLzThreads;
    s[q] = i < n ? sig[o + i] : 0.0;
    v[q] = i < n ? start[o + i] : 0.0;
    u[q] = 0.0;
    ss += v[q] * v[q];
  }
  double nrm = sqrt(block_sum(ss, red));
#pragma unroll
  for (int q = 0; q < kLzPerThread; q++) v[q] /= nrm;
  double beta = 0.0;
  for (int j = 0; j < n; j++) {
    ss = 0.0;
#pragma unroll
    for (int q = 0; q < kLzPerThread; q++) {
      u[q] = s[q] * v[q] - beta * u[q];
      ss += u[q] * u[q];
    }
    const double alpha = fmax(sqrt(block_sum(ss, red)), 1e-300);
#pragma unroll
    for (int q = 0; q < kLzPerThread; q++) u[q] /= alpha;
    if (threadIdx.x == 0) d[o + j] = alpha;
    if (j + 1 == n) break;
    ss = 0.0;
#pragma unroll
    for (int q = 0; q < kLzPerThread; q++) {
      v[q] = s[q] * u[q] - alpha * v[q];
      ss += v[q] * v[q];
    }
    beta = fmax(sqrt(block_sum(ss, red)), 1e-300);
#pragma unroll
    for (int q = 0; q < kLzPerThread; q++) v[q] /= beta;
    if (threadIdx.x == 0) e[o + j] = beta;
  }
}

// Per bidiagonal: the reference's bisection root ||a||^2 + ||b||^2 (sequential sums of squares,
// sqrt, then squared, as bbtsvd.cpp:936 with the reference BLAS nrm2) and the scale
// s = sqrt(sum a^2 + sum b^2). One thread per bidiagonal.
__global__ void k_bidiag_scale(int nb, const int* __restrict__ ns, const long* __restrict__ off,
                               const double* __restrict__ d, const double* __restrict__ e, double* __restrict__ root,
                               double* __restrict__ scale) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= nb) return;
  const int n = ns[b];
  const long o = off[b];
  double sa = 0.0, sb = 0.0;
  for (int i = 0; i < n; i++) sa = sa + d[o + i] * d[o + i];
  for (int i = 0; i + 1 < n; i++) sb = sb + e[o + i] * e[o + i];
  const double na = sqrt(sa), nbv = sqrt(sb);
  root[b] = na * na + nbv * nbv;
  scale[b] = sqrt(sa + sb);
}

// Counting-function features: frac[b * K + k] = nc(scale_b * 10^(-k / 2)) / n_b.
__global__ __launch_bounds__(256) void k_count_features(int nb, int K, const int* __restrict__ ns,
                                                        const long* __restrict__ off, const double* __restrict__ d,
                                                        const double* __restrict__ e,
                                                        const double* __restrict__ scale, float* __restrict__ frac) {
  const long g = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= (long)nb * K) return;
  const int b = (int)(g / K), k = (int)(g - (long)b * K);
  const int n = ns[b];
  const double mu = scale[b] * pow(10.0, -0.5 * k);
  frac[g] = (float)sturm_count(n, d + off[b], e + off[b], mu) / (float)n;
}

// One target per lane: the leaf of the reference's tree that holds the i-th largest singular
// value of bidiagonal tb[j] (t = n - 1 - i from below). A proposed bracket [blo, bhi) is checked
// by one exact count per end that lies strictly inside the root interval: nc(blo) <= t makes blo
// a lower bound and nc(bhi) > t makes bhi an upper bound; an end that fails bounds the value from
// the other side (nc(blo) > t: sigma < blo; nc(bhi) <= t: sigma >= bhi), so a missed bracket
// still narrows one side. Midpoints at or below a lower bound send the target right and those at
// or above an upper bound send it left without a count, as the reference's counts do when they
// are monotone; the others are counted as in the reference. The root's own counts are evaluated
// only for the sides no bound covers. Outputs the leaf midpoint, the leaf's endpoints, the number
// of Sturm counts evaluated and a status (1: bounded on both sides, 2: on one side, 0: from the
// root, -1: the root does not hold the value, as when the reference's root bound is below
// sigma_max). Fallback points flo / fhi (optional) are counted only for a side the bracket left
// open: flo for a missing lower bound, fhi for a missing upper one.
__global__ __launch_bounds__(64) void k_bisect_index(int ntg, const int* __restrict__ ns, const long* __restrict__ off,
                                                     const double* __restrict__ d, const double* __restrict__ e,
                                                     const double* __restrict__ root, double tol,
                                                     const int* __restrict__ tb, const int* __restrict__ ti,
                                                     const double* __restrict__ blo, const double* __restrict__ bhi,
                                                     const double* __restrict__ flo, const double* __restrict__ fhi,
                                                     double* __restrict__ sigma, double* __restrict__ leaf_lo,
                                                     double* __restrict__ leaf_hi, int* __restrict__ iters,
                                                     int* __restrict__ status) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= ntg) return;
  const int b = tb[j];
  const int n = ns[b];
  const double* a = d + off[b];
  const double* bb = e + off[b];
  const int t = n - 1 - ti[j];
  int it = 0;
  double lo = 0.0, hi = root[b];
  bool haveL = false, haveH = false;
  double L = 0.0, H = 0.0;
  if (blo && bhi && blo[j] < bhi[j]) {
    const double pl = blo[j], ph = bhi[j];
    if (pl > lo && pl < hi) {
      const bool below = sturm_count(n, a, bb, pl) <= t;
      it++;
      if (below) { L = pl; haveL = true; }
      else { H = pl; haveH = true; }
    }
    if (ph > lo && ph < hi) {
      const bool below = sturm_count(n, a, bb, ph) <= t;
      it++;
      if (!below) {
        if (!haveH) { H = ph; haveH = true; }
      } else if (!haveL || ph > L) {
        L = ph;
        haveL = true;
      }
    }
    if (haveL && haveH && !(L < H)) haveL = haveH = false;  // counts that are not monotone: use neither
  }
  if (flo && !haveL) {
    const double p = flo[j];
    if (p > lo && p < hi && (!haveH || p < H)) {
      it++;
      if (sturm_count(n, a, bb, p) <= t) { L = p; haveL = true; }
    }
  }
  if (fhi && !haveH) {
    const double p = fhi[j];
    if (p > lo && p < hi && (!haveL || p > L)) {
      it++;
      if (t < sturm_count(n, a, bb, p)) { H = p; haveH = true; }
    }
  }
  if (!haveL || !haveH) {
    bool in_tree = true;
    if (!haveL) {
      in_tree = sturm_count(n, a, bb, lo) <= t;
      it++;
    }
    if (!haveH && in_tree) {
      in_tree = t < sturm_count(n, a, bb, hi);
      it++;
    }
    if (!in_tree) {
      sigma[j] = 0.0;
      leaf_lo[j] = leaf_hi[j] = 0.0;
      iters[j] = it;
      status[j] = -1;
      return;
    }
  }
  for (int level = 0; level < 4096; level++) {
    const double mid = (lo + hi) / 2;
    if ((hi - lo) <= tol || mid == lo || mid == hi) break;
    bool right;
    if (haveL && mid <= L) right = true;
    else if (haveH && mid >= H) right = false;
    else {
      right = sturm_count(n, a, bb, mid) <= t;
      it++;
    }
    if (right) lo = mid;
    else hi = mid;
  }
  sigma[j] = (lo + hi) / 2;
  leaf_lo[j] = lo;
  leaf_hi[j] = hi;
  iters[j] = it;
  status[j] = haveL && haveH ? 1 : (haveL || haveH ? 2 : 0);
}

// ------------------------------------------------------------------ the network
// in (32) -> 256 -> 256 -> 2, ReLU; outputs (c, w): y ~ c with Laplace scale exp(w).
constexpr int kIn = 32, kHid = 256, kOut = 2;
constexpr long kW1 = 0, kB1 = kW1 + (long)kIn * kHid, kW2 = kB1 + kHid, kB2 = kW2 + (long)kHid * kHid,
               kW3 = kB2 + kHid, kB3 = kW3 + (long)kHid * kOut, kParams = kB3 + kOut;

// Caller's float arrays are read 4 at a time with no more than their elements' alignment.
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));

// Z += bias and H = relu(Z) over the B x 256 layer, four columns per thread.
__global__ __launch_bounds__(256) void k_bias_relu(long B, float* __restrict__ Z, const float* __restrict__ bias,
                                                   float* __restrict__ H) {
  const long g = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= B * (kHid / 4)) return;
  const int j = (int)(g % (kHid / 4)) * 4;
  f4u z = *(const f4u*)(Z + 4 * g), h;
#pragma unroll
  for (int q = 0; q < 4; q++) {
    z[q] += bias[j + q];
    h[q] = z[q] > 0.f ? z[q] : 0.f;
  }
  *(f4u*)(Z + 4 * g) = z;
  *(f4u*)(H + 4 * g) = h;
}

// The second hidden layer's bias and ReLU and the output layer in one pass: a wavefront per row,
// four columns per lane. (As a matrix product the two output columns fill 1/64 of a tile.)
constexpr int kHeadRows = 4;  // rows per wavefront
__global__ __launch_bounds__(256) void k_bias_relu_head(long B, float* __restrict__ Z,
                                                        const float* __restrict__ p, float* __restrict__ H,
                                                        float* __restrict__ O) {
  const int lane = threadIdx.x & 63, j = 4 * lane;
  const long r0 = ((long)blockIdx.x * 4 + (threadIdx.x >> 6)) * kHeadRows;
  float w0[4], w1[4], b2[4];
#pragma unroll
  for (int q = 0; q < 4; q++) {
    w0[q] = p[kW3 + (j + q) * kOut];
    w1[q] = p[kW3 + (j + q) * kOut + 1];
    b2[q] = p[kB2 + j + q];
  }
  for (long r = r0; r < min(B, r0 + kHeadRows); r++) {
    f4u z = *(const f4u*)(Z + r * kHid + j), h;
    float o0 = 0.f, o1 = 0.f;
#pragma unroll
    for (int q = 0; q < 4; q++) {
      z[q] += b2[q];
      h[q] = z[q] > 0.f ? z[q] : 0.f;
      o0 += h[q] * w0[q];
      o1 += h[q] * w1[q];
    }
    *(f4u*)(Z + r * kHid + j) = z;
    *(f4u*)(H + r * kHid + j) = h;
    o0 = wave_sum(o0);
    o1 = wave_sum(o1);
    if (lane == 0) {
      O[2 * r] = o0 + p[kB3];
      O[2 * r + 1] = o1 + p[kB3 + 1];
    }
  }
}

// Head of the backward pass over a slab of rows, one column per thread: the Laplace negative
// log-likelihood |y - c| exp(-w) + w averaged over B and its gradient dO, the gradient of the second
// layer's sums dZ2 = (dO W3^T) where H2 > 0, and this slab's share of dW3 = H2^T dO, db2, db3 and
// the loss. `part` holds one row of kHeadPart values per workgroup, summed by k_sum_parts in a
// fixed order.
constexpr int kPartW3 = 0, kPartB2 = kPartW3 + kHid * kOut, kPartB3 = kPartB2 + kHid, kPartLoss = kPartB3 + kOut,
              kHeadPart = kPartLoss + 1;
constexpr int kSlab = 16;  // rows whose dO a workgroup holds at a time
__global__ __launch_bounds__(256) void k_head_back(long B, long rows, const float* __restrict__ O,
                                                   const float* __restrict__ y, const float* __restrict__ H,
                                                   const float* __restrict__ p, float* __restrict__ dZ,
                                                   float* __restrict__ part, float* __restrict__ grad,
                                                   float* __restrict__ loss) {
  __shared__ float d0[kSlab], d1[kSlab], ls[kSlab];
  const int j = threadIdx.x;
  const float w0 = p[kW3 + j * kOut], w1 = p[kW3 + j * kOut + 1];
  float g0 = 0.f, g1 = 0.f, gb = 0.f, s0 = 0.f, s1 = 0.f, sl = 0.f;
  const long end = min(B, (blockIdx.x + 1L) * rows);
  for (long r0 = blockIdx.x * rows; r0 < end; r0 += kSlab) {
    const int n = (int)min((long)kSlab, end - r0);
    float h[kSlab];
#pragma unroll
    for (int q = 0; q < kSlab; q++) h[q] = H[(r0 + min(q, n - 1)) * kHid + j];
    if (j < n) {
      const long r = r0 + j;
      const float c = O[2 * r], w = O[2 * r + 1], e = y[r] - c, ew = expf(-w);
      ls[j] = fabsf(e) * ew + w;
      d0[j] = (e > 0.f ? -ew : (e < 0.f ? ew : 0.f)) / (float)B;
      d1[j] = (1.f - fabsf(e) * ew) / (float)B;
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kSlab; q++)
      if (q < n) {
        const float a = d0[q], b = d1[q];
        const float dz = h[q] > 0.f ? a * w0 + b * w1 : 0.f;
        dZ[(r0 + q) * kHid + j] = dz;
        g0 += h[q] * a;
        g1 += h[q] * b;
        gb += dz;
        s0 += a;
        s1 += b;
        sl += ls[q];
      }
    __syncthreads();
  }
  if (gridDim.x == 1) {  // the slab is the batch
    grad[kW3 + j * kOut] = g0;
    grad[kW3 + j * kOut + 1] = g1;
    grad[kB2 + j] = gb;
    if (j == 0) {
      grad[kB3] = s0;
      grad[kB3 + 1] = s1;
      *loss = sl / (float)B;
    }
    return;
  }
  float* o = part + (long)blockIdx.x * kHeadPart;
  o[kPartW3 + j * kOut] = g0;
  o[kPartW3 + j * kOut + 1] = g1;
  o[kPartB2 + j] = gb;
  if (j == 0) {
    o[kPartB3] = s0;
    o[kPartB3 + 1] = s1;
    o[kPartLoss] = sl / (float)B;
  }
}

// dZ1 = dH1 where H1 > 0 (in place) over a slab of rows, with the slab's column sums.
__global__ __launch_bounds__(256) void k_relu_back(long B, long rows, float* __restrict__ dH,
                                                   const float* __restrict__ H, float* __restrict__ part) {
  const int j = threadIdx.x;
  const long end = min(B, (blockIdx.x + 1L) * rows);
  float s = 0.f;
#pragma unroll 8
  for (long r = blockIdx.x * rows; r < end; r++) {
    const long e = r * kHid + j;
    const float v = H[e] > 0.f ? dH[e] : 0.f;
    dH[e] = v;
    s += v;
  }
  part[(long)blockIdx.x * kHid + j] = s;
}

// Column sums of the n x cols partials: 16 columns per workgroup, 16 threads per column.
// Head partials (loss given) go to the gradient's slots and the loss, others to out.
__global__ __launch_bounds__(256) void k_sum_parts(int n, int cols, const float* __restrict__ part,
                                                   float* __restrict__ out, float* __restrict__ grad,
                                                   float* __restrict__ loss) {
  __shared__ float red[16][17];
  const int c = threadIdx.x & 15, q = threadIdx.x >> 4, col = blockIdx.x * 16 + c;
  float s = 0.f;
  if (col < cols)
#pragma unroll 8
    for (int i = q; i < n; i += 16) s += part[(long)i * cols + col];
  red[q][c] = s;
  __syncthreads();
  if (q != 0 || col >= cols) return;
  s = 0.f;
#pragma unroll
  for (int i = 0; i < 16; i++) s += red[i][c];
  if (!loss) out[col] = s;
  else if (col < kPartB2) grad[kW3 + col] = s;
  else if (col < kPartB3) grad[kB2 + col - kPartB2] = s;
  else if (col < kPartLoss) grad[kB3 + col - kPartB3] = s;
  else *loss = s;
}

__global__ __launch_bounds__(256) void k_adam(long n, float* __restrict__ p, const float* __restrict__ g,
                                              float* __restrict__ m, float* __restrict__ v, float lr, float b1,
                                              float b2, float eps, float c1, float c2) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.f - b1) * gi;
  const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

__global__ __launch_bounds__(256) void k_to_bf16(long n, const float* __restrict__ x, __hip_bfloat16* __restrict__ y) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = __float2bfloat16(x[i]);
}

// BF16 inference: weights and activations in bfloat16, products accumulated in FP32 on
// v_mfma_f32_16x16x32_bf16. A workgroup runs 32 samples through both hidden layers; wavefront w owns
// the units 64 w .. 64 w + 63. An MFMA lane wants 8 consecutive k of one unit, but the weights are
// stored unit-fastest, so each wavefront transposes its 64 x 256 slice of W2 into LDS (8 x 8 blocks
// in registers, 16-byte units XORed by the row against bank conflicts). 4096 samples: 797 us with
// one sample per thread and scalar products, 11 us here.
typedef __bf16 b8 __attribute__((ext_vector_type(8)));
typedef __bf16 b8u __attribute__((ext_vector_type(8), aligned(2)));
typedef float f4 __attribute__((ext_vector_type(4)));
constexpr int kInferRows = 32;
constexpr int kUnits = kHid / 8;  // 16-byte units of a row of 256
__global__ __launch_bounds__(256) void k_mlp_infer_bf16(long B, const float* __restrict__ X,
                                                        const __bf16* __restrict__ P, float* __restrict__ O) {
  __shared__ b8 w2[kHid * kUnits];       // [unit][k], 128 KB
  __shared__ b8 h[kInferRows * kUnits];  // [sample][k] of the first layer, 16 KB
  __shared__ float red[4][kInferRows][2];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, li = lane & 15, lk = lane >> 4;
  const long s0 = (long)blockIdx.x * kInferRows;
  const int u0 = 64 * wave;
  // this wavefront's slice of W2: 8 unit groups x 32 k groups of 8 x 8 blocks, four per lane
#pragma unroll
  for (int z = 0; z < 4; z++) {
    const int blk = lane + 64 * z, ug = blk & 7, kg = blk >> 3;
    b8 in[8];
#pragma unroll
    for (int k = 0; k < 8; k++) in[k] = *(const b8u*)(P + kW2 + (long)(kg * 8 + k) * kHid + u0 + ug * 8);
#pragma unroll
    for (int c = 0; c < 8; c++) {
      b8 o;
#pragma unroll
      for (int k = 0; k < 8; k++) o[k] = in[k][c];
      const int r = u0 + ug * 8 + c;
      w2[r * kUnits + (kg ^ (r & 15))] = o;
    }
  }
  // layer 1: K = 32 is one step; samples are the rows of A, units the columns of B
  b8 xa[2];
#pragma unroll
  for (int a = 0; a < 2; a++) {
    const long s = min(s0 + a * 16 + li, B - 1);
#pragma unroll
    for (int k = 0; k < 8; k++) xa[a][k] = (__bf16)X[s * kIn + lk * 8 + k];
  }
#pragma unroll
  for (int b = 0; b < 4; b++) {
    const int u = u0 + b * 16 + li;
    b8 wb;
#pragma unroll
    for (int k = 0; k < 8; k++) wb[k] = P[kW1 + (long)(lk * 8 + k) * kHid + u];
    const float bias = (float)P[kB1 + u];
#pragma unroll
    for (int a = 0; a < 2; a++) {
      const f4 v = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[a], wb, f4{bias, bias, bias, bias}, 0, 0, 0);
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int s = a * 16 + 4 * lk + q;
        ((__bf16*)h)[(s * kUnits + ((u >> 3) ^ (s & 15))) * 8 + (u & 7)] = (__bf16)(v[q] > 0.f ? v[q] : 0.f);
      }
    }
  }
  __syncthreads();
  // layer 2
  f4 acc[2][4];
#pragma unroll
  for (int b = 0; b < 4; b++) {
    const float bias = (float)P[kB2 + u0 + b * 16 + li];
    acc[0][b] = acc[1][b] = f4{bias, bias, bias, bias};
  }
#pragma unroll
  for (int ks = 0; ks < kHid / 32; ks++) {
    const int ku = ks * 4 + lk;
    b8 ha[2], wb[4];
#pragma unroll
    for (int a = 0; a < 2; a++) ha[a] = h[(a * 16 + li) * kUnits + (ku ^ li)];
#pragma unroll
    for (int b = 0; b < 4; b++) wb[b] = w2[(u0 + b * 16 + li) * kUnits + (ku ^ li)];
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
      for (int b = 0; b < 4; b++) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ha[a], wb[b], acc[a][b], 0, 0, 0);
  }
  // output layer: each lane's four units, then the 16 lanes of a row group, then the wavefronts
  float w30[4], w31[4];
#pragma unroll
  for (int b = 0; b < 4; b++) {
    w30[b] = (float)P[kW3 + (u0 + b * 16 + li) * kOut];
    w31[b] = (float)P[kW3 + (u0 + b * 16 + li) * kOut + 1];
  }
#pragma unroll
  for (int a = 0; a < 2; a++)
#pragma unroll
    for (int q = 0; q < 4; q++) {
      float o0 = 0.f, o1 = 0.f;
#pragma unroll
      for (int b = 0; b < 4; b++) {
        const float v = acc[a][b][q];
        const float hq = (float)(__bf16)(v > 0.f ? v : 0.f);
        o0 += hq * w30[b];
        o1 += hq * w31[b];
      }
#pragma unroll
      for (int off = 8; off > 0; off >>= 1) {
        o0 += __shfl_xor(o0, off, kWave);
        o1 += __shfl_xor(o1, off, kWave);
      }
      if (li == 0) {
        red[wave][a * 16 + 4 * lk + q][0] = o0;
        red[wave][a * 16 + 4 * lk + q][1] = o1;
      }
    }
  __syncthreads();
  if (tid < 2 * kInferRows) {
    const int s = tid >> 1, c = tid & 1;
    if (s0 + s < B)
      O[2 * (s0 + s) + c] = (float)P[kB3 + c] + (red[0][s][c] + red[1][s][c]) + (red[2][s][c] + red[3][s][c]);
  }
}

unsigned grid_for(long n, int per = 256) { return (unsigned)std::max<long>(1, (n + per - 1) / per); }

}  // namespace

extern "C" {

int exc_gk_bidiagonals(int nb, const int* d_n, const long* d_off, const double* d_sigma, const double* d_start,
                       double* d_d, double* d_e, exc_stream_t stream) {
  EXC_REQUIRE(nb >= 0 && (nb == 0 || (d_n && d_off && d_sigma && d_start && d_d && d_e)), EXC_ERR_ARG,
              "exc_gk_bidiagonals: bad arguments");
  if (nb == 0) return EXC_OK;
  hipLaunchKernelGGL(k_gk_lanczos, dim3(nb), dim3(kLzThreads), 0, exc_detail::stream(stream), d_n, d_off, d_sigma,
                     d_start, d_d, d_e);
  EXC_CHECK_HIP(hipGetLastError());
  return EXC_OK;
}

int exc_gk_max_n(void) { return kLzThreads * kLzPerThread; }

int exc_bidiag_scale(int nb, const int* d_n, const long* d_off, const double* d_d, const double* d_e, double* d_root,
                     double* d_scale, exc_stream_t stream) {
  EXC_REQUIRE(nb >= 0 && (nb == 0 || (d_n && d_off && d_d && d_e && d_root && d_scale)), EXC_ERR_ARG,
              "exc_bidiag_scale: bad arguments");
  if (nb == 0) return EXC_OK;
  hipLaunchKernelGGL(k_bidiag_scale, dim3(grid_for(nb, 64)), dim3(64), 0, exc_detail::stream(stream), nb, d_n, d_off,
                     d_d, d_e, d_root, d_scale);
  EXC_CHECK_HIP(hipGetLastError());
  return EXC_OK;
}

int exc_count_features(int nb, int K, const int* d_n, const long* d_off, const double* d_d, const double* d_e,
                       const double* d_scale, float* d_frac, exc_stream_t stream) {
  EXC_REQUIRE(nb >= 0 && K >= 1 && (nb == 0 || (d_n && d_off && d_d && d_e && d_scale && d_frac)), EXC_ERR_ARG,
              "exc_count_features: bad arguments");
  if (nb == 0) return EXC_OK;
  hipLaunchKernelGGL(k_count_features, dim3(grid_for((long)nb * K)), dim3(256), 0, exc_detail::stream(stream), nb, K,
                     d_n, d_off, d_d, d_e, d_scale, d_frac);
  EXC_CHECK_HIP(hipGetLastError());
  return EXC_OK;
}

int exc_bisect_index(int ntg, const int* d_n, const long* d_off, const double* d_d, const double* d_e,
                     const double* d_root, double tol, const int* d_tb, const int* d_ti, const double* d_blo,
                     const double* d_bhi, const double* d_flo, const double* d_fhi, double* d_sigma,
                     double* d_leaf_lo, double* d_leaf_hi, int* d_iters, int* d_status, exc_stream_t stream) {
  EXC_REQUIRE(ntg >= 0 && (ntg == 0 || (d_n && d_off && d_d && d_e && d_root && d_tb && d_ti && d_sigma &&
                                        d_leaf_lo && d_leaf_hi && d_iters && d_status)) &&
                  (!d_blo) == (!d_bhi) && (!d_flo) == (!d_fhi),
              EXC_ERR_ARG, "exc_bisect_index: bad arguments");
  if (ntg == 0) return EXC_OK;
  hipLaunchKernelGGL(k_bisect_index, dim3(grid_for(ntg, 64)), dim3(64), 0, exc_detail::stream(stream), ntg, d_n,
                     d_off, d_d, d_e, d_root, tol, d_tb, d_ti, d_blo, d_bhi, d_flo, d_fhi, d_sigma, d_leaf_lo,
                     d_leaf_hi, d_iters, d_status);
  EXC_CHECK_HIP(hipGetLastError());
  return EXC_OK;
}

long exc_mlp_param_count(void) { return kParams; }
int exc_mlp_dims(int* d_in, int* hidden, int* d_out) {
  if (d_in) *d_in = kIn;
  if (hidden) *hidden = kHid;
  if (d_out) *d_out = kOut;
  return EXC_OK;
}

// Activations of a batch: Z1, H1, Z2, H2 (B x 256 each) and O (B x 2), floats: the hidden layers before
// and after their ReLU, biases added. exc_mlp_backward needs H1 and H2 and writes over Z1 and Z2.
size_t exc_mlp_acts_floats(long B) { return (size_t)B * (4 * kHid + kOut); }

int exc_mlp_forward(long B, const float* d_x, const float* d_p, float* d_acts, float* d_out, void* d_work,
                    size_t work_bytes, exc_stream_t stream) {
  EXC_REQUIRE(B >= 1 && d_x && d_p && d_acts && d_out, EXC_ERR_ARG, "exc_mlp_forward: bad arguments");
  hipStream_t s = exc_detail::stream(stream);
  float* Z1 = d_acts;
  float* H1 = Z1 + B * kHid;
  float* Z2 = H1 + B * kHid;
  float* H2 = Z2 + B * kHid;
  ExcGemmOpts o;
  o.work = d_work;
  o.work_bytes = work_bytes;
  int rc = exc_sgemm_opts(0, 0, B, kHid, kIn, 1.0, d_x, kIn, d_p + kW1, kHid, 0.0, Z1, kHid, o, s);
  if (rc) return rc;
  hipLaunchKernelGGL(k_bias_relu, dim3(grid_for(B * (kHid / 4))), dim3(256), 0, s, B, Z1, d_p + kB1, H1);
  rc = exc_sgemm_opts(0, 0, B, kHid, kHid, 1.0, H1, kHid, d_p + kW2, kHid, 0.0, Z2, kHid, o, s);
  if (rc) return rc;
  hipLaunchKernelGGL(k_bias_relu_head, dim3(grid_for(B, 4 * kHeadRows)), dim3(256), 0, s, B, Z2, d_p, H2, d_out);
  EXC_CHECK_HIP(hipGetLastError());
  return EXC_OK;
}

// Gradient of the mean Laplace negative log-likelihood after exc_mlp_forward on the same batch;
// d_dscratch holds B x (256 + 2) floats. d_loss (one float) receives the loss.
size_t exc_mlp_backward_scratch_floats(long B) { return (size_t)B * (kHid + kOut); }

int exc_mlp_backward(long B, const float* d_x, const float* d_y, const float* d_p, float* d_acts, const float* d_out,
                     float* d_grad, float* d_scratch, float* d_loss, void* d_work, size_t work_bytes,
                     exc_stream_t stream) {
  EXC_REQUIRE(B >= 1 && d_x && d_y && d_p && d_acts && d_out && d_grad && d_scratch && d_loss, EXC_ERR_ARG,
              "exc_mlp_backward: bad arguments");
  hipStream_t s = exc_detail::stream(stream);
  float* Z1 = d_acts;
  float* H1 = Z1 + B * kHid;
  float* Z2 = H1 + B * kHid;
  float* H2 = Z2 + B * kHid;
  // The gradient of a layer's sums: dZ2 in the scratch, dZ1 in Z1's slot (H says where Z was
  // positive). The slabs' partial sums go to Z2's slot (two slabs are over 16 rows, enough for them).
  float* dZ2 = d_scratch;
  float* part = Z2;
  const long rows = std::max<long>(kSlab, (B + 511) / 512);  // of a slab, at most 512 slabs
  const unsigned slabs = grid_for(B, (int)rows);
  ExcGemmOpts o;
  o.work = d_work;
  o.work_bytes = work_bytes;
  hipLaunchKernelGGL(k_head_back, dim3(slabs), dim3(256), 0, s, B, rows, d_out, d_y, H2, d_p, dZ2, part, d_grad,
                     d_loss);
  if (slabs > 1) hipLaunchKernelGGL(k_sum_parts, dim3(grid_for(kHeadPart, 16)), dim3(256), 0, s, (int)slabs, kHeadPart, part,
                     (float*)nullptr, d_grad, d_loss);
  // layer 2: dW2 = H1^T dZ2, dH1 = dZ2 W2^T
  int rc = exc_sgemm_opts(1, 0, kHid, kHid, B, 1.0, H1, kHid, dZ2, kHid, 0.0, d_grad + kW2, kHid, o, s);
  if (rc) return rc;
  rc = exc_sgemm_opts(0, 1, B, kHid, kHid, 1.0, dZ2, kHid, d_p + kW2, kHid, 0.0, Z1, kHid, o, s);
  if (rc) return rc;
  hipLaunchKernelGGL(k_relu_back, dim3(slabs), dim3(256), 0, s, B, rows, Z1, H1, slabs > 1 ? part : d_grad + kB1);
  if (slabs > 1) hipLaunchKernelGGL(k_sum_parts, dim3(grid_for(kHid, 16)), dim3(256), 0, s, (int)slabs, kHid, part, d_grad + kB1,
                     (float*)nullptr, (float*)nullptr);
  // layer 1: dW1 = X^T dZ1
  rc = exc_sgemm_opts(1, 0, kIn, kHid, B, 1.0, d_x, kIn, Z1, kHid, 0.0, d_grad + kW1, kHid, o, s);
  if (rc) return rc;
  EXC_CHECK_HIP(hipGetLastError());
  return EXC_OK;
}

int exc_mlp_adam(float* d_p, const float* d_grad, float* d_m, float* d_v, float lr, float beta1, float beta2,
                 float eps, int step, exc_stream_t stream) {
  EXC_REQUIRE(d_p && d_grad && d_m && d_v && step >= 1, EXC_ERR_ARG, "exc_mlp_adam: bad arguments");
  const float c1 = 1.f - powf(beta1, (float)step), c2 = 1.f - powf(beta2, (float)step);
  hipLaunchKernelGGL(k_adam, dim3(grid_for(kParams)), dim3(256), 0, exc_detail::stream(stream), kParams, d_p, d_grad,
                     d_m, d_v, lr, beta1, beta2, eps, c1, c2);
  EXC_CHECK_HIP(hipGetLastError());
  return EXC_OK;
}

int exc_mlp_to_bf16(const float* d_p, void* d_pbf16, exc_stream_t stream) {
  EXC_REQUIRE(d_p && d_pbf16, EXC_ERR_ARG, "exc_mlp_to_bf16: bad arguments");
  hipLaunchKernelGGL(k_to_bf16, dim3(grid_for(kParams)), dim3(256), 0, exc_detail::stream(stream), kParams, d_p,
                     (__hip_bfloat16*)d_pbf16);
  EXC_CHECK_HIP(hipGetLastError());
  return EXC_OK;
}

int exc_mlp_infer_bf16(long B, const float* d_x, const void* d_pbf16, float* d_out, exc_stream_t stream) {
  EXC_REQUIRE(B >= 1 && d_x && d_pbf16 && d_out, EXC_ERR_ARG, "exc_mlp_infer_bf16: bad arguments");
  hipLaunchKernelGGL(k_mlp_infer_bf16, dim3(grid_for(B, kInferRows)), dim3(256), 0, exc_detail::stream(stream), B, d_x,
                     (const __bf16*)d_pbf16, d_out);
  EXC_CHECK_HIP(hipGetLastError());
  return EXC_OK;
}

}  // extern "C"
