// Givens-rotation masking sweep on gfx950 (the arithmetic of
// givens_mask_cache_optimized_parallel_with_simd, bbtsvd.cpp:781-875).
//
// A workgroup owns a strip of L independent lines (columns for a left mask, rows for a right mask)
// and keeps it in LDS for all passes: one HBM read and one write per element per call, whatever the
// number of passes. Within a pass the rotation pairs are disjoint (a permutation) except, for odd
// K, the extra pair the reference appends; that pair is applied on its own after (mask) or before
// (unmask) the others, which is the order the reference's sequential loop gives it. Each update is
// c*x1 + s'*x2 with separately rounded products and sum, so the result is bit-identical to the
// reference's loop.
//
// What bounds it is the chain of passes: each reads what the last one wrote, through a barrier. So a
// pass is kept short. A thread owns one or two pairs and rotates all L lines of them: the strip is
// stored line-fastest, a pair's two elements are one LDS word of up to 16 bytes each, and the plan
// entry is read once per strip, straight into registers and two passes ahead of its use (it was
// staged in LDS and read again for every line). A strip that one wavefront covers needs no barrier:
// a wavefront's LDS operations complete in order. Both sides of a 1000 x 1000 FP64 mask: 139 -> 52
// us, 2000 x 2000 FP32: 358 -> 97, 100 x 100: 64 -> 19 (HBM would take 3.3, 6.7 and 0.05 us).
#include <algorithm>
#include <type_traits>

#include "exc_common.hpp"

#pragma clang fp contract(off)

namespace {

constexpr int kMaxThreads = 1024;
constexpr size_t kLdsHard = 160 * 1024;

// A plan entry's indices and rotation; no alignment beyond the elements' own is assumed of the plan.
typedef int32_t i2u __attribute__((ext_vector_type(2), aligned(4)));
typedef double d2u __attribute__((ext_vector_type(2), aligned(8)));

template <typename T, int L>
struct Chunk {
  typedef T type __attribute__((ext_vector_type(L)));
};
template <typename T>
struct Chunk<T, 1> {
  typedef T type;
};

// Orders the strip's LDS traffic between the steps of a pass.
__device__ __forceinline__ void strip_sync() {
  if (blockDim.x > kWave) {
    lds_barrier();
  } else {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
}

// odd_mode: 0 none, 1 the special pair is pair 0 (applied first), 2 it is the last pair. NP: pairs
// per thread held in registers; 0: any number, read from the plan in the pass that uses them.
template <typename T, int L, int NP, bool LEFT>
__device__ __forceinline__ void givens_strip(T* __restrict__ x, long m, long n, const int32_t* __restrict__ pairs,
                                             const double* __restrict__ cs, int passes, int half, int mask,
                                             int odd_mode, T* buf) {
  typedef typename Chunk<T, L>::type chunk;
  const int tid = threadIdx.x, nt = blockDim.x;
  const int K = (int)(LEFT ? m : n);
  // neighbouring strips share cache lines: each die takes a contiguous range of them (the
  // dispatcher deals workgroups round-robin over the 8 dies)
  const int g = gridDim.x, x8 = blockIdx.x % 8;
  const long base = ((long)x8 * (g / 8) + min(x8, g % 8) + blockIdx.x / 8) * L;
  const int lines = (int)min((long)L, (LEFT ? n : m) - base);
  chunk* strip = (chunk*)buf;
  if (LEFT) {
    for (int e = tid; e < K * L; e += nt) {
      const int r = e / L, c = e % L;
      buf[e] = c < lines ? x[(long)r * n + base + c] : T(0);
    }
  } else {
    for (int c = 0; c < L; c++)
      for (int q = tid; q < K; q += nt) buf[q * L + c] = c < lines ? x[(base + c) * n + q] : T(0);
  }
  constexpr int NR = NP > 0 ? NP : 4;  // pairs of a thread in flight
  struct Plan {
    i2u r[NR];
    d2u c[NR];
  };
  Plan P0, P1;
  // pairs j0 + u nt of pass p (clamped: entries past the end are read again and not used)
  auto issue = [&](Plan& P, int p, int j0) __attribute__((always_inline)) {
    const long at = (long)min(p, passes - 1) * half;
#pragma unroll
    for (int u = 0; u < NR; u++) {
      const long j = at + min(j0 + u * nt, half - 1);
      P.r[u] = *(const i2u*)(pairs + 2 * j);
      P.c[u] = *(const d2u*)(cs + 2 * j);
    }
  };
  const int special = odd_mode == 1 ? 0 : (odd_mode == 2 ? half - 1 : -1);
  const T sgn = mask ? T(1) : T(-1);
  // sub = 0: every pair; 1: the special pair only; 2: all but the special pair
  auto rotate = [&](const Plan& P, int j0, int sub) __attribute__((always_inline)) {
    chunk a[NR], b[NR];
    bool ok[NR];
#pragma unroll
    for (int u = 0; u < NR; u++) {
      const int j = j0 + u * nt;
      // a malformed plan's out-of-range pair is skipped
      ok[u] = j < half && (unsigned)P.r[u][0] < (unsigned)K && (unsigned)P.r[u][1] < (unsigned)K &&
              (sub == 0 || (j == special) == (sub == 1));
      if (ok[u]) {
        a[u] = strip[P.r[u][0]];
        b[u] = strip[P.r[u][1]];
      }
    }
#pragma unroll
    for (int u = 0; u < NR; u++)
      if (ok[u]) {
        const T c = (T)P.c[u][0], s = (T)P.c[u][1];
        const T ss = sgn * s, nss = -sgn * s;
        strip[P.r[u][0]] = a[u] * c + b[u] * ss;
        strip[P.r[u][1]] = a[u] * nss + b[u] * c;
      }
  };
  auto pass = [&](Plan& P, int p) __attribute__((always_inline)) {
    const int first = odd_mode == 1 ? 1 : (odd_mode == 2 ? 2 : 0);
    for (int sub = first;; sub = 3 - sub) {
      if (NP > 0) {
        rotate(P, tid, sub);
      } else {
        for (int j0 = tid; j0 < half; j0 += NR * nt) {
          issue(P, p, j0);
          rotate(P, j0, sub);
        }
      }
      strip_sync();
      if (first == 0 || sub != first) break;
    }
  };
  if (NP > 0) {
    issue(P0, 0, tid);
    issue(P1, 1, tid);
  }
  strip_sync();
  for (int p = 0; p < passes; p += 2) {
    pass(P0, p);
    if (NP > 0) issue(P0, p + 2, tid);
    if (p + 1 < passes) {
      pass(P1, p + 1);
      if (NP > 0) issue(P1, p + 3, tid);
    }
  }
  if (LEFT) {
    for (int e = tid; e < K * L; e += nt) {
      const int r = e / L, c = e % L;
      if (c < lines) x[(long)r * n + base + c] = buf[e];
    }
  } else {
    for (int c = 0; c < lines; c++)
      for (int q = tid; q < K; q += nt) x[(base + c) * n + q] = buf[q * L + c];
  }
}

template <typename T, int L, int NP, bool LEFT>
__global__ __launch_bounds__(kMaxThreads) void k_givens(T* __restrict__ x, long m, long n,
                                                        const int32_t* __restrict__ pairs,
                                                        const double* __restrict__ cs, int passes, int half, int mask,
                                                        int odd_mode) {
  extern __shared__ __align__(32) unsigned char smem_raw[];
  givens_strip<T, L, NP, LEFT>(x, m, n, pairs, cs, passes, half, mask, odd_mode, reinterpret_cast<T*>(smem_raw));
}

// The same sweep over a batch of matrices of one shape, each with its own plan: blockIdx.y picks
// the matrix.
template <typename T, int L, int NP, bool LEFT>
__global__ __launch_bounds__(kMaxThreads) void k_givens_batched(T* const* __restrict__ xs, long m, long n,
                                                                const int32_t* const* __restrict__ pairs,
                                                                const double* const* __restrict__ cs, int passes,
                                                                int half, int mask, int odd_mode) {
  extern __shared__ __align__(32) unsigned char smem_raw[];
  const int b = blockIdx.y;
  givens_strip<T, L, NP, LEFT>(xs[b], m, n, pairs[b], cs[b], passes, half, mask, odd_mode,
                               reinterpret_cast<T*>(smem_raw));
}

// Shape of a sweep: threads (a pair each, two above 512 pairs so that a thread's LDS accesses
// overlap) and the lines of a strip: as many as make a 16-byte word, while the strips still cover
// three quarters of the CUs and fit in LDS. (With 32-byte words the 1000 x 1000 mask has one strip
// per CU and nothing runs while it waits at its barriers: 26 % slower; with 256 threads of two pairs
// each instead of 512 of one, 46 %.)
struct Sweep {
  int threads, np, l;
};
Sweep sweep_shape(long K, long lines, int half, size_t size) {
  Sweep s;
  const int up = (half + kWave - 1) / kWave * kWave;
  s.np = half <= 512 ? 1 : (half <= 2048 ? 2 : 0);
  s.threads = half <= 512 ? up : (half <= 1024 ? 512 : kMaxThreads);
  s.l = 1;
  while (s.l * 2 * size <= 16 && lines / (s.l * 2) >= 192 && (size_t)K * s.l * 2 * size <= kLdsHard) s.l *= 2;
  return s;
}

// Calls f with the kernel's template arguments as constants.
template <typename T, typename F>
auto with_shape(const Sweep& s, bool left, F f) {
  auto with_l = [&](auto np, auto lf) {
    constexpr int NP = decltype(np)::value;
    constexpr bool LEFT = decltype(lf)::value;
    using std::integral_constant;
    if constexpr (sizeof(T) == 4)
      if (s.l == 4) return f(integral_constant<int, 4>{}, integral_constant<int, NP>{}, integral_constant<bool, LEFT>{});
    if (s.l == 2) return f(integral_constant<int, 2>{}, integral_constant<int, NP>{}, integral_constant<bool, LEFT>{});
    return f(integral_constant<int, 1>{}, integral_constant<int, NP>{}, integral_constant<bool, LEFT>{});
  };
  auto with_np = [&](auto lf) {
    if (s.np == 1) return with_l(std::integral_constant<int, 1>{}, lf);
    if (s.np == 2) return with_l(std::integral_constant<int, 2>{}, lf);
    return with_l(std::integral_constant<int, 0>{}, lf);
  };
  return left ? with_np(std::true_type{}) : with_np(std::false_type{});
}

template <typename K>
int lds_limit(K kernel, size_t lds) {
  if (lds > 64 * 1024)
    EXC_CHECK_HIP(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  return EXC_OK;
}

template <typename T>
int givens_launch(T* x, long m, long n, const int32_t* pairs, const double* cs, long passes, int mask, int is_left,
                  hipStream_t s) {
  EXC_REQUIRE(x && pairs && cs && m >= 1 && n >= 1 && passes >= 0, EXC_ERR_ARG, "exc_givens_apply: bad arguments");
  const long K = is_left ? m : n;
  const long lines = is_left ? n : m;
  if (K <= 1 || passes == 0) return EXC_OK;
  const int half = (int)((K % 2 == 0 ? K : K + 1) / 2);
  const int odd_mode = (K % 2 == 1) ? (mask ? 2 : 1) : 0;
  EXC_REQUIRE((size_t)K * sizeof(T) <= kLdsHard, EXC_ERR_ARG,
              "exc_givens_apply: a line does not fit in LDS (K too large)");
  const Sweep sw = sweep_shape(K, lines, half, sizeof(T));
  const size_t lds = (size_t)K * sw.l * sizeof(T);
  hipEvent_t e0 = exc_prof::mark(s);
  const int rc = with_shape<T>(sw, is_left != 0, [&](auto l, auto np, auto left) -> int {
    auto kernel = k_givens<T, decltype(l)::value, decltype(np)::value, decltype(left)::value>;
    if (int e = lds_limit(kernel, lds)) return e;
    hipLaunchKernelGGL(kernel, dim3(exc_detail::ceil_div(lines, sw.l)), dim3(sw.threads), lds, s, x, m, n, pairs, cs,
                       (int)passes, half, mask, odd_mode);
    return EXC_OK;
  });
  if (rc) return rc;
  EXC_CHECK_HIP(hipGetLastError());
  if (e0) {
    // one read and one write of the matrix; 6 flops per element per rotation
    const double bytes = 2.0 * sizeof(T) * (double)m * (double)n;
    const double flops = 6.0 * (double)passes * half * (double)lines * 2.0 / 2.0 * 2.0 / 2.0;
    exc_prof::book(sizeof(T) == 8 ? "givens_f64" : "givens_f32", e0, exc_prof::mark(s), flops, bytes);
  }
  return EXC_OK;
}

template <typename T>
int givens_batched_launch(int nb, T* const* d_xs, long m, long n, const int32_t* const* d_pairs,
                          const double* const* d_cs, long passes, int mask, int is_left, hipStream_t s) {
  EXC_REQUIRE(nb >= 0 && m >= 1 && n >= 1 && passes >= 0 && (nb == 0 || (d_xs && d_pairs && d_cs)), EXC_ERR_ARG,
              "exc_givens_apply_batched: bad arguments");
  const long K = is_left ? m : n;
  const long lines = is_left ? n : m;
  if (nb == 0 || K <= 1 || passes == 0) return EXC_OK;
  const int half = (int)((K % 2 == 0 ? K : K + 1) / 2);
  const int odd_mode = (K % 2 == 1) ? (mask ? 2 : 1) : 0;
  EXC_REQUIRE((size_t)K * sizeof(T) <= kLdsHard, EXC_ERR_ARG, "exc_givens_apply_batched: K too large");
  const Sweep sw = sweep_shape(K, lines * nb, half, sizeof(T));
  const size_t lds = (size_t)K * sw.l * sizeof(T);
  const int rc = with_shape<T>(sw, is_left != 0, [&](auto l, auto np, auto left) -> int {
    auto kernel = k_givens_batched<T, decltype(l)::value, decltype(np)::value, decltype(left)::value>;
    if (int e = lds_limit(kernel, lds)) return e;
    hipLaunchKernelGGL(kernel, dim3(exc_detail::ceil_div(lines, sw.l), nb), dim3(sw.threads), lds, s, d_xs, m, n,
                       d_pairs, d_cs, (int)passes, half, mask, odd_mode);
    return EXC_OK;
  });
  if (rc) return rc;
  EXC_CHECK_HIP(hipGetLastError());
  return EXC_OK;
}

}  // namespace

extern "C" {

int exc_givens_apply_batched(int nb, double* const* d_xs, long m, long n, const int32_t* const* d_pairs,
                             const double* const* d_cs, long passes, int mask, int is_left, exc_stream_t stream) {
  return givens_batched_launch<double>(nb, d_xs, m, n, d_pairs, d_cs, passes, mask, is_left,
                                       exc_detail::stream(stream));
}

int exc_givens_apply(double* d_x, long m, long n, const int32_t* d_pairs, const double* d_cs, long passes, int mask,
                     int is_left, exc_stream_t stream) {
  return givens_launch<double>(d_x, m, n, d_pairs, d_cs, passes, mask, is_left, exc_detail::stream(stream));
}

int exc_givens_apply_f32(float* d_x, long m, long n, const int32_t* d_pairs, const double* d_cs, long passes,
                         int mask, int is_left, exc_stream_t stream) {
  return givens_launch<float>(d_x, m, n, d_pairs, d_cs, passes, mask, is_left, exc_detail::stream(stream));
}

}  // extern "C"
