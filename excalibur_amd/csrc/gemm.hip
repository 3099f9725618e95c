// Dense GEMM on the gfx950 matrix cores: C = alpha * op(A) op(B) + beta * C, row-major, FP64
// (v_mfma_f64_16x16x4_f64) and FP32 (v_mfma_f32_16x16x4_f32).
//
// Workgroup tiles of 128 x 128 and 64 x 64, chosen per product (gemm_plan); K is staged through
// registers into LDS in steps of 16, one step ahead of the one being multiplied and two ahead of the
// loads. Bound by the MFMAs: FP64 67.9 TFLOP/s at order 4096 and 61.4 on 1000 x 50000 x 1000 (the
// MFMA loop alone 78, the vendor library 71 and 59), FP32 134 at order 8192 and 130 on 2000 x 100000
// x 2000 (156 alone, 149 the library); with scalar loads behind branches, whose merged registers
// waited for every load at once, 55 and 46.6, 111 and 105. Options used by the factorizations: split-K
// (partial tiles summed in a fixed order by a second kernel, so results do not depend on
// scheduling), skipping the zero K range of a triangular op(A), and computing only the lower tiles of a
// symmetric product (mirrored into the upper half by a kernel of its own, in grouped products by the
// reduction).
#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <string>
#include <type_traits>
#include <vector>

#include "exc_common.hpp"
#include "gemm.hpp"

namespace {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

template <typename T>
struct Mfma;
template <>
struct Mfma<double> {
  typedef d4 acc_t;
  __device__ static inline acc_t step(double a, double b, acc_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  // result element v of lane l sits in row (l/16) + 4v, column l%16
  __device__ static inline int row(int lk, int v) { return lk + 4 * v; }
};
template <>
struct Mfma<float> {
  typedef f4 acc_t;
  __device__ static inline acc_t step(float a, float b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  // result element v of lane l sits in row 4(l/16) + v, column l%16
  __device__ static inline int row(int lk, int v) { return 4 * lk + v; }
};


struct GemmArgs {
  long M, N, K;
  const void* A;
  long lda;
  const void* B;
  long ldb;
  void* C;
  long ldc;
  double alpha, beta;
  int tri;        // EXC_TRI_* restriction of the K range per tile
  int lower_only; // compute only tiles with tile_row >= tile_col
  long kchunk;    // split-K chunk (multiple of the K step); 0 = no split
  void* part;     // split-K partials: splits x M x N (type T)
  int bm, bn;     // tile sizes
  long tm;        // tile rows
  long ntile;     // tiles per split (tm x tn, or the lower tiles tm (tm + 1) / 2)
  int pair;       // a workgroup takes the tile rows r and tm - 1 - r (op(A) triangular)
  long total;     // ntile x splits = the 1-D grid
};

constexpr int kXcds = 8;  // dies of the device; the dispatcher deals workgroups round-robin over them

// Tile of workgroup blockIdx.x. The dispatcher sends linear id L to die L % 8, so consecutive tiles
// of the natural order would land on eight dies with eight separate L2s. The remap gives die x a
// contiguous range of the tile order instead, and that order runs the row tiles of one column
// (m fastest) back to back, so their shared B column tile is fetched from HBM once per die and
// the row tiles read it from that die's L2. Splits of K are the slowest index, except where op(A) is
// triangular: its splits differ in their work, so every die takes all splits of its columns (with a
// split or two per die the first ones had 1.75 times the average work).
template <bool TRI>
__device__ inline void tile_of(const GemmArgs& g, long& tile_m, long& tile_n, long& split) {
  const long L = blockIdx.x;
  const long q = g.total / kXcds, r = g.total % kXcds;
  const long x = L % kXcds, j = L / kXcds;
  const long t = x * q + min(x, r) + j;
  if (TRI) {
    const long rows = g.pair ? (g.tm + 1) / 2 : g.tm, column = rows * (g.total / g.ntile);
    tile_n = t / column;
    const long u = t - tile_n * column;
    split = u / rows;
    tile_m = u - split * rows;
    return;
  }
  split = t / g.ntile;
  long u = t - split * g.ntile;
  if (g.lower_only) {
    // column n holds the tm - n tiles m = n .. tm - 1
    long n = 0;
    while (u >= g.tm - n) {
      u -= g.tm - n;
      n++;
    }
    tile_n = n;
    tile_m = n + u;
  } else {
    tile_n = u / g.tm;
    tile_m = u - tile_n * g.tm;
  }
}

// K range [k0, k1) that can contribute to output rows [i0, i0+bm).
__device__ inline void k_range(const GemmArgs& g, long i0, int bm, long& k0, long& k1) {
  k0 = g.tri == EXC_TRI_A_UPPER ? i0 : 0;                   // op(A)[i][k] = 0 for k < i
  k1 = g.tri == EXC_TRI_A_LOWER ? min(g.K, i0 + bm) : g.K;  // op(A)[i][k] = 0 for k > i
}

// 16 bytes of one operand, in registers and in LDS; in global memory only the elements' own
// alignment is assumed (gfx950 loads unaligned 16-byte words).
template <typename T>
struct Unit;
template <>
struct Unit<double> {
  typedef double lds_t __attribute__((ext_vector_type(2)));
  typedef double glb_t __attribute__((ext_vector_type(2), aligned(8)));
};
template <>
struct Unit<float> {
  typedef float lds_t __attribute__((ext_vector_type(4)));
  typedef float glb_t __attribute__((ext_vector_type(4), aligned(4)));
};

// Shape of the kernel: WM x WN wavefronts, each MT x NT MFMA tiles, K staged in steps of kRow bytes'
// worth of elements per operand row.
template <typename T, int WM_, int WN_, int MT_, int NT_, int PER, bool FIRST, int KV_>
struct Shape {
  using elem = T;
  static constexpr int WM = WM_, WN = WN_, MT = MT_, NT = NT_;
  static constexpr int BM = 16 * WM * MT, BN = 16 * WN * NT;
  static constexpr int kThreads = 64 * WM * WN;
  static constexpr bool FRAGS_FIRST = FIRST;  // a step's first fragments are read before its stores
  static constexpr int V = 16 / (int)sizeof(T);        // elements of a 16-byte unit
  static constexpr int kRow = sizeof(T) == 8 ? 128 : 64;  // bytes of K per row and step
  static constexpr int UNITS = kRow / 16;
  static constexpr int BK = kRow / (int)sizeof(T);
  static constexpr int KV = KV_;                        // consecutive k of a lane in a fragment (1 or V)
  static constexpr int GROUPS = BK / (4 * KV);          // a group: KV MFMA steps of 4 k each
  static constexpr int kPerCu = PER;  // resident workgroups (registers and LDS)
};

// One operand's slab of a step, E rows (or columns) by BK, staged through registers into
// LDS as 16-byte units. KMAJ: the operand is contiguous along k in memory (A, or B transposed); LDS
// holds [row][unit of k] with the unit index XORed by the row, so the 16 rows a fragment read
// touches fall into different banks. Otherwise it is contiguous along the rows (A transposed, or
// B) and LDS holds [k][unit of rows], whose fragment reads are whole 256-byte lines.
//
// The contraction may run over k in any order that both operands share. With KV = V the lane group
// lk = lane / 16 takes the V consecutive k of unit lk + 4 g, one per MFMA step, so that one 16-byte
// LDS read feeds V steps; with KV = 1 it takes k = lk + 4 g, which sums in ascending order as
// LAPACK's reference does (the 64 x 64 FP64 tile, the one of small matrices: 2 % slower). Where the
// operand is not KMAJ a read feeds up to V MFMA tiles, whose rows interleave (row_of).
//
// A load is branch-free: its coordinates are clamped into the operand, and what that shifted or
// repeated is put right when the registers are stored (fix). A branch around a load merges two
// definitions of its registers, and the copies that takes wait for the load on the spot.
template <typename T, bool KMAJ, int E, int TT, int UNITS, int KV, int kThreads>
struct Slab {
  typedef typename Unit<T>::lds_t lv;
  typedef typename Unit<T>::glb_t gv;
  static constexpr int V = 16 / (int)sizeof(T);
  static constexpr int Q = E * UNITS / kThreads;    // units per thread
  static constexpr int UPR = KMAJ ? UNITS : E / V;  // units of one LDS row
  static constexpr int STEP = kThreads / UPR;       // rows between a thread's units
  static constexpr int VT = TT < V ? TT : V;        // interleaved MFMA tiles (not KMAJ)
  static constexpr int NP = KMAJ ? Q : 1;
  const T* p[NP];  // KMAJ: this thread's rows at k = 0; else its column at k = 0
  long ld;
  long e0, ext;    // first row of the slab, rows of the operand
  int r0, u;       // first LDS row and unit of this thread
  int sh;          // not KMAJ: elements the clamp moved the unit down by
  lv reg[Q];

  __device__ Slab(const void* P, long ld_, long e0_, long ext_, int tid) : ld(ld_), e0(e0_), ext(ext_) {
    r0 = tid / UPR;
    u = tid % UPR;
    sh = 0;
    if (KMAJ) {
#pragma unroll
      for (int q = 0; q < NP; q++) p[q] = (const T*)P + min(e0 + r0 + q * STEP, ext - 1) * ld;
    } else {
      const long c = e0 + (long)u * V, last = max(ext - V, 0L);
      p[0] = (const T*)P + min(c, last);
      sh = (int)min(max(c - last, 0L), (long)V);
    }
  }
  // The step at kb of the range that ends at k1 (k1 >= V; not KMAJ: ext >= V). What depends on the
  // thread is kept in 32 bits, relative to the step: the registers decide how many workgroups
  // are resident.
  __device__ __forceinline__ void load(long kb, long k1) {
    if (KMAJ) {
      const int k = min(u * V, near(k1 - V - kb));
#pragma unroll
      for (int q = 0; q < Q; q++) reg[q] = *(const gv*)(p[q % NP] + kb + k);
    } else {
      const int last = near(k1 - 1 - kb);
      const T* s = p[0] + kb * ld;
#pragma unroll
      for (int q = 0; q < Q; q++) reg[q] = *(const gv*)(s + min(r0 + q * STEP, last) * ld);
    }
  }
  // a (uniform) distance, saturated far beyond any step
  __device__ static __forceinline__ int near(long d) { return (int)max(min(d, 1L << 24), -(1L << 24)); }
  // The same step element by element, for operands too small for a unit.
  __device__ __forceinline__ void load_checked(long kb, long k1) {
#pragma unroll
    for (int q = 0; q < Q; q++) {
      lv x;
#pragma unroll
      for (int v = 0; v < V; v++) {
        const long row = KMAJ ? e0 + r0 + q * STEP : e0 + (long)u * V + v;
        const long k = KMAJ ? kb + u * V + v : kb + r0 + q * STEP;
        T e = T(0);
        if (row < ext && k < k1) e = KMAJ ? p[q % NP][k] : p[0][k * ld + (row - min(e0 + (long)u * V, max(ext - V, 0L)))];
        x[v] = e;
      }
      reg[q] = x;
    }
  }
  // Elements moved down by s places, zeros behind them (s >= V: all zero).
  __device__ static __forceinline__ lv shifted(lv x, int s) {
    lv y;
#pragma unroll
    for (int v = 0; v < V; v++) {
      T e = T(0);
#pragma unroll
      for (int w = v; w < V; w++) e = w - v == s ? x[w] : e;
      y[v] = e;
    }
    return y;
  }
  // Puts right what the clamps of load did: the step's elements at or beyond k1 become zero.
  __device__ __forceinline__ void fix(long kb, long k1) {
    const int left = near(k1 - kb);
    const int s = KMAJ ? min(max(u * V + V - left, 0), V) : sh;
#pragma unroll
    for (int q = 0; q < Q; q++) reg[q] = shifted(reg[q], !KMAJ && r0 + q * STEP >= left ? V : s);
  }
  // Whether every step needs fix (a unit straddles the end of the rows).
  __device__ __forceinline__ bool ragged() const { return !KMAJ && e0 + E > ext && ext % V != 0; }
  // Zeroes the elements on the far side of the diagonal: k > row (lower) or k < row (upper).
  __device__ __forceinline__ void mask(long kb, bool lower) {
    const int d = near(e0 - kb);
#pragma unroll
    for (int q = 0; q < Q; q++) {
      lv x = reg[q];
#pragma unroll
      for (int v = 0; v < V; v++) {
        const int row = d + (KMAJ ? r0 + q * STEP : u * V + v);
        const int k = KMAJ ? u * V + v : r0 + q * STEP;
        const bool zero = lower ? k > row : k < row;
        x[v] = zero ? T(0) : x[v];
      }
      reg[q] = x;
    }
  }
  __device__ static inline int swz(int row) { return KMAJ ? (row / (16 / UNITS)) & (UNITS - 1) : 0; }
  __device__ __forceinline__ void store(lv* lds) const {
#pragma unroll
    for (int q = 0; q < Q; q++) {
      const int r = r0 + q * STEP;
      lds[r * UPR + (u ^ swz(r))] = reg[q];
    }
  }
  // The wavefront's fragments of group g: f[v][t] is MFMA step v's element for tile t; w0 is the
  // wavefront's first row of the slab.
  __device__ static __forceinline__ void frag(const lv* lds, int w0, int g, int li, int lk, T (*f)[TT]) {
    const int k0 = (lk + 4 * g) * KV;
    const T* l = (const T*)lds;
    if (KMAJ) {
#pragma unroll
      for (int t = 0; t < TT; t++) {
        const int r = w0 + t * 16 + li;
        const int at = r * UPR + ((k0 / V) ^ swz(r));
        if (KV == V) {
          const lv x = lds[at];
#pragma unroll
          for (int v = 0; v < KV; v++) f[v][t] = x[v];
        } else {
          f[0][t] = l[at * V + k0 % V];
        }
      }
    } else {
#pragma unroll
      for (int v = 0; v < KV; v++) {
        const T* line = l + (k0 + v) * E + w0;
#pragma unroll
        for (int t = 0; t < TT; t += VT) {
          if (VT == V) {
            const lv x = *(const lv*)(line + t * 16 + li * VT);
#pragma unroll
            for (int z = 0; z < VT; z++) f[v][t + z] = x[z];
          } else {
#pragma unroll
            for (int z = 0; z < VT; z++) f[v][t + z] = line[t * 16 + li * VT + z];
          }
        }
      }
    }
  }
  // Row of the wavefront's block that element r of MFMA tile t stands for.
  __device__ static __forceinline__ int row_of(int t, int r) {
    return KMAJ ? t * 16 + r : (t / VT) * 16 * VT + r * VT + t % VT;
  }
};

// The 128 x 128 and 64 x 64 workgroup tiles. kStep: measured time of a step on a CU with its
// resident workgroups (us per workgroup), kAlone: with one workgroup on the CU; kTriStep, kTriAlone: the
// same with a triangular op(A), whose mask costs registers (the FP64 128 x 128 kernel of A B reloads a
// few in its loop). The MFMAs alone take
// 1.73 / 0.43 us in FP64 and 0.86 / 0.22 us in FP32. The FP64 tile is split over eight wavefronts
// (four of 64 x 64, whose 256 registers leave two wavefronts per SIMD, are 3 % slower at order 4096); in
// FP32 eight are 5 % slower than four at order 8192. kMaxSum: terms of one running sum
// (its rounding error grows with them) beyond which K is split as far as the workspace allows and,
// in FP64 (kMaxSumFills), as far as two workgroups per CU (and a plan that stays above it counts 10 % more).
template <typename T>
struct Shapes;
template <>
struct Shapes<double> {
  using Big = Shape<double, 4, 2, 2, 4, 2, false, 2>;
  using Small = Shape<double, 2, 2, 2, 2, 4, true, 1>;
  static constexpr double kStep[2] = {1.98, 0.54}, kAlone[2] = {2.09, 0.73};
  static constexpr double kTriStep[2] = {2.10, 0.60}, kTriAlone[2] = {2.65, 1.0};
  static constexpr long kMaxSum = 256;
  static constexpr bool kMaxSumFills = true;
};
template <>
struct Shapes<float> {
  using Big = Shape<float, 2, 2, 4, 4, 3, true, 4>;
  using Small = Shape<float, 2, 2, 2, 2, 4, true, 4>;
  static constexpr double kStep[2] = {1.00, 0.287}, kAlone[2] = {1.18, 0.52};
  static constexpr double kTriStep[2] = {1.09, 0.322}, kTriAlone[2] = {1.58, 0.63};
  static constexpr long kMaxSum = 2048;
  static constexpr bool kMaxSumFills = false;
};

template <class S>
struct Tiles {
  typename Unit<typename S::elem>::lds_t a[2][S::BM * S::UNITS];
  typename Unit<typename S::elem>::lds_t b[2][S::BN * S::UNITS];
};

// One output tile [i0, i0+BM) x [j0, j0+BN) over the K range [k0, k1), k0 a multiple of BK. The result element (gi, gj)
// goes to Cb[(gi - ci0) * ldc + (gj - cj0)]: scaled by alpha (plus beta times the old value) when
// direct, else stored as it is (a split-K partial).
//
// Step c's products read one LDS buffer while the registers, loaded during step c - 1, are stored
// into the other and refilled with step c + 2's loads: a load has a whole step to arrive, and the
// barrier that ends a step waits for no memory. (The stores and loads past the last step, of
// clamped addresses, are not read.)
template <typename T, int TA, int TB, bool TRI, class S>
__device__ __forceinline__ void gemm_tile(const GemmArgs& g, long i0, long j0, long k0, long k1, T* Cb, long ldc,
                                          long ci0, long cj0, bool direct, Tiles<S>& lds) {
  using acc_t = typename Mfma<T>::acc_t;
  constexpr int BK = S::BK, V = S::V, MT = S::MT, NT = S::NT;
  using SA = Slab<T, !TA, S::BM, MT, S::UNITS, S::KV, S::kThreads>;
  using SB = Slab<T, (bool)TB, S::BN, NT, S::UNITS, S::KV, S::kThreads>;
  const int tid = threadIdx.x;
  const int wave = tid >> 6, lane = tid & 63;
  const int li = lane & 15, lk = lane >> 4;
  const int wm = (wave / S::WN) * 16 * MT, wn = (wave % S::WN) * 16 * NT;
  SA sa(g.A, g.lda, i0, g.M, tid);
  SB sb(g.B, g.ldb, j0, g.N, tid);
  acc_t acc[MT][NT];
#pragma unroll
  for (int a = 0; a < MT; a++)
#pragma unroll
    for (int b = 0; b < NT; b++) acc[a][b] = acc_t{0, 0, 0, 0};
  // the last step of a range that ends inside it, operands whose rows end inside a unit, and a
  // triangular operand's steps that cross its diagonal (the k range already excludes the steps
  // wholly on the zero side) are put right between their load and their store
  const bool ragged_a = sa.ragged(), ragged_b = sb.ragged();
  auto store = [&](long kb, int buf, bool fix) __attribute__((always_inline)) {
    if (fix) {
      const bool tail = kb + BK > k1;
      if (tail || ragged_a) sa.fix(kb, k1);
      if (tail || ragged_b) sb.fix(kb, k1);
    }
    if (TRI) {
      const bool lower = g.tri == EXC_TRI_A_LOWER;
      if (lower ? kb + BK > i0 + 1 : g.tri == EXC_TRI_A_UPPER && kb < i0 + S::BM - 1) sa.mask(kb, lower);
    }
    sa.store(lds.a[buf]);
    sb.store(lds.b[buf]);
  };
  T fa[S::KV][MT], fb[S::KV][NT];
  auto frags = [&](int buf, int gr) __attribute__((always_inline)) {
    SA::frag(lds.a[buf], wm, gr, li, lk, fa);
    SB::frag(lds.b[buf], wn, gr, li, lk, fb);
  };
  auto products = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int v = 0; v < S::KV; v++)
#pragma unroll
      for (int a = 0; a < MT; a++)
#pragma unroll
        for (int b = 0; b < NT; b++) acc[a][b] = Mfma<T>::step(fa[v][a], fb[v][b], acc[a][b]);
  };
  if (g.K < V || (TA && g.M < V) || (!TB && g.N < V)) {
    for (long kb = k0; kb < k1; kb += BK) {
      sa.load_checked(kb, k1);
      sb.load_checked(kb, k1);
      store(kb, 0, false);
      lds_barrier();
#pragma unroll
      for (int gr = 0; gr < S::GROUPS; gr++) {
        frags(0, gr);
        products();
      }
      lds_barrier();
    }
  } else if (k0 < k1) {
    sa.load(k0, k1);
    sb.load(k0, k1);
    store(k0, 0, true);
    sa.load(k0 + BK, k1);
    sb.load(k0 + BK, k1);
    lds_barrier();
    int buf = 0;
    for (long kb = k0; kb < k1; kb += BK) {
      if (S::FRAGS_FIRST) frags(buf, 0);
      store(kb + BK, buf ^ 1, true);
      sa.load(kb + 2 * BK, k1);
      sb.load(kb + 2 * BK, k1);
      if (!S::FRAGS_FIRST) frags(buf, 0);
      products();
#pragma unroll
      for (int gr = 1; gr < S::GROUPS; gr++) {
        frags(buf, gr);
        products();
      }
      lds_barrier();
      buf ^= 1;
    }
  }
  // epilogue: operands were supplied as A[lane%16][lane/16], B[lane/16][lane%16]. The VN
  // interleaved tiles of a B that is contiguous along n hold consecutive columns: one store.
  const T alpha = (T)g.alpha, beta = (T)g.beta;
  constexpr int VN = TB ? 1 : SB::VT;
  typedef T cv __attribute__((ext_vector_type(VN == 1 ? 2 : VN), aligned(sizeof(T))));
#pragma unroll
  for (int a = 0; a < MT; a++)
#pragma unroll
    for (int b = 0; b < NT; b += VN)
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const long gi = i0 + wm + SA::row_of(a, Mfma<T>::row(lk, v));
        const long gj = j0 + wn + SB::row_of(b, li);
        if (gi >= g.M || gj >= g.N) continue;
        T* cp = Cb + (gi - ci0) * ldc + (gj - cj0);
        if (VN > 1 && gj + VN <= g.N) {
          cv out;
#pragma unroll
          for (int z = 0; z < VN; z++) out[z] = direct ? alpha * acc[a][b + z][v] : acc[a][b + z][v];
          if (direct && g.beta != 0.0) {
            const cv old = *(const cv*)cp;
#pragma unroll
            for (int z = 0; z < VN; z++) out[z] += beta * old[z];
          }
          *(cv*)cp = out;
        } else {
#pragma unroll
          for (int z = 0; z < VN; z++)
            if (gj + z < g.N) {
              T out = direct ? alpha * acc[a][b + z][v] : acc[a][b + z][v];
              if (direct && g.beta != 0.0) out += beta * cp[z];
              cp[z] = out;
            }
        }
      }
}

// TRI: op(A) is triangular. The general products are a kernel of their own: the triangle's
// code in their loop costs registers, and with them 5 % of their rate.
template <typename T, int TA, int TB, bool TRI, class S>
__global__ __launch_bounds__(S::kThreads, S::kPerCu * S::kThreads / 256) void k_gemm(GemmArgs g) {
  __shared__ Tiles<S> lds;
  long tile_m, tile_n, split;
  tile_of<TRI>(g, tile_m, tile_n, split);
  const long j0 = tile_n * S::BN;
  T* Cb = g.kchunk > 0 ? (T*)g.part + (size_t)split * g.M * g.N : (T*)g.C;
  const long ldc = g.kchunk > 0 ? g.N : g.ldc;
  const long ks = split * g.kchunk, ke = g.kchunk > 0 ? min(g.K, ks + g.kchunk) : g.K;
  if (!TRI) {
    gemm_tile<T, TA, TB, false, S>(g, tile_m * S::BM, j0, ks, ke, Cb, ldc, 0, 0, g.kchunk == 0, lds);
    return;
  }
  for (;;) {
    long k0, k1;
    k_range(g, tile_m * S::BM, S::BM, k0, k1);
    k0 = max(k0, ks);
    k1 = min(k1, ke);
    if (k0 >= k1 && g.kchunk > 0) return;  // the sum of the partials passes over this one
    gemm_tile<T, TA, TB, true, S>(g, tile_m * S::BM, j0, k0, k1, Cb, ldc, 0, 0, g.kchunk == 0, lds);
    // a triangular op(A) gives row r of the tiles a K range that grows or shrinks with r: rows r and
    // tm - 1 - r together are the same work for every workgroup
    if (!g.pair || 2 * tile_m >= g.tm - 1) break;  // the second of a pair, or the middle row
    tile_m = g.tm - 1 - tile_m;
    lds_barrier();  // the next tile restages the slabs
  }
}

// Grouped products: many independent problems of one transposition pattern in one launch. The
// host lays out work items (problem, tile or pair of tiles, K range, partial slot), one workgroup
// each, running the same tile code as k_gemm; the dispatcher balances them over the CUs (a grid that
// strode over them by itself gave every workgroup a fixed share, whatever its items' lengths).
// Items of a tile split over K (or of a mirrored symmetric product) store partial tiles;
// k_grouped_reduce then sums each tile's partials in slot order (deterministic), applies alpha
// and beta, and mirrors lower tiles.
struct GroupProb {
  const void* A;
  const void* B;
  void* C;
  long lda, ldb, ldc, M, N, K;
  int tri, lower_only, mirror, pad;
};
struct GroupItem {
  // slot < 0: the item owns its whole tile and stores it directly; kPaired: and the tile of row
  // tm - 1 - tile_m as well (a triangular op(A), see k_gemm)
  int p, tile_m, tile_n, slot;
  long k0, k1;
};
constexpr int kPaired = -2;
struct GroupRed {
  int p, tile_m, tile_n, first_slot, nslots, pad;
};

// 64 x 64 tiles where op(A) is triangular (they skip more of its zeros, and the large tile's
// registers do not hold the triangle's code: 32 products L^-1 X of order 512 took 7.1 ms with it,
// 6.9 with the small one), 128 x 128 elsewhere.
template <typename T, bool TRI>
using GroupShape = std::conditional_t<TRI, typename Shapes<T>::Small, typename Shapes<T>::Big>;

template <typename T, int TB, bool TRI>
__global__ __launch_bounds__((GroupShape<T, TRI>::kThreads), (GroupShape<T, TRI>::kPerCu * GroupShape<T, TRI>::kThreads / 256)) void k_gemm_grouped(
    const GroupProb* __restrict__ probs, const GroupItem* __restrict__ items, long nitems, T* __restrict__ part,
    double alpha, double beta) {
  using S = GroupShape<T, TRI>;
  constexpr int BM = S::BM, BN = S::BN;
  __shared__ Tiles<S> lds;
  // each die takes a contiguous range of the items, as in tile_of
  const long L = blockIdx.x, q = nitems / kXcds, r = nitems % kXcds;
  const GroupItem w = items[(L % kXcds) * q + min(L % kXcds, r) + L / kXcds];
  const GroupProb pr = probs[w.p];
  GemmArgs g{};
  g.A = pr.A; g.lda = pr.lda; g.B = pr.B; g.ldb = pr.ldb; g.M = pr.M; g.N = pr.N; g.K = pr.K;
  g.tri = pr.tri; g.alpha = alpha; g.beta = beta;
  const bool direct = w.slot < 0;
  const long j0 = (long)w.tile_n * BN;
  T* Cb = direct ? (T*)pr.C : part + (size_t)w.slot * BM * BN;
  const int other_m = (int)((pr.M + BM - 1) / BM) - 1 - w.tile_m;
  for (int tile_m = w.tile_m;;) {
    const long i0 = (long)tile_m * BM;
    long k0 = w.k0, k1 = w.k1;
    if (TRI) {
      k_range(g, i0, BM, k0, k1);
      k0 = max(k0, w.k0);
      k1 = min(k1, w.k1);
    }
    gemm_tile<T, 0, TB, TRI, S>(g, i0, j0, k0, k1, Cb, direct ? pr.ldc : BN, direct ? 0 : i0, direct ? 0 : j0,
                                 direct, lds);
    if (!TRI || w.slot != kPaired || tile_m >= other_m) break;
    tile_m = other_m;
    lds_barrier();  // the next tile restages the slabs
  }
}

template <typename T>
__global__ __launch_bounds__(256) void k_grouped_reduce(const GroupProb* __restrict__ probs,
                                                        const GroupRed* __restrict__ reds, const T* __restrict__ part,
                                                        int tile, double alpha, double beta) {
  const GroupRed r = reds[blockIdx.x];
  const GroupProb pr = probs[r.p];
  T* C = (T*)pr.C;
  for (int e = threadIdx.x; e < tile * tile; e += blockDim.x) {
    const int li = e / tile, lj = e - li * tile;
    const long gi = (long)r.tile_m * tile + li, gj = (long)r.tile_n * tile + lj;
    if (gi >= pr.M || gj >= pr.N) continue;
    if (pr.lower_only && gj > gi) continue;  // the upper part of a diagonal tile comes by mirroring
    T s = T(0);
#pragma unroll 4
    for (int q = 0; q < r.nslots; q++) s += part[(size_t)(r.first_slot + q) * tile * tile + e];
    T out = (T)alpha * s;
    if (beta != 0.0) out += (T)beta * C[gi * pr.ldc + gj];
    C[gi * pr.ldc + gj] = out;
    if (pr.mirror && gj < gi) C[gj * pr.ldc + gi] = out;
  }
}

// Sums split-K partials in split order, applies alpha/beta, and mirrors lower tiles when asked.
template <typename T>
__global__ __launch_bounds__(256) void k_splitk_reduce(GemmArgs g, int splits) {
  const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long total = g.M * g.N;
  if (idx >= total) return;
  const long i = idx / g.N, j = idx - i * g.N;
  if (g.lower_only && (j / g.bn) > (i / g.bm)) return;
  const T* P = (const T*)g.part;
  int z0 = 0, z1 = splits;
  if (g.tri != EXC_TRI_NONE) {  // the splits outside the tile's K range have no partial
    long k0, k1;
    k_range(g, i / g.bm * g.bm, g.bm, k0, k1);
    z0 = (int)(k0 / g.kchunk);
    z1 = (int)((k1 + g.kchunk - 1) / g.kchunk);
  }
  T s = T(0);
#pragma unroll 8
  for (int z = z0; z < z1; z++) s += P[(size_t)z * total + idx];
  T* C = (T*)g.C;
  T out = (T)g.alpha * s;
  if (g.beta != 0.0) out += (T)g.beta * C[i * g.ldc + j];
  C[i * g.ldc + j] = out;
}

// Copies the lower triangle onto the upper one (square C).
template <typename T>
__global__ __launch_bounds__(256) void k_mirror_lower(long n, T* C, long ldc) {
  const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= n * n) return;
  const long i = idx / n, j = idx - i * n;
  if (j > i) C[i * ldc + j] = C[j * ldc + i];
}

// Compute units of the current device (cached per device).
long compute_units() {
  static std::atomic<int> cus[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  int n = cus[dev].load();
  if (n <= 0) {
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    cus[dev].store(n);
  }
  return n;
}

struct GemmPlan {
  int tile;    // 128 or 64
  int splits;  // of K
};

// The least splits of K: they bound the length of a running sum, and with it the rounding error of
// the result. They are those that let 128 x 128 tiles on `slots` resident workgroups end soonest: rounds
// of the chip times steps of about 3 us, and the sum of the partials at 3 TB/s. The faster kernels of
// today would take fewer (1000 x 1000 x 2000 in FP64: 2 instead of 8), but then the sums are longer (1008
// terms instead of 256) and the error of their rounding was 1.7 to 2.9 times as large.
template <typename T>
long least_splits(long M, long N, long K, long tiles, long slots, long room) {
  constexpr int BK = Shapes<T>::Big::BK;
  if (tiles >= slots) return 1;
  long best = 1;
  double best_us = -1.0;
  for (long sp = 1; sp <= std::min({K / BK, 4 * ((slots + tiles - 1) / tiles), room}); sp++) {
    const long rounds = (tiles * sp + slots - 1) / slots, depth = ((K + sp - 1) / sp + BK - 1) / BK;
    const double us = 3.0 * (double)(rounds * depth) + (sp > 1 ? 5.0 + (double)sp * M * N * sizeof(T) / 3.0e6 : 0.0);
    if (best_us < 0.0 || us < best_us) {
      best_us = us;
      best = sp;
    }
  }
  return best;
}

// Tile and split of one product: the pair with the least estimated time. A CU with w workgroups
// takes max(w kStep, kAlone) per step; a split adds the write and the fixed-order sum of its partials
// (about 5 TB/s, they stay in the caches) and 5 us for its launch. Splits need a workspace, and those
// beyond the least keep two steps each (a lone step is all latency); near ties go to the larger tile and
// fewer splits. A triangular product takes the large tile unsplit only: split, its uneven pieces fill the
// chip better as small ones (FP64, order 1000 in 8 splits 52 us against 58, order 2000 in 4 222 against
// 236). Unsplit, L X with L of order 1000 and 50,000 columns takes 1.03 ms with the small tile and 1.10
// with the large, of order 2000 and 40,000 columns 3.08 and 2.85; in FP32 567 and 565 us, 1.67 and 1.46 ms.
template <typename T>
GemmPlan gemm_plan(long M, long N, long K, const ExcGemmOpts& o) {
  constexpr int BK = Shapes<T>::Big::BK;
  constexpr long kMaxSum = Shapes<T>::kMaxSum;
  const long cus = compute_units();
  GemmPlan best{128, 1};
  double best_us = -1.0;
  const bool tri = o.tri != EXC_TRI_NONE;
  const double* step = tri ? Shapes<T>::kTriStep : Shapes<T>::kStep;
  const double* alone = tri ? Shapes<T>::kTriAlone : Shapes<T>::kAlone;
  const long fit = o.work && K > 4 * BK ? (long)std::min<size_t>(K, o.work_bytes / ((size_t)M * N * sizeof(T))) : 1;
  const long room = std::min(fit, K / (2 * BK));
  const long tm128 = (M + 127) / 128, tn128 = (N + 127) / 128;
  const long floor = least_splits<T>(M, N, K, o.lower_only ? tm128 * (tm128 + 1) / 2 : tm128 * tn128,
                                     cus * Shapes<T>::Big::kPerCu, fit);
  for (int c = 0; c < 2; c++) {
    const long tile = c == 0 ? 128 : 64;
    const long tm = (M + tile - 1) / tile, tn = (N + tile - 1) / tile;
    const long tiles = o.lower_only ? tm * (tm + 1) / 2 : tm * tn;
    const long slots = cus * (c == 0 ? Shapes<T>::Big::kPerCu : Shapes<T>::Small::kPerCu);
    const double out = (double)sizeof(T) * M * N * (o.lower_only ? 0.5 : 1.0);
    const long filled = tri ? tiles / 2 + 1 : tiles;  // about half of a split triangle's tiles are empty
    const long most = std::max(1L, std::min(room, 2 * ((slots + filled - 1) / filled)));
    long least = std::min(room, (K + kMaxSum - 1) / kMaxSum);
    if (Shapes<T>::kMaxSumFills) least = std::min(least, 2 * cus / tiles);
    least = std::max(least, floor);
    for (long sp = least; sp <= std::max(least, most); sp++) {
      if (tri && sp > 1 && c == 0) break;
      double depth = (double)(((K + sp - 1) / sp + BK - 1) / BK);
      long units = tiles * sp;
      double sums = (double)sp;
      if (tri && sp == 1) {  // pairs of tile rows, 1 + 1 / tm of K together
        units = (tm + 1) / 2 * tn;
        depth *= 1.0 + 1.0 / (double)tm;
      } else if (tri) {  // half the tiles and partials, and those on the diagonal, are not empty
        units = (tiles * (sp + 1) + 1) / 2;
        sums = 0.5 * (double)(sp + 1);
      }
      const long per_cu = (units + cus - 1) / cus;
      double us = 6.0 + depth * std::max(per_cu * step[c], alone[c]);
      if (sp > 1) us += 5.0 + (2 * sums + 1) * out / 5.0e6;
      if (Shapes<T>::kMaxSumFills && K > sp * kMaxSum) us *= 1.1;
      if (best_us < 0.0 || us < 0.99 * best_us) {
        best_us = us;
        best = GemmPlan{(int)tile, (int)sp};
      }
    }
  }
  return best;
}

template <typename T, bool TRI, class S>
void gemm_launch(int ta, int tb, const GemmArgs& g, hipStream_t s) {
  const dim3 grid((unsigned)g.total), block(S::kThreads);
  if constexpr (!TRI)
    if (tb) {
      if (ta) hipLaunchKernelGGL((k_gemm<T, 1, 1, TRI, S>), grid, block, 0, s, g);
      else hipLaunchKernelGGL((k_gemm<T, 0, 1, TRI, S>), grid, block, 0, s, g);
      return;
    }
  if (ta) hipLaunchKernelGGL((k_gemm<T, 1, 0, TRI, S>), grid, block, 0, s, g);
  else hipLaunchKernelGGL((k_gemm<T, 0, 0, TRI, S>), grid, block, 0, s, g);
}

template <typename T>
int gemm_impl(int ta, int tb, long M, long N, long K, double alpha, const T* A, long lda, const T* B, long ldb,
              double beta, T* C, long ldc, const ExcGemmOpts& o, hipStream_t s) {
  EXC_REQUIRE(M >= 0 && N >= 0 && K >= 0 && C, EXC_ERR_ARG, "exc_gemm: bad shape");
  if (M == 0 || N == 0) return EXC_OK;
  EXC_REQUIRE(o.tri == EXC_TRI_NONE || (!tb && !o.lower_only), EXC_ERR_ARG,
              "exc_gemm: a triangular op(A) takes op(B) = B and a whole C");
  GemmArgs g{};
  g.M = M; g.N = N; g.K = K;
  g.A = A; g.lda = lda; g.B = B; g.ldb = ldb; g.C = C; g.ldc = ldc;
  g.alpha = alpha; g.beta = beta; g.tri = o.tri; g.lower_only = o.lower_only;
  constexpr int BK = Shapes<T>::Big::BK;
  const GemmPlan p = gemm_plan<T>(M, N, K, o);
  g.bm = g.bn = p.tile;
  g.tm = (M + p.tile - 1) / p.tile;
  const long tn = (N + p.tile - 1) / p.tile;
  int splits = p.splits;
  if (splits > 1) {
    long chunk = (K + splits - 1) / splits;
    chunk = ((chunk + BK - 1) / BK) * BK;
    splits = (int)((K + chunk - 1) / chunk);
    g.kchunk = chunk;
    g.part = o.work;
  }
  // an unsplit triangular product's tile rows are paired; a split one's have finer work by themselves
  g.pair = o.tri != EXC_TRI_NONE && splits == 1;
  g.ntile = o.lower_only ? g.tm * (g.tm + 1) / 2 : (g.pair ? (g.tm + 1) / 2 : g.tm) * tn;
  g.total = g.ntile * splits;
  EXC_REQUIRE(g.total < (1L << 31), EXC_ERR_ARG, "exc_gemm: too many tiles");
  hipEvent_t e0 = exc_prof::mark(s);
  const bool tri = o.tri != EXC_TRI_NONE;
  if (p.tile == 128) {
    if (tri) gemm_launch<T, true, typename Shapes<T>::Big>(ta, tb, g, s);
    else gemm_launch<T, false, typename Shapes<T>::Big>(ta, tb, g, s);
  } else {
    if (tri) gemm_launch<T, true, typename Shapes<T>::Small>(ta, tb, g, s);
    else gemm_launch<T, false, typename Shapes<T>::Small>(ta, tb, g, s);
  }
  EXC_CHECK_HIP(hipGetLastError());
  if (e0) {
    // useful flops: a triangular operand halves the products, a symmetric (lower-only) result too
    double flops = 2.0 * (double)M * (double)N * (double)K;
    if (o.tri != EXC_TRI_NONE) flops *= 0.5;
    if (o.lower_only) flops *= 0.5;
    const double bytes = (double)sizeof(T) * ((double)M * K + (double)K * N + (double)M * N * (beta != 0.0 ? 2 : 1));
    exc_prof::book(sizeof(T) == 8 ? "gemm_f64" : "gemm_f32", e0, exc_prof::mark(s), flops, bytes);
  }
  if (splits > 1) {
    hipLaunchKernelGGL(k_splitk_reduce<T>, dim3(exc_detail::ceil_div(M * N, 256)), dim3(256), 0, s, g, splits);
    EXC_CHECK_HIP(hipGetLastError());
  }
  if (o.lower_only && o.mirror) {
    hipLaunchKernelGGL(k_mirror_lower<T>, dim3(exc_detail::ceil_div(M * M, 256)), dim3(256), 0, s, M, C, ldc);
    EXC_CHECK_HIP(hipGetLastError());
  }
  return EXC_OK;
}

// ---- grouped products: tables, launch and the autotuner
struct GroupPlan {
  std::vector<GroupProb> probs;
  std::vector<GroupItem> items;
  std::vector<GroupRed> reds;
  long slots = 0;
  int tile = 128;
  bool tri = false;  // any triangular problem: the kernel for all, with its tile
  double flops = 0.0;
};

GroupPlan group_plan(int nprob, const ExcGemmProblem* P, long kchunk) {
  constexpr int BK = Shapes<double>::Big::BK;
  static_assert(BK == Shapes<float>::Big::BK, "one chunk length for both types");
  GroupPlan g;
  g.tri = std::any_of(P, P + nprob, [](const ExcGemmProblem& q) { return q.tri != EXC_TRI_NONE; });
  g.tile = g.tri ? GroupShape<double, true>::BM : GroupShape<double, false>::BM;
  const int BM = g.tile, BN = g.tile;
  if (kchunk > 0) kchunk = ((kchunk + BK - 1) / BK) * BK;
  for (int p = 0; p < nprob; p++) {
    const ExcGemmProblem& q = P[p];
    GroupProb gp{q.A, q.B, q.C, q.lda, q.ldb, q.ldc, q.M, q.N, q.K, q.tri, q.lower_only, q.mirror, 0};
    g.probs.push_back(gp);
    if (q.M <= 0 || q.N <= 0) continue;
    double f = 2.0 * (double)q.M * q.N * q.K;
    if (q.tri != EXC_TRI_NONE) f *= 0.5;
    if (q.lower_only) f *= 0.5;
    g.flops += f;
    const long tm = (q.M + BM - 1) / BM, tn = (q.N + BN - 1) / BN;
    // chunks of about kchunk, of equal length within a problem
    const long splits = (kchunk > 0 && q.K > kchunk) ? (q.K + kchunk - 1) / kchunk : 1;
    const long chunk = splits == 1 ? q.K : ((q.K + splits - 1) / splits + BK - 1) / BK * BK;
    const bool pair = splits == 1 && !q.lower_only && q.tri != EXC_TRI_NONE;
    for (long b = 0; b < tn; b++)
      for (long a = 0; a < (pair ? (tm + 1) / 2 : tm); a++) {
        if (q.lower_only && a < b) continue;
        if (splits == 1 && !q.mirror) {
          g.items.push_back(GroupItem{p, (int)a, (int)b, pair ? kPaired : -1, 0, q.K});
          continue;
        }
        const long first = g.slots;
        long k0 = 0;
        do {  // an empty K too takes one item: its sum is zero
          g.items.push_back(GroupItem{p, (int)a, (int)b, (int)(g.slots++), k0, std::min(q.K, k0 + chunk)});
          k0 += chunk;
        } while (k0 < q.K);
        g.reds.push_back(GroupRed{p, (int)a, (int)b, (int)first, (int)(g.slots - first), 0});
      }
  }
  return g;
}

size_t group_bytes(const GroupPlan& g, size_t tsize) {
  auto up = [](size_t b) { return (b + 255) / 256 * 256; };
  return up(g.probs.size() * sizeof(GroupProb)) + up(g.items.size() * sizeof(GroupItem)) +
         up(std::max<size_t>(1, g.reds.size()) * sizeof(GroupRed)) + (size_t)g.slots * g.tile * g.tile * tsize;
}

template <typename T>
int group_run(int tb, const GroupPlan& g, double alpha, double beta, void* work, size_t wb,
              hipStream_t s) {
  EXC_REQUIRE(group_bytes(g, sizeof(T)) <= wb, EXC_ERR_SPACE, "exc_gemm_grouped: workspace too small");
  if (g.items.empty()) return EXC_OK;
  EXC_REQUIRE(tb ? !g.tri : g.tri && sizeof(T) == 8, EXC_ERR_ARG, "exc_gemm_grouped: no kernel for this form");
  auto up = [](size_t b) { return (b + 255) / 256 * 256; };
  char* w = (char*)work;
  GroupProb* dp = (GroupProb*)w;
  w += up(g.probs.size() * sizeof(GroupProb));
  GroupItem* di = (GroupItem*)w;
  w += up(g.items.size() * sizeof(GroupItem));
  GroupRed* dr = (GroupRed*)w;
  w += up(std::max<size_t>(1, g.reds.size()) * sizeof(GroupRed));
  T* part = (T*)w;
  // the tables are small; copy them synchronously so no host buffer must outlive the call
  EXC_CHECK_HIP(hipMemcpyAsync(dp, g.probs.data(), g.probs.size() * sizeof(GroupProb), hipMemcpyHostToDevice, s));
  EXC_CHECK_HIP(hipMemcpyAsync(di, g.items.data(), g.items.size() * sizeof(GroupItem), hipMemcpyHostToDevice, s));
  if (!g.reds.empty())
    EXC_CHECK_HIP(hipMemcpyAsync(dr, g.reds.data(), g.reds.size() * sizeof(GroupRed), hipMemcpyHostToDevice, s));
  EXC_CHECK_HIP(hipStreamSynchronize(s));
  const long nitems = (long)g.items.size();
  EXC_REQUIRE(nitems < (1L << 31), EXC_ERR_ARG, "exc_gemm_grouped: too many tiles");
  const dim3 grid((unsigned)nitems), block(g.tri ? GroupShape<T, true>::kThreads : GroupShape<T, false>::kThreads);
  hipEvent_t e0 = exc_prof::mark(s);
  auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, block, 0, s, dp, di, nitems, part, alpha, beta); };
  if (tb) launch(k_gemm_grouped<T, 1, false>);
  else if constexpr (sizeof(T) == 8) launch(k_gemm_grouped<T, 0, true>);
  EXC_CHECK_HIP(hipGetLastError());
  if (!g.reds.empty()) {
    hipLaunchKernelGGL(k_grouped_reduce<T>, dim3((unsigned)g.reds.size()), dim3(256), 0, s, dp, dr, part, g.tile,
                       alpha, beta);
    EXC_CHECK_HIP(hipGetLastError());
  }
  if (e0) exc_prof::book(sizeof(T) == 8 ? "gemm_grouped_f64" : "gemm_grouped_f32", e0, exc_prof::mark(s), g.flops, 0.0);
  return EXC_OK;
}

// Tuning results per problem set: the K chunk that ran fastest and its number of workgroups.
struct TuneEntry {
  long key[8];
  long kchunk;
  int grid;
  double ms;
};
std::vector<TuneEntry> g_tune;
std::mutex g_tune_mu;

template <typename T>
int grouped_impl(int tb, int nprob, const ExcGemmProblem* P, double alpha, double beta, long kchunk,
                 void* work, size_t wb, hipStream_t s) {
  EXC_REQUIRE(nprob >= 0 && (nprob == 0 || P), EXC_ERR_ARG, "exc_gemm_grouped: bad arguments");
  if (kchunk >= 0) return group_run<T>(tb, group_plan(nprob, P, kchunk), alpha, beta, work, wb, s);
  // autotune: one timed run per candidate on the caller's data (each run overwrites the outputs
  // completely, so the last one leaves the result), the fastest kept per problem-set key
  long key[8] = {(long)sizeof(T), 0, tb, nprob, 0, 0, 0, 0};
  for (int p = 0; p < nprob; p++) {
    key[4] += P[p].K;
    key[5] = std::max(key[5], P[p].K);
    key[6] = std::max(key[6], P[p].M * 100003 + P[p].N);
    key[7] = key[7] * 31 + P[p].lower_only * 2 + P[p].tri * 7 + (P[p].beta_zero_hint ? 1 : 0);
  }
  {
    std::lock_guard<std::mutex> lock(g_tune_mu);
    for (const TuneEntry& e : g_tune)
      if (std::equal(e.key, e.key + 8, key))
        return group_run<T>(tb, group_plan(nprob, P, e.kchunk), alpha, beta, work, wb, s);
  }
  EXC_REQUIRE(beta == 0.0, EXC_ERR_ARG, "exc_gemm_grouped: tuning runs need beta = 0 (each run overwrites C)");
  const long chunks[] = {0, 16384, 8192, 4096, 2048};
  hipEvent_t a, b;
  EXC_CHECK_HIP(hipEventCreate(&a));
  EXC_CHECK_HIP(hipEventCreate(&b));
  TuneEntry best{};
  best.ms = -1.0;
  for (long kc : chunks) {
    const GroupPlan g = group_plan(nprob, P, kc);
    if (group_bytes(g, sizeof(T)) > wb) continue;
    int rc = group_run<T>(tb, g, alpha, beta, work, wb, s);  // warm (and tables uploaded)
    if (rc) return rc;
    EXC_CHECK_HIP(hipEventRecord(a, s));
    rc = group_run<T>(tb, g, alpha, beta, work, wb, s);
    if (rc) return rc;
    EXC_CHECK_HIP(hipEventRecord(b, s));
    EXC_CHECK_HIP(hipEventSynchronize(b));
    float ms = 0.f;
    EXC_CHECK_HIP(hipEventElapsedTime(&ms, a, b));
    if (best.ms < 0 || ms < best.ms) {
      best.ms = ms;
      best.kchunk = kc;
      best.grid = (int)g.items.size();
    }
  }
  hipEventDestroy(a);
  hipEventDestroy(b);
  EXC_REQUIRE(best.ms >= 0, EXC_ERR_SPACE, "exc_gemm_grouped: workspace too small for any tuning candidate");
  std::copy(key, key + 8, best.key);
  {
    std::lock_guard<std::mutex> lock(g_tune_mu);
    g_tune.push_back(best);
  }
  return group_run<T>(tb, group_plan(nprob, P, best.kchunk), alpha, beta, work, wb, s);
}

}  // namespace

int exc_gemm_grouped_opts(int dtype, int tb, int nprob, const ExcGemmProblem* probs, double alpha, double beta,
                          long kchunk, void* work, size_t work_bytes, hipStream_t s) {
  EXC_REQUIRE(dtype == 4 || dtype == 8, EXC_ERR_ARG, "exc_gemm_grouped: dtype is 4 (float) or 8 (double)");
  if (dtype == 8) return grouped_impl<double>(tb, nprob, probs, alpha, beta, kchunk, work, work_bytes, s);
  return grouped_impl<float>(tb, nprob, probs, alpha, beta, kchunk, work, work_bytes, s);
}

size_t exc_gemm_grouped_workspace(int dtype, int nprob, const ExcGemmProblem* probs, long kchunk) {
  // the autotuner's smallest chunk needs the most partial slots
  const long kc = kchunk < 0 ? 2048 : kchunk;
  return group_bytes(group_plan(nprob, probs, kc), dtype == 8 ? 8 : 4) + 256;
}

extern "C" int exc_gemm_grouped_tuning(char* buf, size_t cap) {
  std::lock_guard<std::mutex> lock(g_tune_mu);
  std::string out = "[";
  for (size_t i = 0; i < g_tune.size(); i++) {
    char line[256];
    snprintf(line, sizeof line, "%s{\"dtype\": %ld, \"problems\": %ld, \"sum_k\": %ld, \"kchunk\": %ld, \"grid\": %d, \"ms\": %.4f}",
             i ? ", " : "", g_tune[i].key[0], g_tune[i].key[3], g_tune[i].key[4], g_tune[i].kchunk, g_tune[i].grid,
             g_tune[i].ms);
    out += line;
  }
  out += "]";
  if (buf && cap) {
    strncpy(buf, out.c_str(), cap - 1);
    buf[cap - 1] = 0;
  }
  return EXC_OK;
}

int exc_gemm_opts(int ta, int tb, long M, long N, long K, double alpha, const double* A, long lda, const double* B,
                  long ldb, double beta, double* C, long ldc, const ExcGemmOpts& o, hipStream_t s) {
  return gemm_impl<double>(ta, tb, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, o, s);
}

int exc_sgemm_opts(int ta, int tb, long M, long N, long K, double alpha, const float* A, long lda, const float* B,
                   long ldb, double beta, float* C, long ldc, const ExcGemmOpts& o, hipStream_t s) {
  return gemm_impl<float>(ta, tb, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, o, s);
}

extern "C" {

size_t exc_gemm_workspace(long M, long N, long K) {
  (void)K;
  return (size_t)8 * M * N * sizeof(double);
}

int exc_dgemm(int trans_a, int trans_b, long M, long N, long K, double alpha, const double* d_a, long lda,
              const double* d_b, long ldb, double beta, double* d_c, long ldc, void* d_work, size_t work_bytes,
              exc_stream_t stream) {
  ExcGemmOpts o;
  o.work = d_work;
  o.work_bytes = work_bytes;
  return gemm_impl<double>(trans_a, trans_b, M, N, K, alpha, d_a, lda, d_b, ldb, beta, d_c, ldc, o,
                           exc_detail::stream(stream));
}

int exc_sgemm(int trans_a, int trans_b, long M, long N, long K, double alpha, const float* d_a, long lda,
              const float* d_b, long ldb, double beta, float* d_c, long ldc, void* d_work, size_t work_bytes,
              exc_stream_t stream) {
  ExcGemmOpts o;
  o.work = d_work;
  o.work_bytes = work_bytes;
  return gemm_impl<float>(trans_a, trans_b, M, N, K, alpha, d_a, lda, d_b, ldb, beta, d_c, ldc, o,
                          exc_detail::stream(stream));
}

}  // extern "C"
