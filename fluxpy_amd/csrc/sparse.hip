// CSR products and the fused Jacobi radiosity step (solve.py:25-45).
//
// One wave per CSR row; the lanes' partial sums are reduced with cross-lane
// shuffles.  The summation order is fixed, so every product is
// deterministic.
#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>

#include <type_traits>

#include "common.h"

namespace flux {

// SPMM_JACOBI_SCALED: 'right' with X = rho o B kept beside B, so that no
// nonzero multiplies by (or gathers) an albedo.
enum { SPMM_PLAIN = 0, SPMM_JACOBI_RIGHT = 1, SPMM_JACOBI_LEFT = 2, SPMM_JACOBI_SCALED = 3 };

// What a Jacobi step takes beside the matrix and its vector X.  B is the
// iterate X stands for (X itself unless scaled), Xn the next scaled one.
// prev / tol: the column maxima of the step before and their bounds (tol_cols
// of them, 1 or one per column); a step after one that met them all does
// nothing, so a run of steps can be issued without reading the maxima back.
// The maxima are kept in `slots` rows of one value per column, 256 bytes or
// more apart, and workgroups are dealt out over them: atomics on one cache
// line take about 10 ns each, and with the rows the step also needs no cap on
// its workgroups (1 column of 20,402 facets: 36 us with one row and 2,048
// workgroups, 24 with 16 rows; 64 values side by side: 72).
template <typename TX>
struct JacobiArgs {
  const TX *E, *B;
  TX *Xn;
  const TX *rho;
  double rho_s;
  double *colmax;
  const double *prev, *tol;
  int64_t tol_cols;
  int slots;  // a power of two
};

template <typename T>
struct AccOf {
  using type = float;
};
template <>
struct AccOf<double> {
  using type = double;
};

// Matrix values may be stored in BF16 / FP16 (the low-precision inner
// operator of the refined solve); they widen to the accumulation type.
__device__ __forceinline__ float widen(__hip_bfloat16 v) { return __bfloat162float(v); }
__device__ __forceinline__ float widen(__half v) { return __half2float(v); }
__device__ __forceinline__ float widen(float v) { return v; }
__device__ __forceinline__ double widen(double v) { return v; }

template <typename T>
struct WideOf {
  using type = T;
};
template <>
struct WideOf<__hip_bfloat16> {
  using type = float;
};
template <>
struct WideOf<__half> {
  using type = float;
};

__device__ inline void atomic_max_nonneg(double *addr, double v) {
  // Non-negative IEEE doubles order like their bit patterns.
  atomicMax((unsigned long long *)addr, (unsigned long long)__double_as_longlong(v));
}

template <typename T, int V>
struct Vec {
  T v[V];
};

// V consecutive elements from any element-aligned address (one load: global
// loads of 16 bytes need 4-byte alignment).
template <int V, typename T>
__device__ __forceinline__ Vec<T, V> load_vec(const T *p) {
  Vec<T, V> r;
  __builtin_memcpy(&r, p, sizeof(r));
  return r;
}

// A change as the bits that atomic_max_nonneg orders by.  One that is not a
// number is above all others if it counts, else it is no change.
__device__ __forceinline__ unsigned long long change_bits(double v, bool nan_counts) {
  return v == v || nan_counts ? (unsigned long long)__double_as_longlong(v) : 0ull;
}

// Distance of the rows of column maxima, in doubles.
__host__ __device__ __forceinline__ int64_t slot_stride(int64_t nrhs) {
  return (nrhs + 31) / 32 * 32;
}

// True if the step before met its bounds in every column (then its column
// maxima, and this step's, which stay zero, do so for the next step too).
template <typename TX>
__device__ __forceinline__ bool jacobi_met(const JacobiArgs<TX> &jac, int64_t nrhs) {
  if (!jac.prev) return false;
  bool met = true;
  const int lane = threadIdx.x & 63;
  int kk = 1;  // lanes per slot
  while (kk < nrhs && kk < 64) kk <<= 1;
  const int64_t stride = slot_stride(nrhs);
  for (int s = lane / kk; s < jac.slots; s += 64 / kk)
    for (int64_t c = lane & (kk - 1); c < nrhs; c += 64)
      met = met && jac.prev[s * stride + c] <= jac.tol[jac.tol_cols == 1 ? 0 : c];
  return __all(met);
}

// One right-hand side: a wave per row (walking rows so that a workgroup
// issues one atomic per Jacobi step), a lane per nonzero.  Consecutive lanes
// take consecutive nonzeros: their columns are close, so a gather touches few
// cache lines (four consecutive nonzeros per lane load indices and values in
// a third of the instructions, but the gathers of 64 lanes then span 256
// nonzeros: 81 -> 112 us for 35.9 M nonzeros).
template <typename TA, typename TX, typename TAcc, int MODE>
__global__ void __launch_bounds__(256) k_csr_vec(
    int64_t m, const int64_t *__restrict__ indptr, const int32_t *__restrict__ indices,
    const TA *__restrict__ data, const TX *__restrict__ X, TX *__restrict__ Y,
    JacobiArgs<TX> jac, int64_t row0) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (MODE != SPMM_PLAIN && jacobi_met(jac, 1)) return;
  const TX *__restrict__ E = jac.E, *__restrict__ rho = jac.rho, *__restrict__ B = jac.B;
  const double rho_s = jac.rho_s;
  const int64_t step = (int64_t)gridDim.x * (blockDim.x >> 6);
  double rmax = 0.0;
  for (int64_t row = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6; row < m;
       row += step) {
    const int64_t k0 = indptr[row], k1 = indptr[row + 1];
    TAcc acc = 0;
    // kU consecutive strides per pass: the index and value loads of a pass,
    // then its gathers, are all in flight before the first product.  Loads
    // go out unconditionally from clamped addresses (k1 - 1 is a valid entry
    // of this row): a load behind a branch would make the compiler wait for
    // the earlier ones and serialise the pass.
    constexpr int kU = 8;
    for (int64_t kb = k0 + lane; kb < k1; kb += kU * 64) {
      int32_t jj[kU];
      TAcc av[kU], xv[kU];
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        const int64_t k = min(kb + u * 64, k1 - 1);
        jj[u] = indices[k];
        av[u] = (TAcc)widen(data[k]);
      }
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        TAcc x = (TAcc)X[jj[u]];
        if (MODE == SPMM_JACOBI_RIGHT) x = (rho ? (TAcc)rho[jj[u]] : (TAcc)rho_s) * x;
        xv[u] = x;
      }
#pragma unroll
      for (int u = 0; u < kU; ++u)
        if (kb + u * 64 < k1) acc += av[u] * xv[u];
    }
    for (int off = 1; off < 64; off <<= 1) acc += __shfl_xor(acc, off, 64);
    if (lane == 0) {
      const int64_t o = row0 + row;  // row0: first row of a row chunk
      if (MODE == SPMM_PLAIN) {
        Y[o] = (TX)acc;
      } else {
        TAcc y = acc;
        if (MODE == SPMM_JACOBI_LEFT) y = (rho ? (TAcc)rho[o] : (TAcc)rho_s) * y;
        const TX b1 = (TX)((TAcc)E[o] + y);
        Y[o] = b1;
        if (MODE == SPMM_JACOBI_SCALED) jac.Xn[o] = rho[o] * b1;
        rmax = fmax(rmax, fabs((double)b1 - (double)B[o]));
      }
    }
  }
  if (MODE != SPMM_PLAIN) {
    __shared__ double sd[4];
    if (lane == 0) sd[w] = rmax;
    __syncthreads();
    if (threadIdx.x == 0)
      atomic_max_nonneg(jac.colmax + (blockIdx.x & (jac.slots - 1)) * slot_stride(1),
                        fmax(fmax(sd[0], sd[1]), fmax(sd[2], sd[3])));
  }
}

// Products with two or more right-hand sides.  A lane takes V right-hand
// sides of one nonzero in one 16-byte gather (V = 2 in FP64, 4 in FP32), LP
// lanes cover a row of X (or of a tile of it: more than 64 V right-hand sides
// go in equal tiles), and the G = 64 / LP groups of a wave take G nonzeros
// at a time.  The indices and values of 64 S nonzeros are loaded once,
// coalesced, a pass ahead, and handed round through LDS (LP = 1: a lane
// keeps its own), with the albedo of the column multiplied in.
//
// What bounds it: with a lane per right-hand side, every lane loading the
// index, the value and the albedo of its nonzero, it was the rate of the
// address unit (64 lanes in 16 cycles whatever a lane loads: 4 instructions
// per 4 nonzeros at 16 FP64 right-hand sides, 10 per 64 here); now it is the
// gathers from L2 (10.7 M nonzeros, 128 bytes each, in 111 us: 12 TB/s).  10.7
// M nonzeros, product / Jacobi step with per-facet albedo 'right', us:
// FP64 k = 3: 53 / 85 -> 48 / 64, k = 8: 97 / 167 -> 72 / 88, k = 16: 187 / 311
// -> 112 / 134, k = 64: 707 / 1110 -> 390 / 425; FP32 k = 16: 151 / 181 -> 59 /
// 74.  Workgroups of 8 or 16 waves (neighbouring rows on one CU) were slower.
//
// A lane past the end of a row of X loads the row's last V values instead
// (nothing is read outside X) and stores what no other lane has.
//
// With more than 64 right-hand sides a change that is not a number is its
// column's maximum, so an iteration that overflows does not converge; with
// fewer, here and in k_csr_vec, it is passed over.
constexpr int kBlockWaves = 4;

template <typename TA, typename TX, typename TAcc, int MODE, int V, int LP1, int S, int kU>
__global__ void __launch_bounds__(64 * kBlockWaves) k_csr_block(
    int64_t m, const int64_t *__restrict__ indptr, const int32_t *__restrict__ indices,
    const TA *__restrict__ data, const TX *__restrict__ X, int64_t nrhs, int64_t tiles,
    int64_t tile0, int lp_log2, TX *__restrict__ Y, JacobiArgs<TX> jac, int64_t row0) {
  if (MODE != SPMM_PLAIN && jacobi_met(jac, nrhs)) return;
  const TX *__restrict__ E = jac.E, *__restrict__ rho = jac.rho, *__restrict__ B = jac.B;
  const double rho_s = jac.rho_s;
  double *__restrict__ colmax = jac.colmax;
  // this workgroup's right-hand sides: one of `tiles` equal tiles
  const int64_t tile = tile0 + blockIdx.y;
  const int64_t c_lo = nrhs * tile / tiles, c_hi = nrhs * (tile + 1) / tiles;
  const int cols = (int)(c_hi - c_lo);
  X += c_lo;
  Y += c_lo;
  if (MODE != SPMM_PLAIN) {
    E += c_lo;
    B += c_lo;
    colmax += (blockIdx.x & (jac.slots - 1)) * slot_stride(nrhs) + c_lo;
  }
  __shared__ int32_t sidx[LP1 ? 1 : kBlockWaves][LP1 ? 1 : 64 * S];
  __shared__ TAcc sval[LP1 ? 1 : kBlockWaves][LP1 ? 1 : 64 * S];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int LP = LP1 ? 1 : 1 << lp_log2, G = LP1 ? 64 : 64 >> lp_log2;
  const int g = LP1 ? lane : lane >> lp_log2, c = LP1 ? 0 : (lane & (LP - 1)) * V;
  const int col = min(c, cols - V);  // cols >= V
  const int fresh = c - col;         // values below this one belong to another lane
  const int64_t step = (int64_t)gridDim.x * kBlockWaves;
  const bool nan_counts = nrhs > 64;
  unsigned long long rmax[V];
  for (int v = 0; v < V; ++v) rmax[v] = 0;
  for (int64_t row = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6; row < m;
       row += step) {
    const int64_t k0 = indptr[row], k1 = indptr[row + 1];
    TAcc acc[V];
    for (int v = 0; v < V; ++v) acc[v] = 0;
    int32_t idx[S];
    TAcc val[S];
    auto load = [&](int64_t kb) {
#pragma unroll
      for (int u = 0; u < S; ++u) {
        const int64_t k = min(kb + u * 64 + lane, k1 - 1);
        idx[u] = indices[k];
        val[u] = (TAcc)widen(data[k]);
      }
    };
    auto scale = [&]() {
      if (MODE == SPMM_JACOBI_RIGHT) {
#pragma unroll
        for (int u = 0; u < S; ++u) val[u] *= rho ? (TAcc)rho[idx[u]] : (TAcc)rho_s;
      }
    };
    if (k0 < k1) {
      load(k0);
      scale();
    }
    for (int64_t kb = k0; kb < k1; kb += 64 * S) {
      const int cnt = (int)min(k1 - kb, (int64_t)(64 * S));
      if constexpr (LP1) {
        // a lane's own nonzeros
        Vec<TX, V> xv[S];
        TAcc av[S];
#pragma unroll
        for (int u = 0; u < S; ++u) {
          xv[u] = load_vec<V>(X + (int64_t)idx[u] * nrhs + col);
          av[u] = val[u];
        }
        if (kb + 64 * S < k1) load(kb + 64 * S);
#pragma unroll
        for (int u = 0; u < S; ++u)
          if (u * 64 + lane < cnt)
            for (int v = 0; v < V; ++v) acc[v] += av[u] * (TAcc)xv[u].v[v];
        if (kb + 64 * S < k1) scale();
      } else {
#pragma unroll
        for (int u = 0; u < S; ++u) {
          sidx[w][u * 64 + lane] = idx[u];
          sval[w][u * 64 + lane] = val[u];
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        // the next nonzeros, on their way during this pass
        if (kb + 64 * S < k1) load(kb + 64 * S);
        // kU groups of nonzeros at a time, the rest of the pass two at a time
        auto terms = [&](int s, auto groups) {
          constexpr int n = decltype(groups)::value;
          TAcc av[n];
          Vec<TX, V> xv[n];
#pragma unroll
          for (int u = 0; u < n; ++u) {
            const int e = min(s + u * G + g, cnt - 1);
            av[u] = sval[w][e];
            xv[u] = load_vec<V>(X + (int64_t)sidx[w][e] * nrhs + col);
          }
#pragma unroll
          for (int u = 0; u < n; ++u)
            if (s + u * G + g < cnt)
              for (int v = 0; v < V; ++v) acc[v] += av[u] * (TAcc)xv[u].v[v];
        };
        int s = 0;
        for (; s + (kU - 2) * G < cnt; s += kU * G) terms(s, std::integral_constant<int, kU>());
        for (; s < cnt; s += 2 * G) terms(s, std::integral_constant<int, 2>());
        if (kb + 64 * S < k1) scale();
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
      }
    }
    for (int off = LP; off < 64; off <<= 1)
      for (int v = 0; v < V; ++v) acc[v] += __shfl_xor(acc[v], off, 64);
    if (g == 0 && c < cols) {
      const int64_t o = (row0 + row) * nrhs + col;  // row0: first row of a row chunk
      for (int v = 0; v < V; ++v) {
        if (v < fresh) continue;
        if (MODE == SPMM_PLAIN) {
          Y[o + v] = (TX)acc[v];
        } else {
          TAcc y = acc[v];
          if (MODE == SPMM_JACOBI_LEFT) y = (rho ? (TAcc)rho[row0 + row] : (TAcc)rho_s) * y;
          const TX b1 = (TX)((TAcc)E[o + v] + y);
          Y[o + v] = b1;
          if (MODE == SPMM_JACOBI_SCALED) jac.Xn[c_lo + o + v] = rho[row0 + row] * b1;
          rmax[v] = max(rmax[v], change_bits(fabs((double)b1 - (double)B[o + v]), nan_counts));
        }
      }
    }
  }
  if (MODE != SPMM_PLAIN) {
    // one atomic per column and workgroup
    __shared__ unsigned long long sd[kBlockWaves][64 * V];
    if (g == 0)
      for (int v = 0; v < V; ++v) sd[w][(lane & (LP - 1)) * V + v] = rmax[v];
    __syncthreads();
    for (int t = threadIdx.x; t < LP * V; t += blockDim.x) {
      // column of the lane-major slot t, unless another lane has it
      const int cc = t / V * V, base = min(cc, cols - V), v = t - cc;
      if (cc < cols && v >= cc - base) {
        unsigned long long mx = 0;
        for (int q = 0; q < kBlockWaves; ++q) mx = max(mx, sd[q][t]);
        atomicMax((unsigned long long *)colmax + base + v, mx);
      }
    }
  }
}

// Workgroups for m rows: a wave per row, so that rows of uneven length spread
// over the chip as waves end (a wave walking rows took 88 us where this
// takes 81), except in Jacobi steps whose workgroups all end with atomics on
// the same column maxima (2048 workgroups).
template <int MODE>
static unsigned row_blocks(int64_t m, int slots) {
  const int64_t rb = (m + kBlockWaves - 1) / kBlockWaves;
  const int64_t most = MODE == SPMM_PLAIN || slots > 1 ? kMaxGrid1D : 2048;
  return (unsigned)(rb < most ? rb : most);
}

template <typename TA, typename TX, int MODE, int V>
static int launch_block(int64_t m, const int64_t *indptr, const int32_t *indices,
                        const void *data, const void *X, int64_t nrhs, void *Y,
                        const JacobiArgs<TX> &jac, hipStream_t st, int64_t row0) {
  using TAcc = typename AccOf<decltype(typename WideOf<TA>::type() + TX())>::type;
  const int64_t tiles = (nrhs + 64 * V - 1) / (64 * V), width = (nrhs + tiles - 1) / tiles;
  int lp = 0;
  while (((int64_t)V << lp) < width) ++lp;
  const unsigned rows = row_blocks<MODE>(m, jac.slots);
  auto launch = [&](auto kernel) {
    constexpr int64_t most = 65535;  // of a grid's second dimension
    for (int64_t t = 0; t < tiles; t += most)
      hipLaunchKernelGGL(kernel, dim3(rows, (unsigned)(tiles - t < most ? tiles - t : most)),
                         dim3(64 * kBlockWaves), 0, st, m, indptr, indices, (const TA *)data,
                         (const TX *)X, nrhs, tiles, t, lp, (TX *)Y, jac, row0);
  };
  // nonzeros staged per pass: 64 S; groups in flight: kU (kU G <= 64 S)
  if (lp == 0)
    launch(k_csr_block<TA, TX, TAcc, MODE, V, 1, 4, 4>);
  else if (lp == 1)
    launch(k_csr_block<TA, TX, TAcc, MODE, V, 0, 2, 4>);
  else if (lp == 2)
    launch(k_csr_block<TA, TX, TAcc, MODE, V, 0, 2, 8>);
  else
    launch(k_csr_block<TA, TX, TAcc, MODE, V, 0, 1, 8>);
  FLUX_LAUNCH_CHECK();
  return 0;
}

template <typename TA, typename TX, int MODE>
static int launch_rows(int64_t m, const int64_t *indptr, const int32_t *indices,
                       const void *data, const void *X, int64_t nrhs, void *Y,
                       const JacobiArgs<TX> &jac, hipStream_t st, int64_t row0) {
  using TAcc = typename AccOf<decltype(typename WideOf<TA>::type() + TX())>::type;
  constexpr int V = 16 / (int)sizeof(TX);
  if (m <= 0) return 0;
  if (nrhs >= V)
    return launch_block<TA, TX, MODE, V>(m, indptr, indices, data, X, nrhs, Y, jac, st, row0);
  if (nrhs >= 2)
    return launch_block<TA, TX, MODE, 2>(m, indptr, indices, data, X, nrhs, Y, jac, st, row0);
  const unsigned blocks = row_blocks<MODE>(m, jac.slots);
  hipLaunchKernelGGL((k_csr_vec<TA, TX, TAcc, MODE>), dim3(blocks), dim3(256), 0, st, m, indptr,
                     indices, (const TA *)data, (const TX *)X, (TX *)Y, jac, row0);
  FLUX_LAUNCH_CHECK();
  return 0;
}

// A Jacobi step's arguments before the vector type is known.
struct JacobiVoid {
  const void *E, *B, *rho;
  void *Xn;
  double rho_s;
  double *colmax;
  const double *prev, *tol;
  int64_t tol_cols;
  int slots = 1;
  template <typename TX>
  JacobiArgs<TX> as() const {
    return JacobiArgs<TX>{(const TX *)E, (const TX *)B, (TX *)Xn, (const TX *)rho,
                          rho_s,         colmax,        prev,     tol,
                          tol_cols,      slots};
  }
};

template <int MODE>
static int dispatch_rows(int64_t m, const int64_t *indptr, const int32_t *indices,
                         const void *data, int dtype, const void *X, int64_t nrhs, void *Y,
                         int xdtype, const JacobiVoid &jac, hipStream_t st, int64_t row0 = 0) {
  if (dtype == FLUX_F64 && xdtype == FLUX_F64)
    return launch_rows<double, double, MODE>(m, indptr, indices, data, X, nrhs, Y,
                                             jac.as<double>(), st, row0);
  if (dtype == FLUX_F32 && xdtype == FLUX_F64)
    return launch_rows<float, double, MODE>(m, indptr, indices, data, X, nrhs, Y,
                                            jac.as<double>(), st, row0);
  if (dtype == FLUX_F32 && xdtype == FLUX_F32)
    return launch_rows<float, float, MODE>(m, indptr, indices, data, X, nrhs, Y,
                                           jac.as<float>(), st, row0);
  if constexpr (MODE != SPMM_JACOBI_SCALED) {
    if (dtype == FLUX_F64 && xdtype == FLUX_F32)
      return launch_rows<double, float, MODE>(m, indptr, indices, data, X, nrhs, Y,
                                              jac.as<float>(), st, row0);
    if (dtype == FLUX_BF16 && xdtype == FLUX_F32)
      return launch_rows<__hip_bfloat16, float, MODE>(m, indptr, indices, data, X, nrhs, Y,
                                                      jac.as<float>(), st, row0);
    if (dtype == FLUX_F16 && xdtype == FLUX_F32)
      return launch_rows<__half, float, MODE>(m, indptr, indices, data, X, nrhs, Y,
                                              jac.as<float>(), st, row0);
  }
  set_error("csr product: unsupported dtypes (%d, %d)", dtype, xdtype);
  return -2;
}

__global__ void k_fill_f64(double *p, int64_t n, double v) {
  int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n) p[k] = v;
}

__global__ void k_fill_i64(int64_t *p, int64_t n, int64_t v) {
  int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n) p[k] = v;
}

// Deterministic CSR transpose.  Rows are cut into B blocks of R rows.
//  1. cnt[b][j]   = nonzeros of column j inside row block b
//  2. off[b][j]   = col_ptr[j] + sum_{b' < b} cnt[b'][j]
//  3. block b walks its rows in order and places each nonzero (i, j) at
//     off[b][j]++ -- rows of one block are visited in increasing order and a
//     column occurs once per row, so the output rows come out sorted by the
//     original row index without atomics or a sort.
__global__ void k_tr_count(int64_t m, int64_t n, int64_t R, const int64_t *__restrict__ indptr,
                           const int32_t *__restrict__ indices, int64_t *__restrict__ cnt) {
  const int64_t b = blockIdx.x;
  const int64_t r0 = b * R, r1 = min(m, r0 + R);
  for (int64_t k = indptr[r0] + threadIdx.x; k < indptr[r1]; k += blockDim.x)
    atomicAdd((unsigned long long *)&cnt[b * n + indices[k]], 1ull);
}

__global__ void k_tr_colscan(int64_t n, int64_t nb, int64_t *__restrict__ cnt,
                             int64_t *__restrict__ total) {
  const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= n) return;
  int64_t run = 0;
  for (int64_t b = 0; b < nb; ++b) {
    const int64_t c = cnt[b * n + j];
    cnt[b * n + j] = run;
    run += c;
  }
  total[j] = run;
}

template <typename T>
__global__ void k_tr_fill(int64_t m, int64_t n, int64_t R, const int64_t *__restrict__ indptr,
                          const int32_t *__restrict__ indices, const T *__restrict__ data,
                          const int64_t *__restrict__ colptr, int64_t *__restrict__ off,
                          int32_t *__restrict__ oidx, T *__restrict__ odata) {
  const int64_t b = blockIdx.x;
  const int64_t r0 = b * R, r1 = min(m, r0 + R);
  for (int64_t i = r0; i < r1; ++i) {
    for (int64_t k = indptr[i] + threadIdx.x; k < indptr[i + 1]; k += blockDim.x) {
      const int64_t j = indices[k];
      const int64_t pos = colptr[j] + off[b * n + j];
      off[b * n + j] += 1;
      oidx[pos] = (int32_t)i;
      odata[pos] = data[k];
    }
    __syncthreads();
  }
}

}  // namespace flux

using namespace flux;

extern "C" int flux_csr_spmm(int64_t m, int64_t n, const int64_t *indptr,
                             const int32_t *indices, const void *data, int dtype,
                             const void *X, int64_t nrhs, void *Y, int xdtype, void *stream) {
  FLUX_CHECK(m >= 0 && n >= 0 && nrhs >= 0, "flux_csr_spmm: negative sizes");
  if (m == 0 || nrhs == 0) return 0;
  FLUX_CHECK(indptr && X && Y, "flux_csr_spmm: NULL array");
  return dispatch_rows<SPMM_PLAIN>(m, indptr, indices, data, dtype, X, nrhs, Y, xdtype,
                                   JacobiVoid{}, as_stream(stream));
}

// Scan of int64 values (formfactor.hip).
extern "C" int flux_scan_i64(const int64_t *in, int64_t n, int64_t *out, int64_t *total_host,
                             void *stream);

extern "C" int flux_csr_transpose(int64_t m, int64_t n, const int64_t *indptr,
                                  const int32_t *indices, const void *data, int dtype,
                                  int64_t *t_indptr, int32_t *t_indices, void *t_data,
                                  void *stream) {
  FLUX_CHECK(m >= 0 && n >= 0, "flux_csr_transpose: negative sizes");
  FLUX_CHECK(m < ((int64_t)1 << 31), "flux_csr_transpose: m too large for int32 indices");
  FLUX_CHECK(dtype == FLUX_F32 || dtype == FLUX_F64, "flux_csr_transpose: dtype");
  FLUX_CHECK(t_indptr != nullptr && (m == 0 || indptr != nullptr),
             "flux_csr_transpose: NULL array");
  hipStream_t st = as_stream(stream);
  if (n == 0) return 0;
  int64_t R = 256;
  while ((m + R - 1) / R > 1024) R *= 2;
  const int64_t nb = m > 0 ? (m + R - 1) / R : 0;
  int64_t *work = nullptr;
  const int64_t nwork = nb * n + n;
  FLUX_TRY_HIP(hipMalloc(&work, (size_t)(nwork > 0 ? nwork : 1) * sizeof(int64_t)));
  int64_t *cnt = work, *total = work + nb * n;
  int rc = 0;
  do {
    hipLaunchKernelGGL(k_fill_i64, dim3(ceil_div_u(nwork, 256)), dim3(256), 0, st, work, nwork,
                       (int64_t)0);
    if (nb > 0)
      hipLaunchKernelGGL(k_tr_count, dim3((unsigned)nb), dim3(256), 0, st, m, n, R, indptr,
                         indices, cnt);
    hipLaunchKernelGGL(k_tr_colscan, dim3(ceil_div_u(n, 256)), dim3(256), 0, st, n, nb, cnt,
                       total);
    if (hipGetLastError() != hipSuccess) {
      set_error("flux_csr_transpose: count kernels failed");
      rc = -1;
      break;
    }
    rc = flux_scan_i64(total, n, t_indptr, nullptr, stream);
    if (rc) break;
    if (nb > 0) {
      if (dtype == FLUX_F64)
        hipLaunchKernelGGL(k_tr_fill<double>, dim3((unsigned)nb), dim3(256), 0, st, m, n, R,
                           indptr, indices, (const double *)data, t_indptr, cnt, t_indices,
                           (double *)t_data);
      else
        hipLaunchKernelGGL(k_tr_fill<float>, dim3((unsigned)nb), dim3(256), 0, st, m, n, R,
                           indptr, indices, (const float *)data, t_indptr, cnt, t_indices,
                           (float *)t_data);
    }
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    if (e != hipSuccess) {
      set_error("flux_csr_transpose: %s", hipGetErrorString(e));
      rc = -1;
    }
  } while (0);
  (void)hipFree(work);
  return rc;
}

extern "C" int flux_csr_rows_chunk(int64_t m, int64_t row0, const int64_t *indptr,
                                   const int32_t *indices, const void *data, int dtype,
                                   const void *X, int64_t nrhs, void *Y, int xdtype,
                                   const void *E, const void *rho, double rho_scalar, int mode,
                                   double *colmax, void *stream) {
  FLUX_CHECK(m >= 0 && row0 >= 0 && nrhs >= 0, "flux_csr_rows_chunk: negative sizes");
  if (m == 0 || nrhs == 0) return 0;
  FLUX_CHECK(indptr && X && Y, "flux_csr_rows_chunk: NULL array");
  FLUX_CHECK(mode >= 0 && mode <= 2, "flux_csr_rows_chunk: mode must be 0, 1 or 2");
  FLUX_CHECK(mode == 0 || (E && colmax && X != Y),
             "flux_csr_rows_chunk: a Jacobi step needs E, colmax and Y != X");
  hipStream_t st = as_stream(stream);
  const JacobiVoid jac{E, X, rho, nullptr, rho_scalar, colmax, nullptr, nullptr, 0, 1};
  if (mode == 0)
    return dispatch_rows<SPMM_PLAIN>(m, indptr, indices, data, dtype, X, nrhs, Y, xdtype, jac, st,
                                     row0);
  if (mode == 2)
    return dispatch_rows<SPMM_JACOBI_LEFT>(m, indptr, indices, data, dtype, X, nrhs, Y, xdtype,
                                           jac, st, row0);
  return dispatch_rows<SPMM_JACOBI_RIGHT>(m, indptr, indices, data, dtype, X, nrhs, Y, xdtype,
                                          jac, st, row0);
}

extern "C" int flux_csr_jacobi_step(int64_t m, const int64_t *indptr, const int32_t *indices,
                                    const void *data, int dtype, const void *E,
                                    const void *B, int64_t nrhs, const void *rho,
                                    double rho_scalar, int left, void *B1, int xdtype,
                                    double *colmax, void *stream) {
  FLUX_CHECK(m >= 0 && nrhs >= 0, "flux_csr_jacobi_step: negative sizes");
  if (m == 0 || nrhs == 0) return 0;
  FLUX_CHECK(indptr && E && B && B1 && colmax, "flux_csr_jacobi_step: NULL array");
  FLUX_CHECK(B != B1, "flux_csr_jacobi_step: B and B1 must not alias");
  hipStream_t st = as_stream(stream);
  hipLaunchKernelGGL(k_fill_f64, dim3(ceil_div_u(nrhs, 256)), dim3(256), 0, st, colmax, nrhs,
                     0.0);
  FLUX_LAUNCH_CHECK();
  const JacobiVoid jac{E, B, rho, nullptr, rho_scalar, colmax, nullptr, nullptr, 0, 1};
  if (left)
    return dispatch_rows<SPMM_JACOBI_LEFT>(m, indptr, indices, data, dtype, B, nrhs, B1, xdtype,
                                           jac, st);
  return dispatch_rows<SPMM_JACOBI_RIGHT>(m, indptr, indices, data, dtype, B, nrhs, B1, xdtype,
                                          jac, st);
}

extern "C" int flux_csr_jacobi_run(int64_t m, const int64_t *indptr, const int32_t *indices,
                                   const void *data, int dtype, const void *E, void *B0, void *B1,
                                   void *X0, void *X1, int64_t nrhs, const void *rho,
                                   double rho_scalar, int left, int xdtype, const double *tol,
                                   int64_t tol_cols, int64_t first, int64_t nsteps,
                                   int slots, double *colmax, void *stream) {
  FLUX_CHECK(m >= 0 && nrhs >= 0 && first >= 0 && nsteps >= 0,
             "flux_csr_jacobi_run: negative sizes");
  if (m == 0 || nrhs == 0 || nsteps == 0) return 0;
  FLUX_CHECK(indptr && E && B0 && B1 && tol && colmax, "flux_csr_jacobi_run: NULL array");
  FLUX_CHECK(B0 != B1, "flux_csr_jacobi_run: B0 and B1 must not alias");
  FLUX_CHECK(tol_cols == 1 || tol_cols == nrhs, "flux_csr_jacobi_run: tol_cols");
  FLUX_CHECK(slots >= 1 && slots <= 1024 && (slots & (slots - 1)) == 0,
             "flux_csr_jacobi_run: slots must be a power of two up to 1024");
  FLUX_CHECK(!X0 == !X1 && (!X0 || (rho && !left && X0 != X1)),
             "flux_csr_jacobi_run: scaled iterates need rho, 'right' and two buffers");
  hipStream_t st = as_stream(stream);
  const int64_t ns = slots * slot_stride(nrhs), nm = nsteps * ns;
  hipLaunchKernelGGL(k_fill_f64, dim3(ceil_div_u(nm, 256)), dim3(256), 0, st, colmax, nm, 0.0);
  FLUX_LAUNCH_CHECK();
  for (int64_t s = 0; s < nsteps; ++s) {
    const bool odd = (first + s) & 1;
    void *B = odd ? B1 : B0, *Bn = odd ? B0 : B1;
    void *X = X0 ? (odd ? X1 : X0) : B, *Xn = X0 ? (odd ? X0 : X1) : nullptr;
    const JacobiVoid jac{E,          B,
                         rho,        Xn,
                         rho_scalar, colmax + s * ns,
                         s > 0 ? colmax + (s - 1) * ns : nullptr,
                         tol,        tol_cols,
                         slots};
    int rc;
    if (X0)
      rc = dispatch_rows<SPMM_JACOBI_SCALED>(m, indptr, indices, data, dtype, X, nrhs, Bn, xdtype,
                                             jac, st);
    else if (left || !rho)  // F (rho x) = rho (F x) for a scalar
      rc = dispatch_rows<SPMM_JACOBI_LEFT>(m, indptr, indices, data, dtype, X, nrhs, Bn, xdtype,
                                           jac, st);
    else
      rc = dispatch_rows<SPMM_JACOBI_RIGHT>(m, indptr, indices, data, dtype, X, nrhs, Bn, xdtype,
                                            jac, st);
    if (rc) return rc;
  }
  return 0;
}
