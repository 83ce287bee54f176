// Hierarchical compression on the GPU: block statistics of a permuted CSR,
// randomized range sketches of CSR sub-blocks, batched Gram matrices, a
// batched parallel-order Jacobi eigensolver (FP64) and a batched small GEMM.
//
// These replace the per-node work of the reference's tree build
// (compressed_form_factors.py:285-405): spmat.nnz and nbytes(spmat), and the
// ARPACK singular values / vectors of linalg.py:8-50.  The singular values
// of a block A (m x n) come from a Rademacher sketch Y = A W (W: n x l),
// Z = A^T Y, the Gram M = Y^T Y = V D V^T, the orthonormal basis
// Q = Y V D^-1/2 (directions with D_i <= 1e-14 max D dropped) and the
// eigenvalues of K = (Q^T A)(Q^T A)^T = D^-1/2 V^T (Z^T Z) V D^-1/2, whose
// square roots are the singular values of Q^T A.  All of it is FP64.
//
// Block descriptors are int64 rows of 4: r0, r1, c0, c1 (half-open ranges
// of the permuted index space).  Work buffers are addressed by per-block
// int64 offsets computed on the host.
#include "common.h"

namespace flux {

__device__ __forceinline__ int64_t lower_bound_i32(const int32_t *__restrict__ a, int64_t lo,
                                                   int64_t hi, int64_t key) {
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if ((int64_t)a[mid] < key)
      lo = mid + 1;
    else
      hi = mid;
  }
  return lo;
}

// One wave per block: nnz and number of nonzero rows of A[r0:r1, c0:c1].
__global__ void k_block_stats(const int64_t *__restrict__ indptr,
                              const int32_t *__restrict__ indices, int64_t nb,
                              const int64_t *__restrict__ blk, int64_t *__restrict__ nnz,
                              int64_t *__restrict__ nzrows) {
  const int64_t b = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const int lane = threadIdx.x & 63;
  if (b >= nb) return;
  const int64_t r0 = blk[b * 4], r1 = blk[b * 4 + 1], c0 = blk[b * 4 + 2], c1 = blk[b * 4 + 3];
  int64_t cnt = 0, rows = 0;
  for (int64_t r = r0 + lane; r < r1; r += 64) {
    const int64_t s = indptr[r], e = indptr[r + 1];
    const int64_t lo = lower_bound_i32(indices, s, e, c0);
    const int64_t hi = lower_bound_i32(indices, lo, e, c1);
    cnt += hi - lo;
    rows += (hi > lo) ? 1 : 0;
  }
  for (int off = 32; off > 0; off >>= 1) {
    cnt += __shfl_down(cnt, off, 64);
    rows += __shfl_down(rows, off, 64);
  }
  if (lane == 0) {
    nnz[b] = cnt;
    nzrows[b] = rows;
  }
}

__device__ __forceinline__ uint64_t mix64(uint64_t z) {
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
  return z ^ (z >> 31);
}

// Rademacher entry W[j, c] = +-1 from a hash of (seed, global column, c).
__device__ __forceinline__ double rademacher(uint64_t seed, int64_t j, int64_t c) {
  const uint64_t h = mix64(seed ^ mix64((uint64_t)j * 0x9E3779B97F4A7C15ull + (uint64_t)c));
  return (h >> 63) ? -1.0 : 1.0;
}

// Y_b (m_b x l_b, row-major) = A[r0:r1, c0:c1] X_b, where X_b is the
// Rademacher matrix (X == NULL) or a stored (n_b x l_b) block.  One wave per
// (block, row); `rowbase` maps the flat wave id to its block.
template <typename TA>
__global__ void __launch_bounds__(256) k_block_spmm(
    const int64_t *__restrict__ indptr, const int32_t *__restrict__ indices,
    const TA *__restrict__ data, int64_t nb, const int64_t *__restrict__ blk,
    const int64_t *__restrict__ ls, const int64_t *__restrict__ rowstart,
    int64_t total_rows, const double *__restrict__ X, const int64_t *__restrict__ offX,
    double *__restrict__ Y, const int64_t *__restrict__ offY, uint64_t seed,
    int32_t *__restrict__ status) {
  const int64_t w = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const int lane = threadIdx.x & 63;
  if (w >= total_rows) return;
  // binary search the block owning flat row w
  int64_t lo = 0, hi = nb;
  while (hi - lo > 1) {
    const int64_t mid = (lo + hi) >> 1;
    if (rowstart[mid] <= w)
      lo = mid;
    else
      hi = mid;
  }
  const int64_t b = lo;
  const int64_t r0 = blk[b * 4], c0 = blk[b * 4 + 2], c1 = blk[b * 4 + 3];
  const int64_t rl = w - rowstart[b];
  const int64_t r = r0 + rl;
  const int64_t l = ls[b];
  const int64_t s = indptr[r], e = indptr[r + 1];
  const int64_t k0 = lower_bound_i32(indices, s, e, c0);
  const int64_t k1 = lower_bound_i32(indices, k0, e, c1);
  double *yrow = Y + offY[b] + rl * l;
  for (int64_t cb = 0; cb < l; cb += 64) {
    const int64_t c = cb + lane;
    double acc = 0.0;
    if (c < l) {
      for (int64_t k = k0; k < k1; ++k) {
        const int64_t j = indices[k];
        // The column ids of a row are sorted, so [k0, k1) holds only ids in
        // [c0, c1).  An id outside (an unsorted row) would address X outside
        // block b: it is skipped and reported instead of read.
        if (j < c0 || j >= c1) {
          atomicOr(status, 1);
          continue;
        }
        const double x = X ? X[offX[b] + (j - c0) * l + c] : rademacher(seed, j, c);
        acc += (double)data[k] * x;
      }
      yrow[c] = acc;
    }
  }
}

// Batched FP64 products on v_mfma_f64_16x16x4_f64.  A workgroup computes a
// 64 x 64 tile of C = op(A) op(B): K is consumed in slices of 16, staged in
// LDS (A: 64 rows x 16, B: 16 x 64 columns, both zero outside the matrix),
// and wave w owns rows 16 w .. 16 w + 15 of the tile (four 16 x 16 MFMA
// accumulators).  Lane l = 16 g + i holds A[i][g], B[g][i] and D[4 q + g][i].
typedef double v4d __attribute__((ext_vector_type(4)));
constexpr int kGemmTile = 64;
constexpr int kGemmKs = 16;

// a(i, k) and b(k, j) read the operands (bounds already checked).
template <class LA, class LB>
__device__ __forceinline__ void mfma_tile64(LA a, LB b, int64_t M, int64_t N, int64_t K,
                                            int64_t i0, int64_t j0, v4d acc[4]) {
  __shared__ double sa[kGemmTile][kGemmKs + 1];
  __shared__ double sb[kGemmKs][kGemmTile + 1];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int li = lane & 15, lg = lane >> 4;
  for (int c = 0; c < 4; ++c) acc[c] = v4d{0.0, 0.0, 0.0, 0.0};
  for (int64_t k0 = 0; k0 < K; k0 += kGemmKs) {
    // 1024 values of each operand, 4 per thread
    for (int e = tid; e < kGemmTile * kGemmKs; e += 256) {
      const int r = e / kGemmKs, kk = e % kGemmKs;       // A: row r, k kk
      const int64_t gi = i0 + r, gk = k0 + kk;
      sa[r][kk] = (gi < M && gk < K) ? a(gi, gk) : 0.0;
      const int kr = e / kGemmTile, cc = e % kGemmTile;   // B: k kr, column cc
      const int64_t gk2 = k0 + kr, gj = j0 + cc;
      sb[kr][cc] = (gk2 < K && gj < N) ? b(gk2, gj) : 0.0;
    }
    __syncthreads();
    for (int s = 0; s < kGemmKs; s += 4) {
      const double av = sa[16 * wave + li][s + lg];
      for (int c = 0; c < 4; ++c)
        acc[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(av, sb[s + lg][16 * c + li], acc[c], 0, 0,
                                                      0);
    }
    __syncthreads();
  }
}

// G_b = X_b^T X_b (l_b x l_b) for X_b (rows_b x l_b) row-major.  grid.x over
// 64 x 64 tiles (surplus workgroups exit), grid.y over blocks.
__global__ void __launch_bounds__(256) k_batched_gram(
    const int64_t *__restrict__ rows, const int64_t *__restrict__ ls,
    const double *__restrict__ X, const int64_t *__restrict__ offX, double *__restrict__ G,
    const int64_t *__restrict__ offG) {
  const int64_t b = blockIdx.y;
  const int64_t l = ls[b], m = rows[b];
  const int64_t nt = (l + kGemmTile - 1) / kGemmTile;
  const int64_t tile = blockIdx.x;
  if (tile >= nt * nt) return;  // uniform over the workgroup
  const int64_t i0 = (tile / nt) * kGemmTile, j0 = (tile % nt) * kGemmTile;
  const double *Xb = X + offX[b];
  v4d acc[4];
  mfma_tile64([&](int64_t i, int64_t k) { return Xb[k * l + i]; },
              [&](int64_t k, int64_t j) { return Xb[k * l + j]; }, l, l, m, i0, j0, acc);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int li = lane & 15, lg = lane >> 4;
  for (int c = 0; c < 4; ++c)
    for (int q = 0; q < 4; ++q) {
      const int64_t gi = i0 + 16 * wave + 4 * q + lg, gj = j0 + 16 * c + li;
      if (gi < l && gj < l) G[offG[b] + gi * l + gj] = acc[c][q];
    }
}

// C_b = op(A_b) op(B_b), FP64, row-major, per-block shapes.  desc rows of 12
// int64: M, N, K, offA, lda, transA, offB, ldb, transB, offC, ldc, beta_is_1.
__global__ void __launch_bounds__(256) k_batched_gemm(const int64_t *__restrict__ desc,
                                                      const double *__restrict__ A,
                                                      const double *__restrict__ B,
                                                      double *__restrict__ C) {
  const int64_t *d = desc + (int64_t)blockIdx.y * 12;
  const int64_t M = d[0], N = d[1], K = d[2];
  const int64_t ntn = (N + kGemmTile - 1) / kGemmTile;
  const int64_t tile = blockIdx.x;
  if (tile >= ((M + kGemmTile - 1) / kGemmTile) * ntn) return;  // uniform
  const int64_t i0 = (tile / ntn) * kGemmTile, j0 = (tile % ntn) * kGemmTile;
  const double *Ab = A + d[3];
  const double *Bb = B + d[6];
  const int64_t lda = d[4], ldb = d[7];
  const bool ta = d[5] != 0, tb = d[8] != 0;
  v4d acc[4];
  mfma_tile64([&](int64_t i, int64_t k) { return ta ? Ab[k * lda + i] : Ab[i * lda + k]; },
              [&](int64_t k, int64_t j) { return tb ? Bb[j * ldb + k] : Bb[k * ldb + j]; }, M,
              N, K, i0, j0, acc);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int li = lane & 15, lg = lane >> 4;
  for (int c = 0; c < 4; ++c)
    for (int q = 0; q < 4; ++q) {
      const int64_t gi = i0 + 16 * wave + 4 * q + lg, gj = j0 + 16 * c + li;
      if (gi < M && gj < N) {
        double *cp = C + d[9] + gi * d[10] + gj;
        *cp = d[11] ? *cp + acc[c][q] : acc[c][q];
      }
    }
}

// LDS written by some lanes of a wave is read by others of the same wave.
__device__ __forceinline__ void wave_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Tournament pairing of step `step` of a cyclic Jacobi sweep over npad
// (even) indices: index 0 stays, the others rotate; pair k is (p, q), p < q.
__device__ __forceinline__ void jacobi_pair(int k, int step, int npad, int &p, int &q) {
  // both sums are below 2 (npad - 1): k <= npad / 2 - 1, step <= npad - 2
  int x = k - 1 + step, y = npad - 2 - k + step;
  x -= x >= npad - 1 ? npad - 1 : 0;
  y -= y >= npad - 1 ? npad - 1 : 0;
  x = k == 0 ? 0 : x + 1;
  y += 1;
  p = min(x, y);
  q = max(x, y);
}

// Rotation (c, s) that zeroes a_pq of the 2x2 symmetric block.
__device__ __forceinline__ void jacobi_rotation(double app, double aqq, double apq, double &c,
                                                double &s) {
  c = 1.0;
  s = 0.0;
  if (apq != 0.0) {
    const double tau = (aqq - app) / (2.0 * apq);
    const double t = (tau >= 0.0 ? 1.0 : -1.0) / (fabs(tau) + sqrt(1.0 + tau * tau));
    c = 1.0 / sqrt(1.0 + t * t);
    s = t * c;
  }
}

// Batched symmetric eigensolver: cyclic Jacobi in the round-robin
// (tournament) order.  A sweep over a matrix is a serial chain of n - 1
// steps, each with n / 2 rotations that need the matrix as the step before
// left it, so its time is the time of a step in one workgroup, and only what
// the chain needs is in it:
//  * k_eig_sweep rotates the matrix alone, in LDS up to n = kEigLds, one 2 x 2
//    block of (pair, pair) at a time, read and written once (columns, then
//    rows, with a barrier between, read and wrote twice as much, and the
//    eigenvectors from global memory on top).  Both triangles are kept: an
//    element and its mirror image round differently, and the rotations read
//    the upper one.  It leaves the sweep's rotations in global memory.
//  * k_eig_apply applies them to the eigenvectors, whose columns are
//    independent: one wave per two columns, all over the chip.
// A matrix that has converged leaves a flag, and the remaining launches of
// the max_sweeps return at once.  The results are those of the plain order
// (every pair's columns, then its rows), bit for bit.
//
// 12 matrices of n = 88 from a 1,922-facet crater, a call of 6 to 20 sweeps:
// 11.2 ms with one workgroup doing it all in that order, 2.9 ms now (n = 88 to
// 128 in general a quarter to a third of the time; above, where the matrix
// is in L2, three quarters).

// Largest matrix k_eig_sweep holds in LDS (132,096 B).
constexpr int kEigLds = 128;
constexpr int kEigThreads = 1024;

// Sum of v over the workgroup of kEigThreads; every thread gets it.
__device__ __forceinline__ double block_sum_eig(double v, double *red) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double t = 0.0;
  for (int w = 0; w < kEigThreads / 64; ++w) t += red[w];
  __syncthreads();
  return t;
}

struct Rotation {
  double x, y;  // cosine, sine
};

// The sweep's rotations of matrix b: (n - 1) n doubles for even n, n (n - 1)
// for odd n, where the pair with the padding index is left out, and the flag
// in the last of the n^2.  slot(k) of a step: its place without that pair.
__device__ __forceinline__ int64_t rot_at(int step, int k, int n) {
  if (!(n & 1)) return (int64_t)step * (n / 2) + k;
  // the padding index n is x of pair k = n - step, or y of pair k = step
  // (whichever is below (n + 1) / 2)
  const int pad = step < (n + 1) / 2 ? step : n - step;
  return (int64_t)step * (n / 2) + k - (k > pad ? 1 : 0);
}

// The two results of a rotation (c, s) of x, y, each one product and one
// fused step in a fixed order: an element is rounded the same way wherever
// it is rotated.
__device__ __forceinline__ double rot_x(double c, double s, double x, double y) {
  return fma(c, x, -(s * y));
}
__device__ __forceinline__ double rot_y(double c, double s, double x, double y) {
  return fma(s, x, c * y);
}

// Rotation of pair k of a step: into cs, into the sweep's list, and applied
// to the pair's own 2 x 2 block.
template <typename At>
__device__ __forceinline__ void eig_rotation(int n, int npad, int step, int k, At at,
                                             double2 *cs, Rotation *rots) {
  int p, q;
  jacobi_pair(k, step, npad, p, q);
  double c = 1.0, sv = 0.0;
  if (q < n) {
    double &rpp = at(p, p), &rqq = at(q, q), &rpq = at(p, q), &rqp = at(q, p);
    const double app = rpp, aqq = rqq, apq = rpq, aqp = rqp;
    jacobi_rotation(app, aqq, apq, c, sv);
    if (sv != 0.0) {
      const double bpp = rot_x(c, sv, app, apq), bpq = rot_y(c, sv, app, apq);
      const double bqp = rot_x(c, sv, aqp, aqq), bqq = rot_y(c, sv, aqp, aqq);
      rpp = rot_x(c, sv, bpp, bqp);
      rqq = rot_y(c, sv, bpq, bqq);
      rpq = 0.0;
      rqp = 0.0;
    }
    rots[rot_at(step, k, n)] = Rotation{c, sv};
  }
  cs[k] = make_double2(c, sv);
}

// Rotations k1 (rows) and k2 (columns) on their 2 x 2 block.  PAD: the
// matrix has room for the padding index (a zero row and column that stay
// zero).
template <bool PAD, typename At>
__device__ __forceinline__ void eig_block(int n, int npad, int step, int k1, int k2, At at,
                                          const double2 *cs) {
  const double2 r1 = cs[k1], r2 = cs[k2];
  int p, q, r, t;
  jacobi_pair(k1, step, npad, p, q);
  jacobi_pair(k2, step, npad, r, t);
  const bool q_ok = PAD || q < n, t_ok = PAD || t < n;  // at most one is false
  double &ppr = at(p, r);
  double &ppt = t_ok ? at(p, t) : ppr;
  double &pqr = q_ok ? at(q, r) : ppr;
  double &pqt = q_ok ? (t_ok ? at(q, t) : pqr) : ppt;
  const double apr = ppr, apt = t_ok ? ppt : 0.0;
  const double aqr = q_ok ? pqr : 0.0, aqt = q_ok && t_ok ? pqt : 0.0;
  const double xpr = rot_x(r2.x, r2.y, apr, apt), xpt = rot_y(r2.x, r2.y, apr, apt);
  const double xqr = rot_x(r2.x, r2.y, aqr, aqt), xqt = rot_y(r2.x, r2.y, aqr, aqt);
  ppr = rot_x(r1.x, r1.y, xpr, xqr);
  if (t_ok) ppt = rot_x(r1.x, r1.y, xpt, xqt);
  if (q_ok) pqr = rot_y(r1.x, r1.y, xpr, xqr);
  if (q_ok && t_ok) pqt = rot_y(r1.x, r1.y, xpt, xqt);
}

// Blocks that hold the off-diagonal elements of a pair of the next step: next
// pair k joins one index each of pairs k - 1 and k + 1, the outer ones of
// pairs 0 and 1 and of the last two.
__device__ __forceinline__ bool eig_ahead(int k1, int k2, int half) {
  return k2 - k1 == 2 || (k1 == 0 && k2 == 1) || (k1 == half - 2 && k2 == half - 1);
}

// One sweep over the matrix behind at(i, j).  The first wave rotates the
// blocks that the next step's rotations need and computes those (divisions
// and square roots in sequence) while the other waves rotate the rest, so a
// step is one barrier.  The rest is bound by instruction issue (one CU), so
// the blocks are dealt one to a thread, full waves, and their index
// arithmetic is kept short.  cs: two steps' rotations.
template <bool PAD, typename At>
__device__ __forceinline__ void eig_steps(int n, At at, double2 (*cs)[512], Rotation *rots) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int npad = n + (n & 1), half = npad / 2, nsteps = npad - 1;
  // this thread's first item and the stride of kEigThreads - 64 items
  const int d0 = 1 + (tid - 64) / half, k0 = (tid - 64) % half;
  const int dd = (kEigThreads - 64) / half, dk = (kEigThreads - 64) % half;
  if (wave == 0)
    for (int k = lane; k < half; k += 64) eig_rotation(n, npad, 0, k, at, cs[0], rots);
  __syncthreads();
  for (int step = 0; step < nsteps; ++step) {
    const double2 *now = cs[step & 1];
    if (wave == 0) {
      for (int k = lane; k < half; k += 64) {
        const int k1 = k == 0 ? 0 : (k == half - 1 ? half - 2 : k - 1);
        const int k2 = k == 0 ? 1 : (k == half - 1 ? half - 1 : k + 1);
        if (k2 < half && (k == 0 || half > 2)) {
          eig_block<PAD>(n, npad, step, k1, k2, at, now);
          eig_block<PAD>(n, npad, step, k2, k1, at, now);
        }
      }
      wave_order();
      if (step + 1 < nsteps)
        for (int k = lane; k < half; k += 64)
          eig_rotation(n, npad, step + 1, k, at, cs[(step + 1) & 1], rots);
    } else {
      // item (d, k): the block of pairs k and k + d (mod half)
      int d = d0, k = k0;
      while (d < half) {
        const int m = k + d < half ? k + d : k + d - half;
        if (!eig_ahead(min(k, m), max(k, m), half))
          eig_block<PAD>(n, npad, step, k, m, at, now);
        k += dk;
        d += dd;
        if (k >= half) {
          k -= half;
          ++d;
        }
      }
    }
    __syncthreads();
  }
}

__global__ void __launch_bounds__(kEigThreads) k_eig_sweep(
    const int64_t *__restrict__ ns, double *A, const int64_t *__restrict__ offA, double *rot,
    int sweep) {
  __shared__ double a[kEigLds * (kEigLds + 1)];
  __shared__ double2 cs[2][512];
  __shared__ double red[kEigThreads / 64];
  const int64_t b = blockIdx.x;
  const int n = (int)ns[b], tid = threadIdx.x;
  if (n <= 1) return;
  double *ag = A + offA[b];
  double *rb = rot + offA[b];
  double *flag = rb + (int64_t)n * n - 1;
  if (sweep > 0 && *flag == 0.0) return;
  const bool lds = n <= kEigLds;
  const int npad = n + (n & 1), s = npad + 1;  // odd stride
  double off = 0.0, dia = 0.0;
  for (int64_t k = tid; k < (int64_t)n * n; k += kEigThreads) {
    const int i = (int)(k / n), j = (int)(k - (int64_t)i * n);
    const double x = ag[k];
    if (lds) a[i * s + j] = x;
    if (i != j)
      off += x * x;
    else
      dia += x * x;
  }
  const double off_all = block_sum_eig(off, red);
  const double dia_all = block_sum_eig(dia, red);
  const bool done = off_all <= 1e-30 * dia_all || off_all == 0.0;
  if (tid == 0) *flag = done ? 0.0 : 1.0;
  if (done) return;
  if (lds) {
    if (n & 1)
      for (int j = tid; j <= n; j += kEigThreads) a[n * s + j] = a[j * s + n] = 0.0;
    __syncthreads();
    eig_steps<true>(
        n, [&](int i, int j) -> double & { return a[__mul24(i, s) + j]; }, cs, (Rotation *)rb);
    for (int64_t k = tid; k < (int64_t)n * n; k += kEigThreads) {
      const int i = (int)(k / n), j = (int)(k - (int64_t)i * n);
      ag[k] = a[i * s + j];
    }
  } else {
    eig_steps<false>(
        n, [&](int i, int j) -> double & { return ag[(int64_t)i * n + j]; }, cs, (Rotation *)rb);
  }
}

// W <- J^T W for the sweep's rotations (W = V^T, n x n row-major; W = I
// first if init).  A wave keeps two columns in LDS; lane l takes pairs l,
// l + 64, ..., and the next step's rotations are on their way meanwhile.
template <int NI>
__global__ void __launch_bounds__(256) k_eig_apply(const int64_t *__restrict__ ns,
                                                   const int64_t *__restrict__ offA,
                                                   const double *__restrict__ rot,
                                                   double *__restrict__ W, int init, int rotate) {
  extern __shared__ double2 wcols[];  // 4 waves x lds_rows
  const int64_t b = blockIdx.x;
  const int n = (int)ns[b];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int i0 = ((int)blockIdx.y * 4 + wave) * 2;
  if (i0 >= n) return;
  const double *rb = rot + offA[b];
  double *wb = W + offA[b];
  const bool run = rotate && n > 1 && rb[(int64_t)n * n - 1] != 0.0;
  if (!init && !run) return;
  double2 *w = wcols + (int64_t)wave * 64 * 2 * NI;
  const bool two = i0 + 1 < n;
  for (int p = lane; p < n; p += 64) {
    double2 v;
    if (init)
      v = make_double2(p == i0 ? 1.0 : 0.0, p == i0 + 1 ? 1.0 : 0.0);
    else
      v = make_double2(wb[(int64_t)p * n + i0], two ? wb[(int64_t)p * n + i0 + 1] : 0.0);
    w[p] = v;
  }
  wave_order();
  if (run) {
    const Rotation *rots = (const Rotation *)rb;
    const int npad = n + (n & 1), half = npad / 2;
    Rotation next[NI];
#pragma unroll
    for (int u = 0; u < NI; ++u) {
      const int k = lane + 64 * u;
      next[u] = k < half ? rots[rot_at(0, k, n)] : Rotation{1.0, 0.0};
    }
    for (int step = 0; step < npad - 1; ++step) {
      Rotation r[NI];
#pragma unroll
      for (int u = 0; u < NI; ++u) {
        const int k = lane + 64 * u;
        r[u] = next[u];
        if (k < half && step + 1 < npad - 1) next[u] = rots[rot_at(step + 1, k, n)];
      }
#pragma unroll
      for (int u = 0; u < NI; ++u) {
        const int k = lane + 64 * u;
        if (k >= half || r[u].y == 0.0) continue;
        int p, q;
        jacobi_pair(k, step, npad, p, q);
        if (q >= n) continue;  // no rotation stored for the padding index
        const double2 x = w[p], y = w[q];
        w[p] = make_double2(rot_x(r[u].x, r[u].y, x.x, y.x), rot_x(r[u].x, r[u].y, x.y, y.y));
        w[q] = make_double2(rot_y(r[u].x, r[u].y, x.x, y.x), rot_y(r[u].x, r[u].y, x.y, y.y));
      }
      wave_order();
    }
  }
  for (int p = lane; p < n; p += 64) {
    const double2 v = w[p];
    wb[(int64_t)p * n + i0] = v.x;
    if (two) wb[(int64_t)p * n + i0 + 1] = v.y;
  }
}

// Eigenvalues descending (rank by counting, ties by index) and the
// eigenvectors, row i of W, as columns of Vout.
__global__ void __launch_bounds__(256) k_eig_sort(const int64_t *__restrict__ ns,
                                                  const double *__restrict__ A,
                                                  const int64_t *__restrict__ offA,
                                                  const double *__restrict__ W,
                                                  double *__restrict__ Vout,
                                                  double *__restrict__ evals,
                                                  const int64_t *__restrict__ offE) {
  __shared__ double d[1024];
  __shared__ int rank[1024];
  const int64_t b = blockIdx.x;
  const int n = (int)ns[b], tid = threadIdx.x;
  const double *a = A + offA[b];
  for (int i = tid; i < n; i += 256) d[i] = a[(int64_t)i * n + i];
  __syncthreads();
  for (int i = tid; i < n; i += 256) {
    int r = 0;
    for (int j = 0; j < n; ++j) r += (d[j] > d[i]) || (d[j] == d[i] && j < i);
    rank[i] = r;
    if (blockIdx.y == 0) evals[offE[b] + r] = d[i];
  }
  __syncthreads();
  for (int64_t k = (int64_t)blockIdx.y * 256 + tid; k < (int64_t)n * n;
       k += (int64_t)gridDim.y * 256) {
    const int i = (int)(k / n), r = (int)(k - (int64_t)i * n);
    Vout[offA[b] + (int64_t)r * n + rank[i]] = W[offA[b] + k];
  }
}

// G_b <- 1.5 I - 0.5 G_b (n_b x n_b): the factor of one Newton-Schulz step
// Q <- Q (3 I - Q^T Q) / 2 towards orthonormal columns.
__global__ void k_ns_factor(const int64_t *__restrict__ ns, double *__restrict__ G,
                            const int64_t *__restrict__ offG) {
  const int64_t b = blockIdx.y;
  const int64_t n = ns[b];
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < n * n;
       k += (int64_t)gridDim.x * blockDim.x) {
    const double g = G[offG[b] + k];
    G[offG[b] + k] = ((k / n == k % n) ? 1.5 : 0.0) - 0.5 * g;
  }
}

// T_b[:, j] = V_b[:, j] / sqrt(d_j) for d_j > cut * d_0 (d sorted desc),
// else 0;  kept[b] = number of kept columns.
__global__ void k_scale_basis(const int64_t *__restrict__ ns, const double *__restrict__ V,
                              const int64_t *__restrict__ offA, const double *__restrict__ d,
                              const int64_t *__restrict__ offE, double cut,
                              double *__restrict__ T, int64_t *__restrict__ kept) {
  const int64_t b = blockIdx.y;
  const int64_t n = ns[b];
  const double d0 = d[offE[b]];
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < n * n;
       k += (int64_t)gridDim.x * blockDim.x) {
    const int64_t j = k % n;
    const double dj = d[offE[b] + j];
    const bool keep = d0 > 0.0 && dj > cut * d0;
    T[offA[b] + k] = keep ? V[offA[b] + k] / sqrt(dj) : 0.0;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    int64_t c = 0;
    for (int64_t j = 0; j < n; ++j) {
      const double dj = d[offE[b] + j];
      c += (d0 > 0.0 && dj > cut * d0) ? 1 : 0;
    }
    kept[b] = c;
  }
}

// Columns of C_b (l x r) scaled by 1/s_j (s = sqrt of eigenvalues, desc).
__global__ void k_scale_cols_inv_sqrt(const int64_t *__restrict__ dims, double *__restrict__ C,
                                      const int64_t *__restrict__ offC,
                                      const double *__restrict__ lam,
                                      const int64_t *__restrict__ offL) {
  const int64_t b = blockIdx.y;
  const int64_t rows = dims[b * 2], cols = dims[b * 2 + 1];
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < rows * cols;
       k += (int64_t)gridDim.x * blockDim.x) {
    const int64_t j = k % cols;
    const double l = lam[offL[b] + j];
    C[offC[b] + k] = l > 0.0 ? C[offC[b] + k] / sqrt(l) : 0.0;
  }
}

}  // namespace flux

using namespace flux;

extern "C" int flux_block_stats(const int64_t *indptr, const int32_t *indices, int64_t nb,
                                const int64_t *blk, int64_t *nnz, int64_t *nzrows,
                                void *stream) {
  FLUX_CHECK(nb >= 0, "flux_block_stats: negative count");
  if (nb == 0) return 0;
  FLUX_CHECK(indptr && indices && blk && nnz && nzrows, "flux_block_stats: NULL array");
  hipLaunchKernelGGL(k_block_stats, dim3(ceil_div_u(nb, 4)), dim3(256), 0, as_stream(stream),
                     indptr, indices, nb, blk, nnz, nzrows);
  FLUX_LAUNCH_CHECK();
  return 0;
}

extern "C" int flux_block_spmm(const int64_t *indptr, const int32_t *indices, const void *data,
                               int dtype, int64_t nb, const int64_t *blk, const int64_t *ls,
                               const int64_t *rowstart, int64_t total_rows, const double *X,
                               const int64_t *offX, double *Y, const int64_t *offY,
                               uint64_t seed, int32_t *status, void *stream) {
  FLUX_CHECK(nb >= 0 && total_rows >= 0, "flux_block_spmm: bad sizes");
  if (nb == 0 || total_rows == 0) return 0;
  FLUX_CHECK(indptr && indices && data && blk && ls && rowstart && Y && offY && status,
             "flux_block_spmm: NULL array");
  FLUX_CHECK(X == nullptr || offX != nullptr, "flux_block_spmm: offX required with X");
  hipStream_t st = as_stream(stream);
  const unsigned g = ceil_div_u(total_rows, 4);
  if (dtype == FLUX_F64)
    hipLaunchKernelGGL(k_block_spmm<double>, dim3(g), dim3(256), 0, st, indptr, indices,
                       (const double *)data, nb, blk, ls, rowstart, total_rows, X, offX, Y,
                       offY, seed, status);
  else if (dtype == FLUX_F32)
    hipLaunchKernelGGL(k_block_spmm<float>, dim3(g), dim3(256), 0, st, indptr, indices,
                       (const float *)data, nb, blk, ls, rowstart, total_rows, X, offX, Y,
                       offY, seed, status);
  else
    FLUX_CHECK(false, "flux_block_spmm: dtype must be F32/F64");
  FLUX_LAUNCH_CHECK();
  return 0;
}

extern "C" int flux_batched_gram(int64_t nb, const int64_t *rows, const int64_t *ls,
                                 int64_t lmax, const double *X, const int64_t *offX, double *G,
                                 const int64_t *offG, void *stream) {
  FLUX_CHECK(nb >= 0 && nb <= 65535 && lmax >= 0, "flux_batched_gram: bad sizes");
  if (nb == 0 || lmax == 0) return 0;
  const int64_t nt = (lmax + kGemmTile - 1) / kGemmTile;
  hipLaunchKernelGGL(k_batched_gram, dim3((unsigned)(nt * nt), (unsigned)nb), dim3(256), 0,
                     as_stream(stream), rows, ls, X, offX, G, offG);
  FLUX_LAUNCH_CHECK();
  return 0;
}

extern "C" int flux_batched_gemm(int64_t nb, const int64_t *desc, int64_t max_tiles,
                                 const double *A, const double *B, double *C, void *stream) {
  FLUX_CHECK(nb >= 0 && nb <= 65535 && max_tiles >= 0, "flux_batched_gemm: bad sizes");
  if (nb == 0 || max_tiles == 0) return 0;
  hipLaunchKernelGGL(k_batched_gemm, dim3((unsigned)max_tiles, (unsigned)nb), dim3(256), 0,
                     as_stream(stream), desc, A, B, C);
  FLUX_LAUNCH_CHECK();
  return 0;
}

extern "C" int flux_batched_syevj(int64_t nb, const int64_t *ns, int64_t nmax, double *A,
                                  const int64_t *offA, double *Vwork, double *Vout,
                                  double *evals, const int64_t *offE, int max_sweeps,
                                  void *stream) {
  FLUX_CHECK(nb >= 0 && nmax >= 0, "flux_batched_syevj: bad sizes");
  FLUX_CHECK(nmax <= 1024, "flux_batched_syevj: matrices above 1024 x 1024 are not supported");
  FLUX_CHECK(nb <= 0x7fffffff, "flux_batched_syevj: too many matrices");
  if (nb == 0 || nmax == 0) return 0;
  hipStream_t st = as_stream(stream);
  // rotations in Vout until the end, eigenvectors in Vwork
  const dim3 cols((unsigned)nb, (unsigned)((nmax + 7) / 8));
  const int sweeps = max_sweeps > 0 ? max_sweeps : 0;
  for (int k = 0; k < (sweeps ? sweeps : 1); ++k) {
    if (sweeps)
      hipLaunchKernelGGL(k_eig_sweep, dim3((unsigned)nb), dim3(kEigThreads), 0, st, ns, A, offA,
                         Vout, k);
    const int init = k == 0, rotate = sweeps > 0;
    if (nmax <= 128)
      hipLaunchKernelGGL(k_eig_apply<1>, cols, dim3(256), 4 * 128 * sizeof(double2), st, ns, offA,
                         Vout, Vwork, init, rotate);
    else if (nmax <= 256)
      hipLaunchKernelGGL(k_eig_apply<2>, cols, dim3(256), 4 * 256 * sizeof(double2), st, ns, offA,
                         Vout, Vwork, init, rotate);
    else
      hipLaunchKernelGGL(k_eig_apply<8>, cols, dim3(256), 4 * 1024 * sizeof(double2), st, ns,
                         offA, Vout, Vwork, init, rotate);
    FLUX_LAUNCH_CHECK();
  }
  hipLaunchKernelGGL(k_eig_sort, dim3((unsigned)nb, 16), dim3(256), 0, st, ns, A, offA, Vwork,
                     Vout, evals, offE);
  FLUX_LAUNCH_CHECK();
  return 0;
}

extern "C" int flux_batched_ns_factor(int64_t nb, const int64_t *ns, double *G,
                                      const int64_t *offG, void *stream) {
  FLUX_CHECK(nb >= 0 && nb <= 65535, "flux_batched_ns_factor: bad sizes");
  if (nb == 0) return 0;
  FLUX_CHECK(ns && G && offG, "flux_batched_ns_factor: NULL array");
  hipLaunchKernelGGL(k_ns_factor, dim3(64, (unsigned)nb), dim3(256), 0, as_stream(stream), ns,
                     G, offG);
  FLUX_LAUNCH_CHECK();
  return 0;
}

extern "C" int flux_scale_basis(int64_t nb, const int64_t *ns, const double *V,
                                const int64_t *offA, const double *d, const int64_t *offE,
                                double cut, double *T, int64_t *kept, void *stream) {
  FLUX_CHECK(nb >= 0 && nb <= 65535, "flux_scale_basis: bad sizes");
  if (nb == 0) return 0;
  hipLaunchKernelGGL(k_scale_basis, dim3(64, (unsigned)nb), dim3(256), 0, as_stream(stream), ns,
                     V, offA, d, offE, cut, T, kept);
  FLUX_LAUNCH_CHECK();
  return 0;
}

// S[offS[q] + i] = sqrt(max(lam[offL[q] + i], 0)), i < r[q]: the singular
// values of the accepted blocks (the eigenvalues of Z^T Z) in one buffer.
__global__ void k_sigma_from_lambda(int64_t np_, const int64_t *__restrict__ offL,
                                    const int64_t *__restrict__ r,
                                    const int64_t *__restrict__ offS,
                                    const double *__restrict__ lam, double *__restrict__ S) {
  const int64_t q = blockIdx.y;
  if (q >= np_) return;
  for (int64_t i = threadIdx.x + (int64_t)blockIdx.x * blockDim.x; i < r[q];
       i += (int64_t)gridDim.x * blockDim.x)
    S[offS[q] + i] = sqrt(fmax(lam[offL[q] + i], 0.0));
}

extern "C" int flux_sigma_from_lambda(int64_t np_, const int64_t *offL, const int64_t *r,
                                      const int64_t *offS, const double *lam, double *S,
                                      void *stream) {
  FLUX_CHECK(np_ >= 0 && np_ <= 65535, "flux_sigma_from_lambda: bad sizes");
  if (np_ == 0) return 0;
  FLUX_CHECK(offL && r && offS && lam && S, "flux_sigma_from_lambda: NULL array");
  hipLaunchKernelGGL(k_sigma_from_lambda, dim3(1, (unsigned)np_), dim3(256), 0,
                     as_stream(stream), np_, offL, r, offS, lam, S);
  FLUX_LAUNCH_CHECK();
  return 0;
}

extern "C" int flux_scale_cols_inv_sqrt(int64_t nb, const int64_t *dims, double *C,
                                        const int64_t *offC, const double *lam,
                                        const int64_t *offL, void *stream) {
  FLUX_CHECK(nb >= 0 && nb <= 65535, "flux_scale_cols_inv_sqrt: bad sizes");
  if (nb == 0) return 0;
  hipLaunchKernelGGL(k_scale_cols_inv_sqrt, dim3(64, (unsigned)nb), dim3(256), 0,
                     as_stream(stream), dims, C, offC, lam, offL);
  FLUX_LAUNCH_CHECK();
  return 0;
}
