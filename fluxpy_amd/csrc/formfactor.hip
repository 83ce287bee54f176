// Form-factor assembly (form_factors.py:11-72) and mesh geometry
// (shape.py:16-45).
//
// Operation order (all in the mesh dtype T, each operation rounded; this
// file is compiled with -ffp-contract=off):
//   dot3(a, b)  = (a0*b0 + a1*b1) + a2*b2
//   NP_j        = dot3(N_j, P_j)                        (form_factors.py:26)
//   c           = max(0, dot3(N_i, P_j - P_i)) * max(0, dot3(P_i, N_j) - NP_j)
//                                                       (form_factors.py:46-47)
//   keep        c > eps and i != j                      (:50-52)
//   visibility  scene ray test of the backend mode      (:57)
//   s           = pi * (s2 * s2), s2 = (d0^2 + d1^2) + d2^2, d = P_i - P_j
//   F_ij        = (c * A_j) / s, 0 if s == 0            (:62-64)
#include <algorithm>

#include "wide.h"

namespace flux {

template <typename T>
__device__ __forceinline__ T dot3(const T *a, const T *b) {
  return (a[0] * b[0] + a[1] * b[1]) + a[2] * b[2];
}

template <typename T>
__device__ __forceinline__ T pos_part(T x) {
  return x > (T)0 ? x : (T)0;
}

template <typename T>
__device__ __forceinline__ T ff_prefilter(const T *Pi, const T *Ni, const T *Pj,
                                          const T *Nj) {
  T d[3] = {Pj[0] - Pi[0], Pj[1] - Pi[1], Pj[2] - Pi[2]};
  T npj = dot3(Nj, Pj);
  T a = dot3(Ni, d);
  T b = dot3(Pi, Nj) - npj;
  return pos_part(a) * pos_part(b);
}

template <typename T>
__device__ __forceinline__ T ff_value(T c, const T *Pi, const T *Pj, T Aj) {
  T d0 = Pi[0] - Pj[0], d1 = Pi[1] - Pj[1], d2 = Pi[2] - Pj[2];
  T s2 = (d0 * d0 + d1 * d1) + d2 * d2;
  T s = (T)3.141592653589793 * (s2 * s2);
  if (s == (T)0) return (T)0;
  return (c * Aj) / s;
}

// Candidate bits (the pairs that get a ray): one wave per (row p, 64-column
// word w), the waves of the grid striding over all m W words.
template <typename T>
__global__ void __launch_bounds__(256) k_ff_candidates(int64_t nf, const T *__restrict__ P,
                                                       const T *__restrict__ N,
                                                       const int64_t *__restrict__ I, int64_t m,
                                                       const int64_t *__restrict__ J, int64_t n,
                                                       T eps, uint64_t *__restrict__ mask,
                                                       int64_t W) {
  const int lane = threadIdx.x & 63;
  const int64_t nwaves = (int64_t)gridDim.x * (blockDim.x >> 6);
  for (int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6; wave < m * W;
       wave += nwaves) {
    const int64_t p = wave / W, q = (wave % W) * 64 + lane;
    const int64_t i64 = I[p];
    const bool row_ok = i64 >= 0 && i64 < nf;
    const int64_t i = row_ok ? i64 : 0;
    const T Pi[3] = {P[i * 3], P[i * 3 + 1], P[i * 3 + 2]};
    const T Ni[3] = {N[i * 3], N[i * 3 + 1], N[i * 3 + 2]};
    bool bit = false;
    if (q < n && row_ok && J[q] >= 0 && J[q] < nf) {
      const int64_t j = J[q];
      const T Pj[3] = {P[j * 3], P[j * 3 + 1], P[j * 3 + 2]};
      const T Nj[3] = {N[j * 3], N[j * 3 + 1], N[j * 3 + 2]};
      bit = i != j && ff_prefilter(Pi, Ni, Pj, Nj) > eps;
    }
    const uint64_t b = __ballot(bit);
    if (lane == 0) mask[wave] = b;
  }
}

// Candidate pairs a wave keeps in LDS.
constexpr int kPairQueue = 128;  // < 64 left over + one word of 64

// The tiles of a wave.  Large problems draw them from a counter, one atomic
// per 64 words of 64 columns.  Smaller ones have smaller tiles, too many for
// that (an atomic on one address costs the chip about 18 ns: 59,582 one-word
// tiles of 1,922 facets took 1.0 ms drawn and 0.21 ms dealt out): there each
// wave has one tile of every round, in a place that moves from round to
// round (at a fixed place a wave would keep to one column range).
constexpr int64_t kPairTiles = 40960;  // tiles aimed at, 8 a wave
constexpr int64_t kTileShift = 977;    // below 5,120 waves, which rounds need

struct TileWalk {
  int64_t ntiles, base, slot, nwaves;
  unsigned long long *counter;

  __device__ __forceinline__ void init(int64_t n, unsigned long long *c) {
    ntiles = n;
    counter = c;
    nwaves = (int64_t)gridDim.x * 4;
    base = 0;
    slot = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * 4 + (threadIdx.x >> 6)));
  }

  // The next tile, or one past the last.
  __device__ __forceinline__ int64_t next() {
    if (counter) {
      unsigned long long t = 0;
      if ((threadIdx.x & 63) == 0) t = atomicAdd(counter, 1ull);
      return ((int64_t)__builtin_amdgcn_readfirstlane((int)(t >> 32)) << 32) |
             (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)t);
    }
    const int64_t tile = base + slot;
    base += nwaves;
    slot = slot + kTileShift < nwaves ? slot + kTileShift : slot + kTileShift - nwaves;
    return tile < ntiles ? tile : ntiles;
  }
};

static inline int64_t tile_width(int64_t words) {
  return std::max<int64_t>(1, std::min<int64_t>(64, words / kPairTiles));
}

// Rays of the pairs (p, q) of m x n positions for trace_wave (wide.h).  A
// wave takes tiles of one row p, evaluates the prefilter 64 columns at a
// time and keeps the pairs that need a ray in a small queue in LDS, from
// which lanes out of work are served (the prefilter keeps ~1/4 of the pairs
// on terrain).  A visible pair sets its bit in the zeroed mask.  Lanes of a
// wave may work on different rows, so none waits for the end of a row: with
// one wave per row and batches of 64 rays, a row of a small mesh was a
// serial chain of batches and every batch waited for its longest ray.
// Binary walks in such batches took 404 ms for the 41,472-facet terrain
// (seed 5) and 1131 us for a 1,922-facet crater; this took 90.7 ms and
// 214 us before the node step was shortened by a third (wide.h).  It is bound
// by VALU issue (all pairs of the 41,472-facet terrain of the bench: VALUs
// 92 % busy, 57 to 60 % of the lanes active).
template <typename T>
struct PairSource {
  const T *P, *N;
  const int64_t *I, *J;
  int64_t n, W, tile_words, tiles_per_row;
  T eps;
  int mode;
  uint64_t *mask;
  TileWalk tiles;
  int2 *queue;
  // wave state
  int64_t p, w, wend;
  int count, lane;
  bool exhausted;
  T Pi[3], Ni[3];
  int i_row;
  // the lane's ray
  int lp, lq;

  __device__ __forceinline__ bool drained() const { return exhausted && count == 0; }

  __device__ __forceinline__ bool next_tile(const flux_scene &S) {
    const int64_t tile = tiles.next();
    if (tile >= tiles.ntiles) return false;
    p = tile / tiles_per_row;
    w = (tile - p * tiles_per_row) * tile_words;
    wend = min(W, w + tile_words);
    const int64_t i64 = I[p];
    i_row = i64 >= 0 && i64 < S.nf ? (int)i64 : -1;
    const int64_t i = i_row < 0 ? 0 : i_row;
    for (int c = 0; c < 3; ++c) {
      Pi[c] = P[i * 3 + c];
      Ni[c] = N[i * 3 + c];
    }
    if (i_row < 0) w = wend;
    return true;
  }

  // Queue the candidates of the next word; false when no tiles are left.
  __device__ __forceinline__ bool push_word(const flux_scene &S) {
    while (w >= wend) {
      if (!next_tile(S)) {
        exhausted = true;
        return false;
      }
    }
    const int64_t q = w * 64 + lane;
    ++w;
    bool cand = false;
    if (q < n) {
      const int64_t j = J[q];
      if (j >= 0 && j < S.nf && j != i_row) {
        const T Pj[3] = {P[j * 3], P[j * 3 + 1], P[j * 3 + 2]};
        const T Nj[3] = {N[j * 3], N[j * 3 + 1], N[j * 3 + 2]};
        cand = ff_prefilter(Pi, Ni, Pj, Nj) > eps;
      }
    }
    const uint64_t bal = __ballot(cand);
    if (cand) queue[count + lane_rank(bal)] = make_int2((int)p, (int)q);
    count += __popcll(bal);
    return true;
  }

  __device__ __forceinline__ void emit(int a, int b) {
    atomicOr((unsigned long long *)&mask[(int64_t)a * W + (b >> 6)], 1ull << (b & 63));
  }

  __device__ __forceinline__ bool refill(const flux_scene &S, LaneRay &L) {
    if (L.cur == kLaneVisible) emit(lp, lq);
    if (L.cur <= kLaneDone) L.cur = kLaneIdle;
    const uint64_t idle = __ballot(L.cur == kLaneIdle);
    const int want = __popcll(idle);
    while (count < want && push_word(S)) {
    }
    wave_lds_order();
    const int take = min(count, want), rank = lane_rank(idle);
    if (L.cur == kLaneIdle && rank < take) {
      const int2 e = queue[count - 1 - rank];
      lp = e.x;
      lq = e.y;
      const int64_t i = I[lp], j = J[lq];
      const T a[3] = {P[i * 3], P[i * 3 + 1], P[i * 3 + 2]};
      const T b[3] = {P[j * 3], P[j * 3 + 1], P[j * 3 + 2]};
      pair_begin(S, L, (int)i, (int)j, mode, a, b);
    }
    wave_lds_order();
    count -= take;
    return __ballot(L.cur > kLaneIdle) != 0 || !drained();
  }

  __device__ __forceinline__ void leaf(const flux_scene &S, LaneRay &L, const int *stk) {
    lane_leaf(S, L, stk);
  }
};

template <typename T>
__global__ void __launch_bounds__(256, 5) k_ff_mask_rays(
    flux_scene S, const T *__restrict__ P, const T *__restrict__ N,
    const int64_t *__restrict__ I, int64_t m, const int64_t *__restrict__ J, int64_t n, T eps,
    int mode, uint64_t *__restrict__ mask, int64_t W, int64_t tile_words,
    int64_t tiles_per_row, unsigned long long *__restrict__ counter) {
  __shared__ int stack[4][kStackRows][64];
  __shared__ int2 queue[4][kPairQueue];
  const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
  PairSource<T> src;
  src.P = P;
  src.N = N;
  src.I = I;
  src.J = J;
  src.n = n;
  src.W = W;
  src.tile_words = tile_words;
  src.tiles_per_row = tiles_per_row;
  src.eps = eps;
  src.mode = mode;
  src.mask = mask;
  src.tiles.init(m * tiles_per_row, counter);
  src.queue = queue[wv];
  src.p = src.w = src.wend = 0;
  src.count = 0;
  src.lane = lane;
  src.exhausted = false;
  src.lp = src.lq = 0;
  trace_wave<false>(S, src, &stack[wv][0][lane]);
}

// The same for all pairs of one list of n facets in CGAL mode, where the
// rays i -> j and j -> i run along one line: one walk decides both unless
// rounding may (wide.h), so the pairs s < t are walked once.  The list is
// taken in Morton order of the facets (I == NULL: facet ids) or in its own
// order (cluster order elsewhere).  41,472-facet terrain, assembled with a
// walk per direction 131 ms, with one 65.5, with the shorter node step 48.8;
// a 1,922-facet crater, whose waves have about one batch of rays each, 407,
// 412 and 352 us.  Bound by VALU issue like the above (94 to 95 % busy, 60 %
// of the lanes; 0.97 L1 accesses a clock).
template <typename T>
struct BothSource {
  const T *P, *N;
  const int64_t *I;
  int64_t n, W, tile_words, tiles_per_row;
  T eps;
  uint64_t *mask;
  TileWalk tiles;
  int2 *queue;
  int64_t s, w, wend;
  int count, lane;
  bool exhausted;
  T Pi[3], Ni[3];
  int i_row, p_row;
  int lp, lq;

  __device__ __forceinline__ bool drained() const { return exhausted && count == 0; }

  // position and facet of place k of the walking order
  __device__ __forceinline__ int place(const flux_scene &S, int64_t k) const {
    return I ? (int)k : S.order[k];
  }
  __device__ __forceinline__ int facet(const flux_scene &S, int pos) const {
    if (!I) return pos;
    const int64_t i = I[pos];
    return i >= 0 && i < S.nf ? (int)i : -1;
  }

  __device__ __forceinline__ bool next_tile(const flux_scene &S) {
    const int64_t tile = tiles.next();
    if (tile >= tiles.ntiles) return false;
    s = tile / tiles_per_row;
    w = (tile - s * tiles_per_row) * tile_words;
    wend = min(W, w + tile_words);
    w = max(w, (s + 1) >> 6);
    p_row = place(S, s);
    i_row = facet(S, p_row);
    const int64_t i = i_row < 0 ? 0 : i_row;
    for (int c = 0; c < 3; ++c) {
      Pi[c] = P[i * 3 + c];
      Ni[c] = N[i * 3 + c];
    }
    if (i_row < 0) w = wend;
    return true;
  }

  __device__ __forceinline__ bool push_word(const flux_scene &S) {
    while (w >= wend) {
      if (!next_tile(S)) {
        exhausted = true;
        return false;
      }
    }
    const int64_t t = w * 64 + lane;
    ++w;
    bool fwd = false, rev = false;
    int q = 0;
    if (t > s && t < n) {
      q = place(S, t);
      const int64_t j = facet(S, q);
      if (j >= 0 && j != i_row) {
        const T Pj[3] = {P[j * 3], P[j * 3 + 1], P[j * 3 + 2]};
        const T Nj[3] = {N[j * 3], N[j * 3 + 1], N[j * 3 + 2]};
        fwd = ff_prefilter(Pi, Ni, Pj, Nj) > eps;
        rev = ff_prefilter(Pj, Nj, Pi, Ni) > eps;
      }
    }
    const uint64_t bal = __ballot(fwd || rev);
    // bit 30: both directions need a ray; else the pair is stored the way
    // round that does
    if (fwd || rev)
      queue[count + lane_rank(bal)] =
          fwd ? make_int2(p_row | (rev ? 1 << 30 : 0), q) : make_int2(q, p_row);
    count += __popcll(bal);
    return true;
  }

  __device__ __forceinline__ void emit(int a, int b) {
    atomicOr((unsigned long long *)&mask[(int64_t)a * W + (b >> 6)], 1ull << (b & 63));
  }

  __device__ __forceinline__ bool refill(const flux_scene &S, LaneRay &L) {
    bool start = false, both = false;
    if (L.cur == kLaneVisible || L.cur == kLaneBlocked) {
      if (L.cur == kLaneVisible) {
        emit(lp, lq);
        if ((L.flags & (kFlagPair | kFlagReverse)) == kFlagPair) emit(lq, lp);
      }
      if (L.flags & kFlagReverse) {
        const int a = lp;
        lp = lq;
        lq = a;
        start = true;
      }
    }
    if (L.cur <= kLaneDone) L.cur = kLaneIdle;
    const bool free_lane = L.cur == kLaneIdle && !start;
    const uint64_t idle = __ballot(free_lane);
    const int want = __popcll(idle);
    while (count < want && push_word(S)) {
    }
    wave_lds_order();
    const int take = min(count, want), rank = lane_rank(idle);
    if (free_lane && rank < take) {
      const int2 e = queue[count - 1 - rank];
      lp = e.x & ~(1 << 30);
      lq = e.y;
      both = (e.x >> 30) & 1;
      start = true;
    }
    if (start) both_begin(S, L, facet(S, lp), facet(S, lq), both);
    wave_lds_order();
    count -= take;
    return __ballot(L.cur > kLaneIdle) != 0 || !drained();
  }

  __device__ __forceinline__ void leaf(const flux_scene &S, LaneRay &L, const int *stk) {
    both_leaf(S, L, stk);
  }
};

template <typename T>
__global__ void __launch_bounds__(256, 5) k_ff_mask_both(
    flux_scene S, const T *__restrict__ P, const T *__restrict__ N,
    const int64_t *__restrict__ I, int64_t n, T eps, uint64_t *__restrict__ mask, int64_t W,
    int64_t tile_words, int64_t tiles_per_row, unsigned long long *__restrict__ counter) {
  __shared__ int stack[4][kStackRows][64];
  __shared__ int2 queue[4][kPairQueue];
  const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
  BothSource<T> src;
  src.P = P;
  src.N = N;
  src.I = I;
  src.n = n;
  src.W = W;
  src.tile_words = tile_words;
  src.tiles_per_row = tiles_per_row;
  src.eps = eps;
  src.mask = mask;
  src.tiles.init(n * tiles_per_row, counter);
  src.queue = queue[wv];
  src.s = src.w = src.wend = 0;
  src.count = 0;
  src.lane = lane;
  src.exhausted = false;
  src.lp = src.lq = 0;
  trace_wave<false>(S, src, &stack[wv][0][lane]);
}

// mask and the tile counter set to zero (no memset: callers may capture)
__global__ void k_mask_clear(uint64_t *__restrict__ mask, int64_t words,
                             unsigned long long *__restrict__ counter) {
  const int64_t step = (int64_t)gridDim.x * blockDim.x;
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < words; k += step)
    mask[k] = 0ull;
  if (blockIdx.x == 0 && threadIdx.x == 0) *counter = 0ull;
}

// row_nnz[p] = popcount of mask row p; one wave per row.
__global__ void k_row_count(const uint64_t *__restrict__ mask, int64_t m, int64_t W,
                            int64_t *__restrict__ row_nnz) {
  const int64_t p = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const int lane = threadIdx.x & 63;
  if (p >= m) return;
  int64_t c = 0;
  for (int64_t w = lane; w < W; w += 64) c += __popcll(mask[p * W + w]);
  for (int off = 32; off > 0; off >>= 1) c += __shfl_down(c, off, 64);
  if (lane == 0) row_nnz[p] = c;
}

// Exclusive scan of 256 values held one per thread; returns the prefix and
// sets *total.  Uses a 256-entry LDS buffer.
__device__ inline int64_t block_exscan256(int64_t v, int64_t *buf, int64_t *total) {
  const int t = threadIdx.x;
  buf[t] = v;
  __syncthreads();
  for (int off = 1; off < 256; off <<= 1) {
    int64_t a = t >= off ? buf[t - off] : 0;
    __syncthreads();
    buf[t] += a;
    __syncthreads();
  }
  int64_t incl = buf[t];
  *total = buf[255];
  __syncthreads();
  return incl - v;
}

// One 256-thread block per row: CSR columns in ascending order.
template <typename T>
__global__ void __launch_bounds__(256) k_ff_fill(const T *__restrict__ P,
                                                 const T *__restrict__ N,
                                                 const T *__restrict__ A,
                                                 const int64_t *__restrict__ I,
                                                 const int64_t *__restrict__ J, int64_t n,
                                                 const uint64_t *__restrict__ mask, int64_t W,
                                                 const int64_t *__restrict__ indptr,
                                                 int32_t *__restrict__ indices,
                                                 T *__restrict__ data) {
  __shared__ int64_t buf[256];
  const int64_t p = blockIdx.x;
  const int i = (int)I[p];
  T Pi[3] = {P[i * 3], P[i * 3 + 1], P[i * 3 + 2]};
  T Ni[3] = {N[i * 3], N[i * 3 + 1], N[i * 3 + 2]};
  int64_t running = indptr[p];
  for (int64_t w0 = 0; w0 < W; w0 += 256) {
    const int64_t w = w0 + threadIdx.x;
    uint64_t word = w < W ? mask[p * W + w] : 0ull;
    int64_t total;
    int64_t off = block_exscan256((int64_t)__popcll(word), buf, &total);
    int64_t pos = running + off;
    while (word) {
      const int b = __ffsll((unsigned long long)word) - 1;
      word &= word - 1;
      const int64_t q = w * 64 + b;
      const int j = (int)J[q];
      T Pj[3] = {P[(int64_t)j * 3], P[(int64_t)j * 3 + 1], P[(int64_t)j * 3 + 2]};
      T Nj[3] = {N[(int64_t)j * 3], N[(int64_t)j * 3 + 1], N[(int64_t)j * 3 + 2]};
      T c = ff_prefilter(Pi, Ni, Pj, Nj);
      indices[pos] = (int32_t)q;
      data[pos] = ff_value(c, Pi, Pj, A[j]);
      ++pos;
    }
    running += total;
  }
}

__global__ void k_scan_i64(const int64_t *__restrict__ in, int64_t n, int64_t *__restrict__ out) {
  __shared__ int64_t buf[256];
  int64_t carry = 0;
  for (int64_t base = 0; base < n; base += 256) {
    const int64_t k = base + threadIdx.x;
    int64_t v = k < n ? in[k] : 0;
    int64_t total;
    int64_t ex = block_exscan256(v, buf, &total);
    if (k < n) out[k] = carry + ex;
    carry += total;
  }
  if (threadIdx.x == 0) out[n] = carry;
}

template <typename T>
__global__ void k_geometry(const T *__restrict__ V, const int64_t *__restrict__ F, int64_t nf,
                           T *__restrict__ P, T *__restrict__ N, T *__restrict__ A) {
  const int64_t f = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (f >= nf) return;
  const int64_t a = F[f * 3], b = F[f * 3 + 1], c = F[f * 3 + 2];
  T v0[3], v1[3], v2[3];
  for (int k = 0; k < 3; ++k) {
    v0[k] = V[a * 3 + k];
    v1[k] = V[b * 3 + k];
    v2[k] = V[c * 3 + k];
  }
  if (P)
    for (int k = 0; k < 3; ++k) P[f * 3 + k] = ((v0[k] + v1[k]) + v2[k]) / (T)3;
  T e1[3] = {v1[0] - v0[0], v1[1] - v0[1], v1[2] - v0[2]};
  T e2[3] = {v2[0] - v0[0], v2[1] - v0[1], v2[2] - v0[2]};
  T C[3] = {e1[1] * e2[2] - e1[2] * e2[1], e1[2] * e2[0] - e1[0] * e2[2],
            e1[0] * e2[1] - e1[1] * e2[0]};
  T cn = sqrt((C[0] * C[0] + C[1] * C[1]) + C[2] * C[2]);
  if (N)
    for (int k = 0; k < 3; ++k) N[f * 3 + k] = C[k] / cn;
  if (A) A[f] = cn / (T)2;
}

}  // namespace flux

using namespace flux;

extern "C" int flux_ff_mask(const flux_scene *scene, const void *P, const void *N, int dtype,
                            const int64_t *I, int64_t m, const int64_t *J, int64_t n,
                            double eps, int mode, uint64_t *mask, int64_t *row_nnz,
                            void *stream) {
  FLUX_CHECK(scene != nullptr, "flux_ff_mask: NULL scene");
  FLUX_CHECK(m >= 0 && n >= 0, "flux_ff_mask: negative sizes");
  FLUX_CHECK(dtype == FLUX_F32 || dtype == FLUX_F64, "flux_ff_mask: dtype must be F32/F64");
  FLUX_CHECK(mode == FLUX_MODE_CGAL || mode == FLUX_MODE_EMBREE, "flux_ff_mask: bad mode");
  FLUX_CHECK(n < ((int64_t)1 << 31), "flux_ff_mask: n too large for int32 columns");
  if (m == 0) return 0;
  FLUX_CHECK(P && N && I && mask && row_nnz && (n == 0 || J), "flux_ff_mask: NULL array");
  hipStream_t st = as_stream(stream);
  const int64_t W = (n + 63) / 64;
  if (W > 0) {
    FLUX_CHECK(m < ((int64_t)1 << 31), "flux_ff_mask: m too large for int32 rows");
    // row_nnz[0] is the tile counter until k_row_count writes it
    const int64_t tw = tile_width(m * W);
    const int64_t tpr = (W + tw - 1) / tw;
    unsigned long long *counter = (unsigned long long *)row_nnz;
    hipLaunchKernelGGL(k_mask_clear, dim3(grid_1d(m * W, 1024)), dim3(256), 0, st, mask, m * W,
                       counter);
    if (tw < 64) counter = nullptr;
    const unsigned blocks = trace_groups(m * tpr);
    if (dtype == FLUX_F64)
      hipLaunchKernelGGL(k_ff_mask_rays<double>, dim3(blocks), dim3(256), 0, st, *scene,
                         (const double *)P, (const double *)N, I, m, J, n, (double)eps, mode,
                         mask, W, tw, tpr, counter);
    else
      hipLaunchKernelGGL(k_ff_mask_rays<float>, dim3(blocks), dim3(256), 0, st, *scene,
                         (const float *)P, (const float *)N, I, m, J, n, (float)eps, mode,
                         mask, W, tw, tpr, counter);
    FLUX_LAUNCH_CHECK();
  }
  hipLaunchKernelGGL(k_row_count, dim3(ceil_div_u(m, 4)), dim3(256), 0, st, mask, m, W,
                     row_nnz);
  FLUX_LAUNCH_CHECK();
  return 0;
}

extern "C" int flux_ff_mask_square(const flux_scene *scene, const void *P, const void *N,
                                   int dtype, const int64_t *I, int64_t n, double eps,
                                   uint64_t *mask, int64_t *row_nnz, void *stream) {
  FLUX_CHECK(scene != nullptr, "flux_ff_mask_square: NULL scene");
  FLUX_CHECK(n >= 0, "flux_ff_mask_square: negative size");
  FLUX_CHECK(dtype == FLUX_F32 || dtype == FLUX_F64, "flux_ff_mask_square: dtype must be F32/F64");
  FLUX_CHECK(n < ((int64_t)1 << 30), "flux_ff_mask_square: n too large");
  FLUX_CHECK(I || n == scene->nf, "flux_ff_mask_square: without I, n must be the facet count");
  if (n == 0) return 0;
  FLUX_CHECK(P && N && mask && row_nnz, "flux_ff_mask_square: NULL array");
  hipStream_t st = as_stream(stream);
  const int64_t W = (n + 63) / 64;
  const int64_t tw = tile_width(n * W / 2);
  const int64_t tpr = (W + tw - 1) / tw;
  unsigned long long *counter = (unsigned long long *)row_nnz;
  hipLaunchKernelGGL(k_mask_clear, dim3(grid_1d(n * W, 1024)), dim3(256), 0, st, mask, n * W,
                     counter);
  if (tw < 64) counter = nullptr;
  const unsigned blocks = trace_groups(n * tpr);
  if (dtype == FLUX_F64)
    hipLaunchKernelGGL(k_ff_mask_both<double>, dim3(blocks), dim3(256), 0, st, *scene,
                       (const double *)P, (const double *)N, I, n, (double)eps, mask, W, tw, tpr,
                       counter);
  else
    hipLaunchKernelGGL(k_ff_mask_both<float>, dim3(blocks), dim3(256), 0, st, *scene,
                       (const float *)P, (const float *)N, I, n, (float)eps, mask, W, tw, tpr,
                       counter);
  FLUX_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_row_count, dim3(ceil_div_u(n, 4)), dim3(256), 0, st, mask, n, W, row_nnz);
  FLUX_LAUNCH_CHECK();
  return 0;
}

extern "C" int flux_ff_candidates(const flux_scene *scene, const void *P, const void *N,
                                  int dtype, const int64_t *I, int64_t m, const int64_t *J,
                                  int64_t n, double eps, uint64_t *mask, int64_t *row_cnt,
                                  void *stream) {
  FLUX_CHECK(scene != nullptr, "flux_ff_candidates: NULL scene");
  FLUX_CHECK(m >= 0 && n >= 0, "flux_ff_candidates: negative sizes");
  FLUX_CHECK(dtype == FLUX_F32 || dtype == FLUX_F64, "flux_ff_candidates: dtype");
  if (m == 0) return 0;
  FLUX_CHECK(P && N && I && mask && row_cnt && (n == 0 || J), "flux_ff_candidates: NULL array");
  hipStream_t st = as_stream(stream);
  const int64_t W = (n + 63) / 64;
  if (W > 0) {
    const unsigned blocks = (unsigned)std::min<int64_t>((m * W + 3) / 4, 1 << 20);
    if (dtype == FLUX_F64)
      hipLaunchKernelGGL(k_ff_candidates<double>, dim3(blocks), dim3(256), 0, st, scene->nf,
                         (const double *)P, (const double *)N, I, m, J, n, (double)eps, mask, W);
    else
      hipLaunchKernelGGL(k_ff_candidates<float>, dim3(blocks), dim3(256), 0, st, scene->nf,
                         (const float *)P, (const float *)N, I, m, J, n, (float)eps, mask, W);
    FLUX_LAUNCH_CHECK();
  }
  hipLaunchKernelGGL(k_row_count, dim3(ceil_div_u(m, 4)), dim3(256), 0, st, mask, m, W,
                     row_cnt);
  FLUX_LAUNCH_CHECK();
  return 0;
}

extern "C" int flux_ff_fill(const void *P, const void *N, const void *A, int dtype,
                            const int64_t *I, int64_t m, const int64_t *J, int64_t n,
                            const uint64_t *mask, const int64_t *indptr, int32_t *indices,
                            void *data, void *stream) {
  FLUX_CHECK(m >= 0 && n >= 0, "flux_ff_fill: negative sizes");
  FLUX_CHECK(dtype == FLUX_F32 || dtype == FLUX_F64, "flux_ff_fill: dtype must be F32/F64");
  if (m == 0 || n == 0) return 0;
  FLUX_CHECK(P && N && A && I && J && mask && indptr, "flux_ff_fill: NULL array");
  const int64_t W = (n + 63) / 64;
  FLUX_CHECK(m < ((int64_t)1 << 31), "flux_ff_fill: m too large");
  hipStream_t st = as_stream(stream);
  if (dtype == FLUX_F64)
    hipLaunchKernelGGL(k_ff_fill<double>, dim3((unsigned)m), dim3(256), 0, st,
                       (const double *)P, (const double *)N, (const double *)A, I, J, n, mask,
                       W, indptr, indices, (double *)data);
  else
    hipLaunchKernelGGL(k_ff_fill<float>, dim3((unsigned)m), dim3(256), 0, st,
                       (const float *)P, (const float *)N, (const float *)A, I, J, n, mask, W,
                       indptr, indices, (float *)data);
  FLUX_LAUNCH_CHECK();
  return 0;
}

extern "C" int flux_scan_i64(const int64_t *in, int64_t n, int64_t *out, int64_t *total_host,
                             void *stream) {
  FLUX_CHECK(n >= 0 && out != nullptr && (n == 0 || in != nullptr), "flux_scan_i64: bad args");
  hipStream_t st = as_stream(stream);
  hipLaunchKernelGGL(k_scan_i64, dim3(1), dim3(256), 0, st, in, n, out);
  FLUX_LAUNCH_CHECK();
  if (total_host) {
    FLUX_TRY_HIP(hipMemcpyAsync(total_host, out + n, sizeof(int64_t), hipMemcpyDeviceToHost, st));
    FLUX_TRY_HIP(hipStreamSynchronize(st));
  }
  return 0;
}

extern "C" int flux_geometry(const void *V, int64_t nv, const int64_t *F, int64_t nf,
                             int dtype, void *P, void *N, void *A, void *stream) {
  FLUX_CHECK(nv >= 0 && nf >= 0, "flux_geometry: negative sizes");
  FLUX_CHECK(dtype == FLUX_F32 || dtype == FLUX_F64, "flux_geometry: dtype must be F32/F64");
  if (nf == 0) return 0;
  FLUX_CHECK(V && F, "flux_geometry: NULL V or F");
  const int TB = 256;
  hipStream_t st = as_stream(stream);
  if (dtype == FLUX_F64)
    hipLaunchKernelGGL(k_geometry<double>, dim3(ceil_div_u(nf, TB)), dim3(TB), 0, st,
                       (const double *)V, F, nf, (double *)P, (double *)N, (double *)A);
  else
    hipLaunchKernelGGL(k_geometry<float>, dim3(ceil_div_u(nf, TB)), dim3(TB), 0, st,
                       (const float *)V, F, nf, (float *)P, (float *)N, (float *)A);
  FLUX_LAUNCH_CHECK();
  return 0;
}
