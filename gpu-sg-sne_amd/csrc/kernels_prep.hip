// kernels_prep.hip -- construction of P on the GPU: exact kNN, perplexity
// bisection, lambda rescaling, P + P^T, and the COO / hybrid format builds.
//
// Reference (CU = code/cuda/SG-tSNE-CUDA/src, HY = code/cuda/SG-tSNE-HYB/sgtsnepi/src):
//   kNN            CU/allknn.cuh:75-92 (FLANN, approximate; exact here)
//   perplexity     HY/sgtsne.cpp:201-254 (FP64 twin of CU/perplexity_search.cu:18-208)
//   lambda         HY/graph_rescaling.cpp:19-104 (CU/graph_rescaling.cu:11-107)
//   P + P^T        CU/graph_rescaling.cu:266-398, HY/sparsematrix.cpp:69-164,
//                  normalised to sum 1 as HY/sgtsne.cpp:78-85
//   COO rows       CU/prepareMatrix.cu:2-27
//   hybrid         CU/prepareMatrix.cu:56-97, CU/matrix_converter.cpp:106-248
#include "common.hpp"
#include "kernels.hpp"
#include "../../include/sgtsne.h"

#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <climits>
#include <vector>

namespace sgt {

namespace {

// ---- exact kNN -----------------------------------------------------------
// Two kernels over a slab of query slots [0, nq) (slot s is point qlist[s],
// point s without a list): the FP64 distances of every (slot, point) pair,
// then per slot the k smallest (distance, index) keys.
//
// Points stay FP32 on the device; every kernel widens them as it reads them, which
// is exact.
//
// Distances: a 256-thread work-group owns a tile of 16 RQ queries x 16 RR
// references, each thread an RQ x RR micro-tile whose sums run over the
// dimensions in order, acc = fma(diff, diff, acc) (zero-padded dimensions add
// an exact 0), with 16 dimensions of the tile staged in LDS and the next 16 in
// flight.  Bound by FP64 vector issue, two operations per pair and dimension.
// The squared difference does not depend on which point is subtracted from
// which, so when the slab holds every point in order the tiles below the
// diagonal are not computed: tile (a, b) also writes (b, a).
constexpr int kKnnDC = 16;  // dimensions staged per round
constexpr int kKnnThreads = 256;
constexpr int kKnnMaxK = 2048;

template <int RQ, int RR>
__global__ __launch_bounds__(kKnnThreads) void knn_dist_kernel(const float *__restrict__ X, int n, int dim,
                                                               const int *__restrict__ qlist, int s0, int nq,
                                                               int mirror, double *__restrict__ dist) {
  constexpr int TQ = 16 * RQ, TR = 16 * RR;
  constexpr int LQ = TQ * kKnnDC / kKnnThreads, LR = TR * kKnnDC / kKnnThreads;
  static_assert(RQ % 2 == 0 && RR % 2 == 0 && LQ >= 1 && LR >= 1, "micro-tiles of pairs");
  if (mirror && (int)blockIdx.x < (int)blockIdx.y) return;  // square tiles: the mirrored one writes it
  __shared__ double2 qs2[kKnnDC][TQ / 2 + 1], rs2[kKnnDC][TR / 2 + 1];
  double *qs = reinterpret_cast<double *>(qs2), *rs = reinterpret_cast<double *>(rs2);
  constexpr int SQ = TQ + 2, SR = TR + 2;  // doubles per staged dimension
  const int q0 = blockIdx.y * TQ, r0 = blockIdx.x * TR;
  const int tid = threadIdx.x;
  const int tq = tid >> 4, tr = tid & 15;  // queries 2 tq + 32 a, references 2 tr + 32 b (and the next)
  // this thread's share of a staged round: dimension tid % 16 of rows tid / 16 + 16 u
  const int ll = tid & 15;
  const float *qp[LQ], *rp[LR];
#pragma unroll
  for (int u = 0; u < LQ; ++u) {
    const int sl = q0 + (tid >> 4) + 16 * u;
    const int q = sl < nq ? (qlist ? qlist[s0 + sl] : s0 + sl) : -1;
    qp[u] = q >= 0 ? X + (size_t)q * dim : nullptr;
  }
#pragma unroll
  for (int u = 0; u < LR; ++u) {
    const int r = r0 + (tid >> 4) + 16 * u;
    rp[u] = r < n ? X + (size_t)r * dim : nullptr;
  }
  float qb[LQ], rb[LR];
  auto load = [&](int l0) {
    const int l = l0 + ll;
#pragma unroll
    for (int u = 0; u < LQ; ++u) qb[u] = (qp[u] && l < dim) ? qp[u][l] : 0.0f;
#pragma unroll
    for (int u = 0; u < LR; ++u) rb[u] = (rp[u] && l < dim) ? rp[u][l] : 0.0f;
  };
  double acc[RQ][RR];
#pragma unroll
  for (int a = 0; a < RQ; ++a)
#pragma unroll
    for (int b = 0; b < RR; ++b) acc[a][b] = 0.0;
  load(0);
  for (int l0 = 0; l0 < dim; l0 += kKnnDC) {
    __syncthreads();
#pragma unroll
    for (int u = 0; u < LQ; ++u) qs[ll * SQ + (tid >> 4) + 16 * u] = qb[u];
#pragma unroll
    for (int u = 0; u < LR; ++u) rs[ll * SR + (tid >> 4) + 16 * u] = rb[u];
    __syncthreads();
    if (l0 + kKnnDC < dim) load(l0 + kKnnDC);
#pragma unroll 2
    for (int d = 0; d < kKnnDC; ++d) {
      double qv[RQ], rv[RR];
#pragma unroll
      for (int a = 0; a < RQ; a += 2) {
        const double2 v = qs2[d][tq + 8 * a];
        qv[a] = v.x;
        qv[a + 1] = v.y;
      }
#pragma unroll
      for (int b = 0; b < RR; b += 2) {
        const double2 v = rs2[d][tr + 8 * b];
        rv[b] = v.x;
        rv[b + 1] = v.y;
      }
#pragma unroll
      for (int a = 0; a < RQ; ++a)
#pragma unroll
        for (int b = 0; b < RR; ++b) {
          const double df = qv[a] - rv[b];
          acc[a][b] = fma(df, df, acc[a][b]);
        }
    }
  }
#pragma unroll
  for (int a = 0; a < RQ; ++a) {
    const int sl = q0 + 2 * tq + 16 * (a & ~1) + (a & 1);
#pragma unroll
    for (int b = 0; b < RR; ++b) {
      const int r = r0 + 2 * tr + 16 * (b & ~1) + (b & 1);
      if (sl < nq && r < n) {
        dist[(size_t)sl * n + r] = acc[a][b];
        if (mirror) dist[(size_t)r * n + sl] = acc[a][b];
      }
    }
  }
}

// Ascending bitonic sort of P2 (a power of two) (key, index) pairs in LDS by
// the key, then the index; every thread of the work-group calls it.
__device__ void sort_keys(unsigned long long *key, int *id, int P2) {
  for (int size = 2; size <= P2; size <<= 1)
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      __syncthreads();
      for (int t = threadIdx.x; t < P2 / 2; t += blockDim.x) {
        const int i = 2 * stride * (t / stride) + (t & (stride - 1)), j = i + stride;
        const bool up = (i & size) == 0;
        const unsigned long long a = key[i], b = key[j];
        const int ia = id[i], ib = id[j];
        const bool a_after_b = b < a || (b == a && ib < ia);
        if (a_after_b == up) {
          key[i] = b;
          key[j] = a;
          id[i] = ib;
          id[j] = ia;
        }
      }
    }
  __syncthreads();
}

// The k smallest (distance, index) keys of each slot's row of distances, in
// ascending order after the point itself; one work-group per slot.  Distances
// are non-negative, so their bits order as they do; NaN is no neighbour, and a
// row left short ends in (infinity, INT_MAX).  The row is narrowed by
// histograms of 2048 equal ranges of the key between the bounds of the k-th
// smallest, until at most CAP keys lie at or below the upper bound; those are
// sorted.  When the keys tied at the k-th smallest are too many for that, the
// ones of lowest index are taken in index order.  A row costs three passes
// over it (bounds, one histogram, collection) unless its keys crowd.
constexpr int kSelBins = 2048;

template <int CAP>
__global__ __launch_bounds__(kKnnThreads) void knn_select_kernel(const double *__restrict__ dist, int n, int k,
                                                                 const int *__restrict__ qlist, int s0,
                                                                 int32_t *__restrict__ I, double *__restrict__ D) {
  __shared__ unsigned long long key[CAP];
  __shared__ int id[CAP];
  __shared__ int hist[kSelBins];
  __shared__ unsigned long long wlo[kKnnThreads / 64], whi[kKnnThreads / 64];
  __shared__ int wcnt[kKnnThreads / 64];
  __shared__ int total, pick_bin, pick_below;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int q = qlist ? qlist[s0 + blockIdx.x] : s0 + (int)blockIdx.x;
  const unsigned long long *row = reinterpret_cast<const unsigned long long *>(dist) + (size_t)blockIdx.x * n;
  constexpr unsigned long long kInf = 0x7FF0000000000000ull;
  // bounds and count of the row's keys
  unsigned long long lo = ~0ull, hi = 0;
  int cnt = 0;
  for (int r = tid; r < n; r += kKnnThreads) {
    const unsigned long long u = row[r];
    if (u <= kInf && r != q) {
      lo = u < lo ? u : lo;
      hi = u > hi ? u : hi;
      ++cnt;
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const unsigned long long a = __shfl_xor(lo, o, 64), b = __shfl_xor(hi, o, 64);
    lo = a < lo ? a : lo;
    hi = b > hi ? b : hi;
    cnt += __shfl_xor(cnt, o, 64);
  }
  if (lane == 0) {
    wlo[w] = lo;
    whi[w] = hi;
    wcnt[w] = cnt;
  }
  if (tid == 0) total = 0;
  __syncthreads();
  cnt = 0;
#pragma unroll
  for (int v = 0; v < kKnnThreads / 64; ++v) {
    lo = wlo[v] < lo ? wlo[v] : lo;
    hi = whi[v] > hi ? whi[v] : hi;
    cnt += wcnt[v];
  }
  // narrow [lo, hi] around the k-th smallest key; `below` keys lie under lo
  int below = 0, ties = 0;  // ties > 0: that many keys equal to hi, lowest indices first
  if (cnt > CAP)
    for (;;) {
      const unsigned long long range = hi - lo;
      const int bits = 64 - __clzll((long long)(range | 1ull));
      const int shift = bits > 11 ? bits - 11 : 0;
      for (int b = tid; b < kSelBins; b += kKnnThreads) hist[b] = 0;
      __syncthreads();
      for (int r = tid; r < n; r += kKnnThreads) {
        const unsigned long long u = row[r];
        if (u >= lo && u <= hi && u <= kInf && r != q) atomicAdd(&hist[(int)((u - lo) >> shift)], 1);
      }
      __syncthreads();
      if (w == 0) {  // the first bin whose running total reaches k: 32 bins per lane
        int sum = 0;
        for (int b = 0; b < kSelBins / 64; ++b) sum += hist[lane * (kSelBins / 64) + b];
        int pre = sum;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
          const int v = __shfl_up(pre, o, 64);
          if (lane >= o) pre += v;
        }
        const int before = below + pre - sum;
        const unsigned long long reach = __ballot(before + sum >= k);
        if (lane == __ffsll((long long)reach) - 1) {
          int run = before, b = lane * (kSelBins / 64);
          while (run + hist[b] < k) run += hist[b++];
          pick_bin = b;
          pick_below = run;
        }
      }
      __syncthreads();
      const int b = pick_bin, upto = pick_below + hist[b];
      below = pick_below;
      lo += (unsigned long long)b << shift;
      hi = lo + ((1ull << shift) - 1);
      __syncthreads();  // pick_bin and hist are rewritten by the next round
      if (upto <= CAP) break;
      if (shift == 0) {
        ties = k - below;
        break;
      }
    }
  // collect: every key at or below hi, or those under hi and the first ties
  for (int r = tid; r < n; r += kKnnThreads) {
    const unsigned long long u = row[r];
    if (u <= kInf && r != q && (ties ? u < hi : (u <= hi))) {
      const int pos = atomicAdd(&total, 1);
      key[pos] = u;
      id[pos] = r;
    }
  }
  __syncthreads();
  if (ties && w == 0) {
    int have = total;
    for (int r = 0; r < n && have < k; r += 64) {
      const bool eq = r + lane < n && r + lane != q && row[r + lane] == hi;
      const unsigned long long m = __ballot(eq);
      const int pos = have + __popcll(m & ((1ull << lane) - 1ull));
      if (eq && pos < k) {
        key[pos] = hi;
        id[pos] = r + lane;
      }
      have += __popcll(m);
    }
    if (lane == 0) total = have < k ? have : k;
  }
  __syncthreads();
  const int m = total;
  int P2 = 2;
  while (P2 < m) P2 <<= 1;
  for (int t = m + tid; t < P2; t += kKnnThreads) {
    key[t] = ~0ull;
    id[t] = INT_MAX;
  }
  sort_keys(key, id, P2);
  int32_t *Iq = I + (size_t)q * (k + 1);
  double *Dq = D + (size_t)q * (k + 1);
  if (tid == 0) {
    Iq[0] = q;
    Dq[0] = 0.0;
  }
  for (int t = tid; t < k; t += kKnnThreads) {
    Iq[1 + t] = t < m ? id[t] : INT_MAX;
    Dq[1 + t] = t < m ? __longlong_as_double((long long)key[t]) : (double)INFINITY;
  }
}

// ---- exact kNN without a block of distances ---------------------------------
// Work-group tile: 64 queries x 32 references; 256 threads each own a 4x2
// micro-tile of (query, reference) distances, summed as in knn_dist_kernel.
// Candidates below a query's current worst key (distance, index) are queued in
// LDS and merged by one thread per query into a max-heap of k entries kept in
// global memory.  No distance is stored, so the cost per pair does not grow with n
// (200,000 points of 5 dimensions, k = 10: 1.9 ps).  Queries are the slots
// [s0, s0 + nq); heaps are indexed by slot - s0.
constexpr int kHeapQ = 64;
constexpr int kHeapR = 32;

__device__ __forceinline__ bool key_less(double da, int ia, double db, int ib) {
  return da < db || (da == db && ia < ib);
}

__global__ __launch_bounds__(kKnnThreads) void knn_heap_kernel(const float *__restrict__ X, int n,
                                                          int dim, int k, double *__restrict__ hd,
                                                          int *__restrict__ hi, const int *__restrict__ qlist,
                                                          int s0, int nq) {
  __shared__ double qs[kKnnDC][kHeapQ + 1];
  __shared__ double rs[kKnnDC][kHeapR + 1];
  __shared__ double qd[kHeapQ][kHeapR];
  __shared__ int qi[kHeapQ][kHeapR];
  __shared__ int qcnt[kHeapQ];
  __shared__ double thr_d[kHeapQ];
  __shared__ int thr_i[kHeapQ];
  __shared__ int qid[kHeapQ];  // point of each slot (-1: none)

  const int q0 = blockIdx.x * kHeapQ;
  const int tid = threadIdx.x;
  const int tq = tid >> 4;   // 0..15 -> queries tq*4 .. tq*4+3
  const int tr = tid & 15;   // 0..15 -> references tr + 16*c
  if (tid < kHeapQ) {
    qcnt[tid] = 0;
    thr_d[tid] = INFINITY;
    thr_i[tid] = INT_MAX;
    const int slot = q0 + tid;
    qid[tid] = slot < nq ? (qlist ? qlist[s0 + slot] : s0 + slot) : -1;
    if (slot < nq)
      for (int e = 0; e < k; ++e) {
        hd[(size_t)slot * k + e] = INFINITY;
        hi[(size_t)slot * k + e] = INT_MAX;
      }
  }
  __syncthreads();

  for (int r0 = 0; r0 < n; r0 += kHeapR) {
    double acc[4][2];
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b) acc[a][b] = 0.0;
    for (int l0 = 0; l0 < dim; l0 += kKnnDC) {
      for (int idx = tid; idx < kKnnDC * kHeapQ; idx += kKnnThreads) {
        const int qq = idx / kKnnDC, ll = idx % kKnnDC;
        const int q = qid[qq], l = l0 + ll;
        qs[ll][qq] = (q >= 0 && l < dim) ? X[(size_t)q * dim + l] : 0.0;
        if (qq < kHeapR) {
          const int r = r0 + qq;
          rs[ll][qq] = (r < n && l < dim) ? X[(size_t)r * dim + l] : 0.0;
        }
      }
      __syncthreads();
      const int lc = min(kKnnDC, dim - l0);
      for (int ll = 0; ll < lc; ++ll) {
        double qv[4], rv[2];
#pragma unroll
        for (int a = 0; a < 4; ++a) qv[a] = qs[ll][tq * 4 + a];
#pragma unroll
        for (int b = 0; b < 2; ++b) rv[b] = rs[ll][tr + 16 * b];
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
          for (int b = 0; b < 2; ++b) {
            const double df = qv[a] - rv[b];
            acc[a][b] = fma(df, df, acc[a][b]);
          }
      }
      __syncthreads();
    }
    // queue candidates
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      const int ql = tq * 4 + a;
      const int q = qid[ql];
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const int r = r0 + tr + 16 * b;
        if (q >= 0 && r < n && r != q && key_less(acc[a][b], r, thr_d[ql], thr_i[ql])) {
          const int pos = atomicAdd(&qcnt[ql], 1);
          qd[ql][pos] = acc[a][b];
          qi[ql][pos] = r;
        }
      }
    }
    __syncthreads();
    // merge queued candidates into the heaps (one thread per query)
    if (tid < kHeapQ) {
      const int slot = q0 + tid;
      const int cnt = qcnt[tid];
      if (slot < nq && cnt > 0) {
        double *H = hd + (size_t)slot * k;
        int *HI = hi + (size_t)slot * k;
        double rd = H[0];
        int ri = HI[0];
        for (int c = 0; c < cnt; ++c) {
          const double cd = qd[tid][c];
          const int ci = qi[tid][c];
          if (!key_less(cd, ci, rd, ri)) continue;
          int pos = 0;
          for (;;) {
            const int l = 2 * pos + 1, rr = l + 1;
            int m = -1;
            double md = cd;
            int mi = ci;
            if (l < k && key_less(md, mi, H[l], HI[l])) { m = l; md = H[l]; mi = HI[l]; }
            if (rr < k && key_less(md, mi, H[rr], HI[rr])) { m = rr; md = H[rr]; mi = HI[rr]; }
            if (m < 0) break;
            H[pos] = md;
            HI[pos] = mi;
            pos = m;
          }
          H[pos] = cd;
          HI[pos] = ci;
          rd = H[0];
          ri = HI[0];
        }
        thr_d[tid] = rd;
        thr_i[tid] = ri;
      }
      qcnt[tid] = 0;
    }
    __syncthreads();
  }
}

// Heap -> ascending rows with the point itself first (slots as knn_heap_kernel).
__global__ void knn_heap_rows_kernel(int s0, int nq, int k, double *__restrict__ hd, int *__restrict__ hi,
                                     const int *__restrict__ qlist, int32_t *__restrict__ I,
                                     double *__restrict__ D) {
  const int slot = blockIdx.x * blockDim.x + threadIdx.x;
  if (slot >= nq) return;
  const int q = qlist ? qlist[s0 + slot] : s0 + slot;
  double *H = hd + (size_t)slot * k;
  int *HI = hi + (size_t)slot * k;
  int32_t *Iq = I + (size_t)q * (k + 1);
  double *Dq = D + (size_t)q * (k + 1);
  Iq[0] = q;
  Dq[0] = 0.0;
  for (int e = k - 1; e >= 0; --e) {
    Iq[1 + e] = HI[0];
    Dq[1 + e] = H[0];
    const double cd = H[e];
    const int ci = HI[e];
    int pos = 0;
    for (;;) {
      const int l = 2 * pos + 1, rr = l + 1;
      int m = -1;
      double md = cd;
      int mi = ci;
      if (l < e && key_less(md, mi, H[l], HI[l])) { m = l; md = H[l]; mi = HI[l]; }
      if (rr < e && key_less(md, mi, H[rr], HI[rr])) { m = rr; md = H[rr]; mi = HI[rr]; }
      if (m < 0) break;
      H[pos] = md;
      HI[pos] = mi;
      pos = m;
    }
    H[pos] = cd;
    HI[pos] = ci;
  }
}

// ---- kNN through an FP32 matrix-core filter --------------------------------
// The exact distances above cost two FP64 vector operations per (pair,
// dimension).  Here the squared distances of the mean-centred points, rounded
// to FP32, come from matrix-core dot products, |x|^2 + |y|^2 - 2 x.y, and each
// query keeps its k + kFiltSlack nearest candidates under that approximation.
// A rigorous bound on the approximation error then certifies, per query, that
// no point outside the candidate list can be among the exact k nearest; the
// candidates' distances are recomputed with exactly the arithmetic of
// the FP64 kernels and the k smallest (distance, index) keys are kept, so a
// certified row equals their row bit for bit.  Rows that cannot be
// certified (ties or near-ties wider than the slack) go through them.
constexpr int kFiltQ = 64;        // queries per work-group, 16 per wave
constexpr int kFiltR = 64;        // references per tile, 4 blocks of 16
constexpr int kFiltMaxDp = 128;   // padded dimensions (A operands held in registers)
constexpr int kFiltRS = 80;       // LDS row stride of the transposed tile (16 mod 32 banks)
constexpr int kFiltSlack = 16;    // candidates kept beyond k
constexpr int kRerank = 256;      // candidates the re-rank takes at most (k + slack <= 256)

typedef float fv4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ bool key_lessf(float da, int ia, float db, int ib) {
  return da < db || (da == db && ia < ib);
}

// A reference tile is kFiltR rows of NST float4.  Element t of the tile is
// row t % kFiltR, float4 column t / kFiltR: adjacent threads take adjacent
// rows, so the transposed LDS stores are conflict-free.  All of a thread's
// loads are issued before any is used.
template <int T, int NST>
__device__ __forceinline__ void tile_load(const float *__restrict__ Xc, const float *__restrict__ n32, int n, int r0,
                                          float4 (&buf)[kFiltR * NST / T], float &rnv) {
  static_assert((kFiltR * NST) % T == 0, "a tile must split evenly over the work-group");
  const float4 *X4 = reinterpret_cast<const float4 *>(Xc);
#pragma unroll
  for (int u = 0; u < kFiltR * NST / T; ++u) {
    const int t = threadIdx.x + u * T;
    const int j = t % kFiltR, c4 = t / kFiltR;
    buf[u] = r0 + j < n ? X4[(size_t)(r0 + j) * NST + c4] : make_float4(0.f, 0.f, 0.f, 0.f);
  }
  rnv = (threadIdx.x < kFiltR && r0 + (int)threadIdx.x < n) ? n32[r0 + threadIdx.x] : 0.0f;
}

// Stores a loaded tile transposed: rt[c * kFiltRS + j] = Xc[r0 + j][c].
template <int T, int NST>
__device__ __forceinline__ void tile_store(float *rt, float *rn, const float4 (&buf)[kFiltR * NST / T], float rnv) {
#pragma unroll
  for (int u = 0; u < kFiltR * NST / T; ++u) {
    const int t = threadIdx.x + u * T;
    const int j = t % kFiltR, c4 = t / kFiltR;
    float *col = rt + 4 * c4 * kFiltRS + j;
    col[0] = buf[u].x;
    col[kFiltRS] = buf[u].y;
    col[2 * kFiltRS] = buf[u].z;
    col[3 * kFiltRS] = buf[u].w;
  }
  if (threadIdx.x < kFiltR) rn[threadIdx.x] = rnv;
}

// The dot products of a wave's 16 queries with the tile's 64 references:
// acc[t][v] = x(query 16 w + 4 (lane / 16) + v) . x(reference 16 t + lane % 16).
template <int NST>
__device__ __forceinline__ void tile_dots(const float (&areg)[NST], const float *rt, int lane, fv4 (&acc)[4]) {
#pragma unroll
  for (int t = 0; t < 4; ++t) acc[t] = fv4{0.0f, 0.0f, 0.0f, 0.0f};
  // B operand of step s, block t: row (dimension) 4 s + lane / 16, column
  // (reference) 16 t + lane % 16
  const float *rrow = rt + (lane >> 4) * kFiltRS + (lane & 15);
#pragma unroll
  for (int st = 0; st < NST; ++st)
#pragma unroll
    for (int t = 0; t < 4; ++t)
      acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(areg[st], rrow[4 * st * kFiltRS + 16 * t], acc[t], 0, 0, 0);
}

// The filter's preparation.  All of it is bound by the latency of its short
// launches: rows are read by 16 lanes or more each, side by side, and a kernel
// does what can be done on the same rows at once.  With a thread per row and a
// launch per step the preparation of 20,011 points of 50 dimensions took 200 us
// (means 45, centring 24, cells 46, keys 9, counts and offsets 6, reference
// scatter 7, tile spheres 27, frames 11, queries 26), now 65 (13, 13, 18 with
// the keys, tiles 12, frames 8); of a job of 500-8000 points 105 us, now 38.
constexpr int kMeanParts = 128;

// Sums of the columns over a run of rows per work-group: part[work-group][dim].
__global__ __launch_bounds__(256) void knn_mean_kernel(const float *__restrict__ X, int n, int dim,
                                                       double *__restrict__ part) {
  __shared__ double acc[2][kFiltMaxDp];
  const int rows = (n + gridDim.x - 1) / gridDim.x, l = threadIdx.x & 127, h = threadIdx.x >> 7;
  const int r1 = min(n, (int)(blockIdx.x + 1) * rows);
  if (l < dim) {
    double a = 0.0;
#pragma unroll 4
    for (int r = blockIdx.x * rows + h; r < r1; r += 2) a += (double)X[(size_t)r * dim + l];
    acc[h][l] = a;
  }
  __syncthreads();
  if (h == 0 && l < dim) part[(size_t)blockIdx.x * dim + l] = acc[0][l] + acc[1][l];
}

// Sum of squares over the 16 lanes of a row.
__device__ __forceinline__ double row16_sum(double v) {
#pragma unroll
  for (int o = 8; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// The means from their partial sums (every work-group, the first one stores
// them), then the points centred at them in FP32 (zero-padded to dp), their
// squared norms (FP32 of the FP64 sum) and norms, and the largest norm.
constexpr int kCentreRows = 64;
__global__ __launch_bounds__(256) void knn_center_kernel(const float *__restrict__ X, int n, int dim, int dp,
                                                         const double *__restrict__ part, int nparts,
                                                         double *__restrict__ mu, float *__restrict__ Xc,
                                                         float *__restrict__ n32, double *__restrict__ nrm,
                                                         unsigned long long *__restrict__ rmax) {
  __shared__ double acc[2][kFiltMaxDp], m[kFiltMaxDp];
  __shared__ unsigned long long wmax[4];
  {
    const int l = threadIdx.x & 127, h = threadIdx.x >> 7;
    double a = 0.0;
    if (l < dim)
#pragma unroll 8
      for (int k = h; k < nparts; k += 2) a += part[(size_t)k * dim + l];
    acc[h][l] = a;
    __syncthreads();
    if (h == 0 && l < dim) {
      m[l] = (acc[0][l] + acc[1][l]) / (double)n;
      if (blockIdx.x == 0) mu[l] = m[l];
    }
    __syncthreads();
  }
  const int sub = threadIdx.x & 15;
  unsigned long long best = 0;  // norms order as their bits, a NaN above all
#pragma unroll
  for (int u = 0; u < kCentreRows / 16; ++u) {
    const int i = blockIdx.x * kCentreRows + u * 16 + (threadIdx.x >> 4);
    double ss = 0.0;
    if (i < n)
      for (int l = sub; l < dp; l += 16) {
        const float v = l < dim ? (float)((double)X[(size_t)i * dim + l] - m[l]) : 0.0f;
        Xc[(size_t)i * dp + l] = v;
        ss += (double)v * (double)v;
      }
    ss = row16_sum(ss);
    const double r = sqrt(ss);
    if (i < n && sub == 0) {
      n32[i] = (float)ss;
      nrm[i] = r;
    }
    best = max(best, (unsigned long long)__double_as_longlong(r));
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) best = max(best, (unsigned long long)__shfl_xor(best, o, 64));
  if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = best;
  __syncthreads();
  if (threadIdx.x == 0) atomicMax(rmax, max(max(wmax[0], wmax[1]), max(wmax[2], wmax[3])));
}

// ---- block-centred queries ----------------------------------------------------
// The filter's error bound grows with the size of the vectors whose dot
// product it takes, (|a| + |b|)^2, while neighbour gaps are set by local
// distances: with the points centred once globally, clusters far from the
// mean certify no row.  So queries are grouped into blocks of kF2Q that lie
// close together (in the order of a Morton code of a 3-D projection of the
// centred points), and each block is centred at its own mean c_b: the queries
// as fl32(x - c_b), the references of every tile as fl32(fl32(x - mu) -
// fl32(c_b - mu)), with their norms summed in the filter.  The certificate
// then involves only the query's distance to its block's mean.
__device__ __forceinline__ uint32_t spread_bits10(uint32_t v) {
  v &= 1023u;
  v = (v | (v << 16)) & 0x030000FFu;
  v = (v | (v << 8)) & 0x0300F00Fu;
  v = (v | (v << 4)) & 0x030C30C3u;
  v = (v | (v << 2)) & 0x09249249u;
  return v;
}

// +-1/sqrt(dim) entries of three fixed projection directions (a hash of the
// axis and the dimension), so every projection is at most the point's norm.
__device__ __forceinline__ float proj_sign(int axis, int l) {
  uint32_t h = (uint32_t)l * 2654435761u + (uint32_t)axis * 40503u + 0x9E3779B9u;
  h ^= h >> 15;
  h *= 2246822519u;
  h ^= h >> 13;
  return (h & 1u) ? 1.0f : -1.0f;
}

// Cells of the point set: the nearest of P pivots (points (p n) / P, P <= 64;
// FP32 distances of the centred points, ties to the lower pivot), so that
// points of one cluster share cells.  Used only to order the points; any
// assignment gives the same kNN rows.
constexpr int kKnnMaxCells = 64;

// Four lanes per point, each with every fourth pivot; the cells' counts too, and
// the points' sort keys: the cell, then the Morton code of the projections.
__global__ __launch_bounds__(256) void knn_cell_kernel(const float *__restrict__ Xc, int n, int dim, int dp, int P,
                                                       const unsigned long long *__restrict__ rmax,
                                                       int32_t *__restrict__ cell, int *__restrict__ cnt,
                                                       uint32_t *__restrict__ key, int32_t *__restrict__ idx) {
  extern __shared__ float piv[];  // [P][dp]
  __shared__ int hist[kKnnMaxCells];
  for (int t = threadIdx.x; t < P * dp; t += blockDim.x) {
    const int p = t / dp, l = t - p * dp;
    piv[t] = Xc[(size_t)(((int64_t)p * n) / P) * dp + l];
  }
  if (threadIdx.x < kKnnMaxCells) hist[threadIdx.x] = 0;
  __syncthreads();
  const int i = blockIdx.x * 64 + (threadIdx.x >> 2), sub = threadIdx.x & 3;
  const float4 *x4 = reinterpret_cast<const float4 *>(Xc + (size_t)min(i, n - 1) * dp);
  float best = INFINITY;
  int bi = 0;
  for (int p = sub; p < P; p += 4) {
    const float *pp = piv + p * dp;
    float d2 = 0.0f;
    for (int c = 0; c < dp / 4; ++c) {
      const float4 v = x4[c];
      const float a = v.x - pp[4 * c], b = v.y - pp[4 * c + 1], e = v.z - pp[4 * c + 2], f = v.w - pp[4 * c + 3];
      d2 = fmaf(a, a, d2);
      d2 = fmaf(b, b, d2);
      d2 = fmaf(e, e, d2);
      d2 = fmaf(f, f, d2);
    }
    if (d2 < best) {
      best = d2;
      bi = p;
    }
  }
#pragma unroll
  for (int o = 1; o < 4; o <<= 1) {
    const float od = __shfl_xor(best, o, 64);
    const int op = __shfl_xor(bi, o, 64);
    if (od < best || (od == best && op < bi)) {
      best = od;
      bi = op;
    }
  }
  const float R = (float)__longlong_as_double((long long)*rmax);
  const float scale = R > 0.0f ? 512.0f / (R * sqrtf((float)dim)) : 0.0f;
  float p3[3] = {0.0f, 0.0f, 0.0f};
  for (int c = sub; c < dp / 4; c += 4) {  // the padding adds zeros
    const float4 v = x4[c];
#pragma unroll
    for (int a = 0; a < 3; ++a)
      p3[a] += (v.x * proj_sign(a, 4 * c) + v.y * proj_sign(a, 4 * c + 1)) +
               (v.z * proj_sign(a, 4 * c + 2) + v.w * proj_sign(a, 4 * c + 3));
  }
  uint32_t k = 0;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    p3[a] += __shfl_xor(p3[a], 1, 64);
    p3[a] += __shfl_xor(p3[a], 2, 64);
    const float u = fminf(fmaxf(p3[a] * scale + 512.0f, 0.0f), 1023.0f);
    k |= spread_bits10((uint32_t)u) << a;
  }
  if (i < n && sub == 0) {
    cell[i] = bi;
    key[i] = ((uint32_t)bi << 24) | (k >> 6);
    idx[i] = i;
    atomicAdd(&hist[bi], 1);
  }
  __syncthreads();
  if (threadIdx.x < kKnnMaxCells && hist[threadIdx.x]) atomicAdd(&cnt[threadIdx.x], hist[threadIdx.x]);
}

// One work-group per reference tile of kFiltR slots.  The sorted points of each
// cell start a fresh tile; the slots left over are padding (id -1).  Slot ids,
// the id -> slot map, the tile's centred points and its bounding sphere: centre =
// mean of its points, radius = the largest distance to it, in the caller's
// coordinates (FP64); -1 for a tile of padding only.  Each 16 slots are stored
// as the filter's matrix instructions take them: step st (dimensions 4 st .. 4 st
// + 3) of slot j, dimension 4 st + g, belongs to lane 16 g + j, and a lane's
// steps come in pairs, 64 lanes side by side (padding is not written: its
// distances count for nothing).
__global__ __launch_bounds__(256) void knn_tile_kernel(const float *__restrict__ X, const float *__restrict__ Xc,
                                                       int dim, int dp, int P, const int32_t *__restrict__ order,
                                                       const int *__restrict__ cnt, int *__restrict__ slot0,
                                                       float *__restrict__ Xr, int32_t *__restrict__ rid,
                                                       int32_t *__restrict__ rinv, double *__restrict__ tcen,
                                                       double *__restrict__ trad) {
  static_assert(kKnnMaxCells == 64 && kFiltR == 64, "a wave holds the cells, and the slots of a tile");
  __shared__ int ids[kFiltR], valid;
  __shared__ double acc[2][kFiltMaxDp], cen[kFiltMaxDp], wmax[4];
  const int tile = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
  if (tid < 64) {  // first sorted point and first slot of each cell, then of this tile's
    const int c = lane < P ? cnt[lane] : 0, w = (c + kFiltR - 1) / kFiltR;
    int first = c, tiles = w;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int a = __shfl_up(first, o, 64), b = __shfl_up(tiles, o, 64);
      if (lane >= o) {
        first += a;
        tiles += b;
      }
    }
    first -= c;
    tiles -= w;
    if (tile == 0 && lane < P) slot0[lane] = tiles * kFiltR;
    const unsigned long long mine = __ballot(tile >= tiles && tile < tiles + w);
    const int cl = mine ? __builtin_ctzll(mine) : 0;
    const int f0 = __shfl(first, cl, 64), t0 = __shfl(tiles, cl, 64), m = __shfl(c, cl, 64);
    const int k = (tile - t0) * kFiltR + lane;
    const int id = mine && k < m ? order[f0 + k] : -1;
    ids[lane] = id;
    rid[(size_t)tile * kFiltR + lane] = id;
    if (id >= 0) rinv[id] = tile * kFiltR + lane;
    const int nv = __popcll(__ballot(id >= 0));  // the valid slots come first
    if (lane == 0) valid = nv;
  }
  __syncthreads();
  const int nv = valid;
  if (nv == 0) {
    if (tid == 0) trad[tile] = -1.0;
    return;
  }
  {
    const int l = tid & 127, h = tid >> 7;
    double a = 0.0;
    if (l < dim)
#pragma unroll 4
      for (int r = h; r < nv; r += 2) a += (double)X[(size_t)ids[r] * dim + l];
    acc[h][l] = a;
    __syncthreads();
    if (h == 0 && l < dim) {
      const double c = (acc[0][l] + acc[1][l]) / (double)nv;
      cen[l] = c;
      tcen[(size_t)l * gridDim.x + tile] = c;  // by dimension: the filter reads it for many tiles at once
    }
  }
  float2 *out = reinterpret_cast<float2 *>(Xr + (size_t)tile * kFiltR * dp);
  for (int e = tid; e < kFiltR * (dp / 8); e += 256) {
    const int sl = (e & 15) + 16 * ((e >> 4) & 3), h = e >> 6, id = ids[sl];
    if (id < 0) continue;
    const float4 *src = reinterpret_cast<const float4 *>(Xc + (size_t)id * dp) + 2 * h;
    const float4 a = src[0], b = src[1];
    float2 *dst = out + (size_t)(sl >> 4) * dp * 8 + 64 * h + (sl & 15);
    dst[0] = make_float2(a.x, b.x);
    dst[16] = make_float2(a.y, b.y);
    dst[32] = make_float2(a.z, b.z);
    dst[48] = make_float2(a.w, b.w);
  }
  __syncthreads();
  const int sub = tid & 15;
  double best = 0.0;
#pragma unroll
  for (int u = 0; u < kFiltR / 16; ++u) {
    const int r = u * 16 + (tid >> 4);
    double r2 = 0.0;
    if (r < nv)
      for (int l = sub; l < dim; l += 16) {
        const double v = (double)X[(size_t)ids[r] * dim + l] - cen[l];
        r2 = fma(v, v, r2);
      }
    best = fmax(best, row16_sum(r2));
  }
  best = wave_max(best);
  if (lane == 0) wmax[tid >> 6] = best;
  __syncthreads();
  if (tid == 0) trad[tile] = sqrt(fmax(fmax(wmax[0], wmax[1]), fmax(wmax[2], wmax[3])));
}

// One work-group per frame of kF2Q query slots: the frame's mean c_b (FP64),
// delta_b = fl32(c_b - mu) padded to dp, and |delta_b|; then its queries centred
// there: Xq[slot] = fl32(x_q - c_b) (zero-padded), its squared norm (FP32 of the
// FP64 sum) by slot, and by query id its norm |a| and |delta_b| for the
// certificate.
constexpr int kF2Q = 32;  // queries of a frame
__global__ __launch_bounds__(256) void knn_frame_kernel(const float *__restrict__ X, int n, int dim, int dp,
                                                        const int32_t *__restrict__ qorder,
                                                        const double *__restrict__ mu, double *__restrict__ cb,
                                                        float *__restrict__ delta, double *__restrict__ dn,
                                                        float *__restrict__ Xq, float *__restrict__ qn32,
                                                        double *__restrict__ qa, double *__restrict__ qdn) {
  __shared__ int ids[kF2Q];
  __shared__ double acc[2][kFiltMaxDp], cen[kFiltMaxDp], wsum[4];
  const int b = blockIdx.x, tid = threadIdx.x, s0 = b * kF2Q, m = min(kF2Q, n - s0);
  if (tid < kF2Q) ids[tid] = tid < m ? qorder[s0 + tid] : 0;
  __syncthreads();
  const int l = tid & 127, h = tid >> 7;
  double a = 0.0;
  if (l < dim)
#pragma unroll 4
    for (int r = h; r < m; r += 2) a += (double)X[(size_t)ids[r] * dim + l];
  acc[h][l] = a;
  __syncthreads();
  double ss = 0.0;
  if (h == 0 && l < dp) {
    float dv = 0.0f;
    if (l < dim) {
      const double c = (acc[0][l] + acc[1][l]) / (double)m;
      cen[l] = c;
      cb[(size_t)b * dim + l] = c;
      dv = (float)(c - mu[l]);
    }
    delta[(size_t)b * dp + l] = dv;
    ss = (double)dv * (double)dv;
  }
  ss = wave_sum(ss);
  if ((tid & 63) == 0) wsum[tid >> 6] = ss;
  __syncthreads();
  const double dnb = sqrt(wsum[0] + wsum[1] + wsum[2] + wsum[3]);
  if (tid == 0) dn[b] = dnb;
  const int sub = tid & 15;
#pragma unroll
  for (int u = 0; u < kF2Q / 16; ++u) {
    const int r = u * 16 + (tid >> 4);
    double s2 = 0.0;
    if (r < m)
      for (int c = sub; c < dp; c += 16) {
        const float v = c < dim ? (float)((double)X[(size_t)ids[r] * dim + c] - cen[c]) : 0.0f;
        Xq[(size_t)(s0 + r) * dp + c] = v;
        s2 += (double)v * (double)v;
      }
    s2 = row16_sum(s2);
    if (r < m && sub == 0) {
      qn32[s0 + r] = (float)s2;
      qa[ids[r]] = sqrt(s2);
      qdn[ids[r]] = dnb;
    }
  }
}

// Candidate lists: a max-heap of kp (approximate distance, index) keys per
// query in global memory (lists longer than the LDS version holds).  Wave w
// owns queries q0 + 16w .. q0 + 16w + 15.  The points have 4 NST dimensions.
template <int NST>
__global__ __launch_bounds__(256) void knn_filter_kernel(const float *__restrict__ Xc,
                                                         const float *__restrict__ n32, int n, int kp,
                                                         float *__restrict__ hd, int *__restrict__ hi) {
  __shared__ float rt[4 * NST * kFiltRS];
  __shared__ float rn[kFiltR];
  __shared__ float qd[kFiltQ][kFiltR];
  __shared__ int qi[kFiltQ][kFiltR];
  __shared__ int qcnt[kFiltQ];
  __shared__ float thr_d[kFiltQ];
  __shared__ int thr_i[kFiltQ];
  __shared__ float qn[kFiltQ];

  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
  const int q0 = blockIdx.x * kFiltQ;
  // A operand of step s: row (query) lane % 16, column (dimension) 4 s + lane / 16
  float areg[NST];
  {
    const int qa = q0 + 16 * w + (lane & 15);
#pragma unroll
    for (int st = 0; st < NST; ++st) areg[st] = qa < n ? Xc[(size_t)qa * 4 * NST + 4 * st + (lane >> 4)] : 0.0f;
  }
  if (tid < kFiltQ) {
    qcnt[tid] = 0;
    thr_d[tid] = INFINITY;
    thr_i[tid] = INT_MAX;
    const int q = q0 + tid;
    qn[tid] = q < n ? n32[q] : 0.0f;
    if (q < n)
      for (int e = 0; e < kp; ++e) {
        hd[(size_t)q * kp + e] = INFINITY;
        hi[(size_t)q * kp + e] = INT_MAX;
      }
  }
  float4 buf[kFiltR * NST / 256];
  float rnv;
  tile_load<256, NST>(Xc, n32, n, 0, buf, rnv);
  for (int r0 = 0; r0 < n; r0 += kFiltR) {
    __syncthreads();  // the previous tile's LDS is free
    tile_store<256, NST>(rt, rn, buf, rnv);
    __syncthreads();
    // the next tile's loads fly while this one is multiplied and merged
    if (r0 + kFiltR < n) tile_load<256, NST>(Xc, n32, n, r0 + kFiltR, buf, rnv);
    fv4 acc[4];
    tile_dots<NST>(areg, rt, lane, acc);
    // output v of block t: query 16 w + 4 (lane / 16) + v, reference 16 t + lane % 16
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int jl = 16 * t + (lane & 15), r = r0 + jl;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int ql = 16 * w + 4 * (lane >> 4) + v, q = q0 + ql;
        const float dd = (qn[ql] + rn[jl]) - 2.0f * acc[t][v];
        if (q < n && r < n && r != q && key_lessf(dd, r, thr_d[ql], thr_i[ql])) {
          const int pos = atomicAdd(&qcnt[ql], 1);
          qd[ql][pos] = dd;
          qi[ql][pos] = r;
        }
      }
    }
    __syncthreads();
    if (tid < kFiltQ) {
      const int q = q0 + tid;
      const int cnt = qcnt[tid];
      if (q < n && cnt > 0) {
        float *H = hd + (size_t)q * kp;
        int *HI = hi + (size_t)q * kp;
        float rd = H[0];
        int ri = HI[0];
        for (int c = 0; c < cnt; ++c) {
          const float cd = qd[tid][c];
          const int ci = qi[tid][c];
          if (!key_lessf(cd, ci, rd, ri)) continue;
          int pos = 0;
          for (;;) {
            const int l = 2 * pos + 1, rr = l + 1;
            int m = -1;
            float md = cd;
            int mi = ci;
            if (l < kp && key_lessf(md, mi, H[l], HI[l])) { m = l; md = H[l]; mi = HI[l]; }
            if (rr < kp && key_lessf(md, mi, H[rr], HI[rr])) { m = rr; md = H[rr]; mi = HI[rr]; }
            if (m < 0) break;
            H[pos] = md;
            HI[pos] = mi;
            pos = m;
          }
          H[pos] = cd;
          HI[pos] = ci;
          rd = H[0];
          ri = HI[0];
        }
        thr_d[tid] = rd;
        thr_i[tid] = ri;
      }
      qcnt[tid] = 0;
    }
  }
}

// The same filter with the candidate lists in LDS (lists of up to kF2MaxKp).
// A work-group of four waves owns NQ = 16 QB queries of one frame.  The
// references come in tiles of 64, 16 to a wave, stored in the order the matrix
// instructions take them (knn_tile_kernel), so a wave reads its B
// operands straight from memory, coalesced, the next tile's in flight, and
// nothing is staged or transposed in LDS.
//
// A query's list is a buffer of CAP (distance, slot) entries in no order and a
// threshold: a lane appends its pair when the distance is under the threshold
// (ballots give the places).  Once a list holds more than kTrig entries one
// wave cuts it back to the kp smallest (a few spare): the threshold is found by
// bisecting the bits of the distances with ballot counts, and becomes the
// list's new threshold.  An entry dropped or turned away has kp entries at or
// below it, so the list always holds kp smallest values, and the ties dropped
// at the kp-th have that very value: what the certificate needs.  The waves
// meet once a round (a tile; with QB = 1 two, with 16 waves four).  An insertion thus costs a
// few instructions of one wave and a cut about 300 per ~100 insertions; the
// binary heaps this replaces took one lane log2(kp) dependent LDS round trips
// per insertion while both waves of the work-group waited.  20,011 points of 50
// dimensions: 4.09 -> 0.57 ms; a job of 500-8000 points: 1.58 -> 0.12 ms on
// average; the whole kNN of 1.3M points 2.76 -> 1.15 s.
//
// The tiles follow a cell order (see knn_cell_kernel), each with a bounding
// sphere.  A block starts at the tiles around its own queries' (its lists fill
// with near candidates), then visits the others in groups, skipping every tile
// that cannot hold a candidate: with D the distance between the block's and
// the tile's spheres, every query a and reference b of them have a true
// distance of at least D, and the filter value of the pair is within 2^-12 S^2
// of its squared distance (S = block radius + centre distance + tile radius +
// R + |c_b - mu|: more than eight times the certificate's error bounds for the
// rounding of the centred points and the FP32 dot products), so a tile with
// D^2 - 2^-12 S^2 above every query's current threshold holds no candidate.
// Skipped tiles thus leave the lists as a full scan would: the k + kFiltSlack
// smallest values.
constexpr int kF2MaxKp = 128;
constexpr int kFiltHomeBack = 16;  // tiles visited before a block's own
constexpr int kTrig = 192;         // entries beyond which a list is cut
constexpr int kCutSpare = 12;      // entries a cut may leave beyond kp
static_assert(kF2MaxKp + kCutSpare < kTrig, "a cut list is below the trigger");

// Unsigned integers ordered as the floats (none of them NaN), and back.
__device__ __forceinline__ uint32_t float_order(float f) {
  const uint32_t u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float order_float(uint32_t u) {
  return __uint_as_float((u & 0x80000000u) ? (u & 0x7FFFFFFFu) : ~u);
}

// Cuts a list of c >= kp entries to its smallest: at least kp, at most kp +
// spare; returns the new count and, in *thr, a value at or below which at
// least kp of them lie.  One wave; the list's entries must be written.
template <int CAP>
__device__ __forceinline__ int cut_list(float *key, int *id, int c, int kp, int spare, int lane, float *thr) {
  constexpr int E = CAP / 64;
  uint32_t u[E];
  int x[E];
  uint32_t lo = 0xFFFFFFFFu, hi = 0;
#pragma unroll
  for (int i = 0; i < E; ++i) {
    const int e = lane + 64 * i;
    u[i] = e < c ? float_order(key[e]) : 0xFFFFFFFFu;  // above every value (not a float's image)
    x[i] = e < c ? id[e] : -1;
    if (e < c) {
      lo = min(lo, u[i]);
      hi = max(hi, u[i]);
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    lo = min(lo, (uint32_t)__shfl_xor((int)lo, o, 64));
    hi = max(hi, (uint32_t)__shfl_xor((int)hi, o, 64));
  }
  int upto = c;  // entries at or below hi
  while (lo < hi) {
    const uint32_t mid = lo + ((hi - lo) >> 1);
    int m = 0;
#pragma unroll
    for (int i = 0; i < E; ++i) m += __popcll(__ballot(u[i] <= mid));
    if (m >= kp) {
      hi = mid;
      upto = m;
      if (m <= kp + spare) break;
    } else {
      lo = mid + 1;
    }
  }
  int tie_room = CAP;  // entries equal to hi that are kept (all, unless they are too many)
  if (upto > kp + spare) {
    int under = 0;
#pragma unroll
    for (int i = 0; i < E; ++i) under += __popcll(__ballot(u[i] < hi));
    tie_room = kp - under;
  }
  const unsigned long long below = (1ull << lane) - 1ull;
  int pos0 = 0, tie0 = 0;
#pragma unroll
  for (int i = 0; i < E; ++i) {
    const unsigned long long tm = __ballot(u[i] == hi);
    const bool tie = u[i] == hi && tie0 + __popcll(tm & below) < tie_room;
    tie0 += __popcll(tm);
    const bool keep = u[i] < hi || tie;
    const unsigned long long km = __ballot(keep);
    if (keep) {
      const int p = pos0 + __popcll(km & below);
      key[p] = order_float(u[i]);
      id[p] = x[i];
    }
    pos0 += __popcll(km);
  }
  *thr = order_float(hi);
  return pos0;
}

// The reference stream of the LDS-list filter: tiles of kFiltR slots in
// cell order (Xr, -1 ids for padding), their spheres, and the query
// blocks' spheres (centre cb, radius from the queries' norms qa, |c_b - mu|
// in dn; R the largest |x - mu|).
struct RefTiles {
  const float *Xr;
  const int32_t *rid, *rinv;
  int ntiles;
  const double *tcen, *trad;
  const double *cb, *qa, *dn;
  const unsigned long long *rmax;
  int dim;
  const int32_t *cell;  // point -> cell
  const int *slot0;     // cell -> its first slot (a tile boundary)
};

template <int NST, int QB, int NW>
__global__ __launch_bounds__(64 * NW) void knn_filter_list_kernel(const RefTiles rf, const float *__restrict__ Xq,
                                                              const float *__restrict__ qn32,
                                                              const int32_t *__restrict__ qorder,
                                                              const float *__restrict__ delta, int n, int kp,
                                                              float *__restrict__ hd, int *__restrict__ hi) {
  constexpr int NQ = 16 * QB;
  constexpr int TW = NW / 4;                 // tiles taken at once, one per four waves
  constexpr int TPR = NW == 16 ? 4 : QB == 1 ? 2 : 1;  // tiles between the meetings of the waves
  constexpr int CAP = kTrig + 64 * TPR;      // no list overflows in a round
  static_assert(NST % 2 == 0 && kF2Q % NQ == 0 && TPR % TW == 0, "steps come in pairs, work-groups lie in one frame");
  __shared__ float lkey[NQ][CAP];
  __shared__ int lid[NQ][CAP];
  __shared__ int lcnt[NQ];
  __shared__ float lthr[NQ];  // -infinity for a slot without a query: nothing enters
  __shared__ int lqid[NQ];
  __shared__ int need[3];     // round r uses need[r % 3]
  __shared__ unsigned long long gom[4];
  __shared__ int list[256];   // the group's tiles to visit
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = lane >> 4, j = lane & 15;
  const int q0 = blockIdx.x * NQ, frame = q0 / kF2Q;
  const int ntiles = rf.ntiles;
  float areg[QB][NST], dl[NST];
#pragma unroll
  for (int b = 0; b < QB; ++b) {
    const int sa = q0 + 16 * b + j;
#pragma unroll
    for (int st = 0; st < NST; ++st) areg[b][st] = sa < n ? Xq[(size_t)sa * 4 * NST + 4 * st + g] : 0.0f;
  }
#pragma unroll
  for (int st = 0; st < NST; ++st) dl[st] = delta[(size_t)frame * 4 * NST + 4 * st + g];
  if (tid < NQ) {
    const bool in = q0 + tid < n;
    lcnt[tid] = 0;
    lqid[tid] = in ? qorder[q0 + tid] : -1;
    lthr[tid] = in ? INFINITY : -INFINITY;
  }
  if (tid < 3) need[tid] = 0;
  // the block's radius: its queries' largest |x - c_b| (|a| rounded up)
  const double rho =
      wave_max(lane < NQ && q0 + lane < n ? rf.qa[qorder[q0 + lane]] * (1.0 + 0x1p-20) : 0.0);
  __syncthreads();
  // this lane's queries: rows 4 g + v of each block of 16
  float qv[QB][4], th[QB][4];
  int qq[QB][4];
#pragma unroll
  for (int b = 0; b < QB; ++b)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int ql = 16 * b + 4 * g + v;
      qv[b][v] = q0 + ql < n ? qn32[q0 + ql] : 0.0f;
      qq[b][v] = lqid[ql];
      th[b][v] = lthr[ql];
    }
  // the first tile visited: kFiltHomeBack tiles before the block's own, but
  // not before its cell's first tile, so the lists fill from the block's
  // own cell and its threshold prunes the other cells' tiles early
  const int home = rf.rinv[qorder[q0]] / kFiltR;
  const int start = max(home - kFiltHomeBack, rf.slot0[rf.cell[qorder[q0]]] / kFiltR);
  const double R = __longlong_as_double((long long)*rf.rmax);
  const double dnb = rf.dn[frame];
  const double *cbb = rf.cb + (size_t)frame * rf.dim;
  auto visit = [&](int sq) { return (start + sq) % ntiles; };  // the sq-th tile visited
  const float2 *Xr2 = reinterpret_cast<const float2 *>(rf.Xr);
  float2 nb[NST / 2];
  int nid = -1;
  auto load = [&](int tile) {  // this wave's 16 references of a tile
    const size_t t16 = (size_t)tile * 4 + (w & 3);
    const float2 *src = Xr2 + t16 * (NST / 2) * 64 + lane;
#pragma unroll
    for (int u = 0; u < NST / 2; ++u) nb[u] = src[u * 64];
    nid = rf.rid[t16 * 16 + j];
  };
  auto cut = [&](int ql, int spare) {
    float t;
    const int c = cut_list<CAP>(lkey[ql], lid[ql], lcnt[ql], kp, spare, lane, &t);
    if (lane == 0) {
      lcnt[ql] = c;
      lthr[ql] = t;
    }
  };
  auto refresh = [&]() {
#pragma unroll
    for (int b = 0; b < QB; ++b)
#pragma unroll
      for (int v = 0; v < 4; ++v) th[b][v] = lthr[16 * b + 4 * g + v];
  };
  int round = 0;
  // groups of tiles: the first ones small, so that the thresholds prune soon
  for (int g0 = 0, gsz = 32; g0 < ntiles; g0 += gsz, gsz = min(256, g0 >= 64 ? 256 : 2 * gsz)) {
    // tighten every list that has kp entries, then the tiles of the group
    // that some query's threshold reaches
    for (int ql = w; ql < NQ; ql += NW)
      if (lcnt[ql] > kp) cut(ql, kCutSpare);
    __syncthreads();
    refresh();
    const float thr = (float)wave_max(lane < NQ ? (double)lthr[lane] : -INFINITY);
    bool skip = true;
    if (tid < gsz && g0 + tid < ntiles) {
      const int t = visit(g0 + tid);
      const double rt_ = rf.trad[t];
      if (rt_ >= 0.0) {  // not padding only
        skip = false;
        if (thr < INFINITY) {
          const double *tc = rf.tcen + t;
          double d2 = 0.0;
#pragma unroll 8
          for (int l = 0; l < rf.dim; ++l) {
            const double v = cbb[l] - tc[(size_t)l * ntiles];
            d2 = fma(v, v, d2);
          }
          const double dcm = sqrt(d2);
          const double dlb = dcm - rho - rt_;
          const double S = rho + dcm + rt_ + R + dnb;
          skip = dlb > 0.0 && dlb * dlb - 0x1p-12 * S * S > (double)thr;
        }
      }
    }
    // the tiles to visit, in order
    const unsigned long long go = __ballot(!skip);
    if (lane == 0 && w < 4) gom[w] = go;
    __syncthreads();
    const int m0 = __popcll(gom[0]), m1 = m0 + __popcll(gom[1]), m2 = m1 + __popcll(gom[2]), m = m2 + __popcll(gom[3]);
    if (!skip)
      list[(w == 0 ? 0 : w == 1 ? m0 : w == 2 ? m1 : m2) + __popcll(go & ((1ull << lane) - 1ull))] = visit(g0 + tid);
    __syncthreads();
    int k = w / 4;  // the next one of these four waves
    if (k < m) load(list[k]);
    for (int r0 = 0; r0 < m; r0 += TPR) {
#pragma unroll 1
      for (int u = 0; u < TPR / TW; ++u, k += TW) {
        if (k >= m) break;
        float bv[NST];
#pragma unroll
        for (int h = 0; h < NST / 2; ++h) {
          bv[2 * h] = nb[h].x;
          bv[2 * h + 1] = nb[h].y;
        }
        const int rid = nid;
        if (k + TW < m) load(list[k + TW]);
        // into the block's frame, with the squared norms of the references
        float rn = 0.0f;
#pragma unroll
        for (int st = 0; st < NST; ++st) {
          bv[st] -= dl[st];
          rn = fmaf(bv[st], bv[st], rn);
        }
        rn += __shfl_xor(rn, 16, 64);
        rn += __shfl_xor(rn, 32, 64);
        if (rid < 0) rn = INFINITY;  // padding holds anything: under no threshold
        fv4 acc[QB];
#pragma unroll
        for (int b = 0; b < QB; ++b) acc[b] = fv4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int st = 0; st < NST; ++st)
#pragma unroll
          for (int b = 0; b < QB; ++b)
            acc[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(areg[b][st], bv[st], acc[b], 0, 0, 0);
        float dd[QB][4];
        bool any = false;
#pragma unroll
        for (int b = 0; b < QB; ++b)
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            dd[b][v] = (qv[b][v] + rn) - 2.0f * acc[b][v];
            any |= dd[b][v] < th[b][v];
          }
        if (__ballot(any)) {
#pragma unroll
          for (int b = 0; b < QB; ++b) {
            // the 16 references that enter the list of this lane's v-th query;
            // lane v of the 16 takes their places, for the four queries at once
            unsigned gm[4];
            int c = 0;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
              gm[v] = (unsigned)(__ballot(dd[b][v] < th[b][v] && rid != qq[b][v]) >> (16 * g)) & 0xFFFFu;
              if (j == v) c = __popc(gm[v]);
            }
            int base = 0;
            if (c) {
              base = atomicAdd(&lcnt[16 * b + 4 * g + j], c);
              if (base + c > kTrig) need[round % 3] = 1;
            }
#pragma unroll
            for (int v = 0; v < 4; ++v) {
              const int p = __shfl(base, 16 * g + v, 64) + __popc(gm[v] & ((1u << j) - 1u));
              if ((gm[v] >> j) & 1u) {
                lkey[16 * b + 4 * g + v][p] = dd[b][v];
                lid[16 * b + 4 * g + v][p] = rid;
              }
            }
          }
        }
      }
      __syncthreads();
      // every wave reads need[round % 3] before the next meeting; it is
      // cleared after that one, and used again after the one that follows
      const bool full = need[round % 3] != 0;
      if (tid == 0) need[(round + 2) % 3] = 0;
      ++round;
      if (full) {
        for (int ql = w; ql < NQ; ql += NW)
          if (lcnt[ql] > kTrig - 32) cut(ql, kCutSpare);
        __syncthreads();
        refresh();
      }
    }
  }
  __syncthreads();
  for (int ql = w; ql < NQ; ql += NW) {
    const int q = lqid[ql];
    if (q < 0) continue;  // wave-uniform
    if (lcnt[ql] > kp) cut(ql, 0);
    const int c = lcnt[ql];
    for (int e = lane; e < kp; e += 64) {  // a list left short (NaN distances) is not certified
      hd[(size_t)q * kp + e] = e < c ? lkey[ql][e] : INFINITY;
      hi[(size_t)q * kp + e] = e < c ? lid[ql][e] : INT_MAX;
    }
  }
}

// The block-centred arrays of the LDS-list filter (kp <= kF2MaxKp).
struct BlockCentred {
  const float *Xq;         // queries in slot order, centred at their block's mean
  const float *qn32;       // their squared norms
  const int32_t *qorder;   // slot -> query id
  const float *delta;      // per block: fl32(c_b - mu), padded
  RefTiles rf;             // the references in cell order, with tile spheres
};

// Points from which a work-group takes 32 queries instead of 16.  32 halve the
// reads of the references but leave half as many waves per CU (66 KB of lists
// against 41) and half as many work-groups: whole kNN calls at 50 dimensions
// with 16 / 32: 2.24 / 2.46 ms at 10,000 points, 4.23 / 4.58 at 20,000, 82.4 /
// 84.2 at 200,000, 1272 / 1148 at 1.3M.
constexpr int kFiltWide = 1 << 19;

// Points up to which the 16 queries are given 16 waves (a work-group per CU; up to
// 64 dimensions, beyond which 16 waves run out of registers) and eight instead
// of four: the walk over the tiles is then bound by its latency.  The filter alone
// with 8 / 16 waves: 51 / 40 us at 1000 points, 109 / 91 at 4000, 168 / 181 at
// 6000; with 4 / 8: 404 / 354 us at 12,000, 580 / 501 at 20,011, 1495 / 1518 at
// 50,000, 10.0 / 11.6 ms at 200,003.
constexpr int kFiltDeeper = 1 << 12;
constexpr int kFiltDeep = 1 << 15;

template <int NST>
int launch_filter(hipStream_t s, const float *Xc, const float *n32, int n, int kp, const BlockCentred &bc,
                  float *hd, int *hi) {
  if (kp <= kF2MaxKp) {
    if constexpr (NST <= 16) {
      if (n <= kFiltDeeper) {
        knn_filter_list_kernel<NST, 1, 16><<<div_up(n, 16), 1024, 0, s>>>(bc.rf, bc.Xq, bc.qn32, bc.qorder, bc.delta,
                                                                          n, kp, hd, hi);
        SGT_LAUNCH_CHECK();
        return SGTSNE_OK;
      }
    }
    if (n <= kFiltDeep)
      knn_filter_list_kernel<NST, 1, 8><<<div_up(n, 16), 512, 0, s>>>(bc.rf, bc.Xq, bc.qn32, bc.qorder, bc.delta, n,
                                                                      kp, hd, hi);
    else if (n < kFiltWide)
      knn_filter_list_kernel<NST, 1, 4><<<div_up(n, 16), 256, 0, s>>>(bc.rf, bc.Xq, bc.qn32, bc.qorder, bc.delta, n,
                                                                      kp, hd, hi);
    else
      knn_filter_list_kernel<NST, 2, 4><<<div_up(n, 32), 256, 0, s>>>(bc.rf, bc.Xq, bc.qn32, bc.qorder, bc.delta, n,
                                                                      kp, hd, hi);
  } else {
    if constexpr ((kFiltR * NST) % 256 == 0) {
      knn_filter_kernel<NST><<<div_up(n, kFiltQ), 256, 0, s>>>(Xc, n32, n, kp, hd, hi);
    } else {
      SGT_CHECK(false, SGTSNE_ERR_ARG, "no global-heap filter of %d steps", NST);
    }
  }
  SGT_LAUNCH_CHECK();
  return SGTSNE_OK;
}

// float4 steps of the filter's padded dimension.  14 (dims 49-56: the usual
// 50-D PCA input) only with the LDS-list kernel, which takes any even number
// of steps.  The zero padding adds exact zeros, so the FP32 distances, the
// candidates and the rows are the same either way.
int filter_steps(int dim, int kp) {
  const int nst = (dim + 3) / 4;
  if (nst > 12 && nst <= 14 && kp <= kF2MaxKp) return 14;
  return nst <= 4 ? 4 : nst <= 8 ? 8 : nst <= 12 ? 12 : nst <= 16 ? 16 : nst <= 24 ? 24 : 32;
}

int launch_filter_for(hipStream_t s, int nst, const float *Xc, const float *n32, int n, int kp,
                      const BlockCentred &bc, float *hd, int *hi) {
  switch (nst) {
    case 4: return launch_filter<4>(s, Xc, n32, n, kp, bc, hd, hi);
    case 8: return launch_filter<8>(s, Xc, n32, n, kp, bc, hd, hi);
    case 12: return launch_filter<12>(s, Xc, n32, n, kp, bc, hd, hi);
    case 14: return launch_filter<14>(s, Xc, n32, n, kp, bc, hd, hi);
    case 16: return launch_filter<16>(s, Xc, n32, n, kp, bc, hd, hi);
    case 24: return launch_filter<24>(s, Xc, n32, n, kp, bc, hd, hi);
    default: return launch_filter<32>(s, Xc, n32, n, kp, bc, hd, hi);
  }
}

// One wave per query: certify the candidate list, recompute the
// candidates' distances as knn_dist_kernel does (diff = x_q - x_c in FP64,
// acc = fma(diff, diff, acc) over the dimensions in order) and write the row.
//
// The filter compares a = fl32(x_q - c) with b = fl32(fl32(x_c - mu) -
// fl32(c - mu)) for the frame c of the query's block (c = mu, no shift, when
// qdn is 0): F = |a|^2 + |b|^2 - 2 a.b is within E = cE (|a| + |b|)^2 of
// |a - b|^2, and |a - b| is within e = ce (|a| + R + |c - mu| + |b|) of the
// true distance T^(1/2), R the largest |x - mu|.  The k nearest candidates
// (F <= F_k) lie within hi = sqrt(F_k + E) + e with |b| <= |a| + sqrt(F_k) + 1;
// a point outside the list within hi would have |b| <= |a| + hi + e + 1 and
// so F <= (hi + e)^2 + E, yet every non-candidate has F >= F_kp: when F_kp
// exceeds that bound (with a 1e-12 relative margin for the FP64 rounding of
// the recomputed distances), the list holds the k nearest.
//
// A lane holds E of the 64 E candidates: the k-th smallest filter value comes
// from a bisection of its bits with ballot counts, and the recomputed keys are
// sorted by a bitonic network through cross-lane reads, without barriers.  The
// candidates' rows go through LDS, 16 dimensions at a time and 16 lanes to a
// row, so that a load touches few lines while each lane still adds its own
// row's terms in order.  20,011 points of 50 dimensions: a 256-thread work-group
// per query with two sorts of 256 in LDS 505 us, a wave whose lanes read a row
// each 240 us, this 113 us.
template <int E>
__global__ __launch_bounds__(256) void knn_rerank_kernel(
    const float *__restrict__ X, int n, int dim, int k, int kp, const float *__restrict__ hd,
    const int *__restrict__ hi, const double *__restrict__ qa, const double *__restrict__ qdn,
    const unsigned long long *__restrict__ rmax, double cE, double ce, int32_t *__restrict__ I,
    double *__restrict__ D, int *__restrict__ fb_list, int *__restrict__ fb_cnt) {
  __shared__ float stage[4][64][17];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int q = blockIdx.x * 4 + w;
  if (q >= n) return;  // the whole wave leaves
  float(*st)[17] = stage[w];
  uint32_t u[E];
  int id[E];
  bool bad = false;  // a list left short (NaN distances never enter it) is not certified
  uint32_t lo = 0xFFFFFFFFu, hi_ = 0;
#pragma unroll
  for (int i = 0; i < E; ++i) {
    const int e = lane + 64 * i;
    u[i] = e < kp ? float_order(hd[(size_t)q * kp + e]) : 0xFFFFFFFFu;
    id[i] = e < kp ? hi[(size_t)q * kp + e] : INT_MAX;
    if (e < kp) {
      bad |= id[i] < 0 || id[i] >= n;
      lo = min(lo, u[i]);
      hi_ = max(hi_, u[i]);
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    lo = min(lo, (uint32_t)__shfl_xor((int)lo, o, 64));
    hi_ = max(hi_, (uint32_t)__shfl_xor((int)hi_, o, 64));
  }
  bool ok = kp >= n - 1;  // every other point is a candidate
  if (!ok) {
    const double fkp = (double)order_float(hi_);
    while (lo < hi_) {  // the k-th smallest filter value
      const uint32_t mid = lo + ((hi_ - lo) >> 1);
      int m = 0;
#pragma unroll
      for (int i = 0; i < E; ++i) m += __popcll(__ballot(u[i] <= mid));
      if (m >= k) hi_ = mid;
      else lo = mid + 1;
    }
    const double R = __longlong_as_double((long long)*rmax);
    const double a = qa[q], dl = qdn[q];
    const double fk = fmax((double)order_float(lo), 0.0);
    const double bk = a + sqrt(fk) + 1.0;
    const double ek = ce * (a + R + dl + bk);
    const double hik = (sqrt(fk + cE * (a + bk) * (a + bk)) + ek) * (1.0 + 1e-12) + 1e-300;
    const double bn = a + hik + ek + 1.0;
    const double en = ce * (a + R + dl + bn);
    const double fmaxn = (hik + en) * (hik + en) + cE * (a + bn) * (a + bn);
    ok = fkp > fmaxn;  // false for NaN keys too
  }
  if (__ballot(bad)) ok = false;
  // the candidates' distances, as the integers that order the same
  long long d[E];
  const float *xq = X + (size_t)q * dim;
  const int sub = lane & 15, rg = lane >> 4;
#pragma unroll
  for (int i = 0; i < E; ++i) {
    const bool in = id[i] >= 0 && id[i] < n;
    const int row = in ? id[i] : q, rows = min(64, kp - 64 * i);
    double acc = 0.0;
    for (int l0 = 0; l0 < dim; l0 += 16) {
      float v[16];
#pragma unroll
      for (int u = 0; u < 16; ++u) {  // 16 lanes a row, four rows at a time
        const int xr = __shfl(row, 4 * u + rg, 64);
        v[u] = 4 * u + rg < rows && l0 + sub < dim ? X[(size_t)xr * dim + l0 + sub] : 0.0f;
      }
#pragma unroll
      for (int u = 0; u < 16; ++u) st[4 * u + rg][sub] = v[u];
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      const int m = min(16, dim - l0);
      for (int l = 0; l < m; ++l) {
        const double df = (double)xq[l0 + l] - (double)st[lane][l];
        acc = fma(df, df, acc);
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
    d[i] = __double_as_longlong(in ? acc : (double)INFINITY);
    if (!in) id[i] = INT_MAX;
  }
  // ascending bitonic sort; element lane + 64 i of lane's register i
#pragma unroll
  for (int size = 2; size <= 64 * E; size <<= 1)
#pragma unroll
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      if (stride >= 64) {
#pragma unroll
        for (int i = 0; i < E; ++i) {
          const int j = i ^ (stride / 64);
          if (j > i) {
            const bool up = (64 * i & size) == 0;
            if ((d[j] < d[i] || (d[j] == d[i] && id[j] < id[i])) == up) {
              const long long td = d[i];
              d[i] = d[j];
              d[j] = td;
              const int ti = id[i];
              id[i] = id[j];
              id[j] = ti;
            }
          }
        }
      } else {
#pragma unroll
        for (int i = 0; i < E; ++i) {
          const long long od = __shfl_xor(d[i], stride, 64);
          const int oi = __shfl_xor(id[i], stride, 64);
          const bool up = ((lane + 64 * i) & size) == 0, lower = (lane & stride) == 0;
          const bool other_less = od < d[i] || (od == d[i] && oi < id[i]);
          // the lower place keeps the smaller key in an ascending run
          if (other_less == (lower == up)) {
            d[i] = od;
            id[i] = oi;
          }
        }
      }
    }
  int32_t *Iq = I + (size_t)q * (k + 1);
  double *Dq = D + (size_t)q * (k + 1);
  if (lane == 0) {
    Iq[0] = q;
    Dq[0] = 0.0;
    if (!ok) fb_list[atomicAdd(fb_cnt, 1)] = q;
  }
#pragma unroll
  for (int i = 0; i < E; ++i) {
    const int e = lane + 64 * i;
    if (e < k) {
      Iq[1 + e] = id[i];
      Dq[1 + e] = __longlong_as_double(d[i]);
    }
  }
}

template <int E>
int launch_rerank(hipStream_t s, const float *X, int n, int dim, int k, int kp, const float *hd, const int *hi,
                  const double *qa, const double *qdn, const unsigned long long *rmax, double cE, double ce, int32_t *I,
                  double *D, int *fb_list, int *fb_cnt) {
  knn_rerank_kernel<E><<<div_up(n, 4), 256, 0, s>>>(X, n, dim, k, kp, hd, hi, qa, qdn, rmax, cE, ce, I, D, fb_list,
                                                    fb_cnt);
  SGT_LAUNCH_CHECK();
  return SGTSNE_OK;
}

// ---- perplexity bisection (HY/sgtsne.cpp:201-254), LANES lanes per point ----
// The reference's bisection on beta, step for step: the entropy H of the
// point's row at beta against log(u), beta doubled / halved until bracketed,
// then bisected, until |H - log u| < 1e-5 (at most 200 steps).  Each lane of a
// point's group takes the neighbours m = lane, lane + LANES, ..., PER of them
// held in registers (PER = 0: any number, read again at each step); a step's two
// sums (sum_m exp(-beta d_m) and sum_m d_m exp(-beta d_m)) are added over the
// group by a fixed butterfly (deterministic).  Bound by the FP64 exponentials,
// for few points by the latency of a step.  As in the reference, the values
// normalised at the end are those of the last evaluated beta (recomputed from
// it).
template <int LANES, int PER>
__global__ __launch_bounds__(256) void perplexity_kernel2(const double *__restrict__ D, int n, int k, double u,
                                                          float *__restrict__ val, double *__restrict__ beta_out) {
  const int i = (blockIdx.x * blockDim.x + threadIdx.x) / LANES;
  const int l = threadIdx.x & (LANES - 1);
  if (i >= n) return;  // whole groups leave together
  const double *dist = D + (size_t)i * (k + 1) + 1;
  double dm[PER > 0 ? PER : 1];
#pragma unroll
  for (int m = 0; m < PER; ++m) dm[m] = l + m * LANES < k ? dist[l + m * LANES] : 0.0;
  const double tol = 1e-5;
  const double logu = log(u);
  double beta = 1.0, min_beta = -DBL_MAX, max_beta = DBL_MAX;
  double sum_P = 0.0, beta_eval = 1.0;
  bool found = false;
  int iter = 0;
  while (!found && iter < 200) {  // uniform over the group
    beta_eval = beta;
    double sp = 0.0, sh = 0.0;
    if constexpr (PER > 0) {
#pragma unroll
      for (int m = 0; m < PER; ++m)
        if (l + m * LANES < k) {
          const double e = exp(-beta * dm[m]);
          sp += e;
          sh += dm[m] * e;
        }
    } else {
      for (int m = l; m < k; m += LANES) {
        const double e = exp(-beta * dist[m]);
        sp += e;
        sh += dist[m] * e;
      }
    }
#pragma unroll
    for (int o = LANES / 2; o > 0; o >>= 1) {
      sp += __shfl_xor(sp, o, LANES);
      sh += __shfl_xor(sh, o, LANES);
    }
    sum_P = DBL_MIN + sp;
    const double H = (beta * sh) / sum_P + log(sum_P);
    const double Hdiff = H - logu;
    if (Hdiff < tol && -Hdiff < tol) {
      found = true;
    } else if (Hdiff > 0) {
      min_beta = beta;
      beta = (max_beta == DBL_MAX || max_beta == -DBL_MAX) ? beta * 2.0 : (beta + max_beta) / 2.0;
    } else {
      max_beta = beta;
      beta = (min_beta == -DBL_MAX || min_beta == DBL_MAX) ? beta / 2.0 : (beta + min_beta) / 2.0;
    }
    ++iter;
  }
  for (int m = l; m < k; m += LANES) val[(size_t)i * k + m] = (float)(exp(-beta_eval * dist[m]) / sum_P);
  if (beta_out && l == 0) beta_out[i] = beta;
}

// ---- lambda rescaling (one thread per row, FP64) --------------------------
__global__ void lambda_kernel(int n, const int32_t *__restrict__ rowptr, float *__restrict__ val,
                              double lambda, int drop_leaf) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double tolBinary = 1e-5;
  const int maxIter = 100;
  double fval = 1.0 - lambda;
  double sig2 = 1.0, a = -1e3, c = INFINITY;
  int iter = 0;
  const int s = rowptr[i], e = rowptr[i + 1];
  while (fabs(fval) > tolBinary && iter < maxIter) {
    ++iter;
    if (fval > 0) {
      a = sig2;
      sig2 = isinf(c) ? 2 * a : 0.5 * (a + c);
    } else {
      c = sig2;
      sig2 = 0.5 * (a + c);
    }
    double sum_i = 0.0;
    for (int j = s; j < e; ++j) sum_i += exp(log((double)val[j]) * sig2);
    fval = sum_i - lambda;
  }
  double sum_i = 0.0;
  for (int j = s; j < e; ++j) sum_i += exp(log((double)val[j]) * sig2);
  for (int j = s; j < e; ++j) val[j] = (float)(exp(log((double)val[j]) * sig2) / sum_i);
  if (drop_leaf && e - s == 1) val[s] = 0.0f;
}

__global__ void rowids_kernel(int n, const int32_t *__restrict__ rowptr, int32_t *__restrict__ row) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  for (int t = rowptr[i]; t < rowptr[i + 1]; ++t) row[t] = i;
}

// ---- P + P^T, row by row -----------------------------------------------------------
// Row i of the merge holds row i of P and, after it, the entries of column i:
// every entry of P takes its place in its column's row from a counter (which
// starts at the length of P's own row), the places are made offsets by a scan,
// and each row is sorted by column in LDS and its duplicates added in FP64.  An
// entry is one 64-bit word, the column above the bits of the value, so rows
// come out the same whatever order the counters gave: 8 bytes per entry read
// and written twice, where a radix sort of (row, column) keys with FP64 values
// moved 32 bytes in each of 6 passes and took about 25 launches for a small
// job.  16 jobs of 500-8000 points admitted to a batch: 48.9 -> 32.9 ms; a whole
// call on 1203 points 1.89 -> 1.52 ms.
//
// Rows by their length: up to kSymRow entries one wave each; up to kSymRowLds a
// work-group each, from a list of them, so that they spread over the device
// wherever they lie; longer ones (hubs) in ranges of kSymCols columns, a work-group
// each, whose sums are kept by column.
constexpr int kSymRow = 1024;
constexpr int kSymRowLds = 8192;
constexpr int kSymCols = 8192;       // columns of a hub's range (FP64 sums: 64 KB of LDS)
constexpr int kSymBelow = 1 << 19;   // columns of one bitmap of those below a range (64 KB)

__global__ void sym_len_kernel(int n, const int32_t *__restrict__ rowptr, int32_t *__restrict__ cnt, SymLong L,
                               int64_t parts) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i <= n) cnt[i] = i < n ? rowptr[i + 1] - rowptr[i] : 0;
  if (i < 2) L.cnt[i] = 0;
  if (i < parts) L.part[i] = 0.0;
}

// pos[t] = place of entry t in the merged row of its column.  A work-group takes
// kPlaceRun entries and counts equal columns in LDS first (a hash table; an entry
// whose slot another column holds goes to the counter itself), so that a hub's
// counter is increased once per work-group: the 900,000 entries of one column
// took 10.2 ms one by one.
constexpr int kPlaceRun = 2048, kPlaceSlots = 4096;

__global__ __launch_bounds__(256) void sym_place_kernel(int64_t nnz, const int32_t *__restrict__ col,
                                                        int32_t *__restrict__ cnt, int32_t *__restrict__ pos) {
  constexpr int U = kPlaceRun / 256;
  __shared__ int tag[kPlaceSlots], num[kPlaceSlots];
  const int tid = threadIdx.x;
  for (int64_t t0 = (int64_t)blockIdx.x * kPlaceRun; t0 < nnz; t0 += (int64_t)gridDim.x * kPlaceRun) {
    for (int i = tid; i < kPlaceSlots; i += 256) {
      tag[i] = -1;
      num[i] = 0;
    }
    __syncthreads();
    int at[U], slot[U];  // place within the slot's column (slot >= 0) or in the row
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t t = t0 + u * 256 + tid;
      if (t < nnz) {
        const int c = col[t];
        slot[u] = (int)(((unsigned)c * 2654435761u) >> 20);
        const int held = atomicCAS(&tag[slot[u]], -1, c);
        if (held == -1 || held == c) {
          at[u] = atomicAdd(&num[slot[u]], 1);
        } else {
          at[u] = atomicAdd(&cnt[c], 1);
          slot[u] = -1;
        }
      }
    }
    __syncthreads();
    for (int i = tid; i < kPlaceSlots; i += 256)
      if (num[i]) num[i] = atomicAdd(&cnt[tag[i]], num[i]);  // now the first place
    __syncthreads();
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t t = t0 + u * 256 + tid;
      if (t < nnz) pos[t] = slot[u] >= 0 ? num[slot[u]] + at[u] : at[u];
    }
    __syncthreads();
  }
}

__device__ __forceinline__ unsigned long long sym_entry(int col, float v) {
  return ((unsigned long long)(unsigned)col << 32) | __float_as_uint(v);
}

__global__ __launch_bounds__(256) void sym_scatter_kernel(int n, const int32_t *__restrict__ rowptr,
                                                          const int32_t *__restrict__ col,
                                                          const float *__restrict__ val,
                                                          const int32_t *__restrict__ off,
                                                          const int32_t *__restrict__ pos,
                                                          unsigned long long *__restrict__ ent) {
  const int lane = threadIdx.x & 63, nw = (gridDim.x * blockDim.x) >> 6;
  for (int i = (blockIdx.x * blockDim.x + threadIdx.x) >> 6; i < n; i += nw) {
    const int t0 = rowptr[i];
    for (int t = t0 + lane; t < rowptr[i + 1]; t += 64) {
      const int c = col[t];
      const float v = val[t];
      ent[off[i] + (t - t0)] = sym_entry(c, v);
      ent[off[c] + pos[t]] = sym_entry(i, v);
    }
  }
}

// Ascending sort of len words (LDS) by the whole work-group: a bitonic network
// whose merges start with a mirrored step, so every exchange is ascending and
// the places past len need no padding.
__device__ void sort_words(unsigned long long *x, int len) {
  auto exchange = [&](int i, int j) {
    if (j < len) {
      const unsigned long long a = x[i], b = x[j];
      if (b < a) {
        x[i] = b;
        x[j] = a;
      }
    }
  };
  int top = 1;  // log2 of the network's size
  while ((1 << top) < len) ++top;
  const int pairs = 1 << (top - 1);
  for (int lg = 1; lg <= top; ++lg) {
    __syncthreads();
    for (int t = threadIdx.x; t < pairs; t += blockDim.x) {
      const int r = t & ((1 << (lg - 1)) - 1), b = (t >> (lg - 1)) << lg;
      exchange(b + r, b + (1 << lg) - 1 - r);
    }
    for (int ls = lg - 2; ls >= 0; --ls) {
      __syncthreads();
      for (int t = threadIdx.x; t < pairs; t += blockDim.x) {
        const int i = ((t >> ls) << (ls + 1)) + (t & ((1 << ls) - 1));
        exchange(i, i + (1 << ls));
      }
    }
  }
  __syncthreads();
}

// Merges one sorted row (x, in LDS): its columns and summed values to mcol / mval
// at the row's place.  Every thread of the work-group calls it; wsum holds 2 + 2 *
// waves words.
__device__ void merge_row(const unsigned long long *x, int len, int32_t *mcol, double *mval, int32_t *ucnt, double *rowsum,
                          double *wsum) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
  int *wcnt = reinterpret_cast<int *>(wsum + nw);
  double sum = 0.0;
  int done = 0;
  unsigned before = 0xFFFFFFFFu;  // column of the word before the round
  for (int b = 0; b < len; b += blockDim.x) {
    const int i = b + threadIdx.x;
    const unsigned c = i < len ? (unsigned)(x[i] >> 32) : 0xFFFFFFFFu;
    const unsigned prev = threadIdx.x == 0 ? before : i - 1 < len ? (unsigned)(x[i - 1] >> 32) : 0xFFFFFFFFu;
    const unsigned last = (unsigned)(x[min(b + (int)blockDim.x, len) - 1] >> 32);
    const bool head = i < len && (i == 0 || prev != c);
    double v = 0.0;
    if (head)
      for (int j = i; j < len && (unsigned)(x[j] >> 32) == c; ++j) v += (double)__uint_as_float((unsigned)x[j]);
    const unsigned long long m = __ballot(head);
    if (lane == 0) wcnt[w] = __popcll(m);
    __syncthreads();
    int at = done + __popcll(m & ((1ull << lane) - 1ull));
    for (int k = 0; k < nw; ++k) {
      if (k < w) at += wcnt[k];
      done += wcnt[k];
    }
    if (head) {
      mcol[at] = (int32_t)c;
      mval[at] = v;
      sum += v;
    }
    before = last;
    __syncthreads();
  }
  sum = wave_sum(sum);
  if (lane == 0) wsum[w] = sum;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k = 1; k < nw; ++k) sum += wsum[k];
    *ucnt = done;
    *rowsum = sum;
  }
  __syncthreads();
}

// Rows of up to kSymRow entries, one wave each; the others are listed.
__global__ __launch_bounds__(64) void sym_merge_kernel(int n, const int32_t *__restrict__ off,
                                                       const unsigned long long *__restrict__ ent,
                                                       int32_t *__restrict__ mcol, double *__restrict__ mval,
                                                       int32_t *__restrict__ ucnt, double *__restrict__ rowsum,
                                                       SymLong L) {
  __shared__ unsigned long long x[kSymRow];
  __shared__ double wsum[4];
  for (int r = blockIdx.x; r < n; r += gridDim.x) {
    const int o = off[r], len = off[r + 1] - o;
    if (len > kSymRow) {
      if (threadIdx.x == 0) {
        if (len <= kSymRowLds) {
          L.mid[atomicAdd(L.cnt, 1)] = r;
        } else {
          L.hub[atomicAdd(L.cnt + 1, 1)] = r;
          rowsum[r] = 0.0;  // its sum is in its parts
        }
      }
      continue;
    }
    for (int i = threadIdx.x; i < len; i += 64) x[i] = ent[o + i];
    sort_words(x, len);
    merge_row(x, len, mcol + o, mval + o, ucnt + r, rowsum + r, wsum);
  }
}

// The listed rows of up to kSymRowLds entries, a work-group each, bound by the
// barriers of the sort: a job of 20,000 points with rows of 1200 added to a batch 7.1
// ms (28 when a work-group walked the long rows of its 1024 neighbours).
__global__ __launch_bounds__(1024) void sym_merge_mid_kernel(const int32_t *__restrict__ off,
                                                             const unsigned long long *__restrict__ ent,
                                                             int32_t *__restrict__ mcol, double *__restrict__ mval,
                                                             int32_t *__restrict__ ucnt, double *__restrict__ rowsum,
                                                             SymLong L) {
  extern __shared__ unsigned long long xl[];
  __shared__ double wsum[32];
  const int rows = L.cnt[0];
  for (int q = blockIdx.x; q < rows; q += gridDim.x) {
    const int row = L.mid[q], o = off[row], len = off[row + 1] - o;
    for (int i = threadIdx.x; i < len; i += 1024) xl[i] = ent[o + i];
    sort_words(xl, len);
    merge_row(xl, len, mcol + o, mval + o, ucnt + row, rowsum + row, wsum);
  }
}

// Sum over the work-group's 16 waves of a count each thread holds, and the sum
// over the threads before this one.
__device__ int block_scan(int v, int *wcnt, int *before) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  int inc = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int u = __shfl_up(inc, o, 64);
    if (lane >= o) inc += u;
  }
  if (lane == 63) wcnt[w] = inc;
  __syncthreads();
  int all = 0, base = 0;
  for (int k = 0; k < 16; ++k) {
    if (k < w) base += wcnt[k];
    all += wcnt[k];
  }
  __syncthreads();
  *before = base + inc - v;
  return all;
}

// Ranges of kSymCols columns that one work-group of a hub takes in turn, and the
// work-groups of a hub (at most kHubParts).
constexpr int kHubParts = 256;
__host__ __device__ inline int hub_run(int n) { return (n / kSymCols + kHubParts) / kHubParts; }
__host__ __device__ inline int hub_parts(int n) { return (n - 1) / (kSymCols * hub_run(n)) + 1; }

// The hubs: a work-group takes a range of kSymCols columns of one row, reads the
// whole row, adds the values of its columns in LDS by column and counts the
// distinct columns below the range (a bitmap), which is where its part of the
// merged row starts.  No sort, and no limit on the length of a row.  A column has
// two entries (P_ij and P_ji), whose sum does not depend on their order, unless P
// holds an entry more than once: then the FP64 sums are exact, in any order, for
// values within 2^29 of each other.  Bound by the reads of the row, once per range.
// A job of 1M points with a hub of 900,000 added to a batch: 141 ms with the row
// sorted in memory by one work-group, 15 so (its hub 0.75); 200,000 points with
// eight hubs of 100,000: 79 and 3.5.
__global__ __launch_bounds__(1024) void sym_merge_hub_kernel(int n, const int32_t *__restrict__ off,
                                                             const unsigned long long *__restrict__ ent,
                                                             int32_t *__restrict__ mcol, double *__restrict__ mval,
                                                             int32_t *__restrict__ ucnt, SymLong L) {
  extern __shared__ double acc[];  // [kSymCols], then the two bitmaps
  unsigned *mine = reinterpret_cast<unsigned *>(acc + kSymCols), *below = mine + kSymCols / 32;
  __shared__ int wcnt[16];
  __shared__ double wsum[16];
  constexpr int PER = kSymCols / 1024;  // columns of a thread
  static_assert(PER == 8, "a thread's columns are one byte of the bitmap");
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int parts = hub_parts(n), run = hub_run(n);
  const int64_t items = (int64_t)L.cnt[1] * parts;
  for (int64_t it = blockIdx.x; it < items; it += gridDim.x) {
    const int row = L.hub[it / parts], j = (int)(it % parts);
    const int o = off[row], len = off[row + 1] - o;
    int start = 0;  // distinct columns below the range
    double part = 0.0;
    for (int r = 0; r < run; ++r) {
      const unsigned c0 = ((unsigned)j * run + r) * kSymCols;
      if (c0 >= (unsigned)n) break;
      for (int i = tid; i < kSymCols; i += 1024) acc[i] = 0.0;
      if (tid < kSymCols / 32) mine[tid] = 0;
      // the first range counts those below it, one bitmap's columns at a time;
      // each range's own columns are added in the first pass
      const unsigned c1 = r == 0 ? c0 : 0;
      for (unsigned lo = 0;; lo += kSymBelow) {
        const unsigned hi = min(c1, lo + kSymBelow);
        for (unsigned i = tid; i < (hi - lo + 31) / 32; i += 1024) below[i] = 0;
        __syncthreads();
#pragma unroll 4
        for (int i = tid; i < len; i += 1024) {
          const unsigned long long x = ent[o + i];
          const unsigned c = (unsigned)(x >> 32);
          if (c - c0 < (unsigned)kSymCols) {
            if (lo == 0) {
              atomicAdd(&acc[c - c0], (double)__uint_as_float((unsigned)x));
              atomicOr(&mine[(c - c0) / 32], 1u << (c % 32));
            }
          } else if (c - lo < hi - lo) {
            atomicOr(&below[(c - lo) / 32], 1u << (c % 32));
          }
        }
        __syncthreads();
        int cnt = 0, before;
        for (unsigned i = tid; i < (hi - lo + 31) / 32; i += 1024) cnt += __popc(below[i]);
        start += block_scan(cnt, wcnt, &before);
        if (hi == c1) break;
      }
      const unsigned bits = (mine[tid / 4] >> (8 * (tid % 4))) & 0xFFu;
      int at;
      const int total = block_scan(__popc(bits), wcnt, &at);
      at += o + start;
#pragma unroll
      for (int e = 0; e < PER; ++e)
        if ((bits >> e) & 1u) {
          const double v = acc[tid * PER + e];
          mcol[at] = (int32_t)(c0 + tid * PER + e);
          mval[at++] = v;
          part += v;
        }
      start += total;
      __syncthreads();  // the sums are read
    }
    part = wave_sum(part);
    if (lane == 0) wsum[w] = part;
    __syncthreads();
    if (tid == 0) {
      for (int k = 1; k < 16; ++k) part += wsum[k];
      L.part[it] = part;
      L.end[it] = start;
      if (j == parts - 1) ucnt[row] = start;
    }
    __syncthreads();
  }
}

// The merged rows, normalised by the sum of all of them, side by side: a wave for
// each row, a work-group for each part of a hub.
__global__ __launch_bounds__(256) void sym_finish_kernel(int n, const int32_t *__restrict__ off,
                                                         const int32_t *__restrict__ rp,
                                                         const int32_t *__restrict__ mcol,
                                                         const double *__restrict__ mval,
                                                         const double *__restrict__ total,
                                                         int32_t *__restrict__ rowptr, int32_t *__restrict__ col,
                                                         float *__restrict__ val, SymLong L) {
  const int lane = threadIdx.x & 63, nw = (gridDim.x * blockDim.x) >> 6;
  const double tot = *total;
  const int parts = hub_parts(n);
  const int64_t items = (int64_t)L.cnt[1] * parts;
  for (int64_t it = blockIdx.x; it < items; it += gridDim.x) {
    const int row = L.hub[it / parts], o = off[row], p = rp[row];
    for (int e = (it % parts ? L.end[it - 1] : 0) + threadIdx.x; e < L.end[it]; e += blockDim.x) {
      col[p + e] = mcol[o + e];
      val[p + e] = (float)(mval[o + e] / tot);
    }
  }
  for (int i = (blockIdx.x * blockDim.x + threadIdx.x) >> 6; i < n; i += nw) {
    const int o = off[i], p = rp[i], m = rp[i + 1] - p;
    if (lane == 0) rowptr[i] = p;
    if (i == n - 1 && lane == 0) rowptr[n] = rp[n];
    if (off[i + 1] - o > kSymRowLds) continue;
    for (int e = lane; e < m; e += 64) {
      col[p + e] = mcol[o + e];
      val[p + e] = (float)(mval[o + e] / tot);
    }
  }
}

// ---- hybrid ELL + COO tail ----------------------------------------------------
__global__ void build_ell_kernel(int n, int width, const int32_t *__restrict__ rowptr,
                                 const int32_t *__restrict__ col, const float *__restrict__ val,
                                 int32_t *__restrict__ ecol, float *__restrict__ eval,
                                 int32_t *__restrict__ tail_cnt) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n) return;
  const int s = rowptr[r], len = rowptr[r + 1] - s;
  for (int e = 0; e < width; ++e) {
    const int64_t o = (int64_t)e * n + r;
    if (e < len) { ecol[o] = col[s + e]; eval[o] = val[s + e]; }
    else { ecol[o] = r; eval[o] = 0.0f; }
  }
  tail_cnt[r] = len > width ? len - width : 0;
}

__global__ void build_tail_kernel(int n, int width, const int32_t *__restrict__ rowptr,
                                  const int32_t *__restrict__ col, const float *__restrict__ val,
                                  const int32_t *__restrict__ tail_off, int32_t *__restrict__ trow,
                                  int32_t *__restrict__ tcol, float *__restrict__ tval) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n) return;
  const int s = rowptr[r], len = rowptr[r + 1] - s;
  int o = tail_off[r];
  for (int e = width; e < len; ++e, ++o) {
    trow[o] = r;
    tcol[o] = col[s + e];
    tval[o] = val[s + e];
  }
}

// ---- symmetric permutation of P: new row r = old row perm[r], columns
// relabelled by iperm (locality order; the values are untouched) -----------
__global__ void perm_len_kernel(int n, const int32_t *__restrict__ perm, const int32_t *__restrict__ rp,
                                int32_t *__restrict__ len) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n) return;
  const int o = perm[r];
  len[r] = rp[o + 1] - rp[o];
}

__global__ void perm_fill_kernel(int n, const int32_t *__restrict__ perm, const int32_t *__restrict__ iperm,
                                 const int32_t *__restrict__ rp, const int32_t *__restrict__ col,
                                 const float *__restrict__ val, const int32_t *__restrict__ rp2,
                                 int32_t *__restrict__ col2, float *__restrict__ val2) {
  // one wavefront per new row
  const int r = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const int lane = threadIdx.x & 63;
  if (r >= n) return;
  const int o = perm[r];
  const int s0 = rp[o], len = rp[o + 1] - s0, d0 = rp2[r];
  for (int e = lane; e < len; e += 64) {
    col2[d0 + e] = iperm[col[s0 + e]];
    val2[d0 + e] = val[s0 + e];
  }
}

// Columns ascending within each row, in place, on the device alone: one
// work-group per row sorts its (column, value) pairs with a bitonic sort in
// LDS.  Rows longer than kRowSortMax keep their order (the order of a row
// only changes which lanes gather neighbouring points, never the result's
// definition), so nothing here needs the host.
constexpr int kRowSortMax = 4096;

__global__ __launch_bounds__(256) void row_sort_kernel(int n, const int32_t *__restrict__ rp, int32_t *__restrict__ col,
                                                       float *__restrict__ val) {
  __shared__ int32_t kc[kRowSortMax];
  __shared__ float kv[kRowSortMax];
  const int r = blockIdx.x;
  if (r >= n) return;
  const int b = rp[r], len = rp[r + 1] - b;
  if (len < 2 || len > kRowSortMax) return;  // the whole work-group leaves together
  int P = 2;
  while (P < len) P <<= 1;
  for (int t = threadIdx.x; t < P; t += blockDim.x) {
    kc[t] = t < len ? col[b + t] : INT_MAX;
    kv[t] = t < len ? val[b + t] : 0.0f;
  }
  __syncthreads();
  for (int size = 2; size <= P; size <<= 1)
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      for (int t = threadIdx.x; t < P / 2; t += blockDim.x) {
        const int i = 2 * stride * (t / stride) + (t % stride), j = i + stride;
        const bool up = (i & size) == 0;
        const int ci = kc[i], cj = kc[j];
        if ((ci > cj) == up) {
          kc[i] = cj;
          kc[j] = ci;
          const float v = kv[i];
          kv[i] = kv[j];
          kv[j] = v;
        }
      }
      __syncthreads();
    }
  for (int t = threadIdx.x; t < len; t += blockDim.x) {
    col[b + t] = kc[t];
    val[b + t] = kv[t];
  }
}

// ---- spatial order of the embedding -------------------------------------------
// Morton key of each point's position on a 2^B-per-axis lattice over the
// bounding box (B = 16 / 10 / 32 bits per axis for d = 2 / 3 / 1).
__device__ __forceinline__ uint32_t spread_bits2(uint32_t x) {
  x &= 0xffffu;
  x = (x | (x << 8)) & 0x00ff00ffu;
  x = (x | (x << 4)) & 0x0f0f0f0fu;
  x = (x | (x << 2)) & 0x33333333u;
  x = (x | (x << 1)) & 0x55555555u;
  return x;
}
__device__ __forceinline__ uint32_t spread_bits3(uint32_t x) {
  x &= 0x3ffu;
  x = (x | (x << 16)) & 0x030000ffu;
  x = (x | (x << 8)) & 0x0300f00fu;
  x = (x | (x << 4)) & 0x030c30c3u;
  x = (x | (x << 2)) & 0x09249249u;
  return x;
}

__global__ void morton_kernel(int n, int d, int ds, const float *__restrict__ Y, float lo0, float lo1, float lo2,
                              float inv, uint32_t *__restrict__ key, int32_t *__restrict__ idx) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float lo[3] = {lo0, lo1, lo2};
  uint32_t q[3] = {0, 0, 0};
  const float top = d == 1 ? 4294967040.0f : d == 2 ? 65535.0f : 1023.0f;
  for (int a = 0; a < d; ++a) {
    float t = (Y[(size_t)i * ds + a] - lo[a]) * inv * top;
    t = fminf(fmaxf(t, 0.0f), top);  // NaN -> 0
    q[a] = (uint32_t)t;
  }
  uint32_t k;
  if (d == 1) k = q[0];
  else if (d == 2) k = spread_bits2(q[0]) | (spread_bits2(q[1]) << 1);
  else k = spread_bits3(q[0]) | (spread_bits3(q[1]) << 1) | (spread_bits3(q[2]) << 2);
  key[i] = k;
  idx[i] = i;
}

__global__ void invert_perm_kernel(int n, const int32_t *__restrict__ order, int32_t *__restrict__ inv) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r < n) inv[order[r]] = r;
}

__global__ void gather_points_kernel(int n, int ds, const int32_t *__restrict__ order, const float *__restrict__ in,
                                     float *__restrict__ out) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (int64_t)n * ds) return;
  const int r = (int)(t / ds), a = (int)(t % ds);
  out[t] = in[(int64_t)order[r] * ds + a];
}

}  // namespace

namespace {

constexpr size_t kKnnSlabBytes = (size_t)1 << 29;

// Whether the rows of nq slots come sooner from heaps.  Picoseconds per pair,
// fitted to 10,000-400,000 points of 2-200 dimensions, k = 10-1000: a slab's rows
// get fewer as n grows, so the selection leaves the device idle (one work-group
// per row; 24 ps at 200,000 points); the heaps' tiles are small (0.14 against
// 0.06 per dimension), their merges serial (k per row), and a list of few slots
// does not fill the device with work-groups of 64.  All rows, slabs / heaps:
// 20,000 x 50, k = 90 8.3 / 16.8 ms; 60,000 x 5, k = 90 41.6 / 31.1; 200,000 x
// 50, k = 90 1091 / 424; 200,000 x 5, k = 10 957 / 78; 100,000 x 200, k = 90
// 262 / 380; 200,000 x 50, k = 1000 1355 / 1849.  The rule took the slower
// by more than 15 % only below 30,000 points (k below 30 in few dimensions) and
// at 60,000 x 20, k = 90.
bool knn_heaps_better(int n, int dim, int k, int nq) {
  const double slabs = 2.5 + 1.05e-4 * n + 0.064 * dim;
  const double heaps = std::max(1.2 + 0.144 * dim + 4500.0 * k / n, (55000.0 + 4800.0 * dim) / nq);
  return heaps < slabs;
}

// knn_exact_rows by heaps, in groups of slots whose heaps take 512 MB (of fewer
// when there is no memory for that).
int knn_heap_rows(hipStream_t s, ScratchSource &src, const float *X, int n, int dim, int k, const int *qlist, int nq, int32_t *I,
                  double *D) {
  const size_t row = (sizeof(double) + sizeof(int)) * (size_t)k;
  int slab = (int)std::min<int64_t>(nq, (int64_t)(kKnnSlabBytes / row));
  void *block = nullptr;
  for (;;) {
    const int st = src.take(s, row * slab, &block);
    if (st == SGTSNE_OK) break;
    if (slab == 1) return st;
    slab = div_up(slab, 2);
  }
  double *hd = static_cast<double *>(block);
  int *hi = reinterpret_cast<int *>(hd + (size_t)slab * k);
  auto rows = [&](int s0) -> int {
    const int m = std::min(slab, nq - s0);
    knn_heap_kernel<<<div_up(m, kHeapQ), kKnnThreads, 0, s>>>(X, n, dim, k, hd, hi, qlist, s0, m);
    SGT_LAUNCH_CHECK();
    knn_heap_rows_kernel<<<div_up(m, 256), 256, 0, s>>>(s0, m, k, hd, hi, qlist, I, D);
    SGT_LAUNCH_CHECK();
    return SGTSNE_OK;
  };
  int st = SGTSNE_OK;
  for (int s0 = 0; s0 < nq && !st; s0 += slab) st = rows(s0);
  src.give(s, block);
  return st;
}

// Exact kNN of the query slots [0, nq) (points qlist[slot], or all points),
// in slabs of slots whose distances to every point take 512 MB, or of 128 slots
// where those take more (1.3 GB at 1.3M points: whole tiles, and work-groups
// enough for the selection); when there is no memory for that, of fewer.
// All points of a matrix that fits one slab (n <= 8192): mirrored tiles of 128
// x 128.  Lists of up to 256 slots (rows the certificate left) take tiles of
// 32 x 64, which spread a few rows over the device: 128 x 128 tiles would
// leave n / 128 work-groups.  Measured: 6007 points of 784 dimensions 1.40 ms
// for the distances (10 T pair-dimensions/s, of two FP64 operations each: half of
// the 39 T operations/s that FP64 issue allows)
// and 0.17 ms for the selection (one work-group per 64 queries with serial
// heaps: 37.1 ms); the 82 uncertified rows of a 20,011-point 50-D job 0.08 ms
// (11.5 ms).  Slabs of up to 64 slots take the small tiles too.  Where heaps are
// the faster way to the same rows (knn_heaps_better) they are taken.
int knn_exact_rows(hipStream_t s, ScratchSource &src, const float *X, int n, int dim, int k, const int *qlist, int nq, int32_t *I,
                   double *D) {
  if (knn_heaps_better(n, dim, k, nq)) return knn_heap_rows(s, src, X, n, dim, k, qlist, nq, I, D);
  int slab = (int)std::min<int64_t>(nq, std::max<int64_t>(128, (int64_t)(kKnnSlabBytes / 8 / n) / 128 * 128));
  void *block = nullptr;
  for (;;) {
    const int st = src.take(s, sizeof(double) * (size_t)slab * n, &block);
    if (st == SGTSNE_OK) break;
    if (slab == 1) return st;
    slab = slab > 64 ? (slab / 2 + 31) / 32 * 32 : slab / 2;
  }
  const int mirror = !qlist && nq == n && slab == n;
  const bool few = slab <= 64 || (qlist && nq <= 256);
  double *dist = static_cast<double *>(block);
  auto rows = [&](int s0) -> int {
    const int m = std::min(slab, nq - s0);
    if (few)
      knn_dist_kernel<2, 4><<<dim3(div_up(n, 64), div_up(m, 32)), kKnnThreads, 0, s>>>(X, n, dim, qlist, s0, m, 0, dist);
    else
      knn_dist_kernel<8, 8><<<dim3(div_up(n, 128), div_up(m, 128)), kKnnThreads, 0, s>>>(X, n, dim, qlist, s0, m,
                                                                                        mirror, dist);
    SGT_LAUNCH_CHECK();
    if (k <= 256)
      knn_select_kernel<512><<<m, kKnnThreads, 0, s>>>(dist, n, k, qlist, s0, I, D);
    else
      knn_select_kernel<2 * kKnnMaxK><<<m, kKnnThreads, 0, s>>>(dist, n, k, qlist, s0, I, D);
    SGT_LAUNCH_CHECK();
    return SGTSNE_OK;
  };
  int st = SGTSNE_OK;
  for (int s0 = 0; s0 < nq && !st; s0 += slab) st = rows(s0);
  src.give(s, block);
  return st;
}

}  // namespace

int knn_begin(hipStream_t s, ScratchSource &src, const float *X, int n, int dim, int k, int32_t *I, double *D,
              int method, int *count_host, KnnPending *pend) {
  *pend = KnnPending{};
  pend->src = &src;
  SGT_CHECK(n > k && k >= 1 && dim >= 1, SGTSNE_ERR_ARG, "kNN needs n > k >= 1 (n=%d k=%d)", n, k);
  SGT_CHECK(k <= kKnnMaxK, SGTSNE_ERR_ARG, "k too large");
  const bool filter_ok = k + kFiltSlack <= kRerank && dim <= kFiltMaxDp && n >= kFiltQ;
  if (method == SGTSNE_KNN_EXACT_FP64 || (method == SGTSNE_KNN_AUTO && !filter_ok))
    return knn_exact_rows(s, src, X, n, dim, k, nullptr, n, I, D);  // nothing left for knn_end
  SGT_CHECK(filter_ok, SGTSNE_ERR_ARG, "the filtered kNN needs k <= %d, dim <= %d and n >= %d",
            kRerank - kFiltSlack, kFiltMaxDp, kFiltQ);
  const int kp = std::min(k + kFiltSlack, n - 1);
  const int nst = filter_steps(dim, kp), dp = 4 * nst;
  const bool blocked = kp <= kF2MaxKp;  // the list filter centres each query block
  const int nb = div_up(n, kF2Q);
  // point order: cell (nearest of P pivots), then the Morton code of a 3-D
  // projection of the centred points; the query blocks and the reference
  // tiles both follow it, the tiles padded so each lies in one cell
  const int P = std::min(kKnnMaxCells, std::max(1, n / 512));
  const int ntiles = div_up(n + (kFiltR - 1) * P, kFiltR);  // at least the padded slots
  size_t tb = 0;
  if (blocked)
    SGT_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, tb, (uint32_t *)nullptr, (uint32_t *)nullptr,
                                               (int32_t *)nullptr, (int32_t *)nullptr, n, 0, 30, s));
  double *mu, *nrm, *qdn, *cb = nullptr, *dn = nullptr, *qa = nullptr, *tcen = nullptr, *trad = nullptr;
  float *Xc, *n32, *hd, *Xq = nullptr, *qn32 = nullptr, *delta = nullptr, *Xr = nullptr;
  int *hi, *fb;
  int32_t *kidx = nullptr, *qorder = nullptr, *cell = nullptr, *rid = nullptr, *rinv = nullptr;
  int *ccnt, *slot0;  // per cell: points, first slot
  double *parts;
  uint32_t *key0 = nullptr, *key1 = nullptr;
  void *tmp = nullptr;
  unsigned long long *rmax;
  // one block for every temporary: a stream-ordered allocation and its release
  // hold the host for 50 us and more
  for (int pass = 0; pass < 2; ++pass) {
    Carve c{static_cast<char *>(pend->ws)};
    rmax = c.take<unsigned long long>(1);
    ccnt = c.take<int>(kKnnMaxCells);
    fb = c.take<int>((size_t)n + 1);  // [0]: count, then rows
    slot0 = c.take<int>(kKnnMaxCells);
    parts = c.take<double>((size_t)kMeanParts * dim);
    mu = c.take<double>(dim);
    nrm = c.take<double>(n);
    qdn = c.take<double>(n);
    Xc = c.take<float>((size_t)n * dp);
    n32 = c.take<float>(n);
    hd = c.take<float>((size_t)n * kp);
    hi = c.take<int>((size_t)n * kp);
    if (blocked) {
      key0 = c.take<uint32_t>(n);
      key1 = c.take<uint32_t>(n);
      kidx = c.take<int32_t>(n);
      qorder = c.take<int32_t>(n);
      cb = c.take<double>((size_t)nb * dim);
      delta = c.take<float>((size_t)nb * dp);
      dn = c.take<double>(nb);
      Xq = c.take<float>((size_t)n * dp);
      qn32 = c.take<float>(n);
      qa = c.take<double>(n);
      cell = c.take<int32_t>(n);
      rid = c.take<int32_t>((size_t)ntiles * kFiltR);
      rinv = c.take<int32_t>(n);
      Xr = c.take<float>((size_t)ntiles * kFiltR * dp);
      tcen = c.take<double>((size_t)ntiles * dim);
      trad = c.take<double>(ntiles);
      tmp = c.take<char>(tb);
    }
    if (pass == 0) SGT_TRY(src.take(s, c.off, &pend->ws));
  }
  pend->open = true;  // from here on a failure releases the block
  // the largest norm, the cells' counts and the count of uncertified rows
  SGT_HIP(hipMemsetAsync(rmax, 0, reinterpret_cast<char *>(fb + 1) - reinterpret_cast<char *>(rmax), s));
  const int nparts = std::min(kMeanParts, div_up(n, 64));
  knn_mean_kernel<<<nparts, 256, 0, s>>>(X, n, dim, parts);
  SGT_LAUNCH_CHECK();
  knn_center_kernel<<<div_up(n, kCentreRows), 256, 0, s>>>(X, n, dim, dp, parts, nparts, mu, Xc, n32, nrm, rmax);
  SGT_LAUNCH_CHECK();
  BlockCentred bc{};
  if (blocked) {
    knn_cell_kernel<<<div_up(n, 64), 256, sizeof(float) * P * dp, s>>>(Xc, n, dim, dp, P, rmax, cell, ccnt, key0,
                                                                       kidx);
    SGT_LAUNCH_CHECK();
    SGT_HIP(hipcub::DeviceRadixSort::SortPairs(tmp, tb, key0, key1, kidx, qorder, n, 0, 30, s));
    knn_tile_kernel<<<ntiles, 256, 0, s>>>(X, Xc, dim, dp, P, qorder, ccnt, slot0, Xr, rid, rinv, tcen, trad);
    SGT_LAUNCH_CHECK();
    knn_frame_kernel<<<nb, 256, 0, s>>>(X, n, dim, dp, qorder, mu, cb, delta, dn, Xq, qn32, qa, qdn);
    SGT_LAUNCH_CHECK();
    bc = BlockCentred{Xq, qn32, qorder, delta,
                      RefTiles{Xr, rid, rinv, ntiles, tcen, trad, cb, qa, dn, rmax, dim, cell, slot0}};
  } else {
    SGT_HIP(hipMemsetAsync(qdn, 0, sizeof(double) * (size_t)n, s));  // frame of every query: mu
  }
  SGT_TRY(launch_filter_for(s, nst, Xc, n32, n, kp, bc, hd, hi));
  // error constants (unit roundoff u = 2^-24): the squared distance from the
  // filter is within (2 dp + 3) u (|a| + |b|)^2 of that of the FP32 vectors
  // under round-to-nearest; allowing twice that covers directed rounding in
  // the accumulation, and 1e-30 covers underflow.  The FP32 roundings of the
  // centred points move a distance by at most 1.01 u (|a| + R + |c - mu| + |b|).
  const double u = std::ldexp(1.0, -24);
  const double cE = 2.0 * (2.0 * dp + 8.0) * u, ce = 1.05 * u;
  SGT_TRY((kp <= 128 ? launch_rerank<2> : launch_rerank<4>)(s, X, n, dim, k, kp, hd, hi, blocked ? qa : nrm, qdn, rmax, cE,
                                                            ce, I, D, fb + 1, fb));
  SGT_HIP(hipMemcpyAsync(count_host, fb, sizeof(int), hipMemcpyDeviceToHost, s));
  pend->X = X;
  pend->n = n;
  pend->dim = dim;
  pend->k = k;
  pend->I = I;
  pend->D = D;
  pend->fb = fb;
  pend->count_host = count_host;
  return SGTSNE_OK;
}

void knn_release(hipStream_t s, KnnPending *kp) {
  if (kp->ws) kp->src->give(s, kp->ws);
  *kp = KnnPending{};
}

int knn_end(hipStream_t s, KnnPending *kp, int *fallback_rows) {
  if (!kp->open) {  // exact rows throughout
    if (fallback_rows) *fallback_rows = -1;
    return SGTSNE_OK;
  }
  const int nfb = *kp->count_host;
  int st = SGTSNE_OK;
  if (nfb > 0) st = knn_exact_rows(s, *kp->src, kp->X, kp->n, kp->dim, kp->k, kp->fb + 1, nfb, kp->I, kp->D);
  if (fallback_rows) *fallback_rows = nfb;
  knn_release(s, kp);
  return st;
}

int launch_knn(hipStream_t s, const float *X, int n, int dim, int k, int32_t *I, double *D, int method,
               int *fallback_rows) {
  if (fallback_rows) *fallback_rows = -1;
  int nfb = 0;
  KnnPending kp;
  const int st = knn_begin(s, stream_scratch(), X, n, dim, k, I, D, method, &nfb, &kp);
  if (st) {
    knn_release(s, &kp);
    return st;
  }
  if (kp.open && hipStreamSynchronize(s) != hipSuccess) {
    knn_release(s, &kp);
    set_error("kNN failed");
    return SGTSNE_ERR_HIP;
  }
  return knn_end(s, &kp, fallback_rows);
}

int launch_perplexity(hipStream_t s, const double *D, int n, int k, double u, float *val,
                      double *beta_out) {
  // 64 lanes per point would gain 4 us up to 1000 points (27 us) and lose above
  // 1500; held in registers: 40 -> 29 us at 4000 points, 80 -> 70 at 16,000
  const int blocks = div_up(n, 16);
  if (k <= 96) perplexity_kernel2<16, 6><<<blocks, 256, 0, s>>>(D, n, k, u, val, beta_out);
  else if (k <= 160) perplexity_kernel2<16, 10><<<blocks, 256, 0, s>>>(D, n, k, u, val, beta_out);
  else perplexity_kernel2<16, 0><<<blocks, 256, 0, s>>>(D, n, k, u, val, beta_out);
  SGT_LAUNCH_CHECK();
  return SGTSNE_OK;
}

int launch_lambda_rescale(hipStream_t s, int n, const int32_t *rowptr, float *val, double lambda,
                          int drop_leaf) {
  lambda_kernel<<<div_up(n, 128), 128, 0, s>>>(n, rowptr, val, lambda, drop_leaf);
  SGT_LAUNCH_CHECK();
  return SGTSNE_OK;
}

int launch_rowids(hipStream_t s, int n, const int32_t *rowptr, int32_t *row) {
  rowids_kernel<<<div_up(n, 256), 256, 0, s>>>(n, rowptr, row);
  SGT_LAUNCH_CHECK();
  return SGTSNE_OK;
}

// Keeps memory freed to the device's stream-ordered pool cached in the pool:
// with the default release threshold (0) every synchronisation returns it to
// the driver, and the next hipMallocAsync blocks the host to map it again.
// Cross-stream reuse is limited to what stream order and recorded events
// prove: a block freed on one stream is handed to another only through an
// event dependency the caller made, never because the runtime saw the free
// complete (opportunistic) or inserted a wait of its own (internal
// dependencies).
void retain_pool_memory() {
  int dev = 0;
  hipMemPool_t pool = nullptr;
  if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetDefaultMemPool(&pool, dev) != hipSuccess) return;
  uint64_t keep = UINT64_MAX;
  (void)hipMemPoolSetAttribute(pool, hipMemPoolAttrReleaseThreshold, &keep);
  int off = 0;
  (void)hipMemPoolSetAttribute(pool, hipMemPoolReuseAllowOpportunistic, &off);
  (void)hipMemPoolSetAttribute(pool, hipMemPoolReuseAllowInternalDependencies, &off);
}

ScratchSource &stream_scratch() {
  struct Direct final : ScratchSource {
    int take(hipStream_t s, size_t bytes, void **p) override {
      *p = nullptr;
      SGT_HIP(hipMallocAsync(p, bytes > 0 ? bytes : 1, s));
      return SGTSNE_OK;
    }
    void give(hipStream_t s, void *p) override { (void)hipFreeAsync(p, s); }
  };
  static Direct direct;
  return direct;
}

int device_exclusive_scan(hipStream_t s, const int32_t *in, int32_t *out, int n) {
  size_t tb = 0;
  SGT_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, tb, in, out, n, s));
  void *tmp = nullptr;
  SGT_HIP(hipMallocAsync(&tmp, tb > 0 ? tb : 1, s));
  SGT_HIP(hipcub::DeviceScan::ExclusiveSum(tmp, tb, in, out, n, s));
  SGT_HIP(hipFreeAsync(tmp, s));
  return SGTSNE_OK;
}

int sym_begin(hipStream_t s, ScratchSource &src, int n, int64_t nnz, const int32_t *rowptr_d, const int32_t *col_d,
              const float *val_d, int max_row, int *runs_host, SymPending *sp) {
  *sp = SymPending{};
  sp->src = &src;
  const int64_t m2 = 2 * nnz;
  SGT_CHECK(m2 < (int64_t)INT_MAX, SGTSNE_ERR_ARG, "2*nnz exceeds the int32 range");
  size_t tb = 0, tr = 0;
  SGT_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, tb, (int32_t *)nullptr, (int32_t *)nullptr, n + 1, s));
  // the longest merged row: its own entries and, from each other row, one per
  // column (any number if P may hold an entry more than once)
  const int64_t longest = std::min<int64_t>(m2, max_row > 0 ? (int64_t)n + max_row : m2);
  const bool mids = longest > kSymRow, hubs = longest > kSymRowLds;
  const int64_t nhub = hubs ? m2 / kSymRowLds : 0, parts = hub_parts(n);
  SGT_HIP(hipcub::DeviceReduce::Sum(nullptr, tr, (double *)nullptr, (double *)nullptr, (int)(n + nhub * parts), s));
  int32_t *cnt, *off, *pos, *mcol, *ucnt, *rp;
  unsigned long long *ent;
  double *mval, *rowsum, *total;
  SymLong &L = sp->rows;
  void *tmp;
  for (int pass = 0; pass < 2; ++pass) {  // sizes, then the pieces of the block
    Carve c{static_cast<char *>(sp->ws)};
    cnt = c.take<int32_t>((size_t)n + 1);
    off = c.take<int32_t>((size_t)n + 1);
    pos = c.take<int32_t>(nnz);
    ent = c.take<unsigned long long>(m2);
    mcol = c.take<int32_t>(m2);
    mval = c.take<double>(m2);
    L.cnt = c.take<int>(2);
    L.mid = c.take<int32_t>(mids ? m2 / kSymRow : 0);
    L.hub = c.take<int32_t>(nhub);
    L.end = c.take<int32_t>(nhub * parts);
    ucnt = c.take<int32_t>((size_t)n + 1);
    rp = c.take<int32_t>((size_t)n + 1);
    rowsum = c.take<double>((size_t)n + nhub * parts);
    L.part = rowsum + n;
    total = c.take<double>(1);
    tmp = c.take<char>(std::max(tb, tr));
    if (pass == 0) SGT_TRY(src.take(s, c.off, &sp->ws));
  }
  sp->open = true;
  sp->n = n;
  sp->off = off;
  sp->rp = rp;
  sp->mcol = mcol;
  sp->mval = mval;
  sp->total = total;
  sp->runs_host = runs_host;
  const int wblocks = std::min(div_up(n, 4), 16384);  // four waves of a row each
  sym_len_kernel<<<div_up(std::max<int64_t>((int64_t)n + 1, nhub * parts), 256), 256, 0, s>>>(n, rowptr_d, cnt, L, nhub * parts);
  SGT_LAUNCH_CHECK();
  if (nnz > 0) sym_place_kernel<<<(int)std::min<int64_t>((nnz + kPlaceRun - 1) / kPlaceRun, 65536), 256, 0, s>>>(nnz, col_d, cnt, pos);
  SGT_LAUNCH_CHECK();
  SGT_HIP(hipcub::DeviceScan::ExclusiveSum(tmp, tb, cnt, off, n + 1, s));
  sym_scatter_kernel<<<wblocks, 256, 0, s>>>(n, rowptr_d, col_d, val_d, off, pos, ent);
  SGT_LAUNCH_CHECK();
  sym_merge_kernel<<<std::min(n, 65536), 64, 0, s>>>(n, off, ent, mcol, mval, ucnt, rowsum, L);
  SGT_LAUNCH_CHECK();
  if (mids) {  // two work-groups per CU
    sym_merge_mid_kernel<<<(int)std::min<int64_t>(m2 / kSymRow, 512), 1024, sizeof(unsigned long long) * kSymRowLds, s>>>(
        off, ent, mcol, mval, ucnt, rowsum, L);
    SGT_LAUNCH_CHECK();
  }
  if (hubs) {  // one per CU
    sym_merge_hub_kernel<<<(int)std::min<int64_t>(nhub * parts, 256), 1024,
                           sizeof(double) * kSymCols + (kSymCols + kSymBelow) / 8, s>>>(n, off, ent, mcol, mval, ucnt, L);
    SGT_LAUNCH_CHECK();
  }
  SGT_HIP(hipcub::DeviceScan::ExclusiveSum(tmp, tb, ucnt, rp, n + 1, s));  // ucnt[n] is not read into rp
  SGT_HIP(hipcub::DeviceReduce::Sum(tmp, tr, rowsum, total, (int)(n + nhub * parts), s));  // rows, then hubs' parts
  SGT_HIP(hipMemcpyAsync(runs_host, rp + n, sizeof(int), hipMemcpyDeviceToHost, s));
  return SGTSNE_OK;
}

// Gives back the arrays of sym_end.
static void sym_free(hipStream_t s, int32_t *rp, int32_t *cc, float *vv, ScratchSource *out_src) {
  if (out_src) {
    out_src->give(s, rp);  // one block, which starts at rowptr
    return;
  }
  if (rp) (void)hipFree(rp);
  if (cc) (void)hipFree(cc);
  if (vv) (void)hipFree(vv);
}

void sym_release(hipStream_t s, SymPending *sp) {
  if (sp->ws) sp->src->give(s, sp->ws);
  *sp = SymPending{};
}

int sym_end(hipStream_t s, SymPending *sp, int32_t **rowptr_out, int32_t **col_out, float **val_out,
            int64_t *nnz_out, ScratchSource *out_src) {
  SGT_CHECK(sp->open, SGTSNE_ERR_STATE, "no symmetrisation pending");
  const int n = sp->n;
  const int runs = *sp->runs_host;
  int32_t *rp = nullptr, *cc = nullptr;
  float *vv = nullptr;
  if (out_src) {
    void *block = nullptr;
    for (int pass = 0; pass < 2; ++pass) {
      Carve c{static_cast<char *>(block)};
      rp = c.take<int32_t>((size_t)n + 1);
      cc = c.take<int32_t>(runs);
      vv = c.take<float>(runs);
      if (pass == 0) SGT_TRY(out_src->take(s, c.off, &block));
    }
  } else if (hipMalloc((void **)&rp, sizeof(int32_t) * ((size_t)n + 1)) != hipSuccess ||
             hipMalloc((void **)&cc, sizeof(int32_t) * (size_t)(runs > 0 ? runs : 1)) != hipSuccess ||
             hipMalloc((void **)&vv, sizeof(float) * (size_t)(runs > 0 ? runs : 1)) != hipSuccess) {
    (void)hipGetLastError();
    sym_free(s, rp, cc, vv, nullptr);
    set_error("no memory for P + P^T (%d nonzeros)", runs);
    return SGTSNE_ERR_NOMEM;
  }
  sym_finish_kernel<<<std::min(div_up(n, 4), 16384), 256, 0, s>>>(n, sp->off, sp->rp, sp->mcol, sp->mval, sp->total,
                                                                  rp, cc, vv, sp->rows);
  if (const hipError_t e = hipGetLastError(); e != hipSuccess) {
    sym_free(s, rp, cc, vv, out_src);
    set_error("P + P^T failed: %s", hipGetErrorString(e));
    return SGTSNE_ERR_HIP;
  }
  sym_release(s, sp);
  *rowptr_out = rp;
  *col_out = cc;
  *val_out = vv;
  *nnz_out = runs;
  return SGTSNE_OK;
}

int gpu_symmetrize(hipStream_t s, int n, int64_t nnz, const int32_t *rowptr_d, const int32_t *col_d,
                   const float *val_d, int32_t **rowptr_out, int32_t **col_out, float **val_out,
                   int64_t *nnz_out, ScratchSource *out_src) {
  int runs = 0;
  SymPending sp;
  int32_t *rp = nullptr, *cc = nullptr;
  float *vv = nullptr;
  auto wait = [&]() -> int {
    SGT_HIP(hipStreamSynchronize(s));
    return SGTSNE_OK;
  };
  int st = sym_begin(s, out_src ? *out_src : stream_scratch(), n, nnz, rowptr_d, col_d, val_d, 0, &runs, &sp);
  if (!st) st = wait();
  if (!st) st = sym_end(s, &sp, &rp, &cc, &vv, nnz_out, out_src);
  if (st) {
    sym_release(s, &sp);
    return st;
  }
  st = wait();
  if (st) {
    sym_free(s, rp, cc, vv, out_src);
    return st;
  }
  *rowptr_out = rp;
  *col_out = cc;
  *val_out = vv;
  return SGTSNE_OK;
}

int launch_permute_csr(hipStream_t s, int n, int64_t nnz, const int32_t *perm, const int32_t *iperm,
                       const int32_t *rp, const int32_t *col, const float *val, int32_t *rp2,
                       int32_t *col2, float *val2, bool sort_rows, bool device_sort) {
  int32_t *len = nullptr;
  SGT_HIP(hipMallocAsync((void **)&len, sizeof(int32_t) * ((size_t)n + 1), s));
  perm_len_kernel<<<div_up(n, 256), 256, 0, s>>>(n, perm, rp, len);
  SGT_LAUNCH_CHECK();
  SGT_HIP(hipMemsetAsync(len + n, 0, sizeof(int32_t), s));
  SGT_TRY(device_exclusive_scan(s, len, rp2, n + 1));
  if (!sort_rows || device_sort) {
    perm_fill_kernel<<<div_up((int64_t)n * 64, 256), 256, 0, s>>>(n, perm, iperm, rp, col, val, rp2, col2, val2);
    SGT_LAUNCH_CHECK();
    if (sort_rows) {  // in place, without the host (rows above kRowSortMax keep their order)
      row_sort_kernel<<<n, 256, 0, s>>>(n, rp2, col2, val2);
      SGT_LAUNCH_CHECK();
    }
    SGT_HIP(hipFreeAsync(len, s));
    return SGTSNE_OK;
  }
  int32_t *ctmp = nullptr;
  float *vtmp = nullptr;
  SGT_HIP(hipMallocAsync((void **)&ctmp, sizeof(int32_t) * (size_t)std::max<int64_t>(nnz, 1), s));
  SGT_HIP(hipMallocAsync((void **)&vtmp, sizeof(float) * (size_t)std::max<int64_t>(nnz, 1), s));
  perm_fill_kernel<<<div_up((int64_t)n * 64, 256), 256, 0, s>>>(n, perm, iperm, rp, col, val, rp2, ctmp, vtmp);
  SGT_LAUNCH_CHECK();
  // columns ascending within each row: neighbouring lanes gather neighbouring points
  int nbits = 1;
  while ((1ll << nbits) < (long long)n) ++nbits;
  size_t tb = 0;
  SGT_HIP(hipcub::DeviceSegmentedRadixSort::SortPairs(nullptr, tb, ctmp, col2, vtmp, val2, (int)nnz, n, rp2,
                                                      rp2 + 1, 0, nbits, s));
  void *tmp = nullptr;
  SGT_HIP(hipMallocAsync(&tmp, tb > 0 ? tb : 1, s));
  SGT_HIP(hipcub::DeviceSegmentedRadixSort::SortPairs(tmp, tb, ctmp, col2, vtmp, val2, (int)nnz, n, rp2,
                                                      rp2 + 1, 0, nbits, s));
  SGT_HIP(hipFreeAsync(tmp, s));
  SGT_HIP(hipFreeAsync(ctmp, s));
  SGT_HIP(hipFreeAsync(vtmp, s));
  SGT_HIP(hipFreeAsync(len, s));
  return SGTSNE_OK;
}

int spatial_order(hipStream_t s, int n, int d, int ds, const float *Y, const double *lo, double extent,
                  int32_t *order, int32_t *inv) {
  uint32_t *k0 = nullptr, *k1 = nullptr;
  int32_t *i0 = nullptr;
  SGT_HIP(hipMallocAsync((void **)&k0, sizeof(uint32_t) * (size_t)n, s));
  SGT_HIP(hipMallocAsync((void **)&k1, sizeof(uint32_t) * (size_t)n, s));
  SGT_HIP(hipMallocAsync((void **)&i0, sizeof(int32_t) * (size_t)n, s));
  const float invx = extent > 0 ? (float)(1.0 / extent) : 0.0f;
  morton_kernel<<<div_up(n, 256), 256, 0, s>>>(n, d, ds, Y, (float)lo[0], d > 1 ? (float)lo[1] : 0.f,
                                                d > 2 ? (float)lo[2] : 0.f, invx, k0, i0);
  SGT_LAUNCH_CHECK();
  size_t tb = 0;
  SGT_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, tb, k0, k1, i0, order, n, 0, 32, s));
  void *tmp = nullptr;
  SGT_HIP(hipMallocAsync(&tmp, tb > 0 ? tb : 1, s));
  SGT_HIP(hipcub::DeviceRadixSort::SortPairs(tmp, tb, k0, k1, i0, order, n, 0, 32, s));
  SGT_HIP(hipFreeAsync(tmp, s));
  invert_perm_kernel<<<div_up(n, 256), 256, 0, s>>>(n, order, inv);
  SGT_LAUNCH_CHECK();
  SGT_HIP(hipFreeAsync(k0, s));
  SGT_HIP(hipFreeAsync(k1, s));
  SGT_HIP(hipFreeAsync(i0, s));
  return SGTSNE_OK;
}

int launch_gather_points(hipStream_t s, int n, int ds, const int32_t *order, const float *in, float *out) {
  gather_points_kernel<<<div_up((int64_t)n * ds, 256), 256, 0, s>>>(n, ds, order, in, out);
  SGT_LAUNCH_CHECK();
  return SGTSNE_OK;
}

int launch_build_ell(hipStream_t s, int n, int width, const int32_t *rowptr, const int32_t *col,
                     const float *val, int32_t *ecol, float *eval, int32_t *tail_cnt) {
  build_ell_kernel<<<div_up(n, 256), 256, 0, s>>>(n, width, rowptr, col, val, ecol, eval, tail_cnt);
  SGT_LAUNCH_CHECK();
  return SGTSNE_OK;
}

int launch_build_tail(hipStream_t s, int n, int width, const int32_t *rowptr, const int32_t *col,
                      const float *val, const int32_t *tail_off, int32_t *trow, int32_t *tcol,
                      float *tval) {
  build_tail_kernel<<<div_up(n, 256), 256, 0, s>>>(n, width, rowptr, col, val, tail_off, trow, tcol, tval);
  SGT_LAUNCH_CHECK();
  return SGTSNE_OK;
}

}  // namespace sgt
