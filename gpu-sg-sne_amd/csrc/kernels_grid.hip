// kernels_grid.hip -- point <-> grid kernels of the repulsive term, the fused
// update and the device-side reductions of one gradient iteration.
//
// Reference semantics (HY = code/cuda/SG-tSNE-HYB/sgtsnepi/src,
// CU = code/cuda/SG-tSNE-CUDA/src):
//   grid mapping      HY/nuconv.cpp:22-47, CU/nuconv.cu:9-35 (FP32 clamp)
//   Lagrange weights  HY/gridding.cpp:28-40
//   spread (S2G)      HY/gridding.cpp:164-211 / CU/gridding.cu:145-185
//   gather (G2S)      HY/gridding.cpp:508-560 / CU/gridding.cu:187-230
//   forces and Z      HY/qq.cpp:75-106 / CU/Frep.cu:43-80
//   update            CU/gradient_descend.cu:12-44, HY/gradient_descendHYB.cpp:29-78
//
// Reductions: every block writes its partials to rw.part[block * 8 + k], and
// they are combined in a fixed order (deterministic), so no kernel needs a
// device-wide fence: in the iteration by every block of the kernel that uses
// the result (the update adds up Z, the centring the mean and the bounding box:
// at most 2048 partials of 16 bytes and 256 of 64, read from L2), elsewhere by
// a one-block finalize kernel.  An iteration of a small job is a chain of
// kernels of 3-9 us each, so a launch saved is worth more than those reads:
// without the three finalize kernels, the copy of the scalars to the host and
// six timed events an iteration of 2011 points takes 69 us instead of 94, one of
// 60,000 points late in a run 174 instead of 200.
#include "common.hpp"
#include "kernels.hpp"
#include "grid_device.hpp"
#include "spread_fix.hpp"
#include "../../include/sgtsne.h"

namespace sgt {

namespace {

constexpr int kBlock = 256;

enum FinMode { FIN_ZNEU, FIN_ZEXACT, FIN_KL };

// Device clock into stamp[at], by one thread of the launch (NULL: no timing).
__device__ __forceinline__ void stamp_now(DevScalars *sc, int at) {
  if (sc && blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) sc->stamp[at] = wall_clock64();
}
__global__ void stamp_kernel(DevScalars *sc, int at) { stamp_now(sc, at); }

// The scalars the host waits for; the sequence number is released last.
__device__ void publish(HostScalars *hs, const DevScalars *sc, unsigned long long seq) {
  for (int a = 0; a < 4; ++a) {
    hs->minv[a] = sc->minv[a];
    hs->maxv[a] = sc->maxv[a];
  }
  __hip_atomic_store(&hs->seq, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// ---- plain streaming copy (bandwidth / counter calibration) ----------------------
__global__ __launch_bounds__(kBlock) void stream_copy_kernel(const float4 *__restrict__ in, float4 *__restrict__ out,
                                                             int64_t count) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (; i < count; i += stride) out[i] = in[i];
}

// ---- fill ------------------------------------------------------------------
__global__ void fill_kernel(float *__restrict__ p, int64_t count, float v) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (; i < count; i += stride) p[i] = v;
}

// ---- S2G, LDS-privatised whole grid -------------------------------------------
// For grids that fit in LDS: each block spreads a contiguous chunk of points
// into a private LDS copy of the grid and writes it out; a second kernel sums
// the private grids.  No global atomics.  Lanes map to stencil nodes, not to
// points: the 4^d lanes of one point touch 4^d distinct cells, so an LDS
// atomic instruction conflicts only between the 64/4^d points of a wave
// (at most 4-way in 2-D, never in 3-D) even when every point of a clustered
// embedding falls into the same few cells.
constexpr int kS2GBlock = 1024;  // 16 waves share one private grid
constexpr int kS2GUnroll = 4;    // points per lane whose loads are issued together

template <int D>
__global__ __launch_bounds__(kS2GBlock) void s2g_lds_kernel(GridParams g, int n, const float *__restrict__ Y,
                                                            float *__restrict__ part, int chunk, int copies, DevScalars *stamp) {
  stamp_now(stamp, STAMP_S2G);
  extern __shared__ float sgrid[];
  constexpr int M = D + 1;
  constexpr int PPW = NodeLanes<D>::PPW;
  constexpr int NODES = NodeLanes<D>::NODES;
  constexpr int U = kS2GUnroll;
  const int G = grid_cells<D>(g.ng);
  const int MG = M * G;
  for (int e = threadIdx.x; e < copies * MG; e += blockDim.x) sgrid[e] = 0.0f;
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nwaves = blockDim.x >> 6;
  const int node = lane % NODES, slot = lane / NODES;
  const int i0 = blockIdx.x * chunk;
  const int i1 = min(n, i0 + chunk);
  // each point slot of each wave spreads a contiguous run of points, and a
  // lane adds its successive points in registers while they hit the same grid
  // node: in the locality order consecutive points mostly share a cell, so
  // most of the LDS atomics of the plain per-point form become register adds
  const int per_wave = (chunk + nwaves - 1) / nwaves;
  const int per_slot = (per_wave + PPW - 1) / PPW;
  const int w0 = min(i1, i0 + wave * per_wave + slot * per_slot);
  const int w1 = min(min(i1, i0 + (wave + 1) * per_wave), w0 + per_slot);
  float *cp = sgrid + (slot % copies) * MG;  // the point slots of one instruction use different copies
  int cur = -1;
  float acc[M];
#pragma unroll
  for (int a = 0; a < M; ++a) acc[a] = 0.0f;
  for (int base = w0; base < w1; base += U) {
    float y[U][D];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = base + u;
      if (i < w1) load_pt<D>(Y, i, y[u]);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = base + u;
      if (i < w1) {
        int idx;
        float ww;
        node_of_lane<D>(g, y[u], node, idx, ww);
        if (idx != cur) {
          if (cur >= 0) {
#pragma unroll
            for (int a = 0; a < M; ++a) atomicAdd(&cp[a * G + cur], acc[a]);
          }
          cur = idx;
#pragma unroll
          for (int a = 0; a < M; ++a) acc[a] = 0.0f;
        }
        acc[0] += ww;
#pragma unroll
        for (int a = 0; a < D; ++a) acc[a + 1] += (y[u][a] - g.center[a]) * ww;
      }
    }
  }
  if (cur >= 0) {
#pragma unroll
    for (int a = 0; a < M; ++a) atomicAdd(&cp[a * G + cur], acc[a]);
  }
  __syncthreads();
  // sum of the copies -> this block's slice of the partial buffer (coalesced)
  float *dst = part + (int64_t)blockIdx.x * MG;
  for (int e = threadIdx.x; e < MG; e += blockDim.x) {
    float v = 0.0f;
    for (int k = 0; k < copies; ++k) v += sgrid[k * MG + e];
    dst[e] = v;
  }
}

// ---- S2G on the matrix cores (2-D grids of side <= 16 NT) -------------------------
// For 4 points k at a time, the spread of channel c onto a 16 x 16 tile of
// nodes is a rank-4 product, one v_mfma_f32_16x16x4f32:
//   V_c[gx][gy] += sum_k wx_k(gx) * (q_c,k * wy_k(gy))
// with A[gx][k] = wx_k(gx) (lane l holds gx = l % 16 of point k = l / 16),
// B[k][gy] = q_c,k wy_k(gy) (lane l holds gy = l % 16 of the same point), and
// D[gx][gy] in lane l, register v at gx = 4 (l / 16) + v, gy = l % 16.  A
// lane evaluates one Lagrange factor per axis and tile; nodes off a point's
// stencil get weight 0.  Nothing is contended: each wave keeps its points'
// sums in registers whatever the order of the points or how many share a
// cell, the block's 4 waves are added in LDS in a fixed order, and
// grid_reduce_kernel adds the blocks' grids in a fixed order (deterministic).
typedef float mfv4 __attribute__((ext_vector_type(4)));
constexpr int kMfmaBlock = 256;
// points per work-group: about 1024 work-groups whatever N, whole batches of
// 256 (one per wave), between 256 and 4096 points each
inline int mfma_chunk(int n) { return std::min(4096, std::max(256, div_up(div_up(n, 1024), 256) * 256)); }

// Weight of stencil node f + r of a point at f + 1 + dl (the node factor of
// lane_node), 0 when r is not 0..3.
__device__ __forceinline__ float lagrange_node(int r, float dl) {
  const float x = r == 0 ? 1.0f + dl : r == 1 ? dl : r == 2 ? 1.0f - dl : 2.0f - dl;
  const float w = (r == 1 || r == 2) ? lg1(x) : lg2(x);
  return (r >= 0 && r <= 3) ? w : 0.0f;
}

template <int NT>
__global__ __launch_bounds__(kMfmaBlock) void s2g_mfma_kernel(GridParams g, int n, const float *__restrict__ Y,
                                                              float *__restrict__ part, int chunk, DevScalars *stamp) {
  stamp_now(stamp, STAMP_S2G);
  constexpr int T = 16 * NT;  // side of the tiled grid (>= ng)
  __shared__ float red[4][3][T * T];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int k = lane >> 4, node = lane & 15;
  const int i0 = blockIdx.x * chunk;
  const int i1 = min(n, i0 + chunk);
  mfv4 acc[3][NT * NT];
#pragma unroll
  for (int c = 0; c < 3; ++c)
#pragma unroll
    for (int t = 0; t < NT * NT; ++t) acc[c][t] = mfv4{0.0f, 0.0f, 0.0f, 0.0f};
  const float2 *Y2 = reinterpret_cast<const float2 *>(Y);
  // each wave takes 64 consecutive points at a time with one coalesced load
  // (the next 64 are loaded while these are spread); step s of a batch hands
  // point 4 s + k to lanes 16 k .. 16 k + 15 by cross-lane reads
  int base = i0 + 64 * wave;
  float2 nxt = base + lane < i1 ? Y2[base + lane] : make_float2(g.minv[0], g.minv[1]);
  for (; base < i1; base += 256) {
    const float2 cur = nxt;
    const int nb = base + 256;
    nxt = nb + lane < i1 ? Y2[nb + lane] : make_float2(g.minv[0], g.minv[1]);
    const int cnt = min(64, i1 - base);
#pragma unroll 4
    for (int st = 0; st < 16; ++st) {
      if (4 * st >= cnt) break;  // wave-uniform
      const int src = 4 * st + k;
      const float yx = __shfl(cur.x, src), yy = __shfl(cur.y, src);
      const bool in = src < cnt;
      float t0 = (yx - g.minv[0]) * g.scale, t1 = (yy - g.minv[1]) * g.scale;
      t0 = fminf(fmaxf(t0, 0.0f), g.gmax);  // NaN -> 0: never leaves the grid
      t1 = fminf(fmaxf(t1, 0.0f), g.gmax);
      const int f0 = (int)t0, f1 = (int)t1;
      const float d0 = t0 - (float)f0, d1 = t1 - (float)f1;
      float wx[NT], wy[NT];
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        wx[t] = in ? lagrange_node(16 * t + node - f0, d0) : 0.0f;
        wy[t] = lagrange_node(16 * t + node - f1, d1);
      }
      const float q1 = yx - g.center[0], q2 = yy - g.center[1];
#pragma unroll
      for (int ty = 0; ty < NT; ++ty) {
        const float b0 = wy[ty], b1 = q1 * wy[ty], b2 = q2 * wy[ty];
#pragma unroll
        for (int tx = 0; tx < NT; ++tx) {
          acc[0][tx * NT + ty] = __builtin_amdgcn_mfma_f32_16x16x4f32(wx[tx], b0, acc[0][tx * NT + ty], 0, 0, 0);
          acc[1][tx * NT + ty] = __builtin_amdgcn_mfma_f32_16x16x4f32(wx[tx], b1, acc[1][tx * NT + ty], 0, 0, 0);
          acc[2][tx * NT + ty] = __builtin_amdgcn_mfma_f32_16x16x4f32(wx[tx], b2, acc[2][tx * NT + ty], 0, 0, 0);
        }
      }
    }
  }
  // this wave's sums: node (gx, gy) of channel c at red[wave][c][gy * T + gx]
#pragma unroll
  for (int c = 0; c < 3; ++c)
#pragma unroll
    for (int tx = 0; tx < NT; ++tx)
#pragma unroll
      for (int ty = 0; ty < NT; ++ty) {
        float *dst = &red[wave][c][(16 * ty + node) * T + 16 * tx + 4 * k];
        const mfv4 a = acc[c][tx * NT + ty];
        dst[0] = a[0];
        dst[1] = a[1];
        dst[2] = a[2];
        dst[3] = a[3];
      }
  __syncthreads();
  // the block's grid (channel-major, x fastest), waves added in a fixed order
  const int ng = g.ng, G = ng * ng;
  float *out = part + (int64_t)blockIdx.x * 3 * G;
  for (int e = threadIdx.x; e < 3 * G; e += blockDim.x) {
    const int c = e / G, cell = e - c * G;
    const int gy = cell / ng, gx = cell - gy * ng;
    const int sidx = gy * T + gx;
    out[e] = (red[0][c][sidx] + red[1][c][sidx]) + (red[2][c][sidx] + red[3][c][sidx]);
  }
}

// ---- 3-D S2G on the matrix cores (grids of side <= 16) ------------------------------
// A work-group spreads a chunk of points onto its own copy of the grid in LDS.
// It first sorts its points by the base z-cell of their stencils (a stable
// counting sort of (z-cell, position) keys: deterministic) and gives each of its 4
// waves a contiguous quarter of the sorted points, so the work is even however
// the points crowd a few cells.  A wave walks its points in runs of equal base
// z-cell f, 4 at a time; such a step touches slices f .. f + 3 only, and slice
// f + r of channel c gets the rank-4 product
//   V_c[gx][gy][f + r] += sum_k wx_k(gx) (q_c,k wy_k(gy) wz_k(r))
// (one v_mfma_f32_16x16x4f32, layouts as in the 2-D form) into a window of 4
// slice accumulators.  When the base cell moves up, the slices below it are
// final for this wave: they are stored into the LDS grid, which no other wave
// stores to (the waves' runs are disjoint), and the window slides.  The 4
// windows left at the end are added in wave order after a barrier, so the grid
// does not depend on timing; grid_reduce_kernel adds the work-groups' grids in
// a fixed order.
// Points per work-group: whole rounds of 256, up to 2048; fewer for a small job,
// whose few work-groups would each walk a long chain of matrix operations
// (5000 points in 3 work-groups: 127 us; in 20 of them, 44).
constexpr int kMfma3Chunk = 2048;
inline int mfma3_chunk(int n) { return std::min(kMfma3Chunk, std::max(256, div_up(div_up(n, 128), 256) * 256)); }

__global__ __launch_bounds__(kMfmaBlock) void s2g_mfma3_kernel(GridParams g, int n, const float *__restrict__ Y,
                                                               float *__restrict__ part, int chunk, DevScalars *stamp) {
  stamp_now(stamp, STAMP_S2G);
  __shared__ float grid[4 * 16 * 16 * 16];  // [channel][z][y][x], side ng
  __shared__ uint32_t key[kMfma3Chunk];
  __shared__ int zcnt[kMfma3Chunk / kMfmaBlock][4][16];
  __shared__ int zbase[16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int k = lane >> 4, node = lane & 15;
  const int ng = g.ng, G = ng * ng * ng;
  const int i0 = blockIdx.x * chunk;
  const int cnt = min(n, i0 + chunk) - i0;
  const float4 *__restrict__ Y4 = reinterpret_cast<const float4 *>(Y) + i0;
  for (int e = tid; e < 4 * G; e += kMfmaBlock) grid[e] = 0.0f;
  // keys (base z-cell, position) of the chunk's points in ascending order, by
  // a stable counting sort over the at most 16 base z-cells: point i = 256 r
  // + 64 w + lane is ranked among the equal cells of its wave by a ballot,
  // and the (cell, round, wave) counts give its place
  constexpr int kRounds = kMfma3Chunk / kMfmaBlock;
  int fzr[kRounds], rk[kRounds];
#pragma unroll
  for (int r = 0; r < kRounds; ++r) {
    const int i = r * kMfmaBlock + tid;
    fzr[r] = -1;
    if (i < cnt) fzr[r] = (int)fminf(fmaxf((Y4[i].z - g.minv[2]) * g.scale, 0.0f), g.gmax);
    rk[r] = 0;
    for (int v = 0; v < 16; ++v) {
      const unsigned long long m = __ballot(fzr[r] == v);
      if (fzr[r] == v) rk[r] = __popcll(m & ((1ull << lane) - 1ull));
      if (lane == 0) zcnt[r][wave][v] = __popcll(m);
    }
  }
  __syncthreads();
  if (tid < 16) {  // per cell: exclusive prefix over (round, wave), then the cell total
    int run = 0;
    for (int r = 0; r < kRounds; ++r)
      for (int w = 0; w < 4; ++w) {
        const int c = zcnt[r][w][tid];
        zcnt[r][w][tid] = run;
        run += c;
      }
    zbase[tid] = run;
  }
  __syncthreads();
  if (tid == 0) {  // cell totals -> first position of each cell
    int run = 0;
    for (int v = 0; v < 16; ++v) {
      const int c = zbase[v];
      zbase[v] = run;
      run += c;
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kRounds; ++r) {
    const int i = r * kMfmaBlock + tid;
    const int v = fzr[r];
    if (v >= 0) key[zbase[v] + zcnt[r][wave][v] + rk[r]] = ((uint32_t)v << 16) | (uint32_t)i;
  }
  __syncthreads();
  const int pa = (cnt * wave) >> 2, pb = (cnt * (wave + 1)) >> 2;  // this wave's sorted positions
  mfv4 acc[4][4];  // [slice zb + r][channel]
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[r][c] = mfv4{0.0f, 0.0f, 0.0f, 0.0f};
  // slice r of the window -> grid slice z (lane l holds x = 4 (l / 16) + v, y = l % 16)
  auto put = [&](int r, int z, bool add) {
    const int gx0 = 4 * k, gy = node;
    if (z >= ng || gy >= ng) return;
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        if (gx0 + v < ng) {
          float *cell = &grid[((c * ng + z) * ng + gy) * ng + gx0 + v];
          *cell = add ? *cell + acc[r][c][v] : acc[r][c][v];
        }
  };
  auto clear = [&](int r) {
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[r][c] = mfv4{0.0f, 0.0f, 0.0f, 0.0f};
  };
  int zb = pa < pb ? (int)(key[pa] >> 16) : 0;  // window: slices zb .. zb + 3
  int p0 = pa;
  while (p0 < pb) {  // wave-uniform
    const int fz = (int)(key[p0] >> 16);
    if (fz != zb) {  // slices zb .. fz - 1 are final for this wave
      const int sh = fz - zb;
      if (sh == 1) {
        put(0, zb, false);
#pragma unroll
        for (int c = 0; c < 4; ++c) { acc[0][c] = acc[1][c]; acc[1][c] = acc[2][c]; acc[2][c] = acc[3][c]; }
        clear(3);
      } else if (sh == 2) {
        put(0, zb, false);
        put(1, zb + 1, false);
#pragma unroll
        for (int c = 0; c < 4; ++c) { acc[0][c] = acc[2][c]; acc[1][c] = acc[3][c]; }
        clear(2);
        clear(3);
      } else if (sh == 3) {
        put(0, zb, false);
        put(1, zb + 1, false);
        put(2, zb + 2, false);
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[0][c] = acc[3][c];
        clear(1);
        clear(2);
        clear(3);
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          put(r, zb + r, false);
          clear(r);
        }
      }
      zb = fz;
    }
    // end of the run of base cell fz within this wave's positions
    int lo = p0 + 1, hi = pb;
    const uint32_t nextz = (uint32_t)(fz + 1) << 16;
    while (lo < hi) {
      const int m = (lo + hi) >> 1;
      if (key[m] < nextz) lo = m + 1;
      else hi = m;
    }
    const int re = lo;
    for (int ps = p0; ps < re; ps += 4) {
      const int src = ps + k;
      const bool in = src < re;
      const float4 y = Y4[key[in ? src : ps] & 0xFFFFu];
      float t0 = (y.x - g.minv[0]) * g.scale, t1 = (y.y - g.minv[1]) * g.scale, t2 = (y.z - g.minv[2]) * g.scale;
      t0 = fminf(fmaxf(t0, 0.0f), g.gmax);  // NaN -> 0: never leaves the grid
      t1 = fminf(fmaxf(t1, 0.0f), g.gmax);
      t2 = fminf(fmaxf(t2, 0.0f), g.gmax);
      const int f0 = (int)t0, f1 = (int)t1;
      const float d0 = t0 - (float)f0, d1 = t1 - (float)f1, d2 = t2 - (float)(int)t2;
      const float wx = in ? lagrange_node(node - f0, d0) : 0.0f;
      const float wy = lagrange_node(node - f1, d1);
      const float wz[4] = {lg2(1.0f + d2), lg1(d2), lg1(1.0f - d2), lg2(2.0f - d2)};
      const float q1 = y.x - g.center[0], q2 = y.y - g.center[1], q3 = y.z - g.center[2];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float b = wy * wz[r];
        acc[r][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(wx, b, acc[r][0], 0, 0, 0);
        acc[r][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(wx, q1 * b, acc[r][1], 0, 0, 0);
        acc[r][2] = __builtin_amdgcn_mfma_f32_16x16x4f32(wx, q2 * b, acc[r][2], 0, 0, 0);
        acc[r][3] = __builtin_amdgcn_mfma_f32_16x16x4f32(wx, q3 * b, acc[r][3], 0, 0, 0);
      }
    }
    p0 = re;  // the next run starts right after this one
  }
  // the windows left open, added in wave order
  for (int w = 0; w < 4; ++w) {
    __syncthreads();
    if (wave == w && pa < pb) {
#pragma unroll
      for (int r = 0; r < 4; ++r) put(r, zb + r, true);
    }
  }
  __syncthreads();
  float *out = part + (int64_t)blockIdx.x * 4 * G;
  for (int e = tid; e < 4 * G; e += kMfmaBlock) out[e] = grid[e];
}

// ---- S2G with global float atomics (grids too large for LDS) -------------------
// Same lane-per-node mapping; the grid is large here, so contention is low.
template <int D>
__global__ __launch_bounds__(kBlock) void s2g_atomic_kernel(GridParams g, int n,
                                                            const float *__restrict__ Y,
                                                            float *__restrict__ V, DevScalars *stamp) {
  stamp_now(stamp, STAMP_S2G);
  constexpr int PPW = NodeLanes<D>::PPW;
  constexpr int NODES = NodeLanes<D>::NODES;
  const int G = grid_cells<D>(g.ng);
  const int lane = threadIdx.x & 63;
  const int node = lane % NODES, slot = lane / NODES;
  const int gw = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const int nw = (gridDim.x * blockDim.x) >> 6;
  for (int base = gw * PPW; base < n; base += nw * PPW) {
    const int i = base + slot;
    if (i < n) {
      float y[D];
      load_pt<D>(Y, i, y);
      int idx;
      float ww;
      node_of_lane<D>(g, y, node, idx, ww);
      unsafeAtomicAdd(&V[idx], ww);
#pragma unroll
      for (int a = 0; a < D; ++a) unsafeAtomicAdd(&V[(a + 1) * G + idx], (y[a] - g.center[a]) * ww);
    }
  }
}

// Sum of the per-block private grids (deterministic): 64 cells per block,
// 16 partial groups per cell summed in a fixed order, then combined in LDS.
__global__ __launch_bounds__(1024) void grid_reduce_kernel(const float *__restrict__ part, int nparts,
                                                           int cells, float *__restrict__ V, DevScalars *stamp) {
  __shared__ float red[16][64];
  const int c = blockIdx.x * 64 + (threadIdx.x & 63);
  const int gidx = threadIdx.x >> 6;
  float acc = 0.0f;
  if (c < cells) {
    int b = gidx;
    for (; b + 48 < nparts; b += 64) {
      const float v0 = part[(int64_t)b * cells + c], v1 = part[(int64_t)(b + 16) * cells + c];
      const float v2 = part[(int64_t)(b + 32) * cells + c], v3 = part[(int64_t)(b + 48) * cells + c];
      acc += (v0 + v1) + (v2 + v3);
    }
    for (; b < nparts; b += 16) acc += part[(int64_t)b * cells + c];
  }
  red[gidx][threadIdx.x & 63] = acc;
  __syncthreads();
  if (threadIdx.x < 64 && c < cells) {
    float t = 0.0f;
    for (int k = 0; k < 16; ++k) t += red[k][threadIdx.x];
    V[c] = t;
  }
  stamp_now(stamp, STAMP_CONV);  // the spread ends here
}

// ---- G2S + forces + Z ------------------------------------------------------------
// Phi (node-major, see launch_conv) at y_i by the same stencil, the points along
// the tiles of the grid (ord), so that neighbouring lanes read the same nodes:
// 200,003 points late in a 3-D run 68 -> 21 us with both; Frep_i (unnormalised) = ~y_i Phi0 - Phi_{1..d}.
// Z per point, compensated sum over points, FP64:
//   ZDIRECT: z_i = psi_i, the gathered convolution of the unit charges with
//            1/(1 + r^2) (channel D+1), so Z = sum_i psi_i - N;
//   else:    z_i = (1 + 2|~y_i|^2) Phi0 - 2 ~y_i . Phi_{1..d} (HY/qq.cpp:75-106).
// ~y is y minus the charge shift used by S2G (any shift leaves Frep and
// sum z_i unchanged).
template <int D, bool ZDIRECT>
__global__ __launch_bounds__(kBlock) void g2s_force_kernel(GridParams g, int n,
                                                           const float *__restrict__ Y,
                                                           const float *__restrict__ Phi,
                                                           float *__restrict__ Frep, double *part, DevScalars *stamp,
                                                           const int32_t *__restrict__ ord) {
  stamp_now(stamp, STAMP_G2S);
  __shared__ double lds[8];
  const int ng = g.ng;
  const int G = grid_cells<D>(ng);
  constexpr int C = ZDIRECT ? D + 2 : D + 1;
  const float4 *__restrict__ Phi4 = reinterpret_cast<const float4 *>(Phi);
  const float *__restrict__ Phi1 = Phi + 4 * (int64_t)G;
  Neu z{0.0, 0.0};
  for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < n; k += gridDim.x * blockDim.x) {
    const int i = ord ? ord[k] : k;
    float y[D];
    load_pt<D>(Y, i, y);
    int f[D];
    float w[D][4];
    stencil<D>(g, y, f, w);
    float ph[C];
#pragma unroll
    for (int c = 0; c < C; ++c) ph[c] = 0.0f;
    for_stencil<D>(ng, f, w, [&](int idx, float ww) {
      const float4 q = Phi4[idx];
      ph[0] = __builtin_fmaf(q.x, ww, ph[0]);
      ph[1] = __builtin_fmaf(q.y, ww, ph[1]);
      if constexpr (C > 2) ph[2] = __builtin_fmaf(q.z, ww, ph[2]);
      if constexpr (C > 3) ph[3] = __builtin_fmaf(q.w, ww, ph[3]);
      if constexpr (C > 4) ph[4] = __builtin_fmaf(Phi1[idx], ww, ph[4]);
    });
    float fr[D];
    double ysq = 0.0, ydot = 0.0;
#pragma unroll
    for (int a = 0; a < D; ++a) {
      const float yt = y[a] - g.center[a];
      fr[a] = yt * ph[0] - ph[a + 1];
      ysq += (double)yt * (double)yt;
      ydot += (double)yt * (double)ph[a + 1];
    }
    store_pt<D>(Frep, i, fr);
    if constexpr (ZDIRECT) neu_add(z, (double)ph[D + 1]);
    else neu_add(z, (1.0 + 2.0 * ysq) * (double)ph[0] - 2.0 * ydot);
  }
  z = wave_neu(z);
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (lane == 0) { lds[wid * 2] = z.s; lds[wid * 2 + 1] = z.c; }
  __syncthreads();
  if (threadIdx.x == 0) {
    Neu t{lds[0], lds[1]};
    for (int k = 1; k < (int)(blockDim.x >> 6); ++k) neu_merge(t, Neu{lds[2 * k], lds[2 * k + 1]});
    part[(size_t)blockIdx.x * 8 + 0] = t.s;
    part[(size_t)blockIdx.x * 8 + 1] = t.c;
  }
}

// ---- G2S + forces + Z with the grid in LDS (2-D side <= 64, 3-D side <= 16) --------
// The same arithmetic, in the same order, as g2s_force_kernel, with the 4^D
// stencil reads of a point served from LDS instead of L1/L2: each work-group
// (one per CU, 16 waves) first copies the grid into LDS, channels 0..3 of a
// node as one float4 and the fifth (Z-direct in 3-D) in a second array, then
// strides over the points.
constexpr int kG2sLdsCells = 4096;
constexpr int kG2sLdsBlock = 1024;

// Below about 200,000 points the copies of the grid into LDS (and, in 3-D, a
// work-group per CU of 80 KB) cost more than reading the nodes from cache:
// 10,000 points 5.9 (LDS) / 3.8 us, 3-D 20,000 20.5 / 8.4, 200,003 2-D 6.5 / 6.5
// and 3-D 21.3 / 23.1, 400,000 8.4 / 9.3.
inline bool g2s_lds_fits(int d, int ng, int n) {
  return n >= 200000 && ((d == 2 && ng <= 64) || (d == 3 && ng <= 16));
}

template <int D, bool ZDIRECT>
__global__ __launch_bounds__(kG2sLdsBlock) void g2s_lds_kernel(GridParams g, int n, const float *__restrict__ Y,
                                                               const float *__restrict__ Phi,
                                                               float *__restrict__ Frep, double *part, DevScalars *stamp) {
  stamp_now(stamp, STAMP_G2S);
  constexpr int C = ZDIRECT ? D + 2 : D + 1;
  static_assert(C >= 3 && C <= 5, "2-D or 3-D only");
  __shared__ float4 q4[kG2sLdsCells];
  __shared__ float q5[C == 5 ? kG2sLdsCells : 1];
  __shared__ double lds[2 * (kG2sLdsBlock / 64)];
  const int ng = g.ng;
  const int G = grid_cells<D>(ng);
  for (int e = threadIdx.x; e < G; e += blockDim.x) {
    q4[e] = reinterpret_cast<const float4 *>(Phi)[e];
    if constexpr (C == 5) q5[e] = Phi[4 * (int64_t)G + e];
  }
  __syncthreads();
  Neu z{0.0, 0.0};
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    float y[D];
    load_pt<D>(Y, i, y);
    int f[D];
    float w[D][4];
    stencil<D>(g, y, f, w);
    float ph[C];
#pragma unroll
    for (int c = 0; c < C; ++c) ph[c] = 0.0f;
    auto node = [&](int idx, float ww) {
      const float4 v = q4[idx];
      ph[0] = __builtin_fmaf(v.x, ww, ph[0]);
      ph[1] = __builtin_fmaf(v.y, ww, ph[1]);
      ph[2] = __builtin_fmaf(v.z, ww, ph[2]);
      if constexpr (C > 3) ph[3] = __builtin_fmaf(v.w, ww, ph[3]);
      if constexpr (C == 5) ph[4] = __builtin_fmaf(q5[idx], ww, ph[4]);
    };
    if constexpr (D == 3) {
      // for_stencil's order and weights, one z-plane of 16 nodes at a time
      // (the whole stencil unrolled would spill)
#pragma unroll 1
      for (int i2 = 0; i2 < 4; ++i2)
#pragma unroll
        for (int i1 = 0; i1 < 4; ++i1) {
          const float w21 = w[2][i2] * w[1][i1];
#pragma unroll
          for (int i0 = 0; i0 < 4; ++i0) node(((f[2] + i2) * ng + f[1] + i1) * ng + f[0] + i0, w21 * w[0][i0]);
        }
    } else {
      for_stencil<D>(ng, f, w, node);
    }
    float fr[D];
    double ysq = 0.0, ydot = 0.0;
#pragma unroll
    for (int a = 0; a < D; ++a) {
      const float yt = y[a] - g.center[a];
      fr[a] = yt * ph[0] - ph[a + 1];
      ysq += (double)yt * (double)yt;
      ydot += (double)yt * (double)ph[a + 1];
    }
    store_pt<D>(Frep, i, fr);
    if constexpr (ZDIRECT) neu_add(z, (double)ph[D + 1]);
    else neu_add(z, (1.0 + 2.0 * ysq) * (double)ph[0] - 2.0 * ydot);
  }
  z = wave_neu(z);
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (lane == 0) { lds[wid * 2] = z.s; lds[wid * 2 + 1] = z.c; }
  __syncthreads();
  if (threadIdx.x == 0) {
    Neu t{lds[0], lds[1]};
    for (int k = 1; k < (int)(blockDim.x >> 6); ++k) neu_merge(t, Neu{lds[2 * k], lds[2 * k + 1]});
    part[(size_t)blockIdx.x * 8 + 0] = t.s;
    part[(size_t)blockIdx.x * 8 + 1] = t.c;
  }
}

// ---- fused gradient + gains + momentum update ----------------------------------
// dy = alpha Fattr - Frep / Z; gains, uy, y exactly as CU/gradient_descend.cu:29-44;
// per-block sums of the new Y feed the mean of the next centring.

// Sum of nz Neumaier partials (part[8 b], part[8 b + 1]) by threads 0..255 of
// the block, in the finalize kernel's order; every thread receives it.
__device__ Neu block_neu(const double *__restrict__ part, int nz, double (*red)[kBlock]) {
  const int t = threadIdx.x;
  if (t < kBlock) {
    Neu z{0.0, 0.0};
    for (int b = t; b < nz; b += kBlock) neu_merge(z, Neu{part[(size_t)b * 8], part[(size_t)b * 8 + 1]});
    red[0][t] = z.s;
    red[1][t] = z.c;
  }
  __syncthreads();
  for (int s = kBlock / 2; s > 0; s >>= 1) {
    if (t < s) {
      Neu x{red[0][t], red[1][t]};
      neu_merge(x, Neu{red[0][t + s], red[1][t + s]});
      red[0][t] = x.s;
      red[1][t] = x.c;
    }
    __syncthreads();
  }
  return Neu{red[0][0], red[1][0]};
}

// One block's part of the new Y: the sum per dimension, the count of
// non-finite coordinates and the bounds.
struct BoxPart {
  double sum[3], bad;
  float mn[3], mx[3];
  double pad;
};
static_assert(sizeof(BoxPart) == 64, "one partial slot");
constexpr int kMaxBoxParts = 256;  // every wave of the centring reads them all

template <int D>
__device__ __forceinline__ void wave_box(BoxPart &v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
#pragma unroll
    for (int a = 0; a < D; ++a) {
      v.sum[a] += __shfl_xor(v.sum[a], o, 64);
      v.mn[a] = fminf(v.mn[a], __shfl_xor(v.mn[a], o, 64));
      v.mx[a] = fmaxf(v.mx[a], __shfl_xor(v.mx[a], o, 64));
    }
    v.bad += __shfl_xor(v.bad, o, 64);
  }
}

template <int D>
__device__ __forceinline__ void empty_box(BoxPart &v) {
  v = BoxPart{};
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    v.mn[a] = INFINITY;
    v.mx[a] = -INFINITY;
  }
}

template <int D>
__device__ __forceinline__ void merge_box(BoxPart &v, const BoxPart &w) {
#pragma unroll
  for (int a = 0; a < D; ++a) {
    v.sum[a] += w.sum[a];
    v.mn[a] = fminf(v.mn[a], w.mn[a]);
    v.mx[a] = fmaxf(v.mx[a], w.mx[a]);
  }
  v.bad += w.bad;
}

constexpr int kUpdBlock = 1024;  // largest work-group of the update and the centring

template <int D>
__device__ __forceinline__ void add_box(BoxPart &v, const float (&y)[D]) {
#pragma unroll
  for (int a = 0; a < D; ++a) {
    v.sum[a] += (double)y[a];
    v.mn[a] = fminf(v.mn[a], y[a]);
    v.mx[a] = fmaxf(v.mx[a], y[a]);
    v.bad += isfinite(y[a]) ? 0.0 : 1.0;
  }
}

// The block's partial from its threads' (every thread calls it).
template <int D>
__device__ __forceinline__ void block_box(BoxPart &v, BoxPart *__restrict__ box) {
  __shared__ BoxPart wbox[kUpdBlock / 64];
  wave_box<D>(v);
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (lane == 0) wbox[wid] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k = 1; k < (int)(blockDim.x >> 6); ++k) merge_box<D>(v, wbox[k]);
    box[blockIdx.x] = v;
  }
}

template <int D>
__global__ __launch_bounds__(kUpdBlock) void update_kernel(int n, float *__restrict__ Y,
                                                        float *__restrict__ uY,
                                                        float *__restrict__ gains,
                                                        const float *__restrict__ Fattr,
                                                        const float *__restrict__ Frep,
                                                        float alpha, float momentum, float eta,
                                                        const double *__restrict__ zpart, int nz, DevScalars *sc,
                                                        BoxPart *__restrict__ box, int stamp) {
  stamp_now(stamp ? sc : nullptr, STAMP_UPDATE);
  __shared__ double red[2][kBlock];
  const Neu zs = block_neu(zpart, nz, red);
  const double Z = (zs.s + zs.c) - (double)n;
  if (blockIdx.x == 0 && threadIdx.x == 0) sc->Z = Z;
  const float zinv = (float)(1.0 / Z);
  BoxPart v;
  empty_box<D>(v);
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    float y[D], u[D], gn[D], fa[D], fr[D];
    load_pt<D>(Y, i, y);
    load_pt<D>(uY, i, u);
    load_pt<D>(gains, i, gn);
    load_pt<D>(Fattr, i, fa);
    load_pt<D>(Frep, i, fr);
#pragma unroll
    for (int a = 0; a < D; ++a) {
      const float dy = alpha * fa[a] - fr[a] * zinv;
      float gg = (sgnf(dy) != sgnf(u[a])) ? (gn[a] + 0.2f) : (gn[a] * 0.8f);
      if (gg < 0.01f) gg = 0.01f;
      gn[a] = gg;
      u[a] = momentum * u[a] - eta * gg * dy;
      y[a] = y[a] + u[a];
    }
    add_box<D>(v, y);
    store_pt<D>(Y, i, y);
    store_pt<D>(uY, i, u);
    store_pt<D>(gains, i, gn);
  }
  block_box<D>(v, box);
}

// Caller's points into the device's order and layout, with the partials the
// centring needs; the fresh optimiser state along with them.
template <int D>
__global__ __launch_bounds__(kUpdBlock) void set_points_kernel(int n, const float *__restrict__ raw, int aos,
                                                               const int32_t *__restrict__ perm,
                                                               float *__restrict__ Y, int reset,
                                                               float *__restrict__ uY, float *__restrict__ gains,
                                                               BoxPart *__restrict__ box) {
  BoxPart v;
  empty_box<D>(v);
  for (int r = blockIdx.x * blockDim.x + threadIdx.x; r < n; r += gridDim.x * blockDim.x) {
    const int64_t i = perm ? perm[r] : r;
    float y[D];
#pragma unroll
    for (int a = 0; a < D; ++a) y[a] = aos ? raw[i * D + a] : raw[(int64_t)a * n + i];
    store_pt<D>(Y, r, y);
    add_box<D>(v, y);
    if (reset) {
      float z[D], o[D];
#pragma unroll
      for (int a = 0; a < D; ++a) {
        z[a] = 0.0f;
        o[a] = 1.0f;
      }
      store_pt<D>(uY, r, z);
      store_pt<D>(gains, r, o);
    }
  }
  block_box<D>(v, box);
}

template <int D>
__global__ __launch_bounds__(kBlock) void get_points_kernel(int n, const float *__restrict__ in, int aos,
                                                            const int32_t *__restrict__ perm, double scale,
                                                            float *__restrict__ raw) {
  for (int r = blockIdx.x * blockDim.x + threadIdx.x; r < n; r += gridDim.x * blockDim.x) {
    const int64_t i = perm ? perm[r] : r;
    float y[D];
    load_pt<D>(in, r, y);
#pragma unroll
    for (int a = 0; a < D; ++a) raw[aos ? i * D + a : (int64_t)a * n + i] = (float)((double)y[a] * scale);
  }
}

// The centring of the updated Y (HY/gradient_descendHYB.cpp:64-76): every
// block adds up the update's partials in the same fixed order, subtracts the
// mean from its points, and block 0 publishes the centred bounds (rounding is
// monotone, so fl(min y - m) is the minimum of the centred points).
template <int D>
__global__ __launch_bounds__(kUpdBlock) void center_kernel(int n, float *__restrict__ Y,
                                                           const BoxPart *__restrict__ box, int nbox, DevScalars *sc,
                                                           HostScalars *hs, unsigned long long seq, int stamp) {
  // every wave adds all the partials itself, as a binary tree over 256 places:
  // no work-group memory or barrier, and the same bits in every wave
  const int lane = threadIdx.x & 63;
  BoxPart v, w;
  empty_box<D>(v);
  empty_box<D>(w);
  if (lane < nbox) v = box[lane];
  if (lane + 128 < nbox) merge_box<D>(v, box[lane + 128]);
  if (lane + 64 < nbox) w = box[lane + 64];
  if (lane + 192 < nbox) merge_box<D>(w, box[lane + 192]);
  merge_box<D>(v, w);
  wave_box<D>(v);
  float m[D];
#pragma unroll
  for (int a = 0; a < D; ++a) m[a] = (float)(v.sum[a] / (double)n);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    for (int a = 0; a < D; ++a) {
      sc->minv[a] = v.bad > 0.0 ? NAN : (double)(v.mn[a] - m[a]);  // a non-finite coordinate poisons the extent
      sc->maxv[a] = (double)(v.mx[a] - m[a]);
    }
    if (stamp) {
      hs->stamp[0] = sc->stamp[STAMP_END];  // this iteration began where the last one ended
      for (int k = 0; k < 4; ++k) hs->stamp[1 + k] = sc->stamp[k];
    }
    publish(hs, sc, seq);
  }
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    float y[D];
    load_pt<D>(Y, i, y);
#pragma unroll
    for (int a = 0; a < D; ++a) y[a] -= m[a];
    store_pt<D>(Y, i, y);
  }
  // the end of the iteration: all the work-groups are in flight at once with the
  // same work, so the first one's end is the kernel's within its last wave (and its
  // first thread has read the last iteration's).  To the host only where it asks
  // for it.
  if (stamp && blockIdx.x == 0 && threadIdx.x == 0) {
    const unsigned long long t = wall_clock64();
    sc->stamp[STAMP_END] = t;
    if (stamp > 1) hs->end = t;
  }
}

// ---- exact O(N^2) repulsion (validation, CU/compute_error.cu:8-53) -------------
template <int D>
__global__ __launch_bounds__(kBlock) void rep_exact_kernel(int n, const float *__restrict__ Y,
                                                           float *__restrict__ Frep, double *part) {
  __shared__ float tile[kBlock][D];
  __shared__ double lds[4];
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  float yi[D];
#pragma unroll
  for (int a = 0; a < D; ++a) yi[a] = 0.0f;
  if (i < n) load_pt<D>(Y, i, yi);
  double f[D];
#pragma unroll
  for (int a = 0; a < D; ++a) f[a] = 0.0;
  double z = 0.0;
  for (int j0 = 0; j0 < n; j0 += kBlock) {
    const int j = j0 + threadIdx.x;
    float yj[D];
#pragma unroll
    for (int a = 0; a < D; ++a) yj[a] = 0.0f;
    if (j < n) load_pt<D>(Y, j, yj);
#pragma unroll
    for (int a = 0; a < D; ++a) tile[threadIdx.x][a] = yj[a];
    __syncthreads();
    const int cnt = min(kBlock, n - j0);
    for (int t = 0; t < cnt; ++t) {
      if (j0 + t == i) continue;
      double dist = 0.0, df[D];
#pragma unroll
      for (int a = 0; a < D; ++a) {
        df[a] = (double)yi[a] - (double)tile[t][a];
        dist += df[a] * df[a];
      }
      const double q = 1.0 / (1.0 + dist);
#pragma unroll
      for (int a = 0; a < D; ++a) f[a] += df[a] * q * q;
      z += q;
    }
    __syncthreads();
  }
  if (i < n) {
    float fo[D];
#pragma unroll
    for (int a = 0; a < D; ++a) fo[a] = (float)f[a];
    store_pt<D>(Frep, i, fo);
  } else {
    z = 0.0;
  }
  z = wave_sum(z);
  if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = z;
  __syncthreads();
  if (threadIdx.x == 0) part[(size_t)blockIdx.x * 8] = lds[0] + lds[1] + lds[2] + lds[3];
}

// ---- one-block finalisation of the block partials (fixed order) ---------------
__global__ __launch_bounds__(kBlock) void finalize_kernel(int mode, int nblocks, int n,
                                                          const double *__restrict__ part, DevScalars *sc) {
  __shared__ double red[2][kBlock];
  if (mode == FIN_ZNEU) {
    const Neu z = block_neu(part, nblocks, red);
    if (threadIdx.x == 0) sc->Z = (z.s + z.c) - (double)n;
    return;
  }
  const int t = threadIdx.x;
  double acc = 0.0;
  for (int b = t; b < nblocks; b += kBlock) acc += part[(size_t)b * 8];
  red[0][t] = acc;
  __syncthreads();
  for (int s = kBlock / 2; s > 0; s >>= 1) {
    if (t < s) red[0][t] += red[0][t + s];
    __syncthreads();
  }
  if (t == 0) (mode == FIN_ZEXACT ? sc->zexact : sc->kl) = red[0][0];
}

int grid_blocks(int n, int max_blocks) {
  int b = div_up(n > 0 ? n : 1, kBlock);
  return b < max_blocks ? b : max_blocks;
}

int finalize(hipStream_t s, int mode, int nblocks, int n, RedWork rw, DevScalars *sc) {
  finalize_kernel<<<1, kBlock, 0, s>>>(mode, nblocks, n, rw.part, sc);
  SGT_LAUNCH_CHECK();
  return SGTSNE_OK;
}

// Large grids (those no LDS copy or matrix-core tile holds): the points in
// runs of `unit` along the tiles of the grid (ord, see spread_bin_kernel), each
// run's stencil window accumulated in LDS as 64-bit fixed point and added to the
// fixed-point grid Vf (spread_fix.hpp), so the grid is exact and the same
// whatever the order of the points and the atomics.  Bound by the global atomics
// of the windows' cells: in the device order of P a run's window often did not
// fit LDS and every node of every point went to memory.  200,003 points late in
// a run: 3-D 238 -> 69 us, 2-D spread 180 -> 40 us with the order (23 us, renewed
// every 16 evaluations).
template <int D>
__global__ __launch_bounds__(s2g_threads<D>()) void s2g_fix_kernel(GridParams g, float fsf, int n,
                                                                   const float *__restrict__ Y,
                                                                   unsigned long long *__restrict__ Vf, int unit,
                                                                   int lds_slots, const int32_t *__restrict__ ord, DevScalars *stamp) {
  stamp_now(stamp, STAMP_S2G);
  extern __shared__ unsigned long long win[];
  __shared__ int sbox[6];
  const int nunits = (n + unit - 1) / unit;
  for (int u = blockIdx.x; u < nunits; u += gridDim.x)
    spread_fix_unit<D>(g, fsf, Vf, u * unit, min(n, (u + 1) * unit), Y, ord, win, lds_slots, sbox);
}

// V = Vf * 2^-e in FP32 (the FP64 product rounded once), Vf cleared.
__global__ void fix_to_float_kernel(long long *__restrict__ Vf, float *__restrict__ V, int64_t count, double inv,
                                    DevScalars *stamp) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += stride) {
    V[i] = (float)((double)Vf[i] * inv);
    Vf[i] = 0;
  }
  stamp_now(stamp, STAMP_CONV);
}

}  // namespace

int launch_stream_copy(hipStream_t s, const float4 *in, float4 *out, int64_t count) {
  if (count <= 0) return SGTSNE_OK;
  stream_copy_kernel<<<2048, kBlock, 0, s>>>(in, out, count);
  SGT_LAUNCH_CHECK();
  return SGTSNE_OK;
}

int launch_fill(hipStream_t s, float *p, int64_t count, float v) {
  if (count <= 0) return SGTSNE_OK;
  int blocks = (int)std::min<int64_t>((count + kBlock - 1) / kBlock, 4096);
  fill_kernel<<<blocks, kBlock, 0, s>>>(p, count, v);
  SGT_LAUNCH_CHECK();
  return SGTSNE_OK;
}

int launch_stamp(hipStream_t s, DevScalars *sc, int at) {
  stamp_kernel<<<1, 1, 0, s>>>(sc, at);
  SGT_LAUNCH_CHECK();
  return SGTSNE_OK;
}

// LDS grid copies for the spread: one per point slot of a wave when they fit.
int s2g_lds_fits(int d, int ng, size_t *lds_bytes, int *copies) {
  const size_t G = d == 1 ? (size_t)ng : d == 2 ? (size_t)ng * ng : (size_t)ng * ng * ng;
  const size_t one = G * (size_t)(d + 1) * sizeof(float);
  int c = d == 1 ? 16 : d == 2 ? 4 : 1;
  while (c > 1 && one * c > 65536) c >>= 1;
  *copies = c;
  *lds_bytes = one * c;
  return *lds_bytes <= 65536;
}

// Grids that go through the fixed-point windows (and the gather from memory).
bool s2g_takes_order(const GridParams &g, int mode) {
  size_t lds = 0;
  int copies = 1;
  return g.d >= 2 && mode != SGTSNE_SPREAD_ATOMIC && !(g.d == 3 && g.ng <= 16) &&
         !s2g_lds_fits(g.d, g.ng, &lds, &copies);
}

// Tiles of 2^tb cells per axis (at most 32 per axis in 3-D, 128 in 2-D) in
// Morton order: the bin of each point and its place among the bin's points.  A
// work-group counts its 4096 points in LDS first, so a crowded bin takes one
// global atomic per work-group: with one per point, 200,003 points late in a 3-D
// run (1900 in a crowded tile) took 414 us on the serial additions to a bin, now
// 9.
constexpr int kBinPoints = 4;  // per thread

template <int D>
__global__ __launch_bounds__(1024) void spread_bin_kernel(GridParams g, int n, const float *__restrict__ Y, int tb,
                                                          int2 *__restrict__ key, int *__restrict__ cnt) {
  constexpr int B = D == 3 ? 5 : 7, BINS = 1 << (D * B);
  static_assert(BINS <= kSpreadBins, "bins");
  extern __shared__ int bcnt[];
  for (int b = threadIdx.x; b < BINS; b += 1024) bcnt[b] = 0;
  __syncthreads();
  int bin[kBinPoints], rank[kBinPoints];
#pragma unroll
  for (int u = 0; u < kBinPoints; ++u) {
    const int i = (blockIdx.x * kBinPoints + u) * 1024 + threadIdx.x;
    bin[u] = -1;
    if (i < n) {
      float y[D];
      load_pt<D>(Y, i, y);
      int f[D];
      float w[D][4];
      stencil<D>(g, y, f, w);
      int k = 0;
#pragma unroll
      for (int b = 0; b < B; ++b)
#pragma unroll
        for (int a = 0; a < D; ++a) k |= ((f[a] >> (tb + b)) & 1) << (D * b + a);
      bin[u] = k;
      rank[u] = atomicAdd(&bcnt[k], 1);
    }
  }
  __syncthreads();
  for (int b = threadIdx.x; b < BINS; b += 1024) {
    const int c = bcnt[b];
    if (c) bcnt[b] = atomicAdd(&cnt[b], c);
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kBinPoints; ++u)
    if (bin[u] >= 0) key[(blockIdx.x * kBinPoints + u) * 1024 + threadIdx.x] = make_int2(bin[u], bcnt[bin[u]] + rank[u]);
}

// Counts -> first place of each bin (one work-group).
__global__ __launch_bounds__(1024) void spread_scan_kernel(int *__restrict__ cnt) {
  __shared__ int wsum[16];
  constexpr int PER = kSpreadBins / 1024;
  const int t = threadIdx.x, lane = t & 63, wid = t >> 6;
  int v[PER], sum = 0;
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    v[k] = cnt[t * PER + k];
    sum += v[k];
  }
  int inc = sum;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int u = __shfl_up(inc, o, 64);
    if (lane >= o) inc += u;
  }
  if (lane == 63) wsum[wid] = inc;
  __syncthreads();
  int run = inc - sum;
  for (int k = 0; k < wid; ++k) run += wsum[k];
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    cnt[t * PER + k] = run;
    run += v[k];
  }
}

__global__ void spread_place_kernel(int n, const int2 *__restrict__ key, const int *__restrict__ start,
                                    int32_t *__restrict__ ord) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int2 k = key[i];
  ord[start[k.x] + k.y] = i;
}

int launch_spread_order(hipStream_t s, const GridParams &g, int n, const float *Y, int2 *key, int *cnt, int32_t *ord) {
  if (n <= 0) return SGTSNE_OK;
  int tb = 2;
  while ((g.ng >> tb) >= (g.d == 3 ? 32 : 128)) ++tb;
  SGT_TRY(launch_fill(s, reinterpret_cast<float *>(cnt), kSpreadBins, 0.0f));
  const int blocks = div_up(n, kBlock), bblocks = div_up(n, 1024 * kBinPoints);
  if (g.d == 2) spread_bin_kernel<2><<<bblocks, 1024, sizeof(int) << 14, s>>>(g, n, Y, tb, key, cnt);
  else spread_bin_kernel<3><<<bblocks, 1024, sizeof(int) << 15, s>>>(g, n, Y, tb, key, cnt);
  SGT_LAUNCH_CHECK();
  spread_scan_kernel<<<1, 1024, 0, s>>>(cnt);
  SGT_LAUNCH_CHECK();
  spread_place_kernel<<<blocks, kBlock, 0, s>>>(n, key, cnt, ord);
  SGT_LAUNCH_CHECK();
  return SGTSNE_OK;
}

int64_t s2g_scratch_need(const GridParams &g, int n, int mode) {
  int64_t need = 0;
  (void)launch_s2g(nullptr, g, -n, nullptr, nullptr, nullptr, 0, &need, mode);
  return need;
}

int launch_s2g(hipStream_t s, const GridParams &g, int n, const float *Y, float *V, float *scratch,
               int64_t scratch_floats, int64_t *needed, int mode, DevScalars *stamp, const int32_t *ord) {
  const bool query = n < 0;  // size query only
  if (query) n = -n;
  if (n > 0 && g.d == 2 && g.ng <= 32 && mode != SGTSNE_SPREAD_ATOMIC) {
    // matrix cores: no contention however the points crowd the few cells
    const int64_t cells = 3ll * g.ng * g.ng;
    const int chunk = mfma_chunk(n);
    const int blocks = div_up(n, chunk);
    if (needed) *needed = (int64_t)blocks * cells;
    if (query) return SGTSNE_OK;
    SGT_CHECK((int64_t)blocks * cells <= scratch_floats, SGTSNE_ERR_STATE, "spread scratch too small");
    if (g.ng <= 16)
      s2g_mfma_kernel<1><<<blocks, kMfmaBlock, 0, s>>>(g, n, Y, scratch, chunk, stamp);
    else
      s2g_mfma_kernel<2><<<blocks, kMfmaBlock, 0, s>>>(g, n, Y, scratch, chunk, stamp);
    SGT_LAUNCH_CHECK();
    grid_reduce_kernel<<<div_up(cells, 64), 1024, 0, s>>>(scratch, blocks, (int)cells, V, stamp);
    SGT_LAUNCH_CHECK();
    return SGTSNE_OK;
  }
  if (n > 0 && g.d == 3 && g.ng <= 16 && mode != SGTSNE_SPREAD_ATOMIC) {
    const int64_t cells = 4ll * g.ng * g.ng * g.ng;
    const int chunk = mfma3_chunk(n), blocks = div_up(n, chunk);
    if (needed) *needed = (int64_t)blocks * cells;
    if (query) return SGTSNE_OK;
    SGT_CHECK((int64_t)blocks * cells <= scratch_floats, SGTSNE_ERR_STATE, "spread scratch too small");
    s2g_mfma3_kernel<<<blocks, kMfmaBlock, 0, s>>>(g, n, Y, scratch, chunk, stamp);
    SGT_LAUNCH_CHECK();
    grid_reduce_kernel<<<div_up(cells, 64), 1024, 0, s>>>(scratch, blocks, (int)cells, V, stamp);
    SGT_LAUNCH_CHECK();
    return SGTSNE_OK;
  }
  size_t lds = 0;
  int copies = 1;
  const int64_t cells = (int64_t)(g.d == 1 ? g.ng : g.d == 2 ? g.ng * g.ng : g.ng * g.ng * g.ng) * (g.d + 1);
  if (n > 0 && s2g_takes_order(g, mode)) {
    // fixed point in the scratch (2 floats per 64-bit cell): cleared, spread,
    // converted into V and cleared again
    if (needed) *needed = 2 * cells;
    if (query) return SGTSNE_OK;
    SGT_CHECK(2 * cells <= scratch_floats, SGTSNE_ERR_STATE, "spread scratch too small");
    // no cell can exceed 2^61 in magnitude: |weight| <= 1 and the charges
    // are within half the extent of the box centre
    const double maxy = (double)(g.nGrid - 1) / (double)g.scale * (1.0 + 1e-6);
    const double bound = 2.0 * (double)n * (0.5 * maxy + 1.0);
    const int e = std::min(60, std::max(1, 61 - std::ilogb(bound)));
    unsigned long long *Vf = reinterpret_cast<unsigned long long *>(scratch);
    SGT_TRY(launch_fill(s, scratch, 2 * cells, 0.0f));
    // runs long enough to share cells, short enough for two work-groups per CU:
    // 60,000 points late in a 2-D run with runs of 1024 / 128 / 64: 29.9 / 9.4 /
    // 14.0 us; 200,003 points in 3-D with 256 / 128: 68 / 72 us
    const int unit = std::min(g.d == 3 ? kFixUnit3 : 1024, std::max(64, div_up(n, 64 * 512) * 64));
    const int lds_b = 64512;  // two work-groups per CU
    const int blocks = (int)std::min<int64_t>(div_up(n, unit), 2048);
    if (g.d == 2)
      s2g_fix_kernel<2><<<blocks, s2g_threads<2>(), lds_b, s>>>(g, std::ldexp(1.0f, e), n, Y, Vf, unit, lds_b / 8, ord, stamp);
    else
      s2g_fix_kernel<3><<<blocks, s2g_threads<3>(), lds_b, s>>>(g, std::ldexp(1.0f, e), n, Y, Vf, unit, lds_b / 8, ord, stamp);
    SGT_LAUNCH_CHECK();
    fix_to_float_kernel<<<(int)std::min<int64_t>(div_up(cells, 256), 4096), 256, 0, s>>>(
        reinterpret_cast<long long *>(Vf), V, cells, std::ldexp(1.0, -e), stamp);
    SGT_LAUNCH_CHECK();
    return SGTSNE_OK;
  }
  int blocks = 0, chunk = 0;
  if (n > 0 && s2g_lds_fits(g.d, g.ng, &lds, &copies)) {
    // about 64 points per wave, at most 1024 private grids and 64 MiB of them
    int64_t b = std::max<int64_t>(1, div_up(n, (kS2GBlock / 64) * 64));
    b = std::min<int64_t>(b, 1024);
    b = std::min<int64_t>(b, std::max<int64_t>(1, (int64_t)(64ll << 20) / (cells * 4)));
    chunk = div_up(n, b);
    blocks = div_up(n, chunk);
  }
  if (needed) *needed = blocks > 0 ? (int64_t)blocks * cells : 0;
  if (query) return SGTSNE_OK;
  if (blocks > 0 && (int64_t)blocks * cells <= scratch_floats) {
    switch (g.d) {
      case 1: s2g_lds_kernel<1><<<blocks, kS2GBlock, lds, s>>>(g, n, Y, scratch, chunk, copies, stamp); break;
      case 2: s2g_lds_kernel<2><<<blocks, kS2GBlock, lds, s>>>(g, n, Y, scratch, chunk, copies, stamp); break;
      case 3: s2g_lds_kernel<3><<<blocks, kS2GBlock, lds, s>>>(g, n, Y, scratch, chunk, copies, stamp); break;
      default: SGT_CHECK(false, SGTSNE_ERR_ARG, "d must be 1..3");
    }
    SGT_LAUNCH_CHECK();
    grid_reduce_kernel<<<div_up(cells, 64), 1024, 0, s>>>(scratch, blocks, (int)cells, V, stamp);
  } else {
    SGT_TRY(launch_fill(s, V, cells, 0.0f));
    const int ppb = (kBlock / 64) * (g.d == 1 ? 16 : g.d == 2 ? 4 : 1);  // points per block per step
    const int ab = (int)std::min<int64_t>(div_up(n > 0 ? n : 1, ppb), 65536);
    switch (g.d) {
      case 1: s2g_atomic_kernel<1><<<ab, kBlock, 0, s>>>(g, n, Y, V, stamp); break;
      case 2: s2g_atomic_kernel<2><<<ab, kBlock, 0, s>>>(g, n, Y, V, stamp); break;
      case 3: s2g_atomic_kernel<3><<<ab, kBlock, 0, s>>>(g, n, Y, V, stamp); break;
      default: SGT_CHECK(false, SGTSNE_ERR_ARG, "d must be 1..3");
    }
    SGT_LAUNCH_CHECK();
    if (stamp) SGT_TRY(launch_stamp(s, stamp, STAMP_CONV));
  }
  SGT_LAUNCH_CHECK();
  return SGTSNE_OK;
}

int launch_g2s_force(hipStream_t s, const GridParams &g, int n, const float *Y, const float *Phi,
                     float *Frep, int zdirect, RedWork rw, int *nz, DevScalars *stamp, const int32_t *ord) {
  if (g2s_lds_fits(g.d, g.ng, n)) {
    // one 16-wave work-group per CU (the grid copy takes half of its LDS)
    const int lb = std::max(1, std::min({rw.max_blocks, 256, div_up(n > 0 ? n : 1, kG2sLdsBlock)}));
    if (g.d == 2) {
      if (zdirect) g2s_lds_kernel<2, true><<<lb, kG2sLdsBlock, 0, s>>>(g, n, Y, Phi, Frep, rw.part, stamp);
      else g2s_lds_kernel<2, false><<<lb, kG2sLdsBlock, 0, s>>>(g, n, Y, Phi, Frep, rw.part, stamp);
    } else {
      if (zdirect) g2s_lds_kernel<3, true><<<lb, kG2sLdsBlock, 0, s>>>(g, n, Y, Phi, Frep, rw.part, stamp);
      else g2s_lds_kernel<3, false><<<lb, kG2sLdsBlock, 0, s>>>(g, n, Y, Phi, Frep, rw.part, stamp);
    }
    SGT_LAUNCH_CHECK();
    *nz = lb;
    return SGTSNE_OK;
  }
  const int blocks = grid_blocks(n, std::min(rw.max_blocks, 2048));
#define G2S_CASE(DD)                                                                               \
  case DD:                                                                                         \
    if (zdirect) g2s_force_kernel<DD, true><<<blocks, kBlock, 0, s>>>(g, n, Y, Phi, Frep, rw.part, stamp, ord); \
    else g2s_force_kernel<DD, false><<<blocks, kBlock, 0, s>>>(g, n, Y, Phi, Frep, rw.part, stamp, ord);        \
    break;
  switch (g.d) {
    G2S_CASE(1)
    G2S_CASE(2)
    G2S_CASE(3)
    default: SGT_CHECK(false, SGTSNE_ERR_ARG, "d must be 1..3");
  }
#undef G2S_CASE
  SGT_LAUNCH_CHECK();
  *nz = blocks;
  return SGTSNE_OK;
}

int launch_finalize_z(hipStream_t s, int nz, int n, RedWork rw, DevScalars *sc) {
  return finalize(s, FIN_ZNEU, nz, n, rw, sc);
}

int launch_finalize_kl(hipStream_t s, int nblocks, RedWork rw, DevScalars *sc) {
  return finalize(s, FIN_KL, nblocks, 0, rw, sc);
}

// Work-groups of 256 while one per point fits kMaxBoxParts of them, else of
// 1024, so that the few partials still leave four waves per SIMD in flight.
int upd_threads(int n) { return n <= kMaxBoxParts * kBlock ? kBlock : kUpdBlock; }
int upd_blocks(int n) { return std::min(div_up(n > 0 ? n : 1, upd_threads(n)), kMaxBoxParts); }
// the Z partials take the front of the workspace (at most 2048 slots)
BoxPart *box_parts(const RedWork &rw) { return reinterpret_cast<BoxPart *>(rw.part + (size_t)8 * 2048); }

int launch_set_points(hipStream_t s, int d, int n, const float *raw, int layout, const int32_t *perm, float *Y,
                      int reset, float *uY, float *gains, RedWork rw, DevScalars *sc, HostScalars *hs,
                      unsigned long long seq) {
  const int tpb = upd_threads(n), blocks = upd_blocks(n), aos = layout == SGTSNE_LAYOUT_AOS;
  BoxPart *box = box_parts(rw);
#define SET_CASE(DD)                                                                                  \
  case DD:                                                                                            \
    set_points_kernel<DD><<<blocks, tpb, 0, s>>>(n, raw, aos, perm, Y, reset, uY, gains, box);        \
    SGT_LAUNCH_CHECK();                                                                               \
    center_kernel<DD><<<blocks, tpb, 0, s>>>(n, Y, box, blocks, sc, hs, seq, 0);                      \
    break;
  switch (d) {
    SET_CASE(1)
    SET_CASE(2)
    SET_CASE(3)
    default: SGT_CHECK(false, SGTSNE_ERR_ARG, "d must be 1..3");
  }
#undef SET_CASE
  SGT_LAUNCH_CHECK();
  return SGTSNE_OK;
}

int launch_get_points(hipStream_t s, int d, int n, const float *in, int layout, const int32_t *perm, double scale,
                      float *raw) {
  const int blocks = std::min(div_up(n > 0 ? n : 1, kBlock), 4096), aos = layout == SGTSNE_LAYOUT_AOS;
  switch (d) {
    case 1: get_points_kernel<1><<<blocks, kBlock, 0, s>>>(n, in, aos, perm, scale, raw); break;
    case 2: get_points_kernel<2><<<blocks, kBlock, 0, s>>>(n, in, aos, perm, scale, raw); break;
    case 3: get_points_kernel<3><<<blocks, kBlock, 0, s>>>(n, in, aos, perm, scale, raw); break;
    default: SGT_CHECK(false, SGTSNE_ERR_ARG, "d must be 1..3");
  }
  SGT_LAUNCH_CHECK();
  return SGTSNE_OK;
}

int launch_update_center(hipStream_t s, int d, int n, float *Y, float *uY, float *gains, const float *Fattr,
                         const float *Frep, float alpha, float momentum, float eta, int nz, RedWork rw,
                         DevScalars *sc, HostScalars *hs, unsigned long long seq, int stamp) {
  const int tpb = upd_threads(n), blocks = upd_blocks(n);
  SGT_CHECK(nz >= 1 && nz <= 2048 && rw.max_blocks >= 2048 + kMaxBoxParts, SGTSNE_ERR_STATE, "%d partials of Z", nz);
  BoxPart *box = box_parts(rw);
#define UPD_CASE(DD)                                                                                            \
  case DD:                                                                                                      \
    update_kernel<DD><<<blocks, tpb, 0, s>>>(n, Y, uY, gains, Fattr, Frep, alpha, momentum, eta, rw.part, nz, sc, box, \
                                             stamp);                                                            \
    SGT_LAUNCH_CHECK();                                                                                         \
    center_kernel<DD><<<blocks, tpb, 0, s>>>(n, Y, box, blocks, sc, hs, seq, stamp);                            \
    break;
  switch (d) {
    UPD_CASE(1)
    UPD_CASE(2)
    UPD_CASE(3)
    default: SGT_CHECK(false, SGTSNE_ERR_ARG, "d must be 1..3");
  }
#undef UPD_CASE
  SGT_LAUNCH_CHECK();
  return SGTSNE_OK;
}

int launch_rep_exact(hipStream_t s, int d, int n, const float *Y, float *Frep, RedWork rw,
                     DevScalars *sc) {
  const int blocks = div_up(n > 0 ? n : 1, kBlock);
  SGT_CHECK(blocks <= rw.max_blocks, SGTSNE_ERR_ARG, "exact repulsion: n too large for workspace");
  switch (d) {
    case 1: rep_exact_kernel<1><<<blocks, kBlock, 0, s>>>(n, Y, Frep, rw.part); break;
    case 2: rep_exact_kernel<2><<<blocks, kBlock, 0, s>>>(n, Y, Frep, rw.part); break;
    case 3: rep_exact_kernel<3><<<blocks, kBlock, 0, s>>>(n, Y, Frep, rw.part); break;
    default: SGT_CHECK(false, SGTSNE_ERR_ARG, "d must be 1..3");
  }
  SGT_LAUNCH_CHECK();
  return finalize(s, FIN_ZEXACT, blocks, n, rw, sc);
}

}  // namespace sgt
