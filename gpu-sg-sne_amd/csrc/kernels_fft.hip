// kernels_fft.hip -- non-periodic grid convolution of one job with the kernels
// K2 = (1 + h^2 r^2)^-2 and K1 = (1 + h^2 r^2)^-1 by zero-padded FFTs in LDS
// (the passes themselves are in fft_device.hpp, shared with the batched
// engine).
#include "common.hpp"
#include "kernels.hpp"
#include "fft_device.hpp"
#include "../../include/sgtsne.h"

#include <algorithm>
#include <cmath>

namespace sgt {

namespace {

using namespace fft;

template <int IN, int OUT, int MID, bool EC>
__global__ __launch_bounds__(kFftThreads) void fft_pass_kernel(PassArgs a) {
  extern __shared__ float2 lds[];
  pass_body<IN, OUT, MID, EC>(a, blockIdx.x, blockIdx.y, lds);
}

// Two independent passes in one launch: work-groups [0, blocks_k) take a pass
// of the kernel's, the others (blocks_d per channel pair) one of the data's.
template <int KI, int KO, bool KE, int IN, int OUT, bool EC>
__global__ __launch_bounds__(kFftThreads) void fft_two_kernel(PassArgs k, int blocks_k, PassArgs a, int blocks_d) {
  extern __shared__ float2 lds[];
  int b = blockIdx.x;
  if (b < blocks_k) {
    pass_body<KI, KO, MID_FWD, KE>(k, b, 0, lds);
  } else {
    b -= blocks_k;
    pass_body<IN, OUT, MID_FWD, EC>(a, b % blocks_d, b / blocks_d, lds);
  }
}

template <int KI, int KO, bool KE, int IN, int OUT, bool EC>
int run_two(hipStream_t s, const PassArgs &k, const PassArgs &a, int pairs) {
  const int bk = pass_blocks(k), bd = pass_blocks(a);
  const size_t lds = std::max(pass_lds_bytes(k.nl, k.L, k.Lp), pass_lds_bytes(a.nl, a.L, a.Lp));
  fft_two_kernel<KI, KO, KE, IN, OUT, EC><<<bk + bd * pairs, kFftThreads, lds, s>>>(k, bk, a, bd);
  SGT_LAUNCH_CHECK();
  return SGTSNE_OK;
}

// Fills every twiddle table: entry t of the table of length L is
// exp(-2 pi i t / L), evaluated in FP64 and rounded once.
__global__ void twiddle_kernel(float2 *tw, int total) {
  const int g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= total) return;
  int lo = 1, hi = kMaxL / 2 + 1;  // off[lo] <= g < off[hi]; the last such lo is a supported length
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (fft_tables().off[mid] <= g) lo = mid;
    else hi = mid;
  }
  const int t = g - fft_tables().off[lo], L = 2 * lo;
  double sn, cs;
  sincospi(-2.0 * (double)t / (double)L, &sn, &cs);
  tw[g] = make_float2((float)cs, (float)sn);
}

template <int IN, int OUT, int MID, bool EC>
int run_pass(hipStream_t s, const PassArgs &a, int pairs) {
  const int blocks = pass_blocks(a);
  if (blocks == 0) return SGTSNE_OK;
  const size_t lds = pass_lds_bytes(a.nl, a.L, a.Lp);
  dim3 grid(blocks, pairs);
  hipLaunchKernelGGL((fft_pass_kernel<IN, OUT, MID, EC>), grid, dim3(kFftThreads), lds, s, a);
  SGT_LAUNCH_CHECK();
  return SGTSNE_OK;
}

int run_kind(hipStream_t s, int kind, const PassArgs &a, int pairs, bool node_major) {
  switch (kind) {
    case PK_KGEN: return run_pass<IN_KGEN, OUT_KT, MID_FWD, true>(s, a, pairs);
    case PK_W_W_CONV: return run_pass<IN_W, OUT_W, MID_CONV, false>(s, a, pairs);
    case PK_W_PHI:
      return node_major ? run_pass<IN_W, OUT_PHIQ, MID_INV, true>(s, a, pairs)
                        : run_pass<IN_W, OUT_PHIPAIR, MID_INV, true>(s, a, pairs);
    case PK_V_PHI:
      return node_major ? run_pass<IN_VPAIR, OUT_PHIQ, MID_CONV, true>(s, a, pairs)
                        : run_pass<IN_VPAIR, OUT_PHIPAIR, MID_CONV, true>(s, a, pairs);
    case PK_W_W_INV: return run_pass<IN_W, OUT_W, MID_INV, false>(s, a, pairs);
    default: SGT_CHECK(false, SGTSNE_ERR_ARG, "bad FFT pass kind");
  }
}

// ---- small grids: the convolution as a sum ---------------------------------------
// On the grids of a run's first iterations (2-D side <= 32, 3-D side <= 16) the
// transforms are a chain of three (3-D: five) launches whose work is a few
// thousand operations per line; the sum over all pairs of nodes is 262,144
// multiply-adds on a 16 x 16 grid and 84 million on a 16-cube, one launch
// spread over the device.  Sums in FP64 (which issues at the rate of FP32 here)
// of the transforms' FP32 kernel values and charges, in a fixed order: early in a
// run the charges y_i nearly cancel, and FP32 sums of them could be further off
// than the transforms.  Frep against 64 bits, mean over 700-30,000 points,
// transforms / FP32 sums / these: 2-D 2.89e-7 / 2.80e-7 / 2.64e-7, 3-D 3.52e-7 /
// 3.39e-7 / 3.33e-7 (with FP64 kernel values too 2.63e-7 and 3.32e-7).
// 16 x 16 grid: 25.5 us of transforms -> 4.4; 16-cube: 58 -> 12.
// Potentials come node-major; channel 3 (2-D) or 4 (3-D) is the charge with K1.
constexpr int kDirect2 = 32, kDirect3 = 16;  // largest sides
constexpr int kDirectX = 16;                 // outputs of a 2-D work-group

// A work-group per grid row y and kDirectX of its nodes x; thread (x, j) adds the
// nodes of row y' = j.
template <int XP>
__global__ __launch_bounds__(kDirectX *XP) void conv_direct2_kernel(int ng, float hsq, const float *__restrict__ V,
                                                                   float4 *__restrict__ Phi) {
  __shared__ float4 vs[XP][XP];    // charges of (x', y')
  __shared__ double2 ks[XP][XP];   // K2, K1 at (|x - x'|, |y - y'|)
  constexpr int WAVES = kDirectX * XP / 64;
  __shared__ double4 red[WAVES][kDirectX];
  const int xl = threadIdx.x % kDirectX, j = threadIdx.x / kDirectX, x = blockIdx.y * kDirectX + xl, y = blockIdx.x;
  const int G = ng * ng;
#pragma unroll
  for (int t = threadIdx.x; t < XP * XP; t += kDirectX * XP) {
    const int xx = t % XP, jj = t / XP, e = jj * ng + xx;
    vs[jj][xx] = xx < ng && jj < ng ? make_float4(V[e], V[G + e], V[2 * G + e], 0.0f) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    const float k1 = 1.0f / (1.0f + hsq * (float)(xx * xx + (y - jj) * (y - jj)));
    ks[jj][xx] = make_double2((double)(k1 * k1), (double)k1);
  }
  __syncthreads();
  double4 acc = make_double4(0.0, 0.0, 0.0, 0.0);
#pragma unroll 8
  for (int xp = 0; xp < ng; ++xp) {
    const float4 v = vs[j][xp];
    const double2 k = ks[j][abs(x - xp)];
    acc.x = fma(k.x, (double)v.x, acc.x);
    acc.y = fma(k.x, (double)v.y, acc.y);
    acc.z = fma(k.x, (double)v.z, acc.z);
    acc.w = fma(k.y, (double)v.x, acc.w);
  }
  // a wave's four rows y' added across it, then the waves' sums in order
#pragma unroll
  for (int o = kDirectX; o < 64; o <<= 1) {
    acc.x += __shfl_xor(acc.x, o, 64);
    acc.y += __shfl_xor(acc.y, o, 64);
    acc.z += __shfl_xor(acc.z, o, 64);
    acc.w += __shfl_xor(acc.w, o, 64);
  }
  if ((threadIdx.x & 63) < kDirectX) red[threadIdx.x >> 6][xl] = acc;
  __syncthreads();
  if (j == 0 && x < ng) {
#pragma unroll
    for (int k = 1; k < WAVES; ++k) {
      const double4 t = red[k][xl];
      acc.x += t.x;
      acc.y += t.y;
      acc.z += t.z;
      acc.w += t.w;
    }
    Phi[y * ng + x] = make_float4((float)acc.x, (float)acc.y, (float)acc.z, (float)acc.w);
  }
}

// One work-group per row (y, z); thread (y', z') adds the 16 nodes of its row
// to the 16 outputs in registers, and the threads' sums are added across each
// wave and then over the four waves.  Bound by the loads: a lane's row is lines of
// its own, so it is read in 16-byte vectors (11.8 us with them, 18.7 without).
__global__ __launch_bounds__(256) void conv_direct3_kernel(int ng, float hsq, const float *__restrict__ V,
                                                           float *__restrict__ Phi) {
  constexpr int S = kDirect3, C = 5;
  __shared__ double red[4][S * C];
  const int yp = threadIdx.x % S, zp = threadIdx.x / S;
  const int y = blockIdx.x % ng, z = blockIdx.x / ng, G = ng * ng * ng;
  const bool in = yp < ng && zp < ng;
  float k1[S];
  const int r0 = (y - yp) * (y - yp) + (z - zp) * (z - zp);
#pragma unroll
  for (int d = 0; d < S; ++d) k1[d] = 1.0f / (1.0f + hsq * (float)(d * d + r0));
  double acc[S][C];
#pragma unroll
  for (int x = 0; x < S; ++x)
#pragma unroll
    for (int c = 0; c < C; ++c) acc[x][c] = 0.0;
  const float *row = V + (zp * ng + yp) * ng;
  float vr[4][S];
  if (ng % 4 == 0) {  // rows of whole 16-byte vectors (every lane reads lines of its own)
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int h = 0; h < S / 4; ++h) {
        const float4 q = in && 4 * h < ng ? reinterpret_cast<const float4 *>(row + c * G)[h] : make_float4(0.f, 0.f, 0.f, 0.f);
        vr[c][4 * h] = q.x;
        vr[c][4 * h + 1] = q.y;
        vr[c][4 * h + 2] = q.z;
        vr[c][4 * h + 3] = q.w;
      }
  } else {
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int xp = 0; xp < S; ++xp) vr[c][xp] = in && xp < ng ? row[c * G + xp] : 0.0f;
  }
#pragma unroll
  for (int xp = 0; xp < S; ++xp) {
    const float v[4] = {vr[0][xp], vr[1][xp], vr[2][xp], vr[3][xp]};
#pragma unroll
    for (int x = 0; x < S; ++x) {
      const float k = k1[x > xp ? x - xp : xp - x], kk = k * k;
#pragma unroll
      for (int c = 0; c < 4; ++c) acc[x][c] = fma((double)kk, (double)v[c], acc[x][c]);
      acc[x][4] = fma((double)k, (double)v[0], acc[x][4]);
    }
  }
  // across the wave: halves exchanged until 16 groups of four lanes hold 5 sums
  // each (85 shuffles; 80 butterflies would be 480), then added over the four
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  double a[S * C];
#pragma unroll
  for (int x = 0; x < S; ++x)
#pragma unroll
    for (int c = 0; c < C; ++c) a[x * C + c] = acc[x][c];
#pragma unroll
  for (int half = S * C / 2, o = 32; o >= 4; half /= 2, o /= 2) {
    const bool up = lane & o;
#pragma unroll
    for (int i = 0; i < half; ++i) {
      const double keep = up ? a[i + half] : a[i], send = up ? a[i] : a[i + half];
      a[i] = keep + __shfl_xor(send, o, 64);
    }
  }
#pragma unroll
  for (int i = 0; i < C; ++i) {
    a[i] += __shfl_xor(a[i], 2, 64);
    a[i] += __shfl_xor(a[i], 1, 64);
    if ((lane & 3) == 0) red[w][(lane >> 2) * C + i] = a[i];
  }
  __syncthreads();
  for (int o = threadIdx.x; o < S * C; o += blockDim.x) {
    const int x = o / C, c = o - x * C;
    if (x >= ng) continue;
    const double s = (red[0][o] + red[1][o]) + (red[2][o] + red[3][o]);
    const int e = (z * ng + y) * ng + x;
    Phi[c < 4 ? 4 * e + c : 4 * G + e] = (float)s;
  }
}

}  // namespace

size_t twiddle_count() { return (size_t)fft_table_size(); }

int fft_length_for(int ng) { return fft_length(2 * ng - 1); }

int init_twiddles(hipStream_t s, float2 *tw) {
  const int total = fft_table_size();
  twiddle_kernel<<<div_up(total, 256), 256, 0, s>>>(tw, total);
  SGT_LAUNCH_CHECK();
  return SGTSNE_OK;
}

int conv_workspace_bytes(int d, int ng, int L, size_t *w_bytes, size_t *k_bytes) {
  const int pairs = 3;  // at most (1 + ceil(d / 2)) for d <= 3
  const size_t H = (size_t)L / 2 + 1;
  size_t wl = d == 1 ? 0 : d == 2 ? (size_t)ng * L : (size_t)ng * L * L;
  *w_bytes = pairs * wl * sizeof(float2);
  size_t hd = d == 1 ? H : d == 2 ? H * H : H * H * H;
  *k_bytes = hd * sizeof(float2);
  return SGTSNE_OK;
}

int launch_conv(hipStream_t s, const GridParams &g, int zdirect, const float *V, float *Phi,
                const ConvBuffers &b, bool node_major) {
  SGT_CHECK(g.L <= kMaxL && g.L >= 2 * g.ng - 1 && fft_smooth(g.L), SGTSNE_ERR_ARG,
            "FFT length %d invalid for ng %d", g.L, g.ng);
  const float hsq = (float)(g.hgrid * g.hgrid);
  if (node_major && g.d == 2 && g.ng <= kDirect2) {
    float4 *Phi4 = reinterpret_cast<float4 *>(Phi);
    if (g.ng <= 16) conv_direct2_kernel<16><<<g.ng, 16 * kDirectX, 0, s>>>(g.ng, hsq, V, Phi4);
    else conv_direct2_kernel<32><<<dim3(g.ng, 2), 32 * kDirectX, 0, s>>>(g.ng, hsq, V, Phi4);
    SGT_LAUNCH_CHECK();
    return SGTSNE_OK;
  }
  if (node_major && g.d == 3 && g.ng <= kDirect3) {
    conv_direct3_kernel<<<g.ng * g.ng, 256, 0, s>>>(g.ng, hsq, V, Phi);
    SGT_LAUNCH_CHECK();
    return SGTSNE_OK;
  }
  ConvPtrs ptr{V, Phi, b.W, b.Kt1, b.Kt2, b.Kh, b.tw};
  PassArgs args[kMaxPasses];
  int pairs[kMaxPasses], kinds[kMaxPasses];
  const int np = conv_setup(g, zdirect != 0, ptr, args, pairs, kinds);
  // the kernel's passes ride along with the data's they do not depend on
  int i = 0;
  if (g.d == 2) {
    SGT_TRY((run_two<IN_KGEN, OUT_KT, true, IN_VPAIR, OUT_W, true>(s, args[0], args[1], pairs[1])));
    i = 2;
  } else if (g.d == 3) {
    SGT_TRY((run_two<IN_KGEN, OUT_KT, true, IN_VPAIR, OUT_W, true>(s, args[0], args[2], pairs[2])));
    SGT_TRY((run_two<IN_KT, OUT_KT, false, IN_W, OUT_W, false>(s, args[1], args[3], pairs[3])));
    i = 4;
  }
  for (; i < np; ++i) SGT_TRY(run_kind(s, kinds[i], args[i], pairs[i], node_major));
  return SGTSNE_OK;
}

}  // namespace sgt
