// The forward pass and the input gradient of small convolution layers, summed directly over the
// filter taps in one launch.  The three launches of the transform pipeline take 10 to 16 us
// however small the layer is, each waiting for the one before it; where that is longer than
// the sums take (runsSmall, conv_pipeline.hip), nothing is transformed.
#include "common.h"

#include <algorithm>
#include <cmath>

namespace fbfft_amd {
namespace {

constexpr int kWaves = 8;
constexpr int kFilters = 8;          // output planes per workgroup

// n / d for 0 <= n < 2^16 and 0 < d < 2^16: ((n + 1) m) >> 32 with m = floor((2^32 - 1) / d)
struct Divisor {
  unsigned d, m;
};
inline Divisor divisor(int d) { return {(unsigned)d, 0xffffffffu / (unsigned)d}; }
__device__ __forceinline__ int divide(int n, const Divisor& v) {
  return (int)__umulhi((unsigned)n + 1, v.m);
}

struct SmallArgs {
  const float* in;
  const float* w;
  float* out;
  long sB, sC, oB, oM, wM, wC;       // strides in floats
  int sY, sX, oY, oX;
  long wOrigin, wY, wX;              // of the tap that meets window row 0, column 0; wY, wX < 0: reversed
  int C, M, H, W, OH, OW, kH, padY, padX;
  int P;                             // output pixels of all images
  int mGroups;
  Divisor byRow, byTaps;             // kH, C kH KX
};

// filter rows of a wave whose input values are in flight (narrow filters, four instead of two:
// 65 x 6 x 12 x 20, input gradient of 193 filters of 1 x 1 16.0 -> 7.6 us; 8 x 12 x 10 x 7, 55 of 6 x
// 6 9.7 -> 12.6)
constexpr int rowsAhead(int kW) { return kW <= 2 ? 4 : 2; }

// A workgroup: 64 output pixels (a lane each, of any row and image) x 8 output planes.  Its eight
// waves take every eighth filter row (input plane, row of the filter) each and add up in LDS
// in wave order.  The 8 planes' filters wait in LDS, [input plane][row][column][8], and are read
// by all lanes at once; a row's KX input values are in flight under the previous row's
// multiply-adds.  What bounds it is the L1: a load of 64 neighbouring floats, some 15 cycles a
// CU, feeds 8 multiply-adds, 8 cycles.
// PAD: the input gradient, whose windows reach over the edges of the gradient that they read.
template <int KX, bool PAD>
__global__ __launch_bounds__(64 * kWaves) void convSmall(SmallArgs g) {
  constexpr int kAhead = rowsAhead(KX);
  extern __shared__ float lds[];
  const int t = threadIdx.x, lane = t % 64;
  const int wave = __builtin_amdgcn_readfirstlane(t / 64);
  const int m0 = blockIdx.x % g.mGroups * kFilters;
  const int p0 = blockIdx.x / g.mGroups * 64;
  const int plane = g.OH * g.OW;
  const int rows = g.C * g.kH, taps = rows * KX;

  // this lane's pixel; its window relative to the workgroup's first image (in the window's place
  // for lanes behind the last pixel, too: they load and store nothing of their own)
  const int b0 = p0 / plane;
  const int p = min(p0 + lane, g.P - 1);
  const int b = p / plane, y = p % plane / g.OW, x = p % plane % g.OW;
  const int y0 = y - g.padY, x0 = x - g.padX;
  const unsigned at = (unsigned)((b - b0) * g.sB + (long)y * g.sY + (long)x * g.sX) * (unsigned)sizeof(float);
  const char* const image = reinterpret_cast<const char*>(g.in + b0 * g.sB);

  // One filter row's input values: element (c, y0 + ky, x0 + kx).  Those outside are loaded from the
  // lane's own window base (inside) and count as zero.
  auto fetch = [&](float (&v)[KX], int c, int ky) __attribute__((always_inline)) {
#pragma unroll
    for (int kx = 0; kx < KX; ++kx) {
      if constexpr (PAD) {
        const bool inside = (unsigned)(y0 + ky) < (unsigned)g.H && (unsigned)(x0 + kx) < (unsigned)g.W;
        const long off = inside ? (long)(y0 + ky) * g.sY + (long)(x0 + kx) * g.sX : 0;
        const float u = *reinterpret_cast<const float*>(
            image + ((b - b0) * g.sB + (long)c * g.sC + off) * (long)sizeof(float));
        v[kx] = inside ? u : 0.f;
      } else {
        const char* base = image + ((long)c * g.sC + (long)ky * g.sY + (long)kx * g.sX) * (long)sizeof(float);
        v[kx] = *reinterpret_cast<const float*>(base + at);
      }
    }
  };
  // (rows behind the last one are the last one, which nothing multiplies)
  float v[kAhead][KX];
  auto fetchRow = [&](float (&to)[KX], int row) __attribute__((always_inline)) {
    const int r = min(row, rows - 1), c = divide(r, g.byRow);
    fetch(to, c, r - c * g.kH);
  };
#pragma unroll
  for (int u = 0; u < kAhead; ++u) fetchRow(v[u], wave + u * kWaves);

  // the filters: consecutive threads along the taps of one output plane
  for (int f0 = t; f0 < taps * kFilters; f0 += 4 * 64 * kWaves) {
    float w[4];
    int to[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int f = min(f0 + u * 64 * kWaves, taps * kFilters - 1);
      const int m = divide(f, g.byTaps), e = f - m * taps;
      const int row = e / KX, kx = e - row * KX, c = divide(row, g.byRow), ky = row - c * g.kH;
      to[u] = e * kFilters + m;
      // (the last output plane's where there is none: those sums are not stored)
      w[u] = g.w[min(m0 + m, g.M - 1) * g.wM + c * g.wC + g.wOrigin + ky * g.wY + kx * g.wX];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) lds[to[u]] = w[u];
  }
  __syncthreads();

  // (kAhead rows at a time: a chain of a few dozen roundings, not of all the wave's taps)
  float total[kFilters];
#pragma unroll
  for (int j = 0; j < kFilters; ++j) total[j] = 0.f;
  for (int first = wave; first < rows; first += kAhead * kWaves) {
    float sum[kFilters];
#pragma unroll
    for (int j = 0; j < kFilters; ++j) sum[j] = 0.f;
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      const int row = first + u * kWaves;
      if (row < rows) {
        const float4* f = reinterpret_cast<const float4*>(lds + row * KX * kFilters);
#pragma unroll
        for (int kx = 0; kx < KX; ++kx) {
          const float4 lo = f[2 * kx], hi = f[2 * kx + 1];
          sum[0] = __builtin_fmaf(v[u][kx], lo.x, sum[0]);
          sum[1] = __builtin_fmaf(v[u][kx], lo.y, sum[1]);
          sum[2] = __builtin_fmaf(v[u][kx], lo.z, sum[2]);
          sum[3] = __builtin_fmaf(v[u][kx], lo.w, sum[3]);
          sum[4] = __builtin_fmaf(v[u][kx], hi.x, sum[4]);
          sum[5] = __builtin_fmaf(v[u][kx], hi.y, sum[5]);
          sum[6] = __builtin_fmaf(v[u][kx], hi.z, sum[6]);
          sum[7] = __builtin_fmaf(v[u][kx], hi.w, sum[7]);
        }
      }
      fetchRow(v[u], row + kAhead * kWaves);
    }
#pragma unroll
    for (int j = 0; j < kFilters; ++j) total[j] += sum[j];
  }

  __syncthreads();  // the filters are done with
#pragma unroll
  for (int j = 0; j < kFilters; ++j) lds[(wave * kFilters + j) * 64 + lane] = total[j];
  __syncthreads();
  float s = 0.f;
#pragma unroll
  for (int k = 0; k < kWaves; ++k) s += lds[(k * kFilters + wave) * 64 + lane];
  if (p0 + lane < g.P && m0 + wave < g.M)
    g.out[b * g.oB + (m0 + wave) * g.oM + (long)y * g.oY + (long)x * g.oX] = s;
}

}  // namespace

// Estimated us of a pass: the rounds of workgroups on the fullest CU, each with its waves' loads
// (those of rows behind the last one, too) and its filters, and one chain of them.  A load of lanes in
// several images touches more cache lines.  Fitted to 2600 random passes of 1 to 16000 workgroups, half
// of them of at most 9 x 9 pixels: forward within 25 % of nine in ten, input gradients within 15 %.
double convSmallMicroseconds(int pass, int B, int C, int M, int OH, int OW, int kH, int kW) {
  const double pixels = (double)OH * OW;
  const double rounds = std::ceil(std::ceil(B * pixels / 64) * ceilDiv(M, kFilters) / 256);
  const int ahead = rowsAhead(kW), waveRows = ceilDiv(C * kH, kWaves);
  const double loads = (ceilDiv(waveRows, ahead) + 1) * ahead * kW, taps = (double)C * kH * kW;
  const double images = std::max(1.0, std::min(64 / pixels, (double)B)), apart = std::min(1.0, (images - 1) / 31.5);
  if (pass == 0)
    return 2.1 + (1 + 1.18 * apart) * (rounds * (0.45 + loads * (0.0234 + 0.0279 / kW) + 0.003 * taps) +
                                       0.0014 * loads + 0.0035 * taps);
  return 2.35 + (1 + 0.175 * apart) * (rounds * (0.16 + loads * (0.0544 + 0.0283 / kW) + 0.0021 * taps) +
                                       0.0026 * taps);
}

int launchConvSmall(int pass, const float* x, const int* xStride, const int* xSize, const float* y,
                    const int* yStride, const int* ySize, float* out, const int* outStride, const int* outSize,
                    hipStream_t s) {
  const int kH = ySize[2], kW = ySize[3];
  SmallArgs g{};
  g.in = x;
  g.w = y;
  g.out = out;
  g.sB = xStride[0]; g.sC = xStride[1]; g.sY = xStride[2]; g.sX = xStride[3];
  g.oB = outStride[0]; g.oM = outStride[1]; g.oY = outStride[2]; g.oX = outStride[3];
  g.wM = yStride[pass]; g.wC = yStride[1 - pass]; g.wY = yStride[2]; g.wX = yStride[3];
  g.C = xSize[1]; g.M = outSize[1];
  g.H = xSize[2]; g.W = xSize[3]; g.OH = outSize[2]; g.OW = outSize[3];
  g.kH = kH;
  if (pass == 1) {
    g.wOrigin = (kH - 1) * g.wY + (kW - 1) * g.wX;
    g.wY = -g.wY; g.wX = -g.wX;
    g.padY = kH - 1; g.padX = kW - 1;
  }
  g.P = xSize[0] * g.OH * g.OW;
  g.mGroups = ceilDiv(g.M, kFilters);
  g.byRow = divisor(kH);
  g.byTaps = divisor(g.C * kH * kW);
  const size_t bytes = sizeof(float) * kFilters * std::max(g.C * kH * kW, 64 * kWaves);
  const dim3 grid((unsigned)(ceilDiv(g.P, 64) * g.mGroups)), block(64 * kWaves);
  auto go = [&](auto kx) {
    constexpr int KX = decltype(kx)::value;
    if (pass == 1)
      convSmall<KX, true><<<grid, block, bytes, s>>>(g);
    else
      convSmall<KX, false><<<grid, block, bytes, s>>>(g);
  };
  switch (kW) {
    case 1: go(std::integral_constant<int, 1>{}); break;
    case 2: go(std::integral_constant<int, 2>{}); break;
    case 3: go(std::integral_constant<int, 3>{}); break;
    case 4: go(std::integral_constant<int, 4>{}); break;
    case 5: go(std::integral_constant<int, 5>{}); break;
    case 6: go(std::integral_constant<int, 6>{}); break;
    case 7: go(std::integral_constant<int, 7>{}); break;
    case 8: go(std::integral_constant<int, 8>{}); break;
    case 9: go(std::integral_constant<int, 9>{}); break;
    case 10: go(std::integral_constant<int, 10>{}); break;
    case 11: go(std::integral_constant<int, 11>{}); break;
  }
  return launchStatus();
}

}  // namespace fbfft_amd
