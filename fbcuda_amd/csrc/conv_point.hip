// Convolution layers with filters of 1 x 1: each pass is one product of matrices, on the fp32 matrix
// instructions, without transforms.
//
//   forward pass     out[b][m][p]  = sum_c w[m][c] in[b][c][p]      (p: pixel)
//   input gradient   gin[b][c][p]  = sum_m w[m][c] gout[b][m][p]    (the same with the filters transposed)
//   weight gradient  gw[m][c]      = sum_(b, p) gout[b][m][p] in[b][c][p]
#include "common.h"

#include <algorithm>
#include <cmath>

namespace fbfft_amd {
namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
// four floats that start at any float
typedef float __attribute__((ext_vector_type(4), aligned(4))) AnyFour;
typedef const __attribute__((address_space(1))) AnyFour* GlobalFour;

// A wave-uniform address and a lane's 32-bit offset, pinned apart up to the load, which adds them
// (otherwise the sum is widened to 64 bits in vector registers, per load).
__device__ __forceinline__ floatx4 loadFour(const char* base, unsigned offset) {
  asm volatile("" : "+s"(base));
  asm volatile("" : "+v"(offset));
  return *(GlobalFour)(base + offset);
}

struct PointArgs {
  const float* x;
  const float* w;
  float* out;
  long xB, xC, oB, oM, wM, wC;  // strides in floats
  int C, M, pixels, words, total;  // words: groups of four pixels of an image
  int images, rowTiles;
};

constexpr int kPointChunk = 128;  // contracted planes whose filters wait in LDS

// Passes 0 and 1.  A wave: 16 rows (output planes), once or twice, x 16 groups of four neighbouring pixels: a
// lane's 16-byte load of one plane supplies four columns' products, and its results leave as 16-byte
// stores.  (The last four pixels of an image may be some of the four before; both lanes then store the same
// values.)  Nothing but the filters, [plane][row], waits in LDS.  What bounds it is memory; matrix instructions
// take most of the rest.  Nontemporal stores (results of many planes 65 -> 115 us, others +-10 %), rows of 32 on
// 32 x 32 x 2 instructions (0.9 to 1.4 of the time) and 48 or 64 rows (1.0 to 1.5) measured and not kept.
template <int RM>
__global__ __launch_bounds__(256, 2) void pointProducts(PointArgs g) {
  constexpr int MT = 16 * RM, ROW = MT + 1;
  constexpr int AHEAD = 4;  // steps of 4 planes whose pixels are in flight
  __shared__ float filters[kPointChunk * ROW];
  const int t = threadIdx.x, lane = t % 64, r = lane % 16, h = lane / 16;
  const int wave = __builtin_amdgcn_readfirstlane(t / 64);
  const int per = (g.total + 7) / 8;
  const int logical = (blockIdx.x % 8) * per + blockIdx.x / 8;
  if (logical >= g.total) return;
  const int m0 = logical % g.rowTiles * MT;
  const int first = (logical / g.rowTiles * 4 + wave) * 16;  // the wave's first group of pixels

  const int b0 = min(first, g.images * g.words - 1) / g.words;
  const int group = min(first + r, g.images * g.words - 1), b = group / g.words;
  const int p = min(4 * (group - b * g.words), g.pixels - 4);
  const unsigned at = (unsigned)((b - b0) * g.xB + p) * (unsigned)sizeof(float);
  const unsigned planeBytes = (unsigned)g.xC * (unsigned)sizeof(float);
  const char* const image = reinterpret_cast<const char*>(g.x + b0 * g.xB);

  floatx4 sum[RM][4], total[RM][4];
#pragma unroll
  for (int m = 0; m < RM; ++m)
#pragma unroll
    for (int n = 0; n < 4; ++n)
      sum[m][n] = total[m][n] = floatx4{0.f, 0.f, 0.f, 0.f};

  for (int c0 = 0; c0 < g.C; c0 += kPointChunk) {
    const int count = min(kPointChunk, g.C - c0), padded = (count + 3) / 4 * 4, steps = padded / 4;
    // plane c0 + 4 s + h of this lane's pixels (behind the last plane: the last one, times zero)
    floatx4 x[2][AHEAD];
    auto request = [&](int s, int set) __attribute__((always_inline)) {
#pragma unroll
      for (int u = 0; u < AHEAD; ++u) {
        const int k = 4 * min(s + u, steps - 1), own = min(k + h, count - 1) - k;
        x[set][u] = loadFour(image + (long)(c0 + k) * g.xC * (long)sizeof(float), at + (unsigned)own * planeBytes);
      }
    };
    request(0, 0);
    __syncthreads();
    for (int i = t; i < padded * MT; i += 256) {
      // neighbouring lanes along the filters' contiguous side
      const int k = g.wC == 1 ? i % padded : i / MT, m = g.wC == 1 ? i / padded : i % MT;
      const float f = g.w[min(m0 + m, g.M - 1) * g.wM + min(c0 + k, g.C - 1) * g.wC];
      filters[k * ROW + m] = m0 + m < g.M && k < count ? f : 0.f;
    }
    __syncthreads();
    auto multiply = [&](int s, int set) __attribute__((always_inline)) {
#pragma unroll
      for (int u = 0; u < AHEAD; ++u) {
        if (s + u >= steps) break;
        float a[RM];
#pragma unroll
        for (int m = 0; m < RM; ++m) a[m] = filters[(4 * (s + u) + h) * ROW + 16 * m + r];
#pragma unroll
        for (int m = 0; m < RM; ++m)
#pragma unroll
          for (int n = 0; n < 4; ++n) sum[m][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[m], x[set][u][n], sum[m][n], 0, 0, 0);
      }
    };
#pragma unroll 1
    for (int s = 0; s < steps; s += 2 * AHEAD) {
      request(s + AHEAD, 1);
      multiply(s, 0);
      request(s + 2 * AHEAD, 0);
      multiply(s + AHEAD, 1);
      // (chains of a few roundings, not of all planes)
#pragma unroll
      for (int m = 0; m < RM; ++m)
#pragma unroll
        for (int n = 0; n < 4; ++n) {
          total[m][n] += sum[m][n];
          sum[m][n] = floatx4{0.f, 0.f, 0.f, 0.f};
        }
    }
  }

  if (first + r >= g.images * g.words) return;
  float* const to = g.out + b * g.oB + p;
#pragma unroll
  for (int m = 0; m < RM; ++m)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int i = m0 + 16 * m + 4 * h + v;
      if (i < g.M)
        *reinterpret_cast<AnyFour*>(to + i * g.oM) = AnyFour{total[m][0][v], total[m][1][v], total[m][2][v], total[m][3][v]};
    }
}

struct PointGradArgs {
  const float* g;
  const float* x;
  float* part;
  long gB, gM, xB, xC;
  int C, M, pixels, words, groups;  // words: groups of four pixels of an image; groups: of all images
  int mTiles, cTiles, ranges, chunks;  // chunks of kGradPixels pixels
  int total;
};

constexpr int kGradPixels = 64;

// The weight gradient: a workgroup takes 32 WM x 32 WC filters over a range of the pixels of all images, 64 at
// a time through LDS, four waves of 32 x 32; waves that share such a tile take every other (every fourth) eight
// pixels and add up in wave order.  Its partial sums go to part[range][m][c].  The 64 pixels are 16 groups of four
// neighbours of any images, so that small planes, and the ends of others, are not filled up with zeros (us, windows of 8
// points / 64 pixels of one image / so: 3005 x 3412 x 2 x 2, 195 3904 / 5031 / 296; 493 x 828 x 3 x 5, 199 179 / 215 / 68; 128 x 1203 x 6
// x 6, 218 84 / 101 / 57).
template <int WM, int WC>
__global__ __launch_bounds__(256, 3) void pointGradient(PointGradArgs a) {
  constexpr int ROW = kGradPixels + 4, WK = 4 / (WM * WC), LM = 2 * WM, LC = 2 * WC;
  __shared__ __align__(16) float lds[32 * (WM + WC) * ROW];
  static_assert(32 * (WM + WC) * ROW >= (WK - 1) * WM * WC * 1024, "room for the waves' sums");
  float* const ldsC = lds + 32 * WM * ROW;
  const int t = threadIdx.x, lane = t % 64, r = lane % 32, h = lane / 32;
  const int wave = __builtin_amdgcn_readfirstlane(t / 64), wm = wave % WM, wc = wave / WM % WC, wk = wave / (WM * WC);
  const int per = (a.total + 7) / 8;
  const int logical = (blockIdx.x % 8) * per + blockIdx.x / 8;
  if (logical >= a.total) return;
  const int m0 = logical % a.mTiles * 32 * WM, c0 = logical / a.mTiles % a.cTiles * 32 * WC,
            range = logical / a.mTiles / a.cTiles;
  const int first = (int)((long)a.chunks * range / a.ranges), end = (int)((long)a.chunks * (range + 1) / a.ranges);

  // sixteen lanes bring 64 pixels of a row, the workgroup 16 rows at a time
  const int px = 4 * (t % 16), row = t / 16;
  floatx4 vm[LM], vc[LC];
  auto request = [&](int chunk) __attribute__((always_inline)) {
    const int group = chunk * (kGradPixels / 4) + t % 16, known = min(group, a.groups - 1);
    const int b = (unsigned)known / (unsigned)a.words, p = 4 * (known - b * a.words), from = min(p, a.pixels - 4);
#pragma unroll
    for (int i = 0; i < LM; ++i) vm[i] = *(GlobalFour)(a.g + b * a.gB + min(m0 + row + 16 * i, a.M - 1) * a.gM + from);
#pragma unroll
    for (int i = 0; i < LC; ++i) vc[i] = *(GlobalFour)(a.x + b * a.xB + min(c0 + row + 16 * i, a.C - 1) * a.xC + from);
    return group < a.groups ? p - from : 4;
  };
  int d = 0;
  // the last pixels of an image: those that are there, shifted into place, then zeros (behind the last image zeros only)
  auto park = [&](float* to, floatx4 f) __attribute__((always_inline)) {
    floatx4 u = f;
    if (d != 0) {
#pragma unroll
      for (int e = 0; e < 4; ++e) u[e] = e + d == 1 ? f[1] : e + d == 2 ? f[2] : e + d == 3 ? f[3] : 0.f;
    }
    *reinterpret_cast<floatx4*>(to) = u;
  };
  floatx16 sum, total;
#pragma unroll
  for (int e = 0; e < 16; ++e) sum[e] = total[e] = 0.f;
  if (first < end) d = request(first);
  for (int chunk = first; chunk < end; ++chunk) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < LM; ++i) park(lds + (row + 16 * i) * ROW + px, vm[i]);
#pragma unroll
    for (int i = 0; i < LC; ++i) park(ldsC + (row + 16 * i) * ROW + px, vc[i]);
    __syncthreads();
    if (chunk + 1 < end) d = request(chunk + 1);
    const float* const A = lds + (32 * wm + r) * ROW + 8 * wk + 4 * h;
    const float* const B = ldsC + (32 * wc + r) * ROW + 8 * wk + 4 * h;
#pragma unroll
    for (int s = 0; s < kGradPixels / 8 / WK; ++s) {
      const floatx4 f = *reinterpret_cast<const floatx4*>(A + 8 * WK * s), u = *reinterpret_cast<const floatx4*>(B + 8 * WK * s);
#pragma unroll
      for (int e = 0; e < 4; ++e) sum = __builtin_amdgcn_mfma_f32_32x32x2f32(f[e], u[e], sum, 0, 0, 0);
    }
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      total[e] += sum[e];
      sum[e] = 0.f;
    }
  }
  if constexpr (WK > 1) {
    __syncthreads();
    if (wk > 0) {
#pragma unroll
      for (int e = 0; e < 16; ++e) lds[((wave - WM * WC) * 16 + e) * 64 + lane] = total[e];
    }
    __syncthreads();
    if (wk > 0) return;
#pragma unroll
    for (int k = 1; k < WK; ++k)
#pragma unroll
      for (int e = 0; e < 16; ++e) total[e] += lds[((wave + (k - 1) * WM * WC) * 16 + e) * 64 + lane];
  }
  const long Mp = 32L * WM * a.mTiles, Cp = 32L * WC * a.cTiles;
  float* const to = a.part + (range * Mp + m0 + 32 * wm) * Cp + c0 + 32 * wc + r;
#pragma unroll
  for (int e = 0; e < 16; ++e) to[(8 * (e / 4) + 4 * h + e % 4) * Cp] = total[e];
}

// adds the ranges up, 32 lanes to a filter value, in an order that does not depend on timing
constexpr int kAddValues = 16, kAddLanes = 32;
__global__ __launch_bounds__(kAddValues * kAddLanes) void addRanges(const float* part, float* out, long oM, long oC, int M,
                                                                    int C, int Cp, long rangeFloats, int ranges,
                                                                    float scale, bool accumulate) {
  __shared__ float sums[kAddLanes][kAddValues];
  const int v = threadIdx.x % kAddValues, q = threadIdx.x / kAddValues;
  const long i = min((long)blockIdx.x * kAddValues + v, (long)M * C - 1);
  const int m = (int)(i / C), c = (int)(i % C);
  const float* const from = part + (long)m * Cp + c;
  float s = 0.f;
#pragma unroll 4
  for (int k = q; k < ranges; k += kAddLanes) s += from[k * rangeFloats];
  sums[q][v] = s;
  for (int half = kAddLanes / 2; half > 0; half /= 2) {
    __syncthreads();
    if (q < half) sums[q][v] += sums[q + half][v];
  }
  if (q != 0 || (long)blockIdx.x * kAddValues + v >= (long)M * C) return;
  float* const to = out + m * oM + c * oC;
  *to = accumulate ? *to + scale * sums[0][v] : scale * sums[0][v];
}

}  // namespace

// Whether the operands of a pass with filters of 1 x 1 may take this way: planes without gaps of at least one
// 16-byte word, lane offsets of the images that a wave meets in 32 bits, and (passes 0 and 1, which read
// their operands while they write) a result apart from them.
bool pointMayRun(int pass, const float* x, const int* xStride, const int* xSize, const float* y, const int* yStride,
                 const int* ySize, const float* out, const int* outStride, const int* outSize) {
  const auto whole = [](const int* stride, const int* size) {
    return stride[3] == 1 && stride[2] == size[3] && (long)size[2] * size[3] >= 4 && (long)size[2] * size[3] < (1 << 28);
  };
  for (int d = 0; d < 4; ++d)
    if (xStride[d] < 0 || yStride[d] < 0 || outStride[d] < 0) return false;
  if (!whole(xStride, xSize) || !whole(pass == 2 ? yStride : outStride, pass == 2 ? ySize : outSize)) return false;
  // (grids count their lanes in 32 bits)
  const long words = (long)xSize[0] * ((xSize[2] * xSize[3] + 3) / 4);
  if (words > (1 << 28) || (pass == 2 && (long)outSize[0] * outSize[1] > (1 << 26))) return false;
  if (pass == 2) return true;
  if ((words / 64 + 1) * (outSize[1] / 16 + 1) > (1 << 23)) return false;
  const auto last = [](const float* p, const int* stride, const int* size) {
    for (int d = 0; d < 4; ++d) p += (long)stride[d] * (size[d] - 1);
    return p;
  };
  const float* const end = last(out, outStride, outSize);
  if ((out <= last(x, xStride, xSize) && x <= end) || (out <= last(y, yStride, ySize) && y <= end)) return false;
  return 17L * xStride[0] + 3L * xStride[1] + xSize[2] * xSize[3] < (1 << 30);
}

// The ranges of pixels that a weight gradient is cut into, as far as their partial sums fit: workgroups for
// every CU a few times over (us, 45 x 79 x 118 x 118, 50 filters: 128 ranges of one tile 134, 256 124, 512 127; 175
// x 21 x 186 x 187, 21, whose workgroups are smaller: 256 336, 512 229, 1024 218; 69 x 3 x 94 x 94, 45: 256 51, 512 57,
// 1024 75, to add up), of at least four turns each once there are sixteen (3 x 5 x 11 x 11, 249, six turns: one range
// 13.3, six 7.5); and of two, or one up to 32 ranges, while there are no more workgroups than CUs (at least four / so: 138 x 47 x 7 x 7,
// 46 18.1 / 13.2, windows of 8 points 14.8; 12 x 20 x 16 x 16, 50 8.1 / 7.2).
static int pointRanges(const PointGradArgs& a, int wm, int wc, size_t room) {
  const int tiles = a.mTiles * a.cTiles, target = wm * wc == 1 ? 1024 : wm * wc == 2 ? 320 : 640;
  const size_t bytes = sizeof(float) * 1024 * wm * wc * tiles;
  const long fit = (long)std::min<size_t>(room / bytes, 1 << 20);
  const int few = std::min(std::max(a.chunks / 2, std::min(a.chunks, 32)), computeUnits() / tiles);
  return (int)std::max<long>(1, std::min<long>({ceilDiv(target, tiles), fit, std::max({a.chunks / 4, std::min(a.chunks, 16), few})}));
}

// room: bytes of workspace (weight gradients; at least one range fits any pass's workspace, which holds spectra
// of 32 bins of both operands and the result)
int launchConvPoint(int pass, const float* x, const int* xStride, const int* xSize, const float* y, const int* yStride,
                    const int* ySize, float* out, const int* outStride, const int* outSize, float scale, bool accumulate,
                    void* workspace, size_t room, hipStream_t s) {
  const auto padded = [](int total) { return dim3((unsigned)(ceilDiv(total, 8) * 8)); };
  if (pass < 2) {
    PointArgs g{};
    g.x = x; g.w = y; g.out = out;
    g.xB = xStride[0]; g.xC = xStride[1];
    g.oB = outStride[0]; g.oM = outStride[1];
    g.wM = yStride[pass]; g.wC = yStride[1 - pass];
    g.C = xSize[1]; g.M = outSize[1];
    g.pixels = xSize[2] * xSize[3];
    g.words = ceilDiv(g.pixels, 4);
    g.images = xSize[0];
    // 32 rows read each pixel half as often, 16 are twice the workgroups (us, 16 / 32 rows: 133 x 182 x 58 x 58, 57
    // filters, 3496 workgroups of 32 rows, 155 / 134; 55 x 95 x 32 x 32, 300, 2200, 50 / 49; 8 x 25 x 115 x 115, 57,
    // 826, 12.3 / 12.0; 32 x 298 x 29 x 29, 75, 318, 32 / 41; 104 x 45 x 14 x 14, 96, 240, 7.8 / 8.5)
    const int groups = ceilDiv(g.images * g.words, 64);
    const bool two = g.M > 16 && (long)ceilDiv(g.M, 32) * groups >= 8 * 256;
    g.rowTiles = ceilDiv(g.M, two ? 32 : 16);
    g.total = g.rowTiles * groups;
    if (two)
      pointProducts<2><<<padded(g.total), dim3(256), 0, s>>>(g);
    else
      pointProducts<1><<<padded(g.total), dim3(256), 0, s>>>(g);
    return launchStatus();
  }
  PointGradArgs a{};
  a.x = x; a.g = y; a.part = static_cast<float*>(workspace);
  a.xB = xStride[0]; a.xC = xStride[1]; a.gB = yStride[0]; a.gM = yStride[1];
  a.C = xSize[1]; a.M = ySize[1]; a.pixels = xSize[2] * xSize[3];
  a.words = ceilDiv(a.pixels, 4); a.groups = xSize[0] * a.words;
  const int wm = a.M <= 32 ? 1 : 2, wc = a.C <= 32 ? 1 : 2;
  a.mTiles = ceilDiv(a.M, 32 * wm); a.cTiles = ceilDiv(a.C, 32 * wc);
  a.chunks = ceilDiv(a.groups, kGradPixels / 4);
  a.ranges = pointRanges(a, wm, wc, room);
  a.total = a.mTiles * a.cTiles * a.ranges;
  const dim3 grid = padded(a.total), block(256);
  if (wm == 1 && wc == 1)
    pointGradient<1, 1><<<grid, block, 0, s>>>(a);
  else if (wm == 1)
    pointGradient<1, 2><<<grid, block, 0, s>>>(a);
  else if (wc == 1)
    pointGradient<2, 1><<<grid, block, 0, s>>>(a);
  else
    pointGradient<2, 2><<<grid, block, 0, s>>>(a);
  const int Mp = 32 * wm * a.mTiles, Cp = 32 * wc * a.cTiles;
  addRanges<<<dim3((unsigned)(((long)a.M * a.C + kAddValues - 1) / kAddValues)), dim3(kAddValues * kAddLanes), 0, s>>>(
      a.part, out, outStride[0], outStride[1], a.M, a.C, Cp, (long)Mp * Cp, a.ranges, scale, accumulate);
  return launchStatus();
}

}  // namespace fbfft_amd
