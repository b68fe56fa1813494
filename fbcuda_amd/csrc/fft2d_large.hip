// 2D real-to-complex / complex-to-real transforms for N in {64, 128} in ONE
// kernel and one pass over HBM.  The reference needs two kernels and a scratch
// round trip for these sizes (fbfft/FBFFT2D-inl.cuh:230-444,
// fbfft/FBIFFT2D-inl.cuh:252-521).  Output layout cplx[b][kx][ky], kx = 0..N/2:
// the Hermitian-halved axis is the horizontal frequency and the plane is stored
// transposed, as the reference's second pass leaves it.
//
// One workgroup owns one plane, which stays in LDS between the passes (one buffer, reused by every
// stage), and every stage but one belongs to a wave alone:
//   1. a wave loads rows of the plane straight into registers, several lanes per row;
//   2. row pass: N reals as N/2 packed complex values, in two steps of 4 or 8 points with an
//      exchange through LDS between them, left there transposed ([kx][y], before the real-input fix-up);
//   3. workgroup barrier;
//   4. column pass: the lanes of a pair of columns kx and N/2 - kx hold both halves of every
//      fix-up pair (k, N/2 - k), fix them up as they read them and run both columns in two
//      steps; columns kx = 0 and kx = N/2 (both real along y) travel packed as one;
//   5. the wave's columns leave as 16-byte stores, whole columns side by side (stores of 64
//      bytes per column straight from the registers: 87 -> 99 us at 128 points); the packed column is
//      unpacked on the way out.
// The inverse runs the same steps backwards and crops on store; at 128 points it takes one more barrier, to leave
// its rows one after the other.
//
// What bounds them is HBM: 6.2 and 5.9 TB/s (128 points), 6.5 and 6.4 (64).  us, forward / inverse, before
// (fewer lanes with 32 points each, which formed the first butterflies from LDS, every stage between barriers)
// -> this: 4096 planes of 128 x 128 101.5 / 96.5 -> 87.4 / 91.0, 19 planes 8.4 / 8.0 -> 6.2 / 6.2, 3773 windows of
// 73 x 91 87.0 / 85.9 -> 64.7 / 75.2; 16384 of 64 x 64 95.2 / 85.7 -> 84.4 / 84.1, 53 6.6 / 5.7 -> 4.2 / 4.7, 3247 of 36
// x 58 22.0 / 22.8 -> 18.9 / 22.2; buffers from HBM, 5000 of 64 x 64 33.7 / 33.0 -> 29.9 / 31.5, 3000 of 60 x 60 22.5
// / 25.6 -> 21.1 / 23.0, of 50 x 50 21.7 / 23.6 -> 18.5 / 21.6.  At 128 points LDS was the limit while its accesses collided
// (places from column to column 136 apart: 22.4 of 38.3 million active cycles, 94 / 105 us; 130: 3.6 of 19.4).
#include "common.h"
#include "fft_lds.h"
#include "fft_regs.h"

#include <algorithm>

namespace fbfft_amd {
namespace {

// ---- 128 x 128 ----
//
// 512 lanes per plane.  Rows: a wave takes eight at a time,
// eight lanes each, as 64 = 8 x 8 packed values; lane l loads z[l + 8 m] straight into registers and the
// lanes of a row exchange through the row's own places in LDS, which hold [kx][y] in the end.  Columns:
// sixteen lanes take kx and 64 - kx (kx = 0, which carries kx = 64 packed, with 32), which hold both halves of
// every fix-up pair, as 128 = 8 x 16 points: lane l makes the pairs y = l + 16 m, runs 8 points over m
// for both columns, and after the exchange lane (column, ky mod 8) runs 16.  The wave then stores its
// columns, 1 KB each.  The inverse runs backwards.
constexpr int kLanes128 = 512;
// Complex values from column to column.  LDS serves 16 lanes of 8 bytes at a time: the lanes of two rows
// (8 columns) meet 16 different places modulo 16, and so do those of a column.
constexpr int kStride128 = 130;

struct Lane128 {
  int wave, lane;
  int l, r;      // row pass: lane of the row, row of the wave's eight
  int h, pair;   // column pass: lane of the pair, pair
  int k0, k1;    // its columns
  int c, q;      // after the exchange: column (0 or 1) and ky mod 8
};

__device__ __forceinline__ Lane128 lane128(int t) {
  Lane128 a;
  a.wave = __builtin_amdgcn_readfirstlane(t / 64);
  a.lane = t % 64;
  a.l = a.lane % 8;
  a.r = a.lane / 8;
  a.h = a.lane % 16;
  a.pair = a.wave * 4 + a.lane / 16;
  a.k0 = a.pair;
  a.k1 = a.pair ? 64 - a.pair : 32;
  a.c = a.h / 8;
  a.q = a.h % 8;
  return a;
}

// four floats that start at any float
typedef float AnyFour __attribute__((ext_vector_type(4), aligned(4)));

// Planes whose samples, or bins, lie between those of their neighbours share cache lines: an XCD, every eighth workgroup, takes
// consecutive ones.  us, forward / inverse, neighbours on eight XCDs -> on one: 6436 windows of 55 x 40 in 64 points 164 / 172 -> 80 /
// 82, 1652 of 110 x 97 in 128 164 / 232 -> 102 / 111, 100 of 128 x 128 from HBM 23.7 / 22.1 -> 24.8 / 20.4; spectra that do, 5000
// planes of 64 x 64 146 / 154 -> 62 / 52 (one wave a plane, before, 152 / 139), 1300 of 128 x 128 156 / 140 -> 69 / 61 (160 / 128).
__host__ __device__ __forceinline__ bool interleaved(const RealView& r, const CplxView& c) {
  return (abs(r.sb) < 32 || abs(c.sb) < 32) && r.B > 1;
}
__device__ __forceinline__ int planeOf(const RealView& r, const CplxView& c) {
  const int b = blockIdx.x;
  return interleaved(r, c) ? b % 8 * ((r.B + 7) / 8) + b / 8 : b;
}
dim3 planeGrid(const RealView& r, const CplxView& c) { return dim3(interleaved(r, c) ? (r.B + 7) / 8 * 8 : r.B); }

// Whether a spectrum's values of one ky lie closer together than those of one kx: a turned view, [ky][kx] in memory.
// At 128 points these move a ky at a time, 64 columns to an instruction.  us, forward / inverse, a column at a time
// -> so: 236 planes 20.5 / 12.2 -> 10.4 / 10.2, 4000 238 / 130 -> 104 / 96 (four lanes with 32 points each, before, 200 / 109).
// The inverse's last row, read by a lane value after value / by sixteen lanes: 40 windows of 101 x 90 9.9 / 9.1, 1300 planes 35.2 / 32.9.
// (At 64 points a column at a time takes 0.80 and 0.86 of what it took then.)
__device__ __forceinline__ bool nearAcross(const CplxView& c) { return abs(c.sr) < abs(c.sc); }

// The inverse's value of kx = 0 holds even samples in one part and odd ones in the other: multiplied with 1 + 0 i as a complex
// number, even samples beyond the largest float would make NaN of the odd ones.  (64 points, one plane 4.2 -> 4.3 us.)
__device__ __forceinline__ c32 choose(bool first, c32 a, c32 b) { return c32{first ? a.x : b.x, first ? a.y : b.y}; }

// where a row keeps value l of class k between its two steps, and column c of a pair value l of class k
// (of either parity for the two columns): sixteen lanes meet different places on both sides
__device__ __forceinline__ int rowPlace(int k, int l, int y) { return (k * 8 + (l ^ k)) * kStride128 + y; }
__device__ __forceinline__ int columnPlace(int column, int c, int k, int l) {
  return column * kStride128 + k * 16 + (l ^ (2 * k) ^ c);
}
// where the inverse leaves the packed value j of row y: two rows side by side
__device__ __forceinline__ int sampleAt(int y, int j) { return y * 64 + (j ^ (8 * (y & 1))); }

// BY_ROW: a wave takes row after row, 64 samples to an instruction, and turns them in LDS (launchForward128)
template <bool FAST_REAL, bool FAST_CPLX, bool BY_ROW = false>
__global__ __launch_bounds__(kLanes128, 4) void fft2d128Forward(RealView real, CplxView cplx, int padL, int padU) {
  __shared__ __align__(16) c32 cb[64 * kStride128];
  __shared__ __align__(8) c32 tw[256];
  const Lane128 a = lane128(threadIdx.x);
  constexpr bool ANY = !FAST_REAL || !FAST_CPLX;
  const int b = ANY ? planeOf(real, cplx) : blockIdx.x;
  if (ANY && b >= real.B) return;
  // whether a wave's rows 64 i + 8 wave ... + 7 hold a row of the window
  auto any = [&](int i) __attribute__((always_inline)) {
    const int y = 64 * i + 8 * a.wave;
    return FAST_REAL || (real.w > 0 && real.h > 0 && y < padU + real.h && y + 8 > padU);
  };
  const float* const src = real.data + (size_t)b * real.sb;

  c32 z[2][8];
  if constexpr (FAST_REAL) {
    staticFor<2>([&](auto ii) {
      constexpr int i = decltype(ii)::value;
      const c32* row = reinterpret_cast<const c32*>(src + (size_t)(64 * i + 8 * a.wave + a.r) * real.sy) + a.l;
      staticFor<8>([&](auto mm) { z[i][decltype(mm)::value] = row[8 * decltype(mm)::value]; });
    });
  } else {
    // implicit zero padding, any strides: loads at places clamped into the window, no branch
    // between them, and what lies outside counts as zero; whole pairs where the window has only such
    const bool pairs = real.sx == 1 && ((real.sy | real.sb | padL | real.w) & 1) == 0 &&
                       (reinterpret_cast<uintptr_t>(real.data) & 7) == 0;
    if constexpr (BY_ROW) {
      const int left = min(max(a.lane - padL, 0), real.w - 1), right = min(max(a.lane + 64 - padL, 0), real.w - 1);
      staticFor<2>([&](auto ii) {
        constexpr int i = decltype(ii)::value;
        if (!any(i)) return;
        float in[8][2];
        staticFor<8>([&](auto rr) {
          constexpr int r = decltype(rr)::value;
          const float* const row = src + (size_t)min(max(64 * i + 8 * a.wave + r - padU, 0), real.h - 1) * real.sy;
          in[r][0] = row[(size_t)left * real.sx];
          in[r][1] = row[(size_t)right * real.sx];
        });
        staticFor<16>([&](auto rr) {
          constexpr int r = decltype(rr)::value / 2, j = decltype(rr)::value % 2;
          const int x = a.lane + 64 * j;
          reinterpret_cast<float*>(cb + sampleAt(64 * i + 8 * a.wave + r, x / 2))[x % 2] = in[r][j];
        });
      });
      waveExchange();
    }
    staticFor<2>([&](auto ii) {
      constexpr int i = decltype(ii)::value;
      const int y = 64 * i + 8 * a.wave + a.r - padU;
      const bool yIn = (unsigned)y < (unsigned)real.h;
      const float* row = src + (size_t)min(max(y, 0), real.h - 1) * real.sy;
      if constexpr (BY_ROW) {
        if (any(i))
          staticFor<8>([&](auto mm) {
            constexpr int m = decltype(mm)::value;
            z[i][m] = cb[sampleAt(64 * i + 8 * a.wave + a.r, a.l + 8 * m)];
          });
      } else if (any(i) && pairs) {
        staticFor<8>([&](auto mm) {
          const int x = 2 * (a.l + 8 * decltype(mm)::value) - padL;
          z[i][decltype(mm)::value] = *reinterpret_cast<const c32*>(row + min(max(x, 0), real.w - 2));
        });
      } else if (any(i)) {
        staticFor<8>([&](auto mm) {
          const int x = 2 * (a.l + 8 * decltype(mm)::value) - padL;
          z[i][decltype(mm)::value].x = row[(size_t)min(max(x, 0), real.w - 1) * real.sx];
          z[i][decltype(mm)::value].y = row[(size_t)min(max(x + 1, 0), real.w - 1) * real.sx];
        });
      }
      staticFor<8>([&](auto mm) {
        constexpr int m = decltype(mm)::value;
        const int x = 2 * (a.l + 8 * m) - padL;
        z[i][m].x = yIn && (unsigned)x < (unsigned)real.w ? z[i][m].x : 0.0f;
        z[i][m].y = yIn && (unsigned)(x + 1) < (unsigned)real.w ? z[i][m].y : 0.0f;
      });
    });
  }
  fillTwiddles<true>(tw, threadIdx.x, kLanes128);
  __syncthreads();

  // ---- rows ----
  staticFor<2>([&](auto ii) {
    constexpr int i = decltype(ii)::value;
    if (!any(i)) return;
    regFFT<8, true>(z[i]);
    staticFor<8>([&](auto kk) {
      constexpr int k = decltype(kk)::value;
      c32 v = z[i][slot<8>(k)];
      if constexpr (k > 0) v = cmul(v, tw[4 * k * a.l]);
      cb[rowPlace(k, a.l, 64 * i + 8 * a.wave + a.r)] = v;
    });
  });
  waveExchange();
  staticFor<2>([&](auto ii) {
    constexpr int i = decltype(ii)::value;
    if (!any(i)) return;
    staticFor<8>([&](auto jj) {
      constexpr int j = decltype(jj)::value;
      z[i][j] = cb[rowPlace(a.l, j, 64 * i + 8 * a.wave + a.r)];
    });
  });
  waveExchange();
  staticFor<2>([&](auto ii) {
    constexpr int i = decltype(ii)::value;
    if (any(i)) regFFT<8, true>(z[i]);  // (rows outside are zeros)
    staticFor<8>([&](auto kk) {
      constexpr int k = decltype(kk)::value;
      cb[(a.l + 8 * k) * kStride128 + 64 * i + 8 * a.wave + a.r] = z[i][slot<8>(k)];
    });
  });
  __syncthreads();

  // ---- columns ----
  {
    c32 u[8], v[8];
    const c32 root = tw[2 * a.pair], half = c32{0.5f * root.x, 0.5f * root.y};
    staticFor<8>([&](auto mm) {
      constexpr int m = decltype(mm)::value;
      u[m] = cb[a.k0 * kStride128 + a.h + 16 * m];
      v[m] = cb[a.k1 * kStride128 + a.h + 16 * m];
    });
    waveExchange();
    staticFor<8>([&](auto mm) {
      constexpr int m = decltype(mm)::value;
      const c32 p = u[m], q = v[m];
      const c32 e2 = c32{p.x + q.x, p.y - q.y};
      const c32 t = cmul(c32{p.y + q.y, q.x - p.x}, half);
      u[m] = c32{__builtin_fmaf(0.5f, e2.x, t.x), __builtin_fmaf(0.5f, e2.y, t.y)};
      v[m] = c32{__builtin_fmaf(0.5f, e2.x, -t.x), __builtin_fmaf(-0.5f, e2.y, t.y)};
      if (a.wave == 0) {  // (the pair of columns 0 and 32 is in the first wave)
        const bool ends = a.pair == 0;
        u[m] = ends ? c32{p.x + p.y, p.x - p.y} : u[m];
        v[m] = ends ? c32{q.x, -q.y} : v[m];
      }
    });
    regFFT<8, true>(u);
    regFFT<8, true>(v);
    staticFor<8>([&](auto kk) {
      constexpr int k = decltype(kk)::value;
      c32 p = u[slot<8>(k)], q = v[slot<8>(k)];
      if constexpr (k > 0) {
        const c32 w = tw[2 * k * a.h];
        p = cmul(p, w);
        q = cmul(q, w);
      }
      cb[columnPlace(a.k0, 0, k, a.h)] = p;
      cb[columnPlace(a.k1, 1, k, a.h)] = q;
    });
  }
  waveExchange();
  {
    const int column = a.c ? a.k1 : a.k0;
    c32 v[16];
    staticFor<16>([&](auto jj) {
      constexpr int j = decltype(jj)::value;
      v[j] = cb[columnPlace(column, a.c, a.q, j)];
    });
    waveExchange();
    regFFT<16, true>(v);
    staticFor<16>([&](auto kk) {
      constexpr int k = decltype(kk)::value;
      cb[column * kStride128 + a.q + 8 * k] = v[slot<16>(k)];
    });
  }
  float* const dst = cplx.data + (size_t)b * cplx.sb;
  if (!FAST_CPLX && nearAcross(cplx)) {
    // neighbours along kx share cache lines: the workgroup's columns out side by side, a ky at a time
    __syncthreads();
    staticFor<16>([&](auto jj) {
      const int ky = a.wave + 8 * decltype(jj)::value;
      c32 v = cb[a.lane * kStride128 + ky];
      float* const to = dst + (size_t)ky * cplx.sc;
      if (a.lane == 0) {
        const c32 m = cb[(128 - ky) & 127];
        *reinterpret_cast<c32*>(to + (size_t)64 * cplx.sr) = c32{0.5f * (v.y + m.y), 0.5f * (m.x - v.x)};
        v = c32{0.5f * (v.x + m.x), 0.5f * (v.y - m.y)};
      }
      *reinterpret_cast<c32*>(to + (size_t)a.lane * cplx.sr) = v;
    });
    return;
  }
  waveExchange();

  // ---- the wave's columns out; rows 0 and 64 of the result come from packed column 0 ----
  const int ky = 2 * a.lane;
  auto store = [&](int r, float4 o) __attribute__((always_inline)) {
    if constexpr (FAST_CPLX) {
      streamStore(reinterpret_cast<float4*>(dst) + r * 64 + a.lane, o);
    } else {
      float* to = dst + (size_t)r * cplx.sr + (size_t)ky * cplx.sc;
      *reinterpret_cast<float2*>(to) = float2{o.x, o.y};
      *reinterpret_cast<float2*>(to + cplx.sc) = float2{o.z, o.w};
    }
  };
  auto column = [&](int k) __attribute__((always_inline)) {
    return *reinterpret_cast<const float4*>(cb + k * kStride128 + ky);
  };
  staticFor<4>([&](auto ii) {
    constexpr int i = decltype(ii)::value;
    const int k = a.wave * 4 + i;
    if (i == 0 && a.wave == 0) {
      const float4 p = column(0);
      const c32 m0 = cb[(128 - ky) & 127], m1 = cb[127 - ky];
      store(0, float4{0.5f * (p.x + m0.x), 0.5f * (p.y - m0.y), 0.5f * (p.z + m1.x), 0.5f * (p.w - m1.y)});
      store(64, float4{0.5f * (p.y + m0.y), 0.5f * (m0.x - p.x), 0.5f * (p.w + m1.y), 0.5f * (m1.x - p.z)});
      store(32, column(32));
    } else {
      store(k, column(k));
      store(64 - k, column(64 - k));
    }
  });
}

template <bool FAST_REAL, bool FAST_CPLX>
__global__ __launch_bounds__(kLanes128, 4) void fft2d128Inverse(CplxView cplx, RealView real, int padL, int padU) {
  __shared__ __align__(16) c32 cb[64 * kStride128];
  __shared__ __align__(8) c32 tw[256];
  const Lane128 a = lane128(threadIdx.x);
  constexpr bool ANY = !FAST_REAL || !FAST_CPLX;
  const int b = ANY ? planeOf(real, cplx) : blockIdx.x;
  if (ANY && b >= real.B) return;
  // whether a wave's rows 64 i + 8 wave ... + 7 hold a row of the window
  auto any = [&](int i) __attribute__((always_inline)) {
    const int y = 64 * i + 8 * a.wave;
    return FAST_REAL || (real.w > 0 && real.h > 0 && y < padU + real.h && y + 8 > padU);
  };

  // ---- the wave's columns in; column 0 carries 64 as its imaginary part ----
  const int ky = 2 * a.lane;
  const float* const src = cplx.data + (size_t)b * cplx.sb;
  auto load = [&](int r) __attribute__((always_inline)) {
    if constexpr (FAST_CPLX) {
      return reinterpret_cast<const float4*>(src)[r * 64 + a.lane];
    } else {
      const float* from = src + (size_t)r * cplx.sr + (size_t)ky * cplx.sc;
      const float2 p = *reinterpret_cast<const float2*>(from), q = *reinterpret_cast<const float2*>(from + cplx.sc);
      return float4{p.x, p.y, q.x, q.y};
    }
  };
  fillTwiddles<false>(tw, threadIdx.x, kLanes128);
  if (!FAST_CPLX && nearAcross(cplx)) {
    // neighbours along kx share cache lines: the workgroup's columns in side by side, a ky at a time
    c32 in[16];
    staticFor<16>([&](auto jj) {
      constexpr int j = decltype(jj)::value;
      in[j] = *reinterpret_cast<const c32*>(src + (size_t)(a.wave + 8 * j) * cplx.sc + (size_t)a.lane * cplx.sr);
    });
    const int own = a.wave + 8 * (a.lane % 16);  // (16 lanes fold column 64 into column 0)
    const c32 last = *reinterpret_cast<const c32*>(src + (size_t)own * cplx.sc + (size_t)64 * cplx.sr);
    staticFor<16>([&](auto jj) {
      constexpr int j = decltype(jj)::value;
      cb[a.lane * kStride128 + a.wave + 8 * j] = in[j];
    });
    waveExchange();
    if (a.lane < 16) cb[own] = c32{cb[own].x - last.y, cb[own].y + last.x};
    __syncthreads();
  } else {
    float4 in[4][2];
    staticFor<4>([&](auto ii) {
      constexpr int i = decltype(ii)::value;
      const int k = a.wave * 4 + i;
      in[i][0] = load(k);
      in[i][1] = load(k ? 64 - k : 32);
    });
    if (a.wave == 0) {
      const float4 last = load(64);
      in[0][0] = float4{in[0][0].x - last.y, in[0][0].y + last.x, in[0][0].z - last.w, in[0][0].w + last.z};
    }
    staticFor<4>([&](auto ii) {
      constexpr int i = decltype(ii)::value;
      const int k = a.wave * 4 + i;
      *reinterpret_cast<float4*>(cb + k * kStride128 + ky) = in[i][0];
      *reinterpret_cast<float4*>(cb + (k ? 64 - k : 32) * kStride128 + ky) = in[i][1];
    });
    waveExchange();
  }
  {
    const int column = a.c ? a.k1 : a.k0;
    c32 v[16];
    staticFor<16>([&](auto kk) {
      constexpr int k = decltype(kk)::value;
      v[k] = cb[column * kStride128 + a.q + 8 * k];
    });
    waveExchange();
    regFFT<16, false>(v);
    staticFor<16>([&](auto ll) {
      constexpr int l = decltype(ll)::value;
      cb[columnPlace(column, a.c, a.q, l)] = v[slot<16>(l)];
    });
  }
  __syncthreads();  // the roots
  {
    c32 u[8], v[8];
    staticFor<8>([&](auto kk) {
      constexpr int k = decltype(kk)::value;
      u[k] = cb[columnPlace(a.k0, 0, k, a.h)];
      v[k] = cb[columnPlace(a.k1, 1, k, a.h)];
      if constexpr (k > 0) {
        const c32 w = tw[2 * k * a.h];
        u[k] = cmul(u[k], w);
        v[k] = cmul(v[k], w);
      }
    });
    waveExchange();
    regFFT<8, false>(u);
    regFFT<8, false>(v);
    const c32 root = tw[2 * a.pair];
    staticFor<8>([&](auto mm) {
      constexpr int m = decltype(mm)::value;
      const c32 p = u[slot<8>(m)], q = v[slot<8>(m)];
      const c32 e = c32{p.x + q.x, p.y - q.y};
      const c32 o = cmul(c32{p.x - q.x, p.y + q.y}, root);
      c32 zk = c32{e.x - o.y, e.y + o.x}, zh = c32{e.x + o.y, o.x - e.y};
      if (a.wave == 0) {
        const bool ends = a.pair == 0;
        zk = ends ? c32{p.x + p.y, p.x - p.y} : zk;
        zh = ends ? c32{2.0f * q.x, -2.0f * q.y} : zh;
      }
      cb[a.k0 * kStride128 + a.h + 16 * m] = zk;
      cb[a.k1 * kStride128 + a.h + 16 * m] = zh;
    });
  }
  __syncthreads();

  // ---- rows ----
  c32 z[2][8];
  staticFor<2>([&](auto ii) {
    constexpr int i = decltype(ii)::value;
    if (!any(i)) return;
    staticFor<8>([&](auto kk) {
      constexpr int k = decltype(kk)::value;
      z[i][k] = cb[(a.l + 8 * k) * kStride128 + 64 * i + 8 * a.wave + a.r];
    });
  });
  waveExchange();
  staticFor<2>([&](auto ii) {
    constexpr int i = decltype(ii)::value;
    if (!any(i)) return;
    regFFT<8, false>(z[i]);
    staticFor<8>([&](auto ll) {
      constexpr int l = decltype(ll)::value;
      c32 v = z[i][slot<8>(l)];
      if constexpr (l > 0) v = choose(a.l == 0, v, cmul(v, tw[4 * l * a.l]));  // (see choose)
      cb[rowPlace(a.l, l, 64 * i + 8 * a.wave + a.r)] = v;
    });
  });
  waveExchange();
  staticFor<2>([&](auto ii) {
    constexpr int i = decltype(ii)::value;
    if (!any(i)) return;
    staticFor<8>([&](auto kk) {
      constexpr int k = decltype(kk)::value;
      z[i][k] = cb[rowPlace(k, a.l, 64 * i + 8 * a.wave + a.r)];
    });
  });
  __syncthreads();  // every place is free: rows [y][column pair] from here on
  staticFor<2>([&](auto ii) {
    constexpr int i = decltype(ii)::value;
    if (!any(i)) return;
    regFFT<8, false>(z[i]);
    staticFor<8>([&](auto mm) {
      constexpr int m = decltype(mm)::value;
      cb[sampleAt(64 * i + 8 * a.wave + a.r, a.l + 8 * m)] = z[i][slot<8>(m)];
    });
  });
  waveExchange();

  // ---- the wave's rows out, cropped to the window real covers ----
  float* const dst = real.data + (size_t)b * real.sb;
  staticFor<2>([&](auto ii) {
    constexpr int i = decltype(ii)::value;
    if constexpr (FAST_REAL) {
      staticFor<4>([&](auto jj) {
        const int y = 64 * i + 8 * a.wave + 2 * decltype(jj)::value + a.lane / 32, x4 = a.lane % 32;
        streamStore(reinterpret_cast<float4*>(dst + (size_t)y * real.sy) + x4,
                    *reinterpret_cast<const float4*>(cb + sampleAt(y, 2 * x4)));
      });
    } else {
      if (!any(i)) return;
      float v[8][2];
      staticFor<8>([&](auto rr) {
        staticFor<2>([&](auto jj) {
          constexpr int r = decltype(rr)::value, j = decltype(jj)::value;
          const int x = a.lane + 64 * j;
          v[r][j] = reinterpret_cast<const float*>(cb + sampleAt(64 * i + 8 * a.wave + r, x / 2))[x % 2];
        });
      });
      staticFor<8>([&](auto rr) {
        constexpr int r = decltype(rr)::value;
        const int y = 64 * i + 8 * a.wave + r - padU;
        if ((unsigned)y >= (unsigned)real.h) return;
        float* const row = dst + (size_t)y * real.sy;
        staticFor<2>([&](auto jj) {
          constexpr int j = decltype(jj)::value;
          const int x = a.lane + 64 * j - padL;
          if ((unsigned)x < (unsigned)real.w) row[(size_t)x * real.sx] = v[r][j];
        });
      });
    }
  });
}

// ---- 64 x 64 ----
//
// The same with 128 lanes per plane.  Rows: 16 of a wave at a time, four lanes each, as 32 = 4 x 8 packed values:
// lane l loads j = 2 l, 2 l + 1 of every eight, runs 4 points over each, and lane k mod 4 runs 8.  Columns: eight
// lanes take kx and 32 - kx (0 with 16), as 64 = 8 x 8 points.  LDS holds [kx][y] without padding; y is
// permuted by kx so that sixteen lanes meet different places modulo 16 everywhere.  A wave has its own roots, and
// the inverse its samples among the places of its own rows, which leaves one barrier between the passes; the
// forward kernel takes another so that each wave stores half of the plane in sequence (5000 planes to HBM 31.4 ->
// 30.2 us in the median, pairs of columns before).
constexpr int kLanes64 = 128;

// How the real operand moves: whole planes as float4, samples side by side as words of four, others one by one.
// (Decided at run time, these take 2 to 4 % more of small batches.)
enum RealMode { Whole, Words, Single };

struct Lane64 {
  int wave, lane;
  int l, r;     // row pass: lane of the row, row of the wave's sixteen
  int h, pair;  // column pass: lane of the pair, pair
  int k0, k1;   // its columns
};

__device__ __forceinline__ Lane64 lane64(int t) {
  Lane64 a;
  a.wave = __builtin_amdgcn_readfirstlane(t / 64);
  a.lane = t % 64;
  a.l = a.lane % 4;
  a.r = a.lane / 4;
  a.h = a.lane % 8;
  a.pair = a.wave * 8 + a.lane / 8;
  a.k0 = a.pair;
  a.k1 = a.pair ? 32 - a.pair : 16;
  return a;
}

__device__ __forceinline__ constexpr int at64(int column, int y) {
  return column * 64 + (y ^ (8 * (column & 1) + 2 * (column & 2)));
}
// Every exclusive or of columns or of y is one of places, so a lane's places differ from one of them by constants: what
// meets its bits by exclusive or, the rest as the offset of the access.  In bytes, which leaves one instruction or
// none to an access: 998 / 1057 vector instructions, forward / inverse, -> 856 / 915.
__device__ __forceinline__ c32& placed64(c32* cb, int bytes) {
  return *reinterpret_cast<c32*>(reinterpret_cast<char*>(cb) + bytes);
}
// y = h + 8 m of a column, from base = 8 at64(column, h)
__device__ __forceinline__ constexpr int spacedPlace64(int base, int m) { return (base ^ 64 * (m & 1)) + 64 * (m & 6); }
// value j of class k of a row between its two steps is column 8 k + 4 (j & 1) + ((j >> 1) ^ k): from
// base = 8 at64(9 k, y), and of j = 2 l + e from 8 at64(l, y)
__device__ __forceinline__ constexpr int rowValue64(int base, int j) { return (base ^ 8 * at64(j >> 1, 0)) + 2048 * (j & 1); }
__device__ __forceinline__ constexpr int rowClass64(int base, int k, int e) {
  return (base ^ 8 * at64(k, 0)) + 4096 * k + 2048 * e;
}
// value l of class k of a column is y = 8 k + (l ^ k): from base = 8 at64(column, 9 k) base ^ 8 l, and from 8 at64(column, l)
__device__ __forceinline__ constexpr int columnClass64(int base, int k) { return (base ^ 8 * (9 * k & 15)) + 8 * (9 * k & 48); }
// where the packed value j of row 32 i + 16 wave + r waits, before the forward transform and behind the inverse: among the
// places of the wave's rows
__device__ __forceinline__ constexpr int samplePlace64(int wave, int i, int r, int j) {
  return 8 * (1024 * i + 64 * r + 32 * (j >> 4) + 16 * wave + ((j & 15) ^ (8 * (r & 1))));
}

// e^{-/+ 2 pi i m / 64}
template <bool FWD>
__device__ __forceinline__ void fillRoots64(c32* tw, int lane) {
  const int h = (4 * lane) & 127;
  const float sign = lane < 32 ? 1.0f : -1.0f;
  const float c = sign * __builtin_bit_cast(float, kTwiddleBits[2 * h]);
  const float s = sign * __builtin_bit_cast(float, kTwiddleBits[2 * h + 1]);
  tw[lane] = c32{c, FWD ? -s : s};
}

template <int REAL, bool FAST_CPLX>
__global__ __launch_bounds__(kLanes64, 4) void fft2d64Forward(RealView real, CplxView cplx, int padL, int padU) {
  __shared__ __align__(16) c32 cb[32 * 64];
  __shared__ __align__(8) c32 roots[kLanes64 / 64][64];  // a wave's own: no barrier
  const Lane64 a = lane64(threadIdx.x);
  c32* const tw = roots[a.wave];
  constexpr bool ANY = REAL != Whole || !FAST_CPLX;
  const int b = ANY ? planeOf(real, cplx) : blockIdx.x;
  if (ANY && b >= real.B) return;
  // whether a wave's rows 32 i + 16 wave ... + 15 hold a row of the window
  auto any = [&](int i) __attribute__((always_inline)) {
    const int y = 32 * i + 16 * a.wave;
    return REAL == Whole || (real.w > 0 && real.h > 0 && y < padU + real.h && y + 16 > padU);
  };
  const float* const src = real.data + (size_t)b * real.sb;

  float4 z[2][4];  // packed values 2 l + 8 m and the next
  if constexpr (REAL == Whole) {
    staticFor<2>([&](auto ii) {
      constexpr int i = decltype(ii)::value;
      const float4* row = reinterpret_cast<const float4*>(src + (size_t)(32 * i + 16 * a.wave + a.r) * real.sy) + a.l;
      staticFor<4>([&](auto mm) { z[i][decltype(mm)::value] = row[4 * decltype(mm)::value]; });
    });
  } else {
    // implicit zero padding, any strides: loads at places clamped into the window, no branch between them, and
    // what lies outside counts as zero.  Samples side by side move four at a time, from any float on; the words that the
    // window's ends cut (at places that are the same for every row) are shifted into place.  Others move one by
    // one, and where neighbours of a row share cache lines a wave takes row after row and turns them in LDS.  us, four
    // lanes to a row one by one / so: 1763 whole planes 4 bytes off 16 20.2 / 12.6, 2594 windows of 61 x 61 in rows of 64
    // 27.4 / 17.6; 2000 planes of every second float 22.6 / 17.7, every third 22.8 / 21.9, every sixth 35.3 / 35.6, 300 of
    // every fourth 10.2 / 8.5, of every eighth 11.6 / 12.0.
    const int sx = abs(real.sx);
    const bool byRow = REAL == Single && real.w >= 4 && sx > 0 && sx <= 6 && sx <= abs(real.sy);
    auto rowAt = [&](int y) __attribute__((always_inline)) {
      return src + (size_t)min(max(y - padU, 0), real.h - 1) * real.sy;
    };
    if (byRow) {
      const int x = min(max(a.lane - padL, 0), real.w - 1);
      staticFor<2>([&](auto ii) {
        constexpr int i = decltype(ii)::value;
        if (!any(i)) return;
        float in[16];
        staticFor<16>([&](auto rr) {
          constexpr int r = decltype(rr)::value;
          in[r] = rowAt(32 * i + 16 * a.wave + r)[(size_t)x * real.sx];
        });
        staticFor<16>([&](auto rr) {
          constexpr int r = decltype(rr)::value;
          reinterpret_cast<float*>(&placed64(cb, samplePlace64(a.wave, i, r, a.lane / 2)))[a.lane % 2] = in[r];
        });
      });
      waveExchange();
      staticFor<8>([&](auto mm) {
        constexpr int i = decltype(mm)::value / 4, m = decltype(mm)::value % 4;
        z[i][m] = *reinterpret_cast<const float4*>(&placed64(cb, samplePlace64(a.wave, i, a.r, 2 * a.l + 8 * m)));
      });
    } else if constexpr (REAL == Words) {
      staticFor<2>([&](auto ii) {
        constexpr int i = decltype(ii)::value;
        if (!any(i)) return;
        const float* const row = rowAt(32 * i + 16 * a.wave + a.r);
        staticFor<4>([&](auto mm) {
          constexpr int m = decltype(mm)::value;
          const AnyFour f = *reinterpret_cast<const AnyFour*>(row + min(max(4 * a.l + 16 * m - padL, 0), real.w - 4));
          z[i][m] = float4{f[0], f[1], f[2], f[3]};
        });
      });
      const int cutLeft = padL & 3, cutRight = -(padL + real.w) & 3;
      if ((cutLeft | cutRight) != 0) {
        staticFor<8>([&](auto mm) {
          constexpr int i = decltype(mm)::value / 4, m = decltype(mm)::value % 4;
          const int x = 4 * a.l + 16 * m - padL;
          const float4 f = z[i][m];
          if (x > real.w - 4 && x < real.w) {  // from float cutRight on
            z[i][m].x = cutRight == 1 ? f.y : cutRight == 2 ? f.z : f.w;
            z[i][m].y = cutRight == 1 ? f.z : f.w;
            z[i][m].z = f.w;
          }
          if (x < 0 && x > -4) {  // the first float goes to cutLeft
            z[i][m].y = f.x;
            z[i][m].z = cutLeft == 1 ? f.y : f.x;
            z[i][m].w = cutLeft == 1 ? f.z : cutLeft == 2 ? f.y : f.x;
          }
        });
      }
    } else {
      staticFor<2>([&](auto ii) {
        constexpr int i = decltype(ii)::value;
        if (!any(i)) return;
        const float* const row = rowAt(32 * i + 16 * a.wave + a.r);
        staticFor<4>([&](auto mm) {
          constexpr int m = decltype(mm)::value;
          const int x = 4 * a.l + 16 * m - padL;
          z[i][m].x = row[(size_t)min(max(x, 0), real.w - 1) * real.sx];
          z[i][m].y = row[(size_t)min(max(x + 1, 0), real.w - 1) * real.sx];
          z[i][m].z = row[(size_t)min(max(x + 2, 0), real.w - 1) * real.sx];
          z[i][m].w = row[(size_t)min(max(x + 3, 0), real.w - 1) * real.sx];
        });
      });
    }
    staticFor<8>([&](auto mm) {
      constexpr int i = decltype(mm)::value / 4, m = decltype(mm)::value % 4;
      const bool yIn = (unsigned)(32 * i + 16 * a.wave + a.r - padU) < (unsigned)real.h;
      const int x = 4 * a.l + 16 * m - padL;
      z[i][m].x = yIn && (unsigned)x < (unsigned)real.w ? z[i][m].x : 0.0f;
      z[i][m].y = yIn && (unsigned)(x + 1) < (unsigned)real.w ? z[i][m].y : 0.0f;
      z[i][m].z = yIn && (unsigned)(x + 2) < (unsigned)real.w ? z[i][m].z : 0.0f;
      z[i][m].w = yIn && (unsigned)(x + 3) < (unsigned)real.w ? z[i][m].w : 0.0f;
    });
  }
  fillRoots64<true>(tw, a.lane);
  waveExchange();

  // ---- rows ----
  const int values = 8 * at64(a.l, 16 * a.wave + a.r), classes = 8 * at64(9 * a.l, 16 * a.wave + a.r);
  c32 v[2][8];
  staticFor<2>([&](auto ii) {
    constexpr int i = decltype(ii)::value;
    if (!any(i)) return;
    c32 p[4], q[4];
    staticFor<4>([&](auto mm) {
      constexpr int m = decltype(mm)::value;
      p[m] = c32{z[i][m].x, z[i][m].y};
      q[m] = c32{z[i][m].z, z[i][m].w};
    });
    regFFT<4, true>(p);
    regFFT<4, true>(q);
    staticFor<4>([&](auto kk) {
      constexpr int k = decltype(kk)::value;
      c32 f = p[slot<4>(k)], g = q[slot<4>(k)];
      if constexpr (k > 0) {
        f = cmul(f, tw[4 * k * a.l]);
        g = cmul(g, tw[4 * k * a.l + 2 * k]);
      }
      placed64(cb, rowClass64(values, k, 0) + 256 * i) = f;
      placed64(cb, rowClass64(values, k, 1) + 256 * i) = g;
    });
  });
  waveExchange();
  staticFor<2>([&](auto ii) {
    constexpr int i = decltype(ii)::value;
    staticFor<8>([&](auto jj) {
      constexpr int j = decltype(jj)::value;
      v[i][j] = c32{0.0f, 0.0f};
      if (any(i)) v[i][j] = placed64(cb, rowValue64(classes, j) + 256 * i);
    });
  });
  waveExchange();
  staticFor<2>([&](auto ii) {
    constexpr int i = decltype(ii)::value;
    if (any(i)) regFFT<8, true>(v[i]);  // (rows outside are zeros)
    staticFor<8>([&](auto kk) {
      constexpr int k = decltype(kk)::value;
      placed64(cb, values + 2048 * k + 256 * i) = v[i][slot<8>(k)];
    });
  });
  __syncthreads();

  // ---- columns ----
  const int c0 = 8 * at64(a.k0, a.h), c1 = 8 * at64(a.k1, a.h), d0 = 8 * at64(a.k0, 9 * a.h), d1 = 8 * at64(a.k1, 9 * a.h);
  c32 p[8], q[8];
  const c32 root = tw[a.pair], half = c32{0.5f * root.x, 0.5f * root.y};
  staticFor<8>([&](auto mm) {
    constexpr int m = decltype(mm)::value;
    p[m] = placed64(cb, spacedPlace64(c0, m));
    q[m] = placed64(cb, spacedPlace64(c1, m));
  });
  waveExchange();
  staticFor<8>([&](auto mm) {
    constexpr int m = decltype(mm)::value;
    const c32 f = p[m], g = q[m];
    const c32 e2 = c32{f.x + g.x, f.y - g.y};
    const c32 t = cmul(c32{f.y + g.y, g.x - f.x}, half);
    p[m] = c32{__builtin_fmaf(0.5f, e2.x, t.x), __builtin_fmaf(0.5f, e2.y, t.y)};
    q[m] = c32{__builtin_fmaf(0.5f, e2.x, -t.x), __builtin_fmaf(-0.5f, e2.y, t.y)};
    if (a.wave == 0) {  // (the pair of columns 0 and 16 is in the first wave)
      const bool ends = a.pair == 0;
      p[m] = ends ? c32{f.x + f.y, f.x - f.y} : p[m];
      q[m] = ends ? c32{g.x, -g.y} : q[m];
    }
  });
  regFFT<8, true>(p);
  regFFT<8, true>(q);
  staticFor<8>([&](auto kk) {
    constexpr int k = decltype(kk)::value;
    c32 f = p[slot<8>(k)], g = q[slot<8>(k)];
    if constexpr (k > 0) {
      const c32 w = tw[k * a.h];
      f = cmul(f, w);
      g = cmul(g, w);
    }
    placed64(cb, columnClass64(c0, k)) = f;
    placed64(cb, columnClass64(c1, k)) = g;
  });
  waveExchange();
  staticFor<8>([&](auto jj) {
    constexpr int j = decltype(jj)::value;
    p[j] = placed64(cb, d0 ^ 8 * j);
    q[j] = placed64(cb, d1 ^ 8 * j);
  });
  waveExchange();
  regFFT<8, true>(p);
  regFFT<8, true>(q);
  staticFor<8>([&](auto kk) {
    constexpr int k = decltype(kk)::value;
    placed64(cb, spacedPlace64(c0, k)) = p[slot<8>(k)];
    placed64(cb, spacedPlace64(c1, k)) = q[slot<8>(k)];
  });
  __syncthreads();

  // ---- columns out, a half of the plane per wave, 1 KB at a time; rows 0 and 32 of the result come from packed column 0 ----
  const int ky = 2 * (a.lane % 32);
  float* const dst = cplx.data + (size_t)b * cplx.sb;
  auto store = [&](int r, float4 o) __attribute__((always_inline)) {
    if constexpr (FAST_CPLX) {
      streamStore(reinterpret_cast<float4*>(dst) + r * 32 + a.lane % 32, o);
    } else {
      float* to = dst + (size_t)r * cplx.sr + (size_t)ky * cplx.sc;
      *reinterpret_cast<float2*>(to) = float2{o.x, o.y};
      *reinterpret_cast<float2*>(to + cplx.sc) = float2{o.z, o.w};
    }
  };
  staticFor<8>([&](auto ii) {
    constexpr int i = decltype(ii)::value;
    const int column = 16 * a.wave + 2 * i + a.lane / 32;
    float4 o = *reinterpret_cast<const float4*>(cb + at64(column, ky));
    if (i == 0 && a.wave == 0) {
      const c32 m0 = cb[(64 - ky) & 63], m1 = cb[63 - ky];
      if (a.lane < 32) {
        store(32, float4{0.5f * (o.y + m0.y), 0.5f * (m0.x - o.x), 0.5f * (o.w + m1.y), 0.5f * (m1.x - o.z)});
        o = float4{0.5f * (o.x + m0.x), 0.5f * (o.y - m0.y), 0.5f * (o.z + m1.x), 0.5f * (o.w - m1.y)};
      }
    }
    store(column, o);
  });
}

template <int REAL, bool FAST_CPLX>
__global__ __launch_bounds__(kLanes64, 4) void fft2d64Inverse(CplxView cplx, RealView real, int padL, int padU) {
  __shared__ __align__(16) c32 cb[32 * 64];
  __shared__ __align__(8) c32 roots[kLanes64 / 64][64];  // a wave's own: no barrier
  const Lane64 a = lane64(threadIdx.x);
  c32* const tw = roots[a.wave];
  constexpr bool ANY = REAL != Whole || !FAST_CPLX;
  const int b = ANY ? planeOf(real, cplx) : blockIdx.x;
  if (ANY && b >= real.B) return;
  auto any = [&](int i) __attribute__((always_inline)) {
    const int y = 32 * i + 16 * a.wave;
    return REAL == Whole || (real.w > 0 && real.h > 0 && y < padU + real.h && y + 16 > padU);
  };

  // ---- the wave's columns in, two at a time; column 0 carries 32 as its imaginary part ----
  const int ky = 2 * (a.lane % 32);
  const float* const src = cplx.data + (size_t)b * cplx.sb;
  auto load = [&](int r) __attribute__((always_inline)) {
    if constexpr (FAST_CPLX) {
      return reinterpret_cast<const float4*>(src)[r * 32 + a.lane % 32];
    } else {
      const float* from = src + (size_t)r * cplx.sr + (size_t)ky * cplx.sc;
      const float2 f = *reinterpret_cast<const float2*>(from), g = *reinterpret_cast<const float2*>(from + cplx.sc);
      return float4{f.x, f.y, g.x, g.y};
    }
  };
  {
    auto column = [&](int i) __attribute__((always_inline)) {
      const int k = a.wave * 8 + i;
      return a.lane < 32 ? k : k ? 32 - k : 16;
    };
    float4 in[8];
    staticFor<8>([&](auto ii) { in[decltype(ii)::value] = load(column(decltype(ii)::value)); });
    if (a.wave == 0) {
      const float4 last = load(32);
      if (a.lane < 32) in[0] = float4{in[0].x - last.y, in[0].y + last.x, in[0].z - last.w, in[0].w + last.z};
    }
    staticFor<8>([&](auto ii) {
      constexpr int i = decltype(ii)::value;
      *reinterpret_cast<float4*>(cb + at64(column(i), ky)) = in[i];
    });
  }
  fillRoots64<false>(tw, a.lane);
  waveExchange();

  // ---- columns ----
  const int c0 = 8 * at64(a.k0, a.h), c1 = 8 * at64(a.k1, a.h), d0 = 8 * at64(a.k0, 9 * a.h), d1 = 8 * at64(a.k1, 9 * a.h);
  c32 p[8], q[8];
  staticFor<8>([&](auto kk) {
    constexpr int k = decltype(kk)::value;
    p[k] = placed64(cb, spacedPlace64(c0, k));
    q[k] = placed64(cb, spacedPlace64(c1, k));
  });
  waveExchange();
  regFFT<8, false>(p);
  regFFT<8, false>(q);
  staticFor<8>([&](auto ll) {
    constexpr int l = decltype(ll)::value;
    placed64(cb, d0 ^ 8 * l) = p[slot<8>(l)];
    placed64(cb, d1 ^ 8 * l) = q[slot<8>(l)];
  });
  waveExchange();
  staticFor<8>([&](auto kk) {
    constexpr int k = decltype(kk)::value;
    p[k] = placed64(cb, columnClass64(c0, k));
    q[k] = placed64(cb, columnClass64(c1, k));
    if constexpr (k > 0) {
      const c32 w = tw[k * a.h];
      p[k] = cmul(p[k], w);
      q[k] = cmul(q[k], w);
    }
  });
  waveExchange();
  regFFT<8, false>(p);
  regFFT<8, false>(q);
  const c32 root = tw[a.pair];
  staticFor<8>([&](auto mm) {
    constexpr int m = decltype(mm)::value;
    const c32 f = p[slot<8>(m)], g = q[slot<8>(m)];
    const c32 e = c32{f.x + g.x, f.y - g.y};
    const c32 o = cmul(c32{f.x - g.x, f.y + g.y}, root);
    c32 zk = c32{e.x - o.y, e.y + o.x}, zh = c32{e.x + o.y, o.x - e.y};
    if (a.wave == 0) {
      const bool ends = a.pair == 0;
      zk = ends ? c32{f.x + f.y, f.x - f.y} : zk;
      zh = ends ? c32{2.0f * g.x, -2.0f * g.y} : zh;
    }
    placed64(cb, spacedPlace64(c0, m)) = zk;
    placed64(cb, spacedPlace64(c1, m)) = zh;
  });
  __syncthreads();

  // ---- rows ----
  const int values = 8 * at64(a.l, 16 * a.wave + a.r), classes = 8 * at64(9 * a.l, 16 * a.wave + a.r);
  c32 v[2][8];
  staticFor<2>([&](auto ii) {
    constexpr int i = decltype(ii)::value;
    if (!any(i)) return;
    staticFor<8>([&](auto kk) {
      constexpr int k = decltype(kk)::value;
      v[i][k] = placed64(cb, values + 2048 * k + 256 * i);
    });
  });
  waveExchange();
  staticFor<2>([&](auto ii) {
    constexpr int i = decltype(ii)::value;
    if (!any(i)) return;
    regFFT<8, false>(v[i]);
    staticFor<8>([&](auto jj) {
      constexpr int j = decltype(jj)::value;
      c32 f = v[i][slot<8>(j)];
      if constexpr (j > 0) f = choose(a.l == 0, f, cmul(f, tw[2 * j * a.l]));  // (see choose)
      placed64(cb, rowValue64(classes, j) + 256 * i) = f;
    });
  });
  waveExchange();
  const int samples = samplePlace64(a.wave, 0, a.r, 2 * a.l);
  float4 z[2][4];
  staticFor<2>([&](auto ii) {
    constexpr int i = decltype(ii)::value;
    if (!any(i)) return;
    c32 f[4], g[4];
    staticFor<4>([&](auto kk) {
      constexpr int k = decltype(kk)::value;
      f[k] = placed64(cb, rowClass64(values, k, 0) + 256 * i);
      g[k] = placed64(cb, rowClass64(values, k, 1) + 256 * i);
    });
    regFFT<4, false>(f);
    regFFT<4, false>(g);
    staticFor<4>([&](auto mm) {
      constexpr int m = decltype(mm)::value;
      z[i][m] = float4{f[slot<4>(m)].x, f[slot<4>(m)].y, g[slot<4>(m)].x, g[slot<4>(m)].y};
    });
  });
  waveExchange();  // every place of the wave is free: its samples from here on
  staticFor<2>([&](auto ii) {
    constexpr int i = decltype(ii)::value;
    if (!any(i)) return;
    staticFor<4>([&](auto mm) {
      constexpr int m = decltype(mm)::value;
      *reinterpret_cast<float4*>(&placed64(cb, (samples ^ 64 * (m & 1)) + 128 * (m & 2) + 8192 * i)) = z[i][m];
    });
  });
  waveExchange();

  // ---- the wave's rows out, cropped to the window real covers ----
  float* const dst = real.data + (size_t)b * real.sb;
  staticFor<2>([&](auto ii) {
    constexpr int i = decltype(ii)::value;
    if constexpr (REAL == Whole) {
      staticFor<4>([&](auto jj) {
        const int r = 4 * decltype(jj)::value + a.lane / 16, x4 = a.lane % 16;
        streamStore(reinterpret_cast<float4*>(dst + (size_t)(32 * i + 16 * a.wave + r) * real.sy) + x4,
                    *reinterpret_cast<const float4*>(&placed64(cb, samplePlace64(a.wave, i, r, 2 * x4))));
      });
    } else {
      if (!any(i)) return;
      if constexpr (REAL == Words) {
        // words of four to any float; a row's last one may cover some of the one before, of the same values.  us, a row
        // float by float / so: 463 windows of 56 x 56 8.5 / 6.9, 3000 of 50 x 50 to HBM 25.4 / 21.7 (plain stores 23.4), of 60 x
        // 60 27.5 / 23.8, 16384 of 60 x 60 98.7 / 97.0 (99.4), 2669 whole planes 4 bytes off 26.4 / 22.0.  Rows with gaps between
        // them leave cache lines partly written: 3137 of 64 x 64 in rows of 67 25.4 / 22.3, nontemporal 27.5.
        const int w = min(real.w, 64 - padL);
        const int x = min(4 * (a.lane % 16), w - 4), from = padL + x, cut = from & 3;
        const int first = 32 * i + 16 * a.wave + a.lane / 16 - padU;
        auto word = [&](int j, int k) __attribute__((always_inline)) {
          return *reinterpret_cast<const float4*>(&placed64(cb, samplePlace64(a.wave, i, 4 * j + a.lane / 16, 2 * k)));
        };
        float4 o[4];
        staticFor<4>([&](auto jj) { o[decltype(jj)::value] = word(decltype(jj)::value, from / 4); });
        if (((padL | w) & 3) != 0) {
          staticFor<4>([&](auto jj) {
            constexpr int j = decltype(jj)::value;
            const float4 f = o[j], g = word(j, min(from / 4 + 1, 15));
            const bool odd = cut & 1, two = cut & 2;
            const float p0 = odd ? f.y : f.x, p1 = odd ? f.z : f.y, p2 = odd ? f.w : f.z, p3 = odd ? g.x : f.w,
                        p4 = odd ? g.y : g.x, p5 = odd ? g.z : g.y;
            o[j] = float4{two ? p2 : p0, two ? p3 : p1, two ? p4 : p2, two ? p5 : p3};
          });
        }
        if (4 * (a.lane % 16) >= w) return;
        auto rows = [&](auto write) __attribute__((always_inline)) {
          staticFor<4>([&](auto jj) {
            constexpr int j = decltype(jj)::value;
            if ((unsigned)(first + 4 * j) < (unsigned)real.h)
              write(reinterpret_cast<AnyFour*>(dst + (size_t)(first + 4 * j) * real.sy + x), AnyFour{o[j].x, o[j].y, o[j].z, o[j].w});
          });
        };
        if (real.sy == real.w) {
          rows([](AnyFour* to, AnyFour f) { __builtin_nontemporal_store(f, to); });
        } else {
          asm volatile("");  // (or both become plain stores)
          rows([](AnyFour* to, AnyFour f) { *to = f; });
        }
        return;
      }
      float o[16];
      staticFor<16>([&](auto rr) {
        constexpr int r = decltype(rr)::value;
        o[r] = reinterpret_cast<const float*>(&placed64(cb, samplePlace64(a.wave, i, r, a.lane / 2)))[a.lane % 2];
      });
      const int x = a.lane - padL;
      if ((unsigned)x >= (unsigned)real.w) return;
      staticFor<16>([&](auto rr) {
        constexpr int r = decltype(rr)::value;
        const int y = 32 * i + 16 * a.wave + r - padU;
        if ((unsigned)y < (unsigned)real.h) dst[(size_t)y * real.sy + (size_t)x * real.sx] = o[r];
      });
    }
  });
}

bool fastReal(int N, const RealView& r, int padL, int padU) {
  return padL == 0 && padU == 0 && r.h == N && r.w == N && r.sx == 1 && r.sy % 4 == 0 &&
         r.sb % 4 == 0 && aligned(r.data, 16);
}

bool fastCplx(int N, const CplxView& c) {
  return c.sc == 2 && c.sr == 2 * N && c.sb % 4 == 0 && aligned(c.data, 16);
}

// runs f(mode of the real operand, std::bool_constant<fast>{}); width: samples of a row that the transform covers
template <typename F>
void withModes64(const RealView& real, const CplxView& cplx, int padL, int padU, int width, F&& f) {
  const bool fast = fastCplx(64, cplx);
  auto run = [&](auto m) { fast ? f(m, std::true_type{}) : f(m, std::false_type{}); };
  if (fastReal(64, real, padL, padU)) run(std::integral_constant<int, Whole>{});
  else if (real.sx == 1 && width >= 4) run(std::integral_constant<int, Words>{});
  else run(std::integral_constant<int, Single>{});
}

int launchForward64(const RealView& real, const CplxView& cplx, int padL, int padU, hipStream_t s) {
  withModes64(real, cplx, padL, padU, real.w, [&](auto m, auto fc) {
    constexpr int M = decltype(m)::value;
    constexpr bool FC = decltype(fc)::value;
    fft2d64Forward<M, FC><<<M == Whole && FC ? dim3(real.B) : planeGrid(real, cplx), dim3(kLanes64), 0, s>>>(real, cplx, padL, padU);
  });
  return launchStatus();
}

int launchInverse64(const CplxView& cplx, const RealView& real, int padL, int padU, hipStream_t s) {
  withModes64(real, cplx, padL, padU, std::min(real.w, 64 - padL), [&](auto m, auto fc) {
    constexpr int M = decltype(m)::value;
    constexpr bool FC = decltype(fc)::value;
    fft2d64Inverse<M, FC><<<M == Whole && FC ? dim3(real.B) : planeGrid(real, cplx), dim3(kLanes64), 0, s>>>(cplx, real, padL, padU);
  });
  return launchStatus();
}

// Samples four floats apart, in rows of most of the plane: row after row.  (us, one lane of eight rows loads from each / so, four
// lanes of 32 points, which walked down columns, before: one plane 12.7 / 10.5, 11.1; 300 23.1 / 21.6, 22.1; but 300 windows of 101
// x 90 15.4 / 16.6, and 300 planes of every second float 14.5 / 15.7.)
int launchForward128(const RealView& real, const CplxView& cplx, int padL, int padU, hipStream_t s) {
  const bool fr = fastReal(128, real, padL, padU), fc = fastCplx(128, cplx), rows = abs(real.sx) == 4 && real.w >= 104;
  const dim3 grid = fr && fc ? dim3(real.B) : planeGrid(real, cplx), block(kLanes128);
  if (fr && fc)
    fft2d128Forward<true, true><<<grid, block, 0, s>>>(real, cplx, padL, padU);
  else if (fc && rows)
    fft2d128Forward<false, true, true><<<grid, block, 0, s>>>(real, cplx, padL, padU);
  else if (fc)
    fft2d128Forward<false, true><<<grid, block, 0, s>>>(real, cplx, padL, padU);
  else if (fr)
    fft2d128Forward<true, false><<<grid, block, 0, s>>>(real, cplx, padL, padU);
  else if (rows)
    fft2d128Forward<false, false, true><<<grid, block, 0, s>>>(real, cplx, padL, padU);
  else
    fft2d128Forward<false, false><<<grid, block, 0, s>>>(real, cplx, padL, padU);
  return launchStatus();
}

int launchInverse128(const CplxView& cplx, const RealView& real, int padL, int padU, hipStream_t s) {
  const bool fr = fastReal(128, real, padL, padU), fc = fastCplx(128, cplx);
  const dim3 grid = fr && fc ? dim3(real.B) : planeGrid(real, cplx), block(kLanes128);
  if (fr && fc)
    fft2d128Inverse<true, true><<<grid, block, 0, s>>>(cplx, real, padL, padU);
  else if (fc)
    fft2d128Inverse<false, true><<<grid, block, 0, s>>>(cplx, real, padL, padU);
  else if (fr)
    fft2d128Inverse<true, false><<<grid, block, 0, s>>>(cplx, real, padL, padU);
  else
    fft2d128Inverse<false, false><<<grid, block, 0, s>>>(cplx, real, padL, padU);
  return launchStatus();
}

}  // namespace

int launchFft2dLargeForward(int N, const RealView& real, const CplxView& cplx, int padL, int padU,
                            hipStream_t s) {
  if (real.B <= 0) return FBFFT_SUCCESS;
  if (N == 64) return launchForward64(real, cplx, padL, padU, s);
  if (N == 128) return launchForward128(real, cplx, padL, padU, s);
  return FBFFT_UNSUPPORTED_SIZE;
}

int launchFft2dLargeInverse(int N, const CplxView& cplx, const RealView& real, int padL, int padU,
                            hipStream_t s) {
  if (real.B <= 0) return FBFFT_SUCCESS;
  if (N == 64) return launchInverse64(cplx, real, padL, padU, s);
  if (N == 128) return launchInverse128(cplx, real, padL, padU, s);
  return FBFFT_UNSUPPORTED_SIZE;
}

}  // namespace fbfft_amd
