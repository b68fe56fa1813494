// Batched 1D real-to-complex / complex-to-real transforms, N = 2 .. 256
// (replaces decimateInFrequency1DKernel, fbfft/FBFFTCommon.cuh:710-833, and its
// dispatch tables in fbfft/FBFFT-inl.cuh:19-150).
//
// A workgroup (256 lanes; of contiguous rows up to 64 points one wave) stages a row per G lanes in LDS with
// coalesced 8-byte accesses (contiguous rows: 16).  Each row is transformed as an N/2-point complex FFT of the
// even/odd packing z[j] = x[2j] + i x[2j+1]: one lane per row up to N = 64, two
// lanes for N = 128 and four for N = 256 (radix-G split read straight from LDS,
// 32 points per lane in VGPRs, G uniform per wave; contiguous rows of 256 have a kernel of their own,
// below).  The real-input fix-up runs
// on the way out (forward) or on the way in (inverse) with lanes mapped to
// consecutive output elements, so HBM stores are contiguous.  The reference
// instead pairs two rows into one N-point complex transform; results agree to
// rounding and rows never depend on their neighbours here, so odd batch sizes
// need no special case.
#include "common.h"
#include "fft_lds.h"
#include "fft_regs.h"

namespace fbfft_amd {
namespace {

constexpr int k1dThreads = 256;

template <int N>
struct Cfg1D {
  static constexpr int H = N / 2;
  static constexpr int G = (H <= 32) ? 1 : H / 32;
  static constexpr int L = H / G;
  static constexpr int ROWS = k1dThreads / G;
  static constexpr int RS = H + 1;  // LDS row stride in complex (= N + 2 floats)
};

// real [B][N] with strides (sb, sx); cplx [B][N/2+1][2] with strides (cb, ck)
struct Row1D {
  float* real;
  int sb, sx;
  float* cplx;
  int cb, ck;
  int B;
  int padL;
};

template <int N, bool FAST>
__global__ __launch_bounds__(k1dThreads) void fft1dForward(Row1D a) {
  using C = Cfg1D<N>;
  constexpr int H = C::H, G = C::G, L = C::L, ROWS = C::ROWS, RS = C::RS;
  __shared__ __align__(16) c32 lds[ROWS * RS];
  __shared__ __align__(8) c32 tw[256];
  const int t = threadIdx.x;
  const int b0 = blockIdx.x * ROWS;
  fillTwiddles<true>(tw, t, k1dThreads);

  // ---- rows -> LDS as packed complex z[j] = (x[2j], x[2j+1]); every load is
  // issued before the first one is consumed ----
  constexpr int LOADS = (ROWS * H + k1dThreads - 1) / k1dThreads;
  c32 in[LOADS];
  staticFor<LOADS>([&](auto ii) {
    constexpr int i = decltype(ii)::value;
    const int idx = t + k1dThreads * i;
    const int row = min(idx / H, ROWS - 1), j = idx % H;
    const int b = min(b0 + row, a.B - 1);
    if constexpr (FAST) {
      in[i] = *reinterpret_cast<const float2*>(a.real + (size_t)b * a.sb + 2 * j);
    } else {
      const float* src = a.real + (size_t)b * a.sb;
      const int x0 = 2 * j - a.padL, x1 = 2 * j + 1 - a.padL;
      // a right shift that drops the last padL samples (fbfft/FBFFTCommon.cuh:325)
      in[i].x = x0 >= 0 ? src[(size_t)x0 * a.sx] : 0.0f;
      in[i].y = x1 >= 0 ? src[(size_t)x1 * a.sx] : 0.0f;
    }
  });
  staticFor<LOADS>([&](auto ii) {
    constexpr int i = decltype(ii)::value;
    const int idx = t + k1dThreads * i;
    if (idx < ROWS * H) lds[(idx / H) * RS + idx % H] = in[i];
  });
  __syncthreads();

  const int row = t % ROWS, g = t / ROWS;
  c32* zrow = lds + row * RS;
  c32 v[L];
  splitFFT<H, G, true>(zrow, g, tw, v);
  __syncthreads();
  staticFor<L>([&](auto kk) {
    constexpr int k = decltype(kk)::value;
    zrow[G * k + g] = v[slot<L>(k)];
  });
  __syncthreads();

  // ---- fix-up and store: lanes run over consecutive output bins ----
  for (int idx = t; idx < ROWS * (H + 1); idx += k1dThreads) {
    const int r = idx / (H + 1), k = idx % (H + 1);
    const int b = b0 + r;
    if (b >= a.B) break;
    const c32* z = lds + r * RS;
    c32 f;
    if (k == 0 || k == H) {
      c32 z0 = z[0];
      f = c32{k == 0 ? z0.x + z0.y : z0.x - z0.y, 0.0f};
    } else {
      c32 p = z[k], q = z[H - k];
      c32 e = c32{0.5f * (p.x + q.x), 0.5f * (p.y - q.y)};
      c32 o = c32{0.5f * (p.y + q.y), -0.5f * (p.x - q.x)};
      c32 w = tw[k * (256 / N)];
      c32 wo = cmul(o, w);
      f = c32{e.x + wo.x, e.y + wo.y};
    }
    *reinterpret_cast<float2*>(a.cplx + (size_t)b * a.cb + (size_t)k * a.ck) = f;
  }
}

template <int N, bool FAST>
__global__ __launch_bounds__(k1dThreads) void fft1dInverse(Row1D a) {
  using C = Cfg1D<N>;
  constexpr int H = C::H, G = C::G, L = C::L, ROWS = C::ROWS, RS = C::RS;
  __shared__ __align__(16) c32 lds[ROWS * RS];
  __shared__ __align__(8) c32 tw[256];
  const int t = threadIdx.x;
  const int b0 = blockIdx.x * ROWS;
  fillTwiddles<false>(tw, t, k1dThreads);

  // ---- spectra -> LDS, all loads in flight together ----
  constexpr int LOADS = (ROWS * (H + 1) + k1dThreads - 1) / k1dThreads;
  c32 in[LOADS];
  staticFor<LOADS>([&](auto ii) {
    constexpr int i = decltype(ii)::value;
    const int idx = t + k1dThreads * i;
    const int r = min(idx / (H + 1), ROWS - 1), k = idx % (H + 1);
    const int b = min(b0 + r, a.B - 1);
    in[i] = *reinterpret_cast<const float2*>(a.cplx + (size_t)b * a.cb + (size_t)k * a.ck);
  });
  staticFor<LOADS>([&](auto ii) {
    constexpr int i = decltype(ii)::value;
    const int idx = t + k1dThreads * i;
    if (idx < ROWS * (H + 1)) lds[(idx / (H + 1)) * RS + idx % (H + 1)] = in[i];
  });
  __syncthreads();

  // ---- inverse real fix-up in place: bins k and H-k form one work item ----
  for (int idx = t; idx < ROWS * (H / 2 + 1); idx += k1dThreads) {
    const int r = idx / (H / 2 + 1), k = idx % (H / 2 + 1);
    c32* z = lds + r * RS;
    if (k == 0) {
      // only the real parts of F[0] and F[N/2] reach a real result
      const float f0 = z[0].x, fh = z[H].x;
      z[0] = c32{f0 + fh, f0 - fh};
    } else if (2 * k == H) {
      c32 p = z[k];
      z[k] = c32{2.0f * p.x, -2.0f * p.y};
    } else {
      c32 p = z[k], q = z[H - k];
      c32 e = c32{p.x + q.x, p.y - q.y};
      c32 d = c32{p.x - q.x, p.y + q.y};
      c32 o = cmul(d, tw[k * (256 / N)]);
      z[k] = c32{e.x - o.y, e.y + o.x};
      z[H - k] = c32{e.x + o.y, o.x - e.y};
    }
  }
  __syncthreads();

  const int row = t % ROWS, g = t / ROWS;
  c32* zrow = lds + row * RS;
  c32 v[L];
  splitFFT<H, G, false>(zrow, g, tw, v);
  __syncthreads();
  staticFor<L>([&](auto kk) {
    constexpr int k = decltype(kk)::value;
    zrow[G * k + g] = v[slot<L>(k)];
  });
  __syncthreads();

  // ---- store rows ----
  for (int idx = t; idx < ROWS * H; idx += k1dThreads) {
    const int r = idx / H, j = idx % H;
    const int b = b0 + r;
    if (b >= a.B) break;
    c32 val = lds[r * RS + j];
    if constexpr (FAST) {
      *reinterpret_cast<float2*>(a.real + (size_t)b * a.sb + 2 * j) = val;
    } else {
      // the reference writes the first row of each pair at x and the second at
      // x - padL, both only for x >= padL (fbfft/FBFFTCommon.cuh:423-428)
      float* dst = a.real + (size_t)b * a.sb;
      const int shift = (b & 1) ? a.padL : 0;
      const int x0 = 2 * j, x1 = 2 * j + 1;
      if (x0 >= a.padL) dst[(size_t)(x0 - shift) * a.sx] = val.x;
      if (x1 >= a.padL) dst[(size_t)(x1 - shift) * a.sx] = val.y;
    }
  }
}

// ---- N = 8 ... 128 with contiguous, 16-byte aligned operands ----
//
// Same staging as above, but the real-input fix-up never makes a pass of its own
// through LDS: with one lane per row (N <= 64) the whole half-length transform is in
// the lane's registers, and with two lanes per row (N = 128) the split is chosen so
// that the fix-up pairs (k, N/2 - k) stay inside one lane - the forward transform
// splits its outputs by parity, the inverse its inputs (E = IFFT(z even),
// O = IFFT(z odd), x[j] = E[j] + w^j O[j], x[j + N/4] = E[j] - w^j O[j], summed on
// the way out of LDS).  Spectra and rows then move between LDS and HBM as plain 16-byte
// streams.
template <int N, int THREADS>
struct CfgMid {
  static_assert(N >= 8 && N <= 128, "one lane per row up to 64 points, then two");
  static constexpr int H = N / 2;
  static constexpr int G = N <= 64 ? 1 : N / 64;  // lanes per row
  static constexpr int Q = H / G;           // points per lane (32)
  static constexpr int ROWS = THREADS / G;
  static constexpr int RS = H + 1;          // LDS row stride (complex) = spectrum row length
};

template <int N, int THREADS>
__global__ __launch_bounds__(THREADS, 2) void fft1dMidForward(const float* __restrict__ real,
                                                              float* __restrict__ cplx, int B) {
  using C = CfgMid<N, THREADS>;
  constexpr int H = C::H, G = C::G, Q = C::Q, ROWS = C::ROWS, RS = C::RS;
  __shared__ __align__(16) c32 lds[ROWS * RS];
  __shared__ __align__(8) c32 tw[256];
  const int t = threadIdx.x;
  const int b0 = blockIdx.x * ROWS;
  const int rows = min(ROWS, B - b0);
  if constexpr (G > 1) fillTwiddles<true>(tw, t, THREADS);

  // ---- rows -> LDS as packed complex z[j] = (x[2j], x[2j+1]), 16 bytes per load ----
  constexpr int LOADS = ROWS * H / 2 / THREADS;
  const float4* src = reinterpret_cast<const float4*>(real + (size_t)b0 * N);
  float4 in[LOADS];
  staticFor<LOADS>([&](auto ii) {
    constexpr int i = decltype(ii)::value;
    const int idx = t + THREADS * i;               // float4 index: row = idx / (H/2)
    in[i] = src[min(idx, rows * (H / 2) - 1)];
  });
  staticFor<LOADS>([&](auto ii) {
    constexpr int i = decltype(ii)::value;
    const int idx = t + THREADS * i;
    c32* d = lds + (idx / (H / 2)) * RS + 2 * (idx % (H / 2));
    d[0] = c32{in[i].x, in[i].y};
    d[1] = c32{in[i].z, in[i].w};
  });
  __syncthreads();

  // ROWS is a multiple of 64: g is the same for a whole wave, and says so
  const int row = t % ROWS, g = __builtin_amdgcn_readfirstlane(t / ROWS);
  c32* zrow = lds + row * RS;
  c32 v[Q];
  if constexpr (G == 1) {
    splitFFT<H, 1, true>(zrow, 0, tw, v);
    // the row is this lane's alone and is in registers: overwrite it with F[0..H]
    realFixupForwardEmit<H>(v, [&](auto kk, c32 val) {
      constexpr int k = decltype(kk)::value;
      if constexpr (k == 0) {
        zrow[0] = c32{val.x, 0.0f};
        zrow[H] = c32{val.y, 0.0f};
      } else {
        zrow[k] = val;
      }
    });
  } else {
    splitFFT<H, 2, true>(zrow, g, tw, v);   // lane g: Z[2k + g]
    __syncthreads();                        // both lanes of a row have read it
    auto pairOut = [&](auto kp, c32 a, c32 bq) __attribute__((always_inline)) {
      constexpr int k = decltype(kp)::value;  // bin k pairs with H-k
      c32 fk, fhk;
      realPairForward<N, k>(a, bq, fk, fhk);
      zrow[k] = fk;
      zrow[H - k] = fhk;
    };
    if (g == 0) {
      const c32 z0 = v[0];
      zrow[0] = c32{z0.x + z0.y, 0.0f};
      zrow[H] = c32{z0.x - z0.y, 0.0f};
      staticFor<Q / 2 - 1>([&](auto kk) {
        constexpr int k = decltype(kk)::value + 1;  // bins 2k and H-2k
        pairOut(std::integral_constant<int, 2 * k>{}, v[slot<Q>(k)], v[slot<Q>(Q - k)]);
      });
      const c32 m = v[slot<Q>(Q / 2)];  // bin H/2
      zrow[H / 2] = c32{m.x, -m.y};
    } else {
      staticFor<Q / 2>([&](auto kk) {
        constexpr int k = decltype(kk)::value;  // bins 2k+1 and H-2k-1
        pairOut(std::integral_constant<int, 2 * k + 1>{}, v[slot<Q>(k)], v[slot<Q>(Q - 1 - k)]);
      });
    }
  }
  __syncthreads();

  // ---- spectra out: LDS and HBM hold the same [row][H+1] stream ----
  const int total = rows * RS;  // complex values of this workgroup
  float4* dst = reinterpret_cast<float4*>(cplx + (size_t)b0 * 2 * RS);
  const float4* l4 = reinterpret_cast<const float4*>(lds);
  for (int q = t; q < total / 2; q += THREADS) streamStore(dst + q, l4[q]);
  if ((total & 1) && t == 0)
    reinterpret_cast<float2*>(cplx + (size_t)b0 * 2 * RS)[total - 1] = lds[total - 1];
}

template <int N, int THREADS>
__global__ __launch_bounds__(THREADS, 2) void fft1dMidInverse(const float* __restrict__ cplx,
                                                              float* __restrict__ real, int B) {
  using C = CfgMid<N, THREADS>;
  constexpr int H = C::H, G = C::G, Q = C::Q, ROWS = C::ROWS, RS = C::RS;
  __shared__ __align__(16) c32 lds[ROWS * RS];
  const int t = threadIdx.x;
  const int b0 = blockIdx.x * ROWS;
  const int rows = min(ROWS, B - b0);

  // ---- spectra -> LDS, the same [row][H+1] stream in both places ----
  const int total = rows * RS;
  constexpr int LOADS = (ROWS * RS / 2 + THREADS - 1) / THREADS;
  const float4* src = reinterpret_cast<const float4*>(cplx + (size_t)b0 * 2 * RS);
  float in[4 * LOADS];  // plain floats: always promoted to registers
  staticFor<LOADS>([&](auto ii) {
    constexpr int i = decltype(ii)::value;
    const float4 v = src[min(t + THREADS * i, max(total / 2 - 1, 0))];
    in[4 * i] = v.x;
    in[4 * i + 1] = v.y;
    in[4 * i + 2] = v.z;
    in[4 * i + 3] = v.w;
  });
  float4* l4 = reinterpret_cast<float4*>(lds);
  staticFor<LOADS>([&](auto ii) {
    constexpr int i = decltype(ii)::value;
    const int q = t + THREADS * i;
    if (q < total / 2) l4[q] = float4{in[4 * i], in[4 * i + 1], in[4 * i + 2], in[4 * i + 3]};
  });
  if ((total & 1) && t == 0)
    lds[total - 1] = reinterpret_cast<const float2*>(cplx + (size_t)b0 * 2 * RS)[total - 1];
  __syncthreads();

  // ROWS is a multiple of 64: g is the same for a whole wave, and says so
  const int row = t % ROWS, g = __builtin_amdgcn_readfirstlane(t / ROWS);
  c32* zrow = lds + row * RS;
  float* frow = reinterpret_cast<float*>(zrow);
  c32 zz[Q];
  if constexpr (G == 1) {
    // only the real parts of F[0] and F[H] reach a real result
    realFixupInverseFetch<H>(
        [&](auto kk) {
          constexpr int k = decltype(kk)::value;
          if constexpr (k == 0)
            return c32{zrow[0].x, zrow[H].x};
          else
            return zrow[k];
        },
        zz);
    regFFT<H, false>(zz);
    // private row, all of it in registers: store x[2j], x[2j+1]
    staticFor<Q>([&](auto jj) {
      constexpr int j = decltype(jj)::value;
      zrow[j] = zz[slot<Q>(j)];
    });
  } else {
    auto pairFix = [&](auto kk, c32& zk, c32& zhk) __attribute__((always_inline)) {
      constexpr int k = decltype(kk)::value;
      const c32 a = zrow[k], bb = zrow[H - k];
      const c32 e = c32{a.x + bb.x, a.y - bb.y};
      const c32 d = c32{a.x - bb.x, a.y + bb.y};
      const c32 o = mulRoot<N, k, false>(d);
      zk = c32{e.x - o.y, e.y + o.x};
      zhk = c32{e.x + o.y, o.x - e.y};
    };
    if (g == 0) {
      const float f0 = zrow[0].x, fh = zrow[H].x;
      zz[0] = c32{f0 + fh, f0 - fh};
      staticFor<Q / 2 - 1>([&](auto mm) {
        constexpr int k = 2 * (decltype(mm)::value + 1);  // 2, 4, ..., H/2 - 2
        pairFix(std::integral_constant<int, k>{}, zz[k / 2], zz[(H - k) / 2]);
      });
      const c32 a = zrow[H / 2];
      zz[Q / 2] = c32{2.0f * a.x, -2.0f * a.y};
    } else {
      staticFor<Q / 2>([&](auto mm) {
        constexpr int k = 2 * decltype(mm)::value + 1;    // 1, 3, ..., H/2 - 1
        pairFix(std::integral_constant<int, k>{}, zz[(k - 1) / 2], zz[(H - k - 1) / 2]);
      });
    }
    regFFT<Q, false>(zz);
    if (g == 1) {
      staticFor<Q>([&](auto jj) {
        constexpr int j = decltype(jj)::value;
        zz[slot<Q>(j)] = mulRoot<H, j, false>(zz[slot<Q>(j)]);
      });
    }
    __syncthreads();  // both lanes of a row have read it
    // E as floats [0, H) of the row, w^j O as floats [H, N)
    staticFor<Q>([&](auto jj) {
      constexpr int j = decltype(jj)::value;
      reinterpret_cast<c32*>(frow + H * g)[j] = zz[slot<Q>(j)];
    });
  }
  __syncthreads();

  // ---- rows out, 16 bytes per store ----
  float4* dst = reinterpret_cast<float4*>(real + (size_t)b0 * N);
  for (int q = t; q < rows * (N / 4); q += THREADS) {
    const int r = q / (N / 4), c4 = q % (N / 4);
    const float* base = reinterpret_cast<const float*>(lds + r * RS);
    float4 o;
    if constexpr (G == 1) {
      o = float4{base[4 * c4], base[4 * c4 + 1], base[4 * c4 + 2], base[4 * c4 + 3]};
    } else {
      const int f = (4 * c4) % H;
      const float sg = 4 * c4 < H ? 1.0f : -1.0f;
      o = float4{base[f] + sg * base[H + f], base[f + 1] + sg * base[H + f + 1],
                 base[f + 2] + sg * base[H + f + 2], base[f + 3] + sg * base[H + f + 3]};
    }
    streamStore(dst + q, o);
  }
}

// ---- N = 256 with contiguous, 16-byte aligned operands ----
//
// A wave transforms eight rows by itself, eight lanes each, as 128 = 16 x 8 points: lane l
// loads z[l + 8 m] straight into registers and runs 16 points over m, the wave exchanges through
// LDS, and lane p runs the two 8-point transforms of k mod 16 = p and 16 - p (lane 0: 0 and 8),
// which hold both halves of every fix-up pair (k, 128 - k).  The inverse runs backwards.
// What bounds it is HBM.  Four waves of a workgroup share a table of roots and nothing else, and
// 35 KB of LDS leave room for 16 waves per CU that load, compute and store on their own.  Four
// lanes per row with the rows in LDS, two workgroups of 66 KB per CU in three phases each, took (us,
// forward / inverse, before -> this) 98.1 / 90.5 -> 83.6 / 86.7 on 262144 rows (6.5 and 6.2 TB/s),
// 7.9 / 7.9 -> 4.9 / 5.3 on 8192 and 7.3 / 7.2 -> 4.2 / 4.4 on 687, one chain of instructions each.
constexpr int kWaveRows = 8, kRowBins = 129;

struct Rows256 {
  int wave, lane, p, row;  // p: lane of the row
  int second;              // the second k mod 16 of this lane; the first one is p
  int rest;                // k of pair i < 4 is p + 16 i, of the others rest + 16 i
};

__device__ __forceinline__ Rows256 rows256(int t) {
  Rows256 c;
  c.wave = __builtin_amdgcn_readfirstlane(t / 64);
  c.lane = t % 64;
  c.p = c.lane % 8;
  c.row = c.lane / 8;
  c.second = c.p ? 16 - c.p : 8;
  c.rest = c.p ? c.p : -56;
  return c;
}

// value l of class k (mod 16) of a row, between the two steps: no two lanes of a bank
__device__ __forceinline__ int exchangeAt(const Rows256& c, int k, int l) {
  return k * 64 + c.row * 8 + (l ^ (k & 7));
}

__device__ __forceinline__ c32 choose(bool first, c32 a, c32 b) {
  return c32{first ? a.x : b.x, first ? a.y : b.y};
}

__global__ __launch_bounds__(k1dThreads, 4) void fft1d256Forward(const float* __restrict__ real,
                                                                 float* __restrict__ cplx, int B) {
  __shared__ __align__(16) c32 lds[k1dThreads / 64][kWaveRows * kRowBins];
  __shared__ __align__(8) c32 tw[256];
  const Rows256 c = rows256(threadIdx.x);
  const int first = (blockIdx.x * (k1dThreads / 64) + c.wave) * kWaveRows;
  const int rows = min(kWaveRows, B - first);
  const c32* const src = reinterpret_cast<const c32*>(real) + (size_t)min(first + c.row, B - 1) * 128 + c.p;
  c32 v[16];
  staticFor<16>([&](auto mm) {
    constexpr int m = decltype(mm)::value;
    v[m] = src[8 * m];
  });
  fillTwiddles<true>(tw, threadIdx.x, k1dThreads);
  __syncthreads();
  if (rows <= 0) return;

  regFFT<16, true>(v);
  c32* const buf = lds[c.wave];
  staticFor<16>([&](auto kk) {
    constexpr int k = decltype(kk)::value;
    c32 a = v[slot<16>(k)];
    if constexpr (k > 0) a = cmul(a, tw[2 * k * c.p]);
    buf[exchangeAt(c, k, c.p)] = a;
  });
  waveExchange();
  c32 u[8], w[8];
  staticFor<8>([&](auto jj) {
    constexpr int j = decltype(jj)::value;
    u[j] = buf[exchangeAt(c, c.p, j)];
    w[j] = buf[exchangeAt(c, c.second, j)];
  });
  waveExchange();
  regFFT<8, true>(u);
  regFFT<8, true>(w);

  // F[k] and F[128 - k] from Z[k], Z[128 - k], the halvings on the root and the final multiply-adds
  c32* const out = buf + c.row * kRowBins;
  const bool lane0 = c.p == 0;
  staticFor<8>([&](auto ii) {
    constexpr int i = decltype(ii)::value;
    c32 a = u[slot<8>(i)], b = w[slot<8>(7 - i)];
    if constexpr (i < 4) {
      b = choose(lane0, u[slot<8>((8 - i) % 8)], b);
    } else {
      a = choose(lane0, w[slot<8>(i - 4)], a);
      b = choose(lane0, w[slot<8>(11 - i)], b);
    }
    const int k0 = i < 4 ? c.p : c.rest;
    const c32 e2 = c32{a.x + b.x, a.y - b.y};
    const c32 root = tw[(k0 + 16 * i) & 255];
    const c32 t = cmul(c32{a.y + b.y, b.x - a.x}, c32{0.5f * root.x, 0.5f * root.y});
    c32 f = c32{__builtin_fmaf(0.5f, e2.x, t.x), __builtin_fmaf(0.5f, e2.y, t.y)};
    c32 fh = c32{__builtin_fmaf(0.5f, e2.x, -t.x), __builtin_fmaf(-0.5f, e2.y, t.y)};
    if constexpr (i == 0) {  // F[0] and F[128] are real, whatever Z[0] is, and overflow only with their own sums
      f = choose(lane0, c32{a.x + a.y, 0.0f}, f);
      fh = choose(lane0, c32{a.x - a.y, 0.0f}, fh);
    }
    out[k0 + 16 * i] = f;
    out[128 - k0 - 16 * i] = fh;
  });
  if (lane0) out[64] = cconj(u[slot<8>(4)]);
  waveExchange();

  // the rows of the wave are one stream in LDS and in HBM
  const int total = rows * kRowBins;
  float4* const dst = reinterpret_cast<float4*>(cplx + (size_t)first * 2 * kRowBins);
  const float4* const l4 = reinterpret_cast<const float4*>(buf);
  for (int q = c.lane; q < total / 2; q += 64) streamStore(dst + q, l4[q]);
  if ((total & 1) && c.lane == 0)
    reinterpret_cast<float2*>(cplx + (size_t)first * 2 * kRowBins)[total - 1] = buf[total - 1];
}

__global__ __launch_bounds__(k1dThreads, 4) void fft1d256Inverse(const float* __restrict__ cplx,
                                                                 float* __restrict__ real, int B) {
  __shared__ __align__(16) c32 lds[k1dThreads / 64][kWaveRows * kRowBins];
  __shared__ __align__(8) c32 tw[256];
  const Rows256 c = rows256(threadIdx.x);
  const int first = (blockIdx.x * (k1dThreads / 64) + c.wave) * kWaveRows;
  const int rows = min(kWaveRows, B - first);
  c32* const buf = lds[c.wave];
  if (rows > 0) {
    const int total = rows * kRowBins;
    const float4* const src = reinterpret_cast<const float4*>(cplx + (size_t)first * 2 * kRowBins);
    constexpr int LOADS = (kWaveRows * kRowBins / 2 + 63) / 64;
    float in[4 * LOADS];  // plain floats: always promoted to registers
    staticFor<LOADS>([&](auto ii) {
      constexpr int i = decltype(ii)::value;
      const float4 f = src[min(c.lane + 64 * i, total / 2 - 1)];
      in[4 * i] = f.x;
      in[4 * i + 1] = f.y;
      in[4 * i + 2] = f.z;
      in[4 * i + 3] = f.w;
    });
    float4* const l4 = reinterpret_cast<float4*>(buf);
    staticFor<LOADS>([&](auto ii) {
      constexpr int i = decltype(ii)::value;
      const int q = c.lane + 64 * i;
      if (q < total / 2) l4[q] = float4{in[4 * i], in[4 * i + 1], in[4 * i + 2], in[4 * i + 3]};
    });
    if ((total & 1) && c.lane == 0)
      buf[total - 1] = reinterpret_cast<const float2*>(cplx + (size_t)first * 2 * kRowBins)[total - 1];
  }
  fillTwiddles<false>(tw, threadIdx.x, k1dThreads);
  __syncthreads();
  if (rows <= 0) return;

  // Z[k] and Z[128 - k] from F[k], F[128 - k] (gain 2); rows behind the last one are what LDS held
  const c32* const from = buf + c.row * kRowBins;
  const bool lane0 = c.p == 0;
  c32 zk[8], zh[8];
  staticFor<8>([&](auto ii) {
    constexpr int i = decltype(ii)::value;
    const int k0 = i < 4 ? c.p : c.rest;
    c32 a = from[k0 + 16 * i], b = from[128 - k0 - 16 * i];
    if constexpr (i == 0) {  // only the real parts of F[0] and F[128] reach a real result
      a.y = lane0 ? 0.0f : a.y;
      b.y = lane0 ? 0.0f : b.y;
    }
    const c32 e = c32{a.x + b.x, a.y - b.y};
    const c32 o = cmul(c32{a.x - b.x, a.y + b.y}, tw[(k0 + 16 * i) & 255]);
    zk[i] = c32{e.x - o.y, e.y + o.x};
    zh[i] = c32{e.x + o.y, o.x - e.y};
    if constexpr (i == 0) zk[0] = choose(lane0, c32{a.x + b.x, a.x - b.x}, zk[0]);  // (no products with zeros)
  });
  const c32 middle = from[64];
  waveExchange();
  c32 u[8], w[8];
  staticFor<8>([&](auto jj) {
    constexpr int j = decltype(jj)::value;
    if constexpr (j < 4)
      u[j] = zk[j];
    else if constexpr (j == 4)
      u[j] = choose(lane0, c32{2.0f * middle.x, -2.0f * middle.y}, zk[j]);
    else
      u[j] = choose(lane0, zh[8 - j], zk[j]);
    w[j] = choose(lane0, j < 4 ? zk[(j + 4) % 8] : zh[(11 - j) % 8], zh[7 - j]);
  });
  regFFT<8, false>(u);
  regFFT<8, false>(w);
  staticFor<8>([&](auto ll) {
    constexpr int l = decltype(ll)::value;
    c32 a = u[slot<8>(l)], b = w[slot<8>(l)];
    if constexpr (l > 0) {
      a = choose(lane0, a, cmul(a, tw[2 * l * c.p]));  // an infinite F[0] or F[128] stays one in every sample
      b = cmul(b, tw[2 * l * c.second]);
    }
    buf[exchangeAt(c, c.p, l)] = a;
    buf[exchangeAt(c, c.second, l)] = b;
  });
  waveExchange();
  c32 z[16];
  staticFor<16>([&](auto kk) {
    constexpr int k = decltype(kk)::value;
    z[k] = buf[exchangeAt(c, k, c.p)];
  });
  waveExchange();
  regFFT<16, false>(z);
  // z[p + 8 m]; the rows' 16-byte words are permuted so that no bank holds two rows' columns
  staticFor<16>([&](auto mm) {
    constexpr int m = decltype(mm)::value;
    buf[c.row * 128 + 8 * (m ^ c.row) + c.p] = z[slot<16>(m)];
  });
  waveExchange();
  float4* const dst = reinterpret_cast<float4*>(real + (size_t)first * 256);
  const float4* const l4 = reinterpret_cast<const float4*>(buf);
  staticFor<kWaveRows>([&](auto rr) {
    constexpr int r = decltype(rr)::value;
    if (r < rows) streamStore(dst + r * 64 + c.lane, l4[r * 64 + (c.lane ^ (4 * r))]);
  });
}

template <int N>
int launch1d(bool forward, const Row1D& a, bool fast, hipStream_t s) {
  dim3 grid(ceilDiv(a.B, Cfg1D<N>::ROWS)), block(k1dThreads);
  if (forward) {
    if (fast)
      fft1dForward<N, true><<<grid, block, 0, s>>>(a);
    else
      fft1dForward<N, false><<<grid, block, 0, s>>>(a);
  } else {
    if (fast)
      fft1dInverse<N, true><<<grid, block, 0, s>>>(a);
    else
      fft1dInverse<N, false><<<grid, block, 0, s>>>(a);
  }
  return launchStatus();
}

}  // namespace

int launchFft1d(bool forward, int N, float* real, int sb, int sx, float* cplx, int cb, int ck,
                int B, int padL, hipStream_t s) {
  if (B <= 0) return FBFFT_SUCCESS;
  Row1D a{real, sb, sx, cplx, cb, ck, B, padL};
  const bool fast = padL == 0 && sx == 1 && sb % 2 == 0 && aligned(real, 8);
  if (N >= 8 && padL == 0 && sx == 1 && sb == N && ck == 2 && cb == N + 2 && aligned(real, 16) &&
      aligned(cplx, 16)) {
    auto mid = [&](auto n, auto threads) {
      constexpr int NN = decltype(n)::value, TT = decltype(threads)::value;
      const dim3 grid(ceilDiv(B, CfgMid<NN, TT>::ROWS)), block(TT);
      if (forward)
        fft1dMidForward<NN, TT><<<grid, block, 0, s>>>(real, cplx, B);
      else
        fft1dMidInverse<NN, TT><<<grid, block, 0, s>>>(cplx, real, B);
    };
    // Workgroups of one wave up to 64 points: rows of 64, both transforms, us with 256 lanes / 64: 600 rows
    // 9.1 / 8.0, 32768 10.8 / 9.5, 131072 24.9 / 22.0, 1048576 197 / 187; of 32, 4096 6.0 / 5.4 (in a graph; 7.1
    // launched one by one either way); 8 and 16 points 0.93 to 1.0.  At 128 points a wave takes one half of its
    // rows' transforms, so two waves are the fewest, while 256 lanes leave CUs idle: 600 rows 10.9 / 10.0,
    // 28000 15.9 / 13.1, 40000 18.6 / 18.3, but 50000 20.3 / 21.9, 65536 23.3 / 25.3.
    const std::integral_constant<int, 64> oneWave;
    switch (N) {
      case 8: mid(std::integral_constant<int, 8>{}, oneWave); break;
      case 16: mid(std::integral_constant<int, 16>{}, oneWave); break;
      case 32: mid(std::integral_constant<int, 32>{}, oneWave); break;
      case 64: {
        // (9 waves per CU; forward, a round of them, 147456 rows, to 1.8, 256 lanes / 64: 160000 14.6 / 15.3, 200000 15.9 / 17.2, 262000 20.2 /
        // 20.8, but 140000 13.5 / 10.3, 275000 22.7 / 21.5)
        const long waves = ceilDiv(B, 64), round = 9L * computeUnits();
        if (forward && waves > round && 5 * waves <= 9 * round)
          mid(std::integral_constant<int, 64>{}, std::integral_constant<int, 256>{});
        else
          mid(std::integral_constant<int, 64>{}, oneWave);
        break;
      }
      case 128:
        if (ceilDiv(B, 128) <= computeUnits())
          mid(std::integral_constant<int, 128>{}, std::integral_constant<int, 128>{});
        else
          mid(std::integral_constant<int, 128>{}, std::integral_constant<int, 256>{});
        break;
      case 256: {
        const dim3 grid(ceilDiv(B, kWaveRows * (k1dThreads / 64))), block(k1dThreads);
        if (forward)
          fft1d256Forward<<<grid, block, 0, s>>>(real, cplx, B);
        else
          fft1d256Inverse<<<grid, block, 0, s>>>(cplx, real, B);
      }
    }
    return launchStatus();
  }
  switch (N) {
    case 2: return launch1d<2>(forward, a, fast, s);
    case 4: return launch1d<4>(forward, a, fast, s);
    case 8: return launch1d<8>(forward, a, fast, s);
    case 16: return launch1d<16>(forward, a, fast, s);
    case 32: return launch1d<32>(forward, a, fast, s);
    case 64: return launch1d<64>(forward, a, fast, s);
    case 128: return launch1d<128>(forward, a, fast, s);
    case 256: return launch1d<256>(forward, a, fast, s);
  }
  return FBFFT_UNSUPPORTED_SIZE;
}

}  // namespace fbfft_amd
