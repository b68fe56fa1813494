// Fused tiled FFT convolution: FFT -> multiply-accumulate -> IFFT in one kernel
// with no device scratch (replaces updateOutputIteratedKernel*,
// updateGradInputIteratedKernel* and accGradParametersIteratedKernel*,
// fbfft/FFTIteratedConvolution.cuh:97-570, and the entry points at :624-755).
//
// All three passes are one scheme: planes "A_a" and "W_w" are transformed for
// each step of a reduction and acc[a][w] += A_a (x) W_w is accumulated per
// frequency bin, then every acc plane is inverse-transformed and cropped into
// its destination window.
//
//   pass             step       A_a               W_w               acc -> destination
//   updateOutput     cin        ins[t](n_a, c)    weight(f_w, c)    a * conj(w) -> outs[t](n_a, f_w) / N^2
//   updateGradInput  cout       outs[t](n_a, f)   weight(f, c_w)    a * w       -> ins[t](n_a, c_w)  / N^2
//   accGradParams    tile, n    ins[t](n, c_a)    outs[t](n, f_w)   a * conj(w) -> weight(f_w, c_a) * scale / N^2
//
// updateOutput and updateGradInput run one workgroup per (A group, W group).
// accGradParameters reduces over all tiles and images; its reduction is also cut
// into ranges that separate workgroups accumulate and add atomically into the
// zeroed weight gradient, so that the chip is filled.
//
// The reference gives every (batch, plane) pair its own lanes and recomputes
// both forward transforms for each of them.  Here a 512-lane workgroup owns
// BN x FO products (8 x 8 for N = 32, 16 x 16 for N = 16, 32 x 32 for N = 8) and
// takes two reduction steps per iteration: its 1024/N plane slots hold the BN + FO
// forward transforms of both steps, so every lane transforms in every iteration
// and 2 (BN + FO) transforms feed 2 BN FO products (one transform per 4, 8, 16
// products).  A planes of passes 0 and 1 are the (image, tile) pairs of the call, whatever
// the batch: a workgroup's A planes come from several tiles when the batch is small.
//
// The products run on the matrix cores: v_mfma_f32_4x4x1 multiplies sixteen independent
// 4 x 4 blocks, one block per frequency bin, so a wave accumulates 4 A planes x 4 W planes
// of sixteen neighbouring bins per instruction, four instructions per complex product,
// and the bins cost no vector arithmetic (which the transforms need all of).  Spectra pass
// through LDS once; the 64 complex accumulators of a lane stay in registers across the
// whole reduction.  Spectral rows 0 and N/2 of a real plane are Hermitian along x: after
// the row pass they become N "virtual bins" in the place of packed row 0 (x: row 0 at x,
// N/2 + x: row N/2 at x, and at 0 and N/2 the pairs of real values of each row), which
// multiply like any other bin except for the two pairs, whose lanes drop the cross terms
// by a zero factor.
#include "common.h"

#include <algorithm>
#include "fft2d_core.h"
#include "fft_regs.h"

namespace fbfft_amd {
namespace {

constexpr int kThreads = 512;
typedef float floatx4 __attribute__((ext_vector_type(4)));

struct ConvArgs {
  const fbfft_tile* ins;
  const fbfft_tile* outs;
  float* weight;
  int ws[4];  // weight strides (floats)
  int wn[4];  // weight sizes: Cout, Cin, kH, kW
  int batch;
  int numTiles;
  int splits;  // accGradParameters: workgroups sharing one reduction
  int aGroups, wGroups;  // workgroups of this launch along A and W planes
  int firstA, firstW;    // its first A and W plane; passes 0, 1: A planes count from ...
  int image0;            // ... tile 0 of this image
  int aPlanes;           // passes 0, 1: A planes per workgroup, at most BN
  float scale;
};

// workgroups of one launch: a grid counts its lanes along x in 32 bits, and every XCD takes
// the same number of workgroups
constexpr long kMaxWorkgroups = 0xffffffffL / kThreads / 8 * 8;

struct PlaneRef {
  float* p;
  int sy, sx, h, w, padL, padU;
  bool valid;
};

__device__ __forceinline__ PlaneRef tilePlane(const fbfft_tile& t, int n, int c, int batch) {
  PlaneRef r;
  r.valid = n < batch && n < t.size[0] && c < t.size[1];
  // the plane pointer comes out of a descriptor in memory: say that it is device memory,
  // or every access through it is a flat instruction
  typedef __attribute__((address_space(1))) float* GlobalPtr;
  r.p = (float*)(GlobalPtr)(t.data + (size_t)n * t.stride[0] + (size_t)c * t.stride[1]);
  r.sy = t.stride[2];
  r.sx = t.stride[3];
  r.h = t.size[2];
  r.w = t.size[3];
  r.padL = t.padL;
  r.padU = t.padU;
  return r;
}

__device__ __forceinline__ PlaneRef weightPlane(const ConvArgs& a, int f, int c) {
  PlaneRef r;
  r.valid = f < a.wn[0] && c < a.wn[1];
  r.p = a.weight + (size_t)f * a.ws[0] + (size_t)c * a.ws[1];
  r.sy = a.ws[2];
  r.sx = a.ws[3];
  r.h = a.wn[2];
  r.w = a.wn[3];
  r.padL = 0;
  r.padU = 0;
  return r;
}

template <int N>
struct ConvCfg {
  static constexpr int H = N / 2;
  static constexpr int T = N / 2;                  // lanes per plane transform
  static constexpr int SLOTS = kThreads / T;       // concurrent plane transforms
  static constexpr int SPI = 2;                    // reduction steps per iteration
  static constexpr int FO = SLOTS / (2 * SPI);     // W planes per workgroup
  static constexpr int BN = FO;                    // A planes per workgroup
  static constexpr int RA = SLOTS / FO;            // A planes per round of inverse transforms
  static constexpr int RS = PlaneCfg<N>::RS;
  // packed plane in LDS (complex), padded so that the product loop's reads - half a wave
  // takes 8 bins (64 bytes) of four planes at once - meet 64 different banks
  static constexpr int PSZ = (H * RS + 23) / 32 * 32 + 8;
  static constexpr int PB = H * N;                 // bins per plane
  static constexpr int BLOCKS = PB / 16;           // groups of 16 bins, one per MFMA block
  static constexpr int WAVES = kThreads / 64;
  static constexpr int NBW = BLOCKS >= WAVES ? BLOCKS / WAVES : 1;  // bin groups per wave
  static constexpr int SHARE = BLOCKS >= WAVES ? 1 : WAVES / BLOCKS;  // waves sharing a bin group
  static constexpr int AB = BN / 4 / SHARE;        // blocks of 4 A planes per wave
  static constexpr int WB = FO / 4;                // blocks of 4 W planes per wave
  static_assert(PSZ >= H * RS && PSZ % 32 == 8, "plane stride");
  static_assert(NBW * AB * WB == 16, "64 complex accumulators per lane");
  static_assert(SPI * BN * T == kThreads / 2, "one half of the waves transforms A planes");
  static_assert(RA == 4, "a round of inverse transforms takes one block of A planes");
};

// Makes LDS writes of the whole workgroup visible to it.  Only LDS is fenced: global loads
// in flight (the next iteration's planes) stay in flight.
__device__ __forceinline__ void ldsBarrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// How the planes of one wave are fetched.  Their windows usually lie in one tensor: then a
// row's address is a scalar base (step and row) plus a lane's 32-bit offset that never
// changes, and a load costs no vector arithmetic.
template <int N>
struct WaveLoader {
  // Whole: every window covers the whole transform plane.  Pairs, Singles: the windows cover
  // the same rows (scalar tests), a lane's two columns as one 8-byte word or as two loads.
  // Ragged: rows differ from plane to plane.  Scattered: so do strides, or the planes lie
  // too far apart.
  enum Mode { Empty, Whole, Pairs, Singles, Ragged, Scattered };
  const char* base;  // of the wave, lowered so that every lane's offset is positive
  int rowBytes;
  unsigned off;      // of the lane's first column in row 0 of its transform plane
  int mode, first, last;  // the same for the whole wave; Pairs, Singles: rows [first, last)
  // rows [lo, lo + rows) of the lane's two columns lie in the window; three bytes, because
  // registers are what this kernel is shortest of
  unsigned window;

  __device__ __forceinline__ unsigned lo() const { return window & 255u; }
  __device__ __forceinline__ unsigned rowsA() const { return window >> 8 & 255u; }
  __device__ __forceinline__ unsigned rowsB() const { return window >> 16; }

  // ref: the lane's plane, valid or not
  __device__ __forceinline__ void plan(const PlaneRef& ref, int l) {
    const int xa = 2 * l - ref.padL;
    const bool va = ref.valid && (unsigned)xa < (unsigned)ref.w;
    const bool vb = ref.valid && (unsigned)(xa + 1) < (unsigned)ref.w;
    const unsigned rows = min(max(ref.h, 0), N);
    window = min((unsigned)ref.padU, (unsigned)N) | (va ? rows << 8 : 0u) | (vb ? rows << 16 : 0u);
    // the first lane with a plane sets the base
    const unsigned long long have = __builtin_amdgcn_ballot_w64(ref.valid && ref.h > 0 && ref.w > 0);
    mode = Empty;
    if (have == 0) return;
    const int lead = __builtin_ctzll(have);
    const unsigned long long p = (unsigned long long)ref.p;
    const unsigned long long p0 =
        (unsigned long long)(unsigned)__builtin_amdgcn_readlane((int)(unsigned)p, lead) |
        (unsigned long long)(unsigned)__builtin_amdgcn_readlane((int)(unsigned)(p >> 32), lead) << 32;
    const int sy = __builtin_amdgcn_readlane(ref.sy, lead);
    rowBytes = sy * (int)sizeof(float);
    // a window starts at most N rows and N columns inside its plane
    const long lower = ((long)(sy < 0 ? 0 : sy) * N + N) * (long)sizeof(float);
    const long rel = (long)(p - p0) + lower + ((long)xa - (long)ref.padU * sy) * (long)sizeof(float);
    base = (const char*)p0 - lower;
    off = (unsigned)rel;
    const bool here = (va || vb) && ref.h > 0;
    const bool near = ref.sx == 1 && ref.sy == sy && sy >= 0 && sy < (1 << 22) && rel >= 0 &&
                      rel < (1L << 31) - 8 && ref.padU >= 0 && ref.padU <= N;
    const unsigned lead1 = __builtin_amdgcn_readlane((int)(rows << 8 | lo()), lead);
    first = lead1 & 255u;
    last = min(first + (int)(lead1 >> 8), N);
    // rows on 8-byte boundaries, even left edge and width: the lane's two columns are one
    // 8-byte word per row, inside or outside the window together
    const bool pairs = ((sy | ref.padL | ref.w) & 1) == 0 && (p & 7) == 0;
    const bool whole = window == ((unsigned)N << 8 | (unsigned)N << 16);
    mode = __builtin_amdgcn_ballot_w64(here && !near) != 0 ? Scattered
           : __builtin_amdgcn_ballot_w64(here && (rows << 8 | lo()) != lead1) != 0 ? Ragged
           : __builtin_amdgcn_ballot_w64(here && !pairs) != 0 ? Singles
           : __builtin_amdgcn_ballot_w64(!whole) != 0 ? Pairs : Whole;
  }

  // the two columns as z0[j] = (X[2j][x], X[2j+1][x]), x = 2l, and z1 the same for x = 2l + 1.
  // stepBytes: how far the wave's planes have moved since plan().
  __device__ __forceinline__ void load(long stepBytes, c32 (&z0)[N / 2], c32 (&z1)[N / 2]) const {
    typedef float Pair __attribute__((ext_vector_type(2)));
    typedef const __attribute__((address_space(1))) Pair* GlobalPair;
    typedef const __attribute__((address_space(1))) float* GlobalFloat;
    // The empty statements keep scalar base and lane offset apart up to the load, and the
    // base a running sum (left alone the compiler keeps a scalar offset per row alive across
    // the whole reduction).
    unsigned o = off;
    const char* rowBase = base + stepBytes;
    auto pin = [&]() __attribute__((always_inline)) {
      asm volatile("" : "+s"(rowBase));
      asm volatile("" : "+v"(o));
    };
    auto set = [](c32& z, int odd, float v) __attribute__((always_inline)) { (odd ? z.y : z.x) = v; };
    if (mode == Whole) {
      staticFor<N>([&](auto yy) {
        constexpr int y = decltype(yy)::value;
        pin();
        const Pair v = *(GlobalPair)(rowBase + o);
        rowBase += rowBytes;
        set(z0[y / 2], y % 2, v.x);
        set(z1[y / 2], y % 2, v.y);
      });
    } else {
      staticFor<N / 2>([&](auto jj) {
        z0[decltype(jj)::value] = z1[decltype(jj)::value] = c32{0.0f, 0.0f};
      });
      if (mode == Pairs) {
        if (rowsA() != 0) {
          staticFor<N>([&](auto yy) {
            constexpr int y = decltype(yy)::value;
            pin();
            if (y >= first && y < last) {
              const Pair v = *(GlobalPair)(rowBase + o);
              set(z0[y / 2], y % 2, v.x);
              set(z1[y / 2], y % 2, v.y);
            }
            rowBase += rowBytes;
          });
        }
      } else if (mode == Singles) {
        const char* const rowBase0 = rowBase;
        if (rowsA() != 0) {
          staticFor<N>([&](auto yy) {
            constexpr int y = decltype(yy)::value;
            pin();
            if (y >= first && y < last) set(z0[y / 2], y % 2, *(GlobalFloat)(rowBase + o));
            rowBase += rowBytes;
          });
        }
        rowBase = rowBase0 + sizeof(float);
        if (rowsB() != 0) {
          staticFor<N>([&](auto yy) {
            constexpr int y = decltype(yy)::value;
            pin();
            if (y >= first && y < last) set(z1[y / 2], y % 2, *(GlobalFloat)(rowBase + o));
            rowBase += rowBytes;
          });
        }
      } else if (mode == Ragged) {
        const unsigned lo = this->lo(), rowsA = this->rowsA(), rowsB = this->rowsB();
        staticFor<N>([&](auto yy) {
          constexpr int y = decltype(yy)::value;
          pin();
          GlobalFloat p = (GlobalFloat)(rowBase + o);
          if (y - lo < rowsA) set(z0[y / 2], y % 2, p[0]);
          if (y - lo < rowsB) set(z1[y / 2], y % 2, p[1]);
          rowBase += rowBytes;
        });
      }
    }
  }

  // mode Scattered: every lane its own pointer and strides
  __device__ __forceinline__ void loadScattered(const PlaneRef& ref, int l, c32 (&z0)[N / 2],
                                                c32 (&z1)[N / 2]) const {
    typedef const __attribute__((address_space(1))) float* GlobalFloat;
    const int xa = 2 * l - ref.padL;
    const bool va = ref.valid && (unsigned)xa < (unsigned)ref.w;
    const bool vb = ref.valid && (unsigned)(xa + 1) < (unsigned)ref.w;
    GlobalFloat p = (GlobalFloat)(ref.p + (long)xa * ref.sx - (long)ref.padU * ref.sy);
    staticFor<N>([&](auto yy) {
      constexpr int y = decltype(yy)::value;
      const bool vy = (unsigned)(y - ref.padU) < (unsigned)ref.h;
      float a = 0.0f, b = 0.0f;
      if (vy && va) a = p[0];
      if (vy && vb) b = p[ref.sx];
      (y % 2 ? z0[y / 2].y : z0[y / 2].x) = a;
      (y % 2 ? z1[y / 2].y : z1[y / 2].x) = b;
      p += ref.sy;
    });
  }
};

template <int N, int PASS>
__global__ __launch_bounds__(kThreads) void iteratedConvKernel(ConvArgs a) {
  using C = ConvCfg<N>;
  constexpr int H = C::H, T = C::T, SLOTS = C::SLOTS, FO = C::FO, BN = C::BN, RS = C::RS,
                PSZ = C::PSZ, SPI = C::SPI, RA = C::RA, NBW = C::NBW, AB = C::AB, WB = C::WB;
  static_assert((BN + FO) * SPI == SLOTS && BN % RA == 0, "slot layout");
  constexpr bool CONJ = (PASS != 1);
  __shared__ __align__(16) c32 lds[SLOTS * PSZ];

  const int t = threadIdx.x;
  const int s = t / T, l = t % T;
  const int wave = __builtin_amdgcn_readfirstlane(t / 64);
  const int lane = t % 64;

  const int Cout = a.wn[0], Cin = a.wn[1];
  const int steps = PASS == 0 ? Cin : PASS == 1 ? Cout : a.numTiles * a.batch;
  // Passes 0, 1: one workgroup per (A group, W group).  Pass 2: the reduction is also cut
  // into a.splits ranges whose results meet in an atomic add.  Workgroups are dealt
  // round-robin to the 8 XCDs; every XCD takes a contiguous range of logical ids, W groups
  // fastest, so that the workgroups that transform the same A planes share an L2.
  const int total = a.splits * a.aGroups * a.wGroups;
  const int per = (total + 7) / 8;
  const int logical = (blockIdx.x % 8) * per + blockIdx.x / 8;
  if (logical >= total) return;
  const int w0 = a.firstW + logical % a.wGroups * FO;              // first W plane
  const int aPlanes = PASS == 2 ? BN : a.aPlanes;
  const int a0 = a.firstA + logical / a.wGroups % a.aGroups * aPlanes;  // first A plane
  const int perSplit = PASS == 2 ? ((steps + a.splits - 1) / a.splits + SPI - 1) / SPI * SPI : steps;
  const int stepBegin = PASS == 2 ? logical / (a.wGroups * a.aGroups) * perSplit : 0;
  const int stepEnd = min(steps, stepBegin + perSplit);

  // acc[bin group][block of A][block of W]: lane (b, j) of a wave holds, at bin b of the
  // group, W plane j of the block and its four A planes
  floatx4 accR[NBW][AB][WB], accI[NBW][AB][WB];
#pragma unroll
  for (int n = 0; n < NBW; ++n)
#pragma unroll
    for (int i = 0; i < AB; ++i)
#pragma unroll
      for (int j = 0; j < WB; ++j) accR[n][i][j] = accI[n][i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

  c32* plane = lds + s * PSZ;
  // Slots: A planes of every step first, then W planes, so that each SIMD's two waves are
  // one of either kind.  Slot s transforms plane sj of reduction step SPI * it + su.
  const bool isA = s < SPI * BN;
  const int su = isA ? s / BN : (s - SPI * BN) / FO, sj = isA ? s % BN : (s - SPI * BN) % FO;
  // (su is the same for the planes of a wave)
  const int suw = __builtin_amdgcn_readfirstlane(su);
  // Passes 0 and 1: the wave's planes move by one stride from step to step, and how they are
  // fetched is planned once.  (Planes whose strides differ - tiles of several tensors - are
  // planned again at every step, like the tiles of pass 2.)
  WaveLoader<N> loader;
  auto planeAt = [&](int step, bool isA, int sj) __attribute__((always_inline)) {
    if (PASS == 2) {
      // past the last step the tile index is clamped; the plane is marked absent
      const int tl = __builtin_amdgcn_readfirstlane(min(step / a.batch, a.numTiles - 1)), n = step % a.batch;
      return isA ? tilePlane(a.ins[tl], n, a0 + sj, a.batch) : tilePlane(a.outs[tl], n, w0 + sj, a.batch);
    }
    if (isA) {
      const int row = a0 + sj;
      const fbfft_tile& d = (PASS == 0 ? a.ins : a.outs)[row % a.numTiles];
      return tilePlane(d, a.image0 + row / a.numTiles, step, a.batch);
    }
    return PASS == 0 ? weightPlane(a, w0 + sj, step) : weightPlane(a, step, w0 + sj);
  };
  long stride = 0;       // floats from step to step
  int planned = 0;       // steps [0, planned) of the wave's planes follow the plan
  if (PASS != 2) {
    int mine = PASS == 0 ? a.ws[1] : a.ws[0], held = steps;
    if (isA) {
      const fbfft_tile& d = (PASS == 0 ? a.ins : a.outs)[(a0 + sj) % a.numTiles];
      mine = d.stride[1];
      held = d.size[1];
    }
    const int stride0 = __builtin_amdgcn_readfirstlane(mine);
    const bool same = __builtin_amdgcn_ballot_w64(mine != stride0 || held < steps) == 0;
    loader.plan(planeAt(0, isA, sj), l);
    stride = stride0;
    // (an odd stride moves the planes off their 8-byte boundaries)
    if (same && loader.mode != WaveLoader<N>::Scattered &&
        (loader.mode == WaveLoader<N>::Singles || loader.mode == WaveLoader<N>::Ragged || stride0 % 2 == 0))
      planned = steps;
  }
  c32 z0[H], z1[H];
  auto load = [&](int it) __attribute__((always_inline)) {
    const int step = SPI * it + suw;
    long stepBytes = (long)step * stride * (long)sizeof(float);
    // the lane's plane where the plan does not cover the step; past the last step nothing is
    // there.  (The lane's place is worked out afresh: nothing of this stays in registers.)
    auto unplanned = [&](int& column) __attribute__((always_inline)) {
      int tt = t;
      asm volatile("" : "+v"(tt));
      const int s2 = tt / T;
      const bool isA2 = s2 < SPI * BN;
      column = tt % T;
      PlaneRef ref = planeAt(step, isA2, (isA2 ? s2 : s2 - SPI * BN) % BN);
      ref.valid = ref.valid && step < stepEnd;
      return ref;
    };
    int column;
    if (step >= planned) {
      const PlaneRef ref = unplanned(column);
      loader.plan(ref, column);
      stepBytes = 0;
    }
    // (one chain of branches with no early exit: every path sets all of z0 and z1, and the
    // compiler sees that they need no registers before)
    if (loader.mode == WaveLoader<N>::Scattered) {
      const PlaneRef ref = unplanned(column);
      loader.loadScattered(ref, column, z0, z1);
    } else {
      loader.load(stepBytes, z0, z1);
    }
  };

  // product loop: lane (b, j) supplies plane j of a block of four at bin b of a group
  const int b16 = lane / 4, j4 = lane % 4;
  const int group0 = C::SHARE == 1 ? wave * NBW : wave % C::BLOCKS;  // first bin group
  const int aBlock0 = C::SHARE == 1 ? 0 : wave / C::BLOCKS * AB;     // first block of A planes
  const int bin0 = 16 * group0 + b16;
  const int laneBin = bin0 / N * RS + bin0 % N;   // where the lane's bin sits in a plane
  // ... and bin group n of the wave relative to it (more than one group only at N = 32)
  auto groupOff = [](int n) { return n / 2 * RS + n % 2 * 16; };
  static_assert(NBW == 1 || N == 32, "bin groups of a wave");
  // the bins of real pairs: 0 and N/2 (at N = 32: the first bin of groups 0 and 1)
  const bool pair = bin0 == 0 || (N < 32 && bin0 == H);
  const float keep = pair ? 0.f : 1.f;

  const int itBegin = stepBegin / SPI, itEnd = (stepEnd + SPI - 1) / SPI;
  // (one more turn ahead of the first iteration, which only fetches)
  for (int it = itBegin - 1; it < itEnd; ++it) {
    if (it >= itBegin) {
      // ---- forward transforms of this iteration's A and W planes ----
      __builtin_amdgcn_s_setprio(0);
      {
        c32 p0[H], p1[H];
        columnTransformForward<N>(z0, z1, p0, p1);
        ldsBarrier();  // the spectra of the previous iteration are consumed by everybody
        storeColumns<N>(p0, p1, plane, l);
      }
      waveExchange();
      rowPassInPlace<N, true>(plane, l);
      waveExchange();
      {  // packed row 0, P[x] = F0[x] + i FH[x], to its virtual bins
        const c32 p = plane[l], m = plane[l == 0 ? H : N - l];
        waveExchange();
        plane[l] = l == 0 ? c32{p.x, m.x} : c32{0.5f * (p.x + m.x), 0.5f * (p.y - m.y)};
        plane[H + l] = l == 0 ? c32{p.y, m.y} : c32{0.5f * (p.y + m.y), 0.5f * (m.x - p.x)};
      }
      ldsBarrier();
    }
    // On every SIMD the W wave takes its products first and goes on to its next transforms
    // while the A wave multiplies: vector and matrix instructions of the two overlap instead
    // of taking turns (16 x 32 x 256 x 256 image, 32 filters of 9 x 9: 555 -> 480 us; the
    // A wave first 510 us, the W wave first throughout 475 us forward but 520 us for the
    // weight gradient).
    if (wave >= C::WAVES / 2) __builtin_amdgcn_s_setprio(3);
    // the next iteration's planes travel under this iteration's products
    load(it + 1);
    __builtin_amdgcn_sched_barrier(0);
    if (it < itBegin) continue;

    // ---- acc[a][w] += A_a (x) W_w ----
    // a * conj(w) or a * w as re += ar wr +- ai wi, im += ai wr -+ ar wi; the bins of real
    // pairs take (ar wr, ai wi): the cross terms' A is zeroed, the second product takes wi
    // Operands are read one bin group ahead of the instructions that take them; the barriers
    // keep the compiler from reading all of them first, which spills.
    struct Operands {
      c32 a[AB], w[WB];
    };
    // (two base addresses and constant offsets: the compiler's own choice is an address per
    // read, kept alive across the reduction)
    typedef const __attribute__((address_space(3))) vfloat2* LdsPair;
    LdsPair baseA = (LdsPair)(lds + (4 * aBlock0 + j4) * PSZ + laneBin);
    LdsPair baseW = (LdsPair)(lds + (SPI * BN + j4) * PSZ + laneBin);
    asm volatile("" : "+v"(baseA), "+v"(baseW));
    auto read = [&](auto gg) __attribute__((always_inline)) {
      constexpr int u = decltype(gg)::value / NBW, n = decltype(gg)::value % NBW;
      Operands o;
#pragma unroll
      for (int i = 0; i < AB; ++i) {
        const vfloat2 v = baseA[(u * BN + 4 * i) * PSZ + groupOff(n)];
        o.a[i] = c32{v.x, v.y};
      }
#pragma unroll
      for (int j = 0; j < WB; ++j) {
        const vfloat2 v = baseW[(u * FO + 4 * j) * PSZ + groupOff(n)];
        o.w[j] = c32{v.x, v.y};
      }
      return o;
    };
    Operands ops[2];
    ops[0] = read(std::integral_constant<int, 0>{});
    staticFor<SPI * NBW>([&](auto gg) {
      constexpr int g = decltype(gg)::value, n = g % NBW;
      if constexpr (g + 1 < SPI * NBW) ops[(g + 1) % 2] = read(std::integral_constant<int, g + 1>{});
      __builtin_amdgcn_sched_barrier(0);
      const Operands& o = ops[g % 2];
      constexpr bool mayPair = n < 2;
      const float cross = mayPair ? keep : 1.f;
      // (first products of every accumulator, then second ones: no instruction waits for the
      // one before it)
#pragma unroll
      for (int i = 0; i < AB; ++i)
#pragma unroll
        for (int j = 0; j < WB; ++j) {
          accR[n][i][j] = __builtin_amdgcn_mfma_f32_4x4x1f32(o.a[i].x, o.w[j].x, accR[n][i][j], 0, 0, 0);
          accI[n][i][j] = __builtin_amdgcn_mfma_f32_4x4x1f32(o.a[i].y, mayPair && pair ? o.w[j].y : o.w[j].x, accI[n][i][j], 0, 0, 0);
        }
#pragma unroll
      for (int i = 0; i < AB; ++i) {
        const float ai = (CONJ ? cross : -cross) * o.a[i].y, ar = (CONJ ? -cross : cross) * o.a[i].x;
#pragma unroll
        for (int j = 0; j < WB; ++j) {
          accR[n][i][j] = __builtin_amdgcn_mfma_f32_4x4x1f32(ai, o.w[j].y, accR[n][i][j], 0, 0, 0);
          accI[n][i][j] = __builtin_amdgcn_mfma_f32_4x4x1f32(ar, o.w[j].y, accI[n][i][j], 0, 0, 0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    });
  }

  // ---- inverse transforms, RA = 4 A planes (one block) x FO W planes per round ----
  const float norm = (PASS == 2 ? a.scale : 1.0f) / (float)(N * N);
  // (the lane's place is worked out afresh, so that nothing of it occupies registers above)
  int te = t;
  asm volatile("" : "+v"(te));
  const int se = te / T, le = te % T, je = te % 4, be = te % 64 / 4;
  c32* planeE = lds + se * PSZ;
  const int binE = 16 * group0 + be, laneBinE = binE / N * RS + binE % N;
#pragma unroll
  for (int rd = 0; rd < BN / RA; ++rd) {
    if (RA * rd >= aPlanes) break;
    ldsBarrier();
    if (C::SHARE == 1 || aBlock0 / AB == rd / AB) {
#pragma unroll
      for (int n = 0; n < NBW; ++n)
#pragma unroll
        for (int j = 0; j < WB; ++j)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            lds[(i * FO + 4 * j + je) * PSZ + laneBinE + groupOff(n)] =
                c32{accR[n][rd % AB][j][i], accI[n][rd % AB][j][i]};
    }
    ldsBarrier();
    {  // virtual bins back to the packed row: Q[x] = S0[x] + i SH[x], Q[N-x] = conj(S0[x]) +
       // i conj(SH[x]); lane 0 sorts the four real values into Q[0] and Q[N/2]
      const c32 c0 = planeE[le], cH = planeE[H + le];
      c32 q = c32{c0.x - cH.y, c0.y + cH.x}, qm = c32{c0.x + cH.y, cH.x - c0.y};
      if (le == 0) {
        q = c32{c0.x, cH.x};
        qm = c32{c0.y, cH.y};
      }
      waveExchange();
      planeE[le] = q;
      planeE[le == 0 ? H : N - le] = qm;
    }
    waveExchange();
    rowPassInPlace<N, false>(planeE, le);
    waveExchange();
    {
      columnPassInverse<N>(planeE, le, z0, z1);
      const int ai = a0 + RA * rd + se / FO;
      const int wi = w0 + se % FO;
      PlaneRef ref;
      if (PASS == 2) {
        ref = weightPlane(a, wi, ai);
      } else {
        const fbfft_tile& d = PASS == 0 ? a.outs[ai % a.numTiles] : a.ins[ai % a.numTiles];
        ref = tilePlane(d, a.image0 + ai / a.numTiles, wi, a.batch);
        ref.valid = ref.valid && wi < (PASS == 0 ? Cout : Cin) && RA * rd + se / FO < aPlanes;
      }
      if (ref.valid) {
        if (PASS == 2 && a.splits > 1)
          storeColumnsWindow<N, true, true>(ref.p, ref.sy, ref.sx, ref.h, ref.w, ref.padL, ref.padU,
                                            le, z0, z1, norm);
        else
          storeColumnsWindow<N>(ref.p, ref.sy, ref.sx, ref.h, ref.w, ref.padL, ref.padU, le, z0, z1,
                                norm);
      }
    }
  }
}

// weight[f][c][y][x] = 0 through its strides (a fill kernel, so that the call
// stays capturable in a graph)
__global__ void zeroWeight(ConvArgs a) {
  const long total = (long)a.wn[0] * a.wn[1] * a.wn[2] * a.wn[3];
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (long)gridDim.x * blockDim.x) {
    long r = i;
    const int x = r % a.wn[3];
    r /= a.wn[3];
    const int y = r % a.wn[2];
    r /= a.wn[2];
    const int c = r % a.wn[1];
    const int f = r / a.wn[1];
    a.weight[(long)f * a.ws[0] + (long)c * a.ws[1] + (long)y * a.ws[2] + (long)x * a.ws[3]] = 0.0f;
  }
}

template <int N>
int launchPass(int pass, ConvArgs a, bool deterministic, hipStream_t s) {
  using C = ConvCfg<N>;
  const int Cout = a.wn[0], Cin = a.wn[1];
  const long rows = (long)a.numTiles * a.batch;  // (image, tile) pairs
  const long wGroups = ceilDiv(pass == FBFFT_UPDATE_GRAD_INPUT ? Cin : Cout, C::FO);
  // Passes 0 and 1 over a few pairs leave most of the CUs idle when every workgroup takes BN of
  // them; with a short reduction the first loads, the inverse transforms and the stores are most
  // of a workgroup's time, and that is spread over the CUs instead (one workgroup per CU: 256
  // VGPRs).  Slots beyond aPlanes transform the next workgroup's planes and drop the result.
  // BN planes / spread, us: 3 x 1 x 24 x 32, 21 filters of 2 x 2, 8 points 23.9 / 8.8 (one
  // workgroup per tile 21.8); 2 x 4 x 72 x 80, 17 of 7 x 7, 32 points, every other column 36.6 /
  // 26.8 (31.4).  In a longer reduction the iterations are the time, and more workgroups only
  // transform more: 10 x 81 x 113 x 110, 20 of 5 x 5, 32 points 263 / 306.  Around the line, 32
  // points: 18 steps 94 / 85 (1 x 15 x 148 x 148, input gradient of 18 filters of 6 x 6), 20
  // steps 78 / 83 (3 x 20 x 97 x 98, 53 of 11 x 11), 23 steps 89 / 97.
  a.aPlanes = C::BN;
  const int steps = pass == FBFFT_UPDATE_OUTPUT ? Cin : Cout;
  if (pass != FBFFT_ACC_GRAD_PARAMETERS && steps <= 18) {
    const long groups = std::max(1L, computeUnits() / wGroups);
    a.aPlanes = (int)std::min<long>(C::BN, (rows + groups - 1) / groups);
    // ... where that leaves out a round of inverse transforms (5 of 8 planes and both rounds,
    // 79 x 8 x 111 x 108, input gradient of 8 filters of 5 x 5: 44.6 / 48.7)
    if (ceilDiv(a.aPlanes, C::RA) * C::RA == C::BN) a.aPlanes = C::BN;
  }
  const long aGroups = pass == FBFFT_ACC_GRAD_PARAMETERS ? ceilDiv(Cin, C::BN) : (rows + a.aPlanes - 1) / a.aPlanes;
  if (pass == FBFFT_ACC_GRAD_PARAMETERS) {
    // The reference runs one block per group of planes over the whole reduction
    // (fbfft/FFTIteratedConvolution.cuh:600-613).  With 256 CUs that leaves most of the
    // chip idle, so the reduction is also split until there are about two
    // workgroups per CU; the partial gradients are then added atomically into a
    // zeroed weight tensor (summation order, hence the last bits, vary from run to
    // run).  A single split stores directly.
    // deterministic: the reference's schedule, one workgroup per plane group over the
    // whole reduction in a fixed order, no atomics (and most of the chip idle)
    const long groups = aGroups * wGroups;
    a.splits = deterministic
                   ? 1
                   : (int)std::max(1L, std::min((512 + groups - 1) / groups, (rows + 2 * C::SPI - 1) / (2 * C::SPI)));
    // Ranges hold whole iterations, so the last of them can be empty: those are not launched.
    // (The ranges of an XCD are neighbours, and empty ones would all fall to the last XCD while
    // the first takes a third round of workgroups: 34 x 29 x 35 x 35 images, 37 filters of 4 x 4,
    // 26 ranges of which 23 hold something, 110.7 us with all of them launched, 77.4 us without.)
    const long range = ((rows + a.splits - 1) / a.splits + C::SPI - 1) / C::SPI * C::SPI;
    a.splits = (int)((rows + range - 1) / range);
    if (a.splits > 1) {
      const long total = (long)a.wn[0] * a.wn[1] * a.wn[2] * a.wn[3];
      zeroWeight<<<dim3((unsigned)std::min<long>((total + 255) / 256, 4096)), 256, 0, s>>>(a);
    }
  }
  // one launch, unless its grid would be too large (more than one split has no such number
  // of plane groups); then ranges of W groups and, below those, of A groups
  const long wStep = std::min(wGroups, kMaxWorkgroups);
  const long aStep = std::min(aGroups, kMaxWorkgroups / (wStep * a.splits));
  for (long w = 0; w < wGroups; w += wStep) {
    for (long g = 0; g < aGroups; g += aStep) {
      a.wGroups = (int)std::min(wStep, wGroups - w);
      a.aGroups = (int)std::min(aStep, aGroups - g);
      a.firstW = (int)(w * C::FO);
      const long firstA = g * a.aPlanes;
      a.firstA = (int)(pass == FBFFT_ACC_GRAD_PARAMETERS ? firstA : firstA % a.numTiles);
      a.image0 = (int)(pass == FBFFT_ACC_GRAD_PARAMETERS ? 0 : firstA / a.numTiles);
      const long total = (long)a.splits * a.aGroups * a.wGroups;
      const dim3 grid((unsigned)((total + 7) / 8 * 8));
      if (pass == FBFFT_UPDATE_OUTPUT)
        iteratedConvKernel<N, 0><<<grid, kThreads, 0, s>>>(a);
      else if (pass == FBFFT_UPDATE_GRAD_INPUT)
        iteratedConvKernel<N, 1><<<grid, kThreads, 0, s>>>(a);
      else
        iteratedConvKernel<N, 2><<<grid, kThreads, 0, s>>>(a);
      const int rc = launchStatus();
      if (rc != FBFFT_SUCCESS) return rc;
    }
  }
  return FBFFT_SUCCESS;
}

}  // namespace

// returns 1 launched, 0 nothing matched, -FBFFT_HIP_ERROR on launch failure
int launchIteratedConv(int N, const fbfft_tile* ins, const fbfft_tile* outs, float* weight,
                       const int* wStride, const int* wSize, int pass, float scale, int batch,
                       size_t numTiles, bool deterministic, hipStream_t s) {
  if (!(N == 8 || N == 16 || N == 32)) return 0;
  if (pass < 0 || pass > 2) return 0;
  ConvArgs a;
  a.ins = ins;
  a.outs = outs;
  a.weight = weight;
  for (int d = 0; d < 4; ++d) {
    a.ws[d] = wStride[d];
    a.wn[d] = wSize[d];
  }
  a.batch = batch;
  a.numTiles = (int)numTiles;
  a.splits = 1;
  a.scale = scale;
  if (batch <= 0 || numTiles == 0 || wSize[0] <= 0 || wSize[1] <= 0) return 1;  // nothing to do
  // The kernels count a reduction over (tile, image) pairs, and the tiles and the pairs of one
  // launch (kMaxWorkgroups groups of up to 32), in 32 bits.  A weight gradient over more pairs
  // than that came out as zeros.
  if (numTiles > (pass == FBFFT_ACC_GRAD_PARAMETERS ? 0x7fff0000u / (unsigned)batch : 1u << 30)) return 0;
  int rc = N == 8    ? launchPass<8>(pass, a, deterministic, s)
           : N == 16 ? launchPass<16>(pass, a, deterministic, s)
                     : launchPass<32>(pass, a, deterministic, s);
  return rc == FBFFT_SUCCESS ? 1 : -rc;
}

}  // namespace fbfft_amd
