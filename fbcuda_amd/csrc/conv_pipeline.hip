// The three passes of an FFT convolution layer (valid cross-correlation forward,
// its gradient with respect to the input, its gradient with respect to the
// weights), each as three kernels that hand spectra to each other in a layout
// chosen for the matrix cores.
//
// The reference's external callers run fbfft2D -> transposeMM -> fbifft2D on
// plane-major spectra [plane][bin] (MM-inl.cuh:188-196), which makes the
// frequency bin - the batch index of the contraction - the innermost dimension
// and caps the contraction's tile size (accumulators are needed for every bin of
// a cache line at once).  Here the spectra never take that shape:
//
//   1. forwardBinMajor:  planes -> S[bin][k][row]   (row = image / output plane)
//      a 256-lane workgroup transforms SLOTS = 512/N planes with consecutive
//      `row` and the same k and writes each bin as one contiguous run.
//   2. binGemmDirect:    C[bin][i][j] = sum_k A[bin][k][i] * conj(B[bin][k][j])
//      one workgroup = one bin x (128 x 64) or (64 x 64) tile; k-slices of A and B
//      are contiguous in HBM and are copied verbatim into LDS by global_load_lds;
//      4 waves of MFMA 32x32x2 sub-tiles, three real products per complex one;
//      counters show A + B fetched
//      from HBM exactly once (the tiles of a bin share an L2: workgroup ids are
//      remapped per XCD) and C written once with coalesced stores.
//      binGemmSplit: the same product on the bf16 matrix instructions, fp32 operands
//      split into three bf16 values each.
//      binGemmRegsWide / binGemmRegsNarrow / binGemmRegsSplitK: the same product without LDS for
//      products with a side of up to 32 (planGemm picks kernel, tiles and the
//      ranges a long reduction is cut into).
//   3. inverseBinMajor:  C[bin][i][j] -> planes, gathering runs of SLOTS
//      consecutive j per bin, inverse transform, crop on store.
//
// The planes of an operand are a PlaneSet: whole tensors, overlapping windows of
// images larger than the transform (the layer entry points), or the tile
// descriptors of FFTIteratedConvolution in device memory (fbfft_iterated_conv_ws).
//
// Spectral rows 0 and N/2 of a real plane are both Hermitian along kx, so their
// 2 N complex values carry N complex worth of information; they travel as N
// "virtual bins": v = x (0 < x < N/2) is row 0 at x, v = N/2 + x is row N/2 at x, and
// v = 0 / v = N/2 hold the four real values (row 0 at 0 and N/2) / (row N/2 at 0 and
// N/2) as (re, im) pairs.  The contraction is then a plain complex GEMM on N^2/2 bins;
// only the two bins of real pairs multiply component by component instead (the product
// rule of fbfft/FFTIteratedConvolution.cuh:161-186 with the unpacking done once, when
// the forward transform stores the spectrum).
//
// All three passes are the same product P[i][j] = sum_k X[i][k] * op(Y[j][k]) with
// the roles of MM-inl.cuh:188-196: forward (i, j, k) = (image, output plane, input
// plane), op = conj; input gradient (image, input plane, output plane), op =
// identity; weight gradient (input plane, output plane, image), op = conj.  The
// kernels always compute sum_k A * conj(B); the forward transforms store a
// spectrum conjugated where the pass needs it.
//
// Figures below name two layers: the 27 x 27 layer, 128 x 64 x 27 x 27 images and 192 filters
// of 5 x 5, and the 256 x 256 layer, 16 x 32 x 256 x 256 images and 32 filters of 9 x 9.
#include "common.h"
#include "fft2d_core.h"
#include "fft_regs.h"

#include <algorithm>
#include <cmath>
#include <utility>

namespace fbfft_amd {
namespace {

constexpr int kT = 256;
// lanes of a transform workgroup: 16 planes of 32 x 32, so that a bin leaves or arrives as
// a 128-byte run (measured at the 27 x 27 / the 256 x 256 layer: 128 lanes, 64-byte runs,
// +10 % / +12 % per pass; 512 lanes, one workgroup per CU, +8 % / +6 %)
constexpr int kTF = 256;
typedef float floatx16 __attribute__((ext_vector_type(16)));

template <int N>
struct BMCfg {
  static constexpr int H = N / 2;
  static constexpr int T = N / 2;
  static constexpr int SLOTS = kTF / T;                // planes per workgroup
  static constexpr int RS = PlaneCfg<N>::RS;
  // plane stride in LDS (complex): 16-byte aligned, and 4 banks mod 32 so that the
  // transposed accesses (16 or more planes at the same bin) spread over the banks
  static constexpr int PSZ = (H + 1) * RS;
  static_assert((2 * PSZ) % 32 == 4 && PSZ % 2 == 0, "plane stride");
  static constexpr int BINS = H * N;      // N virtual bins of rows 0 and N/2, then rows 1 .. N/2-1
};

// A family of planes indexed by (row, k).  Plain: plane (row, k) is the h x w window at
// base + row*sRow + k*sK.  Tiled (images larger than the transform): one of the two
// indices is the composite (image, tileY, tileX), image-major; its stride is the
// image stride, h x w is the whole image, and tile (ty, tx) is the winH x winW
// window at (orgY + ty*stepY, orgX + tx*stepX) clipped to the image - rows and
// columns clipped off above / left become the plane's padU / padL, so the window
// keeps its place inside the FFT plane.  padU0 / padL0 shift every window further
// (where a cropped result sits inside the inverse transform's plane).  Described
// (FFTIteratedConvolution's interface, fbfft/FFTIteratedConvolution.cuh:71-88): one of
// the two indices is the composite (image, tile), image-major, and every tile is a
// descriptor in device memory - a [batch][planes][h][w] view with its own strides and
// pads; the other index is the plane within the view.
struct PlaneSet {
  float* base;
  long sRow, sK;
  int sy, sx, h, w;
  int R, K;         // valid rows / k
  int tiled;        // 0: plain, 1: row is the composite index, 2: k is
  int tilesY, tilesX, stepY, stepX, orgY, orgX, winH, winW;
  int padU0, padL0;
  const fbfft_tile* tiles;  // described sets: the descriptors
  int described;            // 0: no, 1: row is the composite (image, tile), 2: k is
  int numTiles;             // tiles per image
};

struct PlaneWindow {
  float* p;
  int h, w, padL, padU;
  int sy, sx;
  bool valid;  // described sets: the view holds this image and plane and is not empty
};

// DESCRIBED is a compile-time fact (the kernels' PAIRS == 2 instantiations): carried as a
// run-time test it cost the tiled sets 2 % (the 256 x 256 layer: 290 against 284 us).
template <bool DESCRIBED>
__device__ __forceinline__ PlaneWindow planeWindow(const PlaneSet& ps, int row, int k) {
  if constexpr (DESCRIBED) {
    const int comp = ps.described == 1 ? row : k, other = ps.described == 1 ? k : row;
    // image-major: consecutive composites are consecutive tiles of one image - in a
    // row-major tiling neighbours in memory, which is what 16 planes of a workgroup should
    // be (tile-major, 16 images of one tile: 345 instead of 296 us at the 256 x 256 layer)
    const fbfft_tile& d = ps.tiles[comp % ps.numTiles];
    const int n = comp / ps.numTiles;
    PlaneWindow win;
    win.valid = n < d.size[0] && other < d.size[1] && d.size[2] > 0 && d.size[3] > 0;
    // a plane the view does not hold takes the place of one it does, and loads nothing
    // (no row passes the window test, and with padU = 0 no batch of rows is asked for)
    typedef __attribute__((address_space(1))) float* GlobalPtr;
    win.p = (float*)(GlobalPtr)(d.data + (long)min(n, max(d.size[0] - 1, 0)) * d.stride[0] +
                                (long)min(other, max(d.size[1] - 1, 0)) * d.stride[1]);
    win.h = max(d.size[2], 0);
    win.w = max(d.size[3], 0);
    win.padU = win.valid ? d.padU : 0;
    win.padL = d.padL;
    win.sy = d.stride[2];
    win.sx = d.stride[3];
    return win;
  }
  if (ps.tiled == 0)
    return PlaneWindow{ps.base + (long)row * ps.sRow + (long)k * ps.sK, ps.h, ps.w, ps.padL0,
                       ps.padU0, ps.sy, ps.sx, true};
  const int comp = ps.tiled == 1 ? row : k, other = ps.tiled == 1 ? k : row;
  const long sImg = ps.tiled == 1 ? ps.sRow : ps.sK, sOther = ps.tiled == 1 ? ps.sK : ps.sRow;
  const int perImage = ps.tilesY * ps.tilesX;
  const int img = comp / perImage, t = comp % perImage;
  const int y0 = ps.orgY + (t / ps.tilesX) * ps.stepY, x0 = ps.orgX + (t % ps.tilesX) * ps.stepX;
  const int ya = max(y0, 0), xa = max(x0, 0);
  PlaneWindow win;
  win.p = ps.base + (long)img * sImg + (long)other * sOther + (long)ya * ps.sy + (long)xa * ps.sx;
  win.h = min(y0 + ps.winH, ps.h) - ya;
  win.w = min(x0 + ps.winW, ps.w) - xa;
  win.padU = ps.padU0 + ya - y0;
  win.padL = ps.padL0 + xa - x0;
  win.sy = ps.sy;
  win.sx = ps.sx;
  win.valid = true;
  return win;
}

// ---- 1. planes -> S[bin][k][row] ----
// One operand of the product: its planes, where its spectra go, and how many
// workgroups (row groups x Kp) transform it.
struct ForwardJob {
  PlaneSet ps;
  float2* S;
  int Rp, Kp;
  float imSign;
  int rowGroups;  // workgroups per k: Rp / SLOTS, or half of that (rounded up) when a
                  // workgroup takes two runs of rows
  int stream;     // spectra leave with nontemporal stores
};

// Both operands of a pass in one launch: workgroups [0, a.rowGroups * a.Kp) transform
// a's planes, the rest b's.  PAIRS_x: every plane of that set passes
// windowMovesAsPairs() (8-byte words per row).  GROUPS (1 or 2): runs of SLOTS
// consecutive rows per workgroup; with two, the second run's planes are requested as
// soon as the first run's columns have left the registers and fly under the first
// run's row pass and stores.
template <int N, int PAIRS, int GROUPS>
__device__ __forceinline__ void forwardBinMajorBody(const ForwardJob& job, int wg, c32* lds);

template <int N, int PAIRS_A, int PAIRS_B, int GROUPS>
__global__ __launch_bounds__(kTF) void forwardBinMajor(ForwardJob a, ForwardJob b) {
  __shared__ __align__(16) c32 lds[BMCfg<N>::SLOTS * BMCfg<N>::PSZ];
  const int nA = a.rowGroups * a.Kp;
  if ((int)blockIdx.x < nA)
    forwardBinMajorBody<N, PAIRS_A, GROUPS>(a, blockIdx.x, lds);
  else
    forwardBinMajorBody<N, PAIRS_B, GROUPS>(b, blockIdx.x - nA, lds);
}

template <int N, int PAIRS, int GROUPS>
__device__ __forceinline__ void forwardBinMajorBody(const ForwardJob& job, int wg, c32* lds) {
  using C = BMCfg<N>;
  constexpr int H = C::H, T = C::T, SLOTS = C::SLOTS, RS = C::RS, PSZ = C::PSZ;
  const PlaneSet& ps = job.ps;
  float2* S = job.S;
  const int Rp = job.Rp, Kp = job.Kp;
  const float imSign = job.imSign;
  const int t = threadIdx.x;
  const int s = t / T, l = t % T;
  const int k = wg / job.rowGroups;
  c32* plane = lds + s * PSZ;

  auto load = [&](int r0, c32 (&z0)[H], c32 (&z1)[H]) __attribute__((always_inline)) {
    // padding planes (row >= R, k >= K) take the window of an existing plane and load nothing
    const int row = r0 + s;
    const PlaneWindow win = planeWindow<PAIRS == 2>(ps, min(row, ps.R - 1), min(k, ps.K - 1));
    const bool present = row < ps.R && k < ps.K && win.valid;
    // 4-byte loads (odd widths or strides): the lane takes columns l and l + N/2, so that
    // a load instruction reads neighbouring floats (the 27 x 27 layer: input gradient 108.0 ->
    // 101.6 us, weight gradient 108.0 -> 104.1 us; forward pass unchanged).  PAIRS = 2
    // (described sets: the windows are only known on the device) decides per plane
    // between 8-byte and 4-byte loads of columns 2l and 2l + 1.
    loadColumnsWindow<N, PAIRS, PAIRS == 0>(win.p, win.sy, win.sx, win.h, win.w, win.padL, win.padU,
                                            l, z0, z1, present);
  };
  // lanes: sp = t % SLOTS walks the run (consecutive rows), bq = t / SLOTS in [0, T)
  // walks bins: lane (sp, bq) stores columns x = bq and bq + T of every spectral row,
  // so LDS and HBM offsets are compile-time constants on top of one per-lane base.
  auto copyOutAs = [&](int r0, auto streamTag) __attribute__((always_inline)) {
    const int sp = t % SLOTS, bq = t / SLOTS;
    const c32* src = lds + sp * PSZ + bq;
    const long binStride = (long)Kp * Rp;
    float2* dst = S + (long)k * Rp + r0 + sp + bq * binStride;
    auto put = [&](int bin, c32 v) __attribute__((always_inline)) {
      if constexpr (decltype(streamTag)::value)
        streamStore(dst + bin * binStride, v);
      else
        dst[bin * binStride] = v;
    };
    // Packed row 0 holds P[x] = F0[x] + i FH[x]: F0[x] = (P[x] + conj P[N-x]) / 2,
    // FH[x] = (P[x] - conj P[N-x]) / 2i.  Lane bq stores virtual bins bq (F0) and
    // T + bq (FH); bq = 0 stores the real pairs (F0[0], F0[N/2]) and (FH[0], FH[N/2]),
    // which no conjugation touches.
    {
      const c32 a = src[0], m = lds[sp * PSZ + (bq == 0 ? H : N - bq)];
      c32 f0 = c32{0.5f * (a.x + m.x), 0.5f * (a.y - m.y) * imSign};
      c32 fh = c32{0.5f * (a.y + m.y), 0.5f * (m.x - a.x) * imSign};
      if (bq == 0) {
        f0 = c32{a.x, m.x};
        fh = c32{a.y, m.y};
      }
      put(0, f0);
      put(T, fh);
    }
    staticFor<H - 1>([&](auto rr) {
      constexpr int r = decltype(rr)::value + 1;
      const c32 u = src[r * RS], v = src[r * RS + T];
      put(r * N, c32{u.x, u.y * imSign});
      put(r * N + T, c32{v.x, v.y * imSign});
    });
  };
  // Spectra larger than the last-level cache can hold until the contraction reads them
  // leave with the nontemporal hint (job.stream, the same for the whole launch): the
  // weight gradient of a 16 x 32 x 256 x 256 layer in 1936 windows (2 x 254 MB of spectra)
  // 310 -> 269 us; spectra that do fit (84 MB for 128 x 64 x 27 x 27 * 192 x 64 x 5 x 5)
  // lose 2-7 % with it, because the contraction then fetches them from HBM.
  auto copyOut = [&](int r0) __attribute__((always_inline)) {
    if (job.stream)
      copyOutAs(r0, std::true_type{});
    else
      copyOutAs(r0, std::false_type{});
  };

  const int ra = (wg % job.rowGroups) * GROUPS * SLOTS;
  c32 za0[H], za1[H];
  load(ra, za0, za1);
  columnPassForward<N, PAIRS == 0>(za0, za1, plane, l);
  waveExchange();  // the lanes of a plane sit in one wave
  if constexpr (GROUPS == 2) {
    const int rb = ra + SLOTS;
    const bool second = rb < Rp;  // the same for the whole workgroup
    c32 zb0[H], zb1[H];
    if (second) load(rb, zb0, zb1);
    rowPassInPlace<N, true>(plane, l);
    __syncthreads();
    copyOut(ra);
    if (second) {
      __syncthreads();  // every wave has copied the first run out of the plane buffers
      columnPassForward<N, PAIRS == 0>(zb0, zb1, plane, l);
      waveExchange();
      rowPassInPlace<N, true>(plane, l);
      __syncthreads();
      copyOut(rb);
    }
  } else {
    rowPassInPlace<N, true>(plane, l);
    __syncthreads();
    copyOut(ra);
  }
}

// ---- 3. C[bin][i][j] -> planes (i, j), cropped ----
// A workgroup takes GROUPS (1 or 2) runs of SLOTS consecutive j of one i.  With two, the
// second run's spectra are requested as soon as the first run's have been parked in
// LDS, and fly under the first run's transforms and stores.
template <int N, bool ACC, int GROUPS, int PAIRS>
__global__ __launch_bounds__(kTF) void inverseBinMajor(const float2* Cs, int I, int Jp, PlaneSet out,
                                                       float scale, int splits, long splitStride,
                                                       int runGroups) {
  using C = BMCfg<N>;
  constexpr int H = C::H, T = C::T, SLOTS = C::SLOTS, RS = C::RS, PSZ = C::PSZ;
  constexpr int PER = C::BINS / T;
  static_assert(C::BINS % T == 0, "bins divide evenly over the lane groups");
  __shared__ __align__(16) c32 lds[SLOTS * PSZ];
  const int t = threadIdx.x;
  const int s = t / T, l = t % T;
  // one grid index for (i, group of runs), runs fastest: a batch on i may exceed what a
  // second grid dimension can count
  const int i = blockIdx.x / runGroups, runGroup = blockIdx.x % runGroups;
  const int sp = t % SLOTS, bq = t / SLOTS;
  const long binStride = (long)I * Jp;
  c32* plane = lds + s * PSZ;

  // gather: every load of a run is issued before its first LDS store
  auto request = [&](int j0, c32 (&in)[PER]) __attribute__((always_inline)) {
    const float2* src = Cs + (long)i * Jp + j0 + sp;
    staticFor<PER>([&](auto uu) {
      constexpr int u = decltype(uu)::value;
      in[u] = src[(bq + T * u) * binStride];
    });
    // partial products of a reduction cut into ranges: added in range order
    for (int sp2 = 1; sp2 < splits; ++sp2) {
      src += splitStride;
      staticFor<PER>([&](auto uu) {
        constexpr int u = decltype(uu)::value;
        const c32 v = src[(bq + T * u) * binStride];
        in[u].x += v.x;
        in[u].y += v.y;
      });
    }
  };
  auto park = [&](const c32 (&in)[PER]) __attribute__((always_inline)) {
    c32* dstp = lds + sp * PSZ;
    staticFor<PER>([&](auto uu) {
      constexpr int u = decltype(uu)::value;  // bin = bq + T*u: row u/2, column bq + T*(u%2)
      dstp[(u / 2) * RS + T * (u % 2) + bq] = in[u];
    });
  };
  auto transformAndStore = [&](int j0) __attribute__((always_inline)) {
    // where the result goes: asked for up front, so that a described set's descriptor
    // (device memory) arrives under the transforms instead of ahead of the stores
    const int j = j0 + s;
    const PlaneWindow win = planeWindow<PAIRS == 2>(out, i, min(j, out.K - 1));
    {  // virtual bins of row 0 back to the packed row: Q[x] = C0[x] + i CH[x],
       // Q[N-x] = conj(C0[x]) + i conj(CH[x]); lane 0 sorts the four real values into
       // Q[0] = (C0[0], CH[0]) and Q[N/2] = (C0[N/2], CH[N/2]).  The T lanes of a plane
       // sit in one wave: all of them have read before any of them writes.
      const c32 c0 = plane[l], cH = plane[T + l];
      c32 q = c32{c0.x - cH.y, c0.y + cH.x}, qm = c32{c0.x + cH.y, cH.x - c0.y};
      if (l == 0) {
        q = c32{c0.x, cH.x};
        qm = c32{c0.y, cH.y};
      }
      plane[l] = q;
      plane[l == 0 ? H : N - l] = qm;
    }
    waveExchange();
    rowPassInPlace<N, false>(plane, l);
    waveExchange();
    c32 z0[H], z1[H];
    // PAIRS = 0, no 8-byte stores: a lane takes columns l and l + N/2, so that each store
    // instruction writes a contiguous run per plane (the 27 x 27 layer: 102.4 -> 101.5 us).
    // PAIRS = 2 (described sets): columns 2l and 2l + 1, 8-byte or 4-byte stores decided
    // per plane.
    columnPassInverse<N, PAIRS == 0>(plane, l, z0, z1);
    // (Parking the cropped planes in LDS and writing them out as 16-byte runs - one
    // contiguous stream for dense outputs, row quads for windows of a tiled image - was
    // measured and is slower, 35.9 -> 36.6 us at the 27 x 27 layer and 112 -> 131 us at
    // the 256 x 256 layer: the kernel waits on its own chain of phases, not on store requests.
    // The dense case again with each wave parking its own four planes - one aligned run
    // of memory, no workgroup barrier - and nontemporal 16-byte stores: 106.8-108.3 us
    // per forward pass at the 27 x 27 layer against 106.7-108.2, no change.)
    if (j < out.K) {  // out.K: number of valid output planes along j
      if (win.valid) {
        if constexpr (PAIRS == 2) {
          if (windowMovesAsPairs(win.p, win.sy, win.sx, win.w, win.padL))
            storeColumnsWindow<N, ACC, false, true, false>(win.p, win.sy, win.sx, win.h, win.w,
                                                           win.padL, win.padU, l, z0, z1, scale);
          else
            storeColumnsWindow<N, ACC, false, false, false>(win.p, win.sy, win.sx, win.h, win.w,
                                                            win.padL, win.padU, l, z0, z1, scale);
        } else {
          storeColumnsWindow<N, ACC, false, PAIRS == 1, PAIRS == 0>(
              win.p, win.sy, win.sx, win.h, win.w, win.padL, win.padU, l, z0, z1, scale);
        }
      }
    }
  };

  const int ja = runGroup * GROUPS * SLOTS;
  c32 in[PER];
  request(ja, in);
  park(in);
  __syncthreads();
  if constexpr (GROUPS == 2) {
    const int jb = ja + SLOTS;
    const bool second = jb < Jp;  // the same for the whole workgroup
    if (second) request(jb, in);
    transformAndStore(ja);
    if (second) {
      __syncthreads();  // every wave has read the first run out of the plane buffers
      park(in);
      __syncthreads();
      transformAndStore(jb);
    }
  } else {
    transformAndStore(ja);
  }
}

// ---- 2. batched complex GEMM, bin-major ----
constexpr int GI = 128;

struct GemmArgs {
  const float2* A;  // [bins][Kp][Ip]
  const float2* B;  // [bins][Kp][Jp]
  float2* C;        // [bins][I][Jp]
  int bins, I, Ip, Jp, Kp;
  int IT, JT;       // tiles per bin
  int N;            // transform size: bins 0 and N/2 hold pairs of real values
  // register kernels only: the reduction is cut into `splits` ranges of slicesPerSplit
  // k-slices (blockIdx.y names the range); range s writes its partial product to
  // C + s * splitStride and the inverse kernel adds the partials in range order
  int splits, slicesPerSplit;
  long splitStride;
};

// The k-slices go from HBM straight into LDS (global_load_lds, 16 bytes per lane,
// no staging registers or LDS store instructions) through a ring of three stages:
// slice s+2 is requested before slice s is multiplied, one barrier per slice.  A
// wave instruction moves 1 KiB: one k-row of 128 complex or two k-rows of 64
// complex; LDS has exactly the HBM layout.  Requires Kp % 8 == 0 with the padding
// rows zeroed; rows / columns beyond Ip / Jp are clamped (they only feed
// accumulators that are never stored).
constexpr int GJ2 = 64, GK2 = 8;

// A wave-uniform address, pinned in scalar registers: the empty statement keeps the
// compiler from folding it into a lane's offset, so that "scalar base + 32-bit lane
// offset" reaches the memory instruction as its two operands and costs no vector
// arithmetic.
template <class T>
__device__ __forceinline__ T* scalarBase(T* p) {
  asm volatile("" : "+s"(p));
  return p;
}

// ... and a lane's 32-bit offset kept apart from it up to the instruction (otherwise its
// widening to 64 bits is hoisted and the sum becomes a vector addition per access).
// (By value: the copy costs a move per access.  Marking the long-lived register itself
// instead saves the moves and measured 1.5 us slower on the weight gradient of a
// 128 x 64 x 27 x 27 * 192 x 64 x 5 x 5 layer, the same elsewhere.)
__device__ __forceinline__ unsigned laneOffset(unsigned o) {
  asm volatile("" : "+v"(o));
  return o;
}

// plain vectors in global memory (float2's members take a generic `this`)
typedef float __attribute__((ext_vector_type(2))) PlainPair;
typedef __attribute__((address_space(1))) PlainPair GlobalPair;
typedef float __attribute__((ext_vector_type(4))) PlainQuad;
typedef __attribute__((address_space(1))) PlainQuad GlobalQuad;

__device__ __forceinline__ void loadToLds(const float2* src, float2* ldsWaveBase) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                   (__attribute__((address_space(3))) void*)ldsWaveBase, 16, 0, 0);
}

template <int TI>
struct GemmStage {
  float2 A[GK2][TI];
  float2 B[GK2][GJ2];
};

// TI = 128: wave w owns rows 32w.. and both 32-column halves of the 64 columns.
// TI = 64 (few rows, or too few 128-row tiles to balance the chip): wave w owns rows
// 32 (w % 2).. and columns 32 (w / 2)..
template <int TI>
__global__ __launch_bounds__(kT, TI == 128 ? 4 : 6) void binGemmDirect(GemmArgs g) {
  static_assert(TI == 128 || TI == 64, "tile rows");
  constexpr int NQ = TI == 128 ? 2 : 1;
  constexpr int LOADS = TI == 128 ? 3 : 2;  // global->LDS instructions per wave and slice
  using Stage = GemmStage<TI>;
  // three separate variables, not one array: the compiler tracks pending
  // global->LDS loads per LDS variable, so reading one stage does not wait for the
  // loads still in flight into the other three
  __shared__ __align__(16) Stage stage0, stage1, stage2;
  const int t = threadIdx.x;
  const int lane = t % 64;
  // the wave's number in a scalar register: everything below that depends only on it
  // (LDS destinations, row offsets of the loads and of the result) is scalar arithmetic
  const int w = __builtin_amdgcn_readfirstlane(t / 64);
  const int r = lane % 32, h = lane / 32;

  const int total = g.bins * g.IT * g.JT;
  const int per = (total + 7) / 8;
  const int logical = (blockIdx.x % 8) * per + blockIdx.x / 8;
  if (logical >= total) return;
  const int bin = logical / (g.IT * g.JT);
  const int rem = logical % (g.IT * g.JT);
  const int i0 = (rem / g.JT) * TI, j0 = (rem % g.JT) * GJ2;
  const int rb = TI == 128 ? w : w % 2;  // 32-row block of this wave
  const int cb = TI == 128 ? 0 : w / 2;  // first 32-column block of this wave
  // bins of real pairs: (ar br, ai bi) instead of a complex product; k1 and k3 hold them
  const bool pairs = bin == 0 || 2 * bin == g.N;
  const float cross = pairs ? 0.f : 1.f;

  // this workgroup's range of the reduction (blockIdx.y; no range is empty)
  const int sliceFirst = blockIdx.y * g.slicesPerSplit;
  const float2* Ab = g.A + ((long)bin * g.Kp + (long)sliceFirst * GK2) * g.Ip;
  const float2* Bb = g.B + ((long)bin * g.Kp + (long)sliceFirst * GK2) * g.Jp;
  // per-lane source columns, clamped into the padded arrays
  const int ia = min(i0 + 2 * (TI == 128 ? lane : lane % 32), g.Ip - 2);
  const int jb = min(j0 + 2 * (lane % 32), g.Jp - 2);

  // Three real products per complex product instead of four: with a = ar + i ai and
  // b = br + i bi,  a conj(b) = (k1 - k3) + i (k1 + k2)  for
  //   k1 = (ar + ai) br,  k2 = -ar (br + bi),  k3 = ai (br - bi).
  // The sums cost three VALU adds per operand pair; the matrix pipeline, which
  // bounds this kernel, does a quarter less work.
  // (Cleared by 48 moves per sub-tile.  Giving the first slice's products a constant
  // zero addend instead takes that slice out of the loop, and there the compiler waits
  // for every load in flight before the first LDS read: 101 -> 107 us on a
  // 128 x 64 x 27 x 27 * 192 x 64 x 5 x 5 forward pass.)
  floatx16 k1[NQ], k2[NQ], k3[NQ];
#pragma unroll
  for (int q = 0; q < NQ; ++q)
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      k1[q][v] = 0.f;
      k2[q][v] = 0.f;
      k3[q][v] = 0.f;
    }

  const int slices = min(g.slicesPerSplit, g.Kp / GK2 - sliceFirst);
  // wave w moves rows 2w, 2w+1 of A and rows 2w, 2w+1 of B of a slice: LOADS instructions.
  // An address is a scalar base (slice and wave) plus a lane's 32-bit byte offset that
  // never changes, so a step spends no vector instructions on addresses.
  const unsigned laneA = (unsigned)((TI == 128 ? 0 : h * g.Ip) + ia) * (unsigned)sizeof(float2);
  const unsigned laneB = (unsigned)(h * g.Jp + jb) * (unsigned)sizeof(float2);
  const char* const waveA = (const char*)(Ab + (long)(2 * w) * g.Ip);
  const char* const waveB = (const char*)(Bb + (long)(2 * w) * g.Jp);
  const long sliceA = (long)GK2 * g.Ip * sizeof(float2), sliceB = (long)GK2 * g.Jp * sizeof(float2);
  auto issue = [&](Stage& st, int sl) __attribute__((always_inline)) {
    loadToLds((const float2*)(scalarBase(waveA + sl * sliceA) + laneOffset(laneA)), &st.A[2 * w][0]);
    if constexpr (TI == 128)
      loadToLds((const float2*)(scalarBase(waveA + sl * sliceA + g.Ip * sizeof(float2)) + laneOffset(laneA)),
                &st.A[2 * w + 1][0]);
    loadToLds((const float2*)(scalarBase(waveB + sl * sliceB) + laneOffset(laneB)), &st.B[2 * w][0]);
  };

  // One slice: wait for it, let everybody see it, request the slice two ahead into
  // the stage that was multiplied last time round, multiply.  Every step issues
  // exactly LOADS loads (past the end it re-requests the last slice into a stage
  // nobody reads), so "all but the newest LOADS have landed" always means "slice sl
  // has landed" and the compiler can count the loads in flight at every LDS read.
  // (Three stages of 8 KB let six workgroups of the 64-row kernel share a CU, 74
  // registers per lane allowing it; a fourth stage with five workgroups measured 0.6 /
  // 0.8 / 2.5 us slower on the three passes of a 128 x 64 x 27 x 27 * 192 x 64 x 5 x 5
  // layer - while the kernel needed 89 registers and five workgroups were the most
  // either way, the fourth stage was the faster form by 2 us on the weight gradient.)
  auto step = [&](Stage& cur, Stage& refill, int sl) __attribute__((always_inline)) {
    __builtin_amdgcn_s_waitcnt(0x0F70 | LOADS);  // vmcnt(LOADS): all but the newest slice
    // ... and so have everybody else's, and slice sl-1 is consumed.  A bare barrier:
    // the fences of __syncthreads() would wait for every load in flight, and no wave
    // stores to LDS with anything but these loads.
    __builtin_amdgcn_s_barrier();
    issue(refill, min(sl + 2, slices - 1));
    float2 av[GK2 / 2], bv[GK2 / 2][NQ];
#pragma unroll
    for (int s2 = 0; s2 < GK2 / 2; ++s2) {
      av[s2] = cur.A[2 * s2 + h][32 * rb + r];
#pragma unroll
      for (int q = 0; q < NQ; ++q) bv[s2][q] = cur.B[2 * s2 + h][32 * (cb + q) + r];
    }
#pragma unroll
    for (int s2 = 0; s2 < GK2 / 2; ++s2) {
      const float2 a = av[s2];
      const float as = __builtin_fmaf(cross, a.y, a.x);
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        const float2 b = bv[s2][q];
        const float nbs = -b.x - b.y, bd = __builtin_fmaf(cross, b.x, -b.y);
        k1[q] = __builtin_amdgcn_mfma_f32_32x32x2f32(as, b.x, k1[q], 0, 0, 0);
        k2[q] = __builtin_amdgcn_mfma_f32_32x32x2f32(a.x, nbs, k2[q], 0, 0, 0);
        k3[q] = __builtin_amdgcn_mfma_f32_32x32x2f32(a.y, bd, k3[q], 0, 0, 0);
      }
    }
  };

  issue(stage0, 0);
  issue(stage1, min(1, slices - 1));
  int sl = 0;
  for (; sl + 3 <= slices; sl += 3) {
    step(stage0, stage2, sl);
    step(stage1, stage0, sl + 1);
    step(stage2, stage1, sl + 2);
  }
  if (sl < slices) {
    step(stage0, stage2, sl);
    if (sl + 1 < slices) step(stage1, stage0, sl + 1);
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): nothing may land in LDS after this wave is gone

  // The sums leave unscaled; the inverse transform's factor carries 1 / N^2.
  float2* Cb = g.C + blockIdx.y * g.splitStride + (long)bin * g.I * g.Jp;
  if (i0 + 32 * rb + 32 <= g.I && j0 + 32 * (cb + NQ) <= g.Jp) {
    // the wave's whole block lies inside C: a scalar base per accumulator row plus the
    // lane's fixed offset, no tests
    const unsigned laneC = (unsigned)(4 * h * g.Jp + r) * (unsigned)sizeof(float2);
    char* const waveC = (char*)(Cb + (long)(i0 + 32 * rb) * g.Jp + j0 + 32 * cb);
    const long rowC = (long)g.Jp * sizeof(float2);
    auto store = [&](auto realPairs) __attribute__((always_inline)) {
#pragma unroll
      for (int q = 0; q < NQ; ++q)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          // (global address space spelled out: behind the pinned base the compiler no
          // longer sees where the pointer came from and would store through flat addresses)
          typedef float __attribute__((ext_vector_type(2))) Pair;  // a plain vector: float2's assignment takes a generic `this`
          auto* dst = (__attribute__((address_space(1))) Pair*)(
              scalarBase(waveC + (8 * (v / 4) + v % 4) * rowC + q * 32 * (long)sizeof(float2)) +
              laneOffset(laneC));
          if constexpr (decltype(realPairs)::value)
            *dst = Pair{k1[q][v], -k3[q][v]};
          else
            *dst = Pair{k1[q][v] - k3[q][v], k1[q][v] + k2[q][v]};
        }
    };
    if (pairs)
      store(std::true_type{});
    else
      store(std::false_type{});
    return;
  }
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    const int j = j0 + 32 * (cb + q) + r;
    if (j >= g.Jp) continue;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int i = i0 + 32 * rb + 8 * (v / 4) + 4 * h + v % 4;
      if (i < g.I)
        Cb[(long)i * g.Jp + j] = pairs ? float2{k1[q][v], -k3[q][v]}
                                       : float2{k1[q][v] - k3[q][v], k1[q][v] + k2[q][v]};
    }
  }
}

// The same product with no LDS in the loop and no barriers there: a wave loads exactly
// the operand values its own MFMA lanes supply - lane (r, h) of v_mfma_f32_32x32x2_f32
// supplies row / column r at k = h, so one 8-byte load per lane fetches k-rows 2s and
// 2s+1 of 32 consecutive rows (two 256-byte runs per wave instruction).  Slices of 8 k
// ride a ring of three register sets, two in flight while one is multiplied; the
// scheduling barriers keep each slice's loads ahead of the products of the slice two
// before it (left alone the compiler sinks the loads below the products and then waits
// for all of them at the top of the loop).
template <class Slice, class Fetch, class Multiply>
__device__ __forceinline__ void ringOfThree(int first, int step, int n, Fetch fetch,
                                            Multiply multiply) {
  // slices first, first + step, ...: n of them
  if (n <= 0) return;
  Slice s0, s1, s2;
  fetch(s0, first);
  fetch(s1, first + step * min(1, n - 1));
  int sl = 0;
  for (; sl + 3 <= n; sl += 3) {
    fetch(s2, first + step * min(sl + 2, n - 1));
    __builtin_amdgcn_sched_barrier(0);
    multiply(s0);
    __builtin_amdgcn_sched_barrier(0);
    fetch(s0, first + step * min(sl + 3, n - 1));
    __builtin_amdgcn_sched_barrier(0);
    multiply(s1);
    __builtin_amdgcn_sched_barrier(0);
    fetch(s1, first + step * min(sl + 4, n - 1));
    __builtin_amdgcn_sched_barrier(0);
    multiply(s2);
    __builtin_amdgcn_sched_barrier(0);
  }
  if (sl < n) {
    multiply(s0);
    if (sl + 1 < n) multiply(s1);
  }
}

// The same with two register sets: one slice in flight while one is multiplied.
template <class Slice, class Fetch, class Multiply>
__device__ __forceinline__ void ringOfTwo(int first, int step, int n, Fetch fetch, Multiply multiply) {
  if (n <= 0) return;
  Slice s0, s1;
  fetch(s0, first);
  int sl = 0;
  for (; sl + 2 <= n; sl += 2) {
    fetch(s1, first + step * (sl + 1));
    __builtin_amdgcn_sched_barrier(0);
    multiply(s0);
    __builtin_amdgcn_sched_barrier(0);
    fetch(s0, first + step * min(sl + 2, n - 1));
    __builtin_amdgcn_sched_barrier(0);
    multiply(s1);
    __builtin_amdgcn_sched_barrier(0);
  }
  if (sl < n) multiply(s0);
}

// Both sides short (up to 32 rows and 32 columns per bin, any K - the weight gradient
// of a layer with few planes reduces over every image and window), and products too small to
// fill the chip with larger tiles (planGemm): one workgroup per 32 x 32 tile of a
// bin and range of the reduction; its four waves take every fourth k-slice each and
// wave 0 adds the four 32 x 32 partial tiles in wave order (through LDS) before it
// stores, so the result does not depend on timing.
struct GemmSlice {
  float2 a[GK2 / 2], b[GK2 / 2];
};

__global__ __launch_bounds__(kT, 4) void binGemmRegsSplitK(GemmArgs g) {
  __shared__ float red[3][48][64];
  const int t = threadIdx.x;
  // (the wave's number in a scalar register: its slices and their addresses are scalar)
  const int lane = t % 64, w = __builtin_amdgcn_readfirstlane(t / 64);
  const int r = lane % 32, h = lane / 32;
  const int total = g.bins * g.IT * g.JT;
  const int per = (total + 7) / 8;
  const int logical = (blockIdx.x % 8) * per + blockIdx.x / 8;
  if (logical >= total) return;
  const int bin = logical / (g.IT * g.JT);
  const int rem = logical % (g.IT * g.JT);
  const int i0 = rem / g.JT * 32, j0 = rem % g.JT * 32;
  const bool pairs = bin == 0 || 2 * bin == g.N;  // bins of real pairs: (ar br, ai bi)
  const float cross = pairs ? 0.f : 1.f;

  // operand columns beyond the padded arrays are clamped (they feed accumulators that
  // are never stored).  An address is a scalar base (bin, k-rows) plus the lane's fixed
  // 32-bit offset: no vector arithmetic per load.
  const unsigned laneA = (unsigned)(h * g.Ip + min(i0 + r, g.Ip - 1)) * (unsigned)sizeof(float2);
  const unsigned laneB = (unsigned)(h * g.Jp + min(j0 + r, g.Jp - 1)) * (unsigned)sizeof(float2);
  const char* const binA = (const char*)(g.A + (long)bin * g.Kp * g.Ip);
  const char* const binB = (const char*)(g.B + (long)bin * g.Kp * g.Jp);
  const long sa = 2L * g.Ip * sizeof(float2), sb = 2L * g.Jp * sizeof(float2);  // two k-rows

  floatx16 k1, k2, k3;
#pragma unroll
  for (int v = 0; v < 16; ++v) k1[v] = k2[v] = k3[v] = 0.f;

  auto fetch = [&](GemmSlice& s, int sl) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < GK2 / 2; ++u) {
      const long k2rows = (long)sl * (GK2 / 2) + u;
      const PlainPair va = *(const GlobalPair*)(scalarBase(binA + k2rows * sa) + laneOffset(laneA));
      const PlainPair vb = *(const GlobalPair*)(scalarBase(binB + k2rows * sb) + laneOffset(laneB));
      s.a[u] = float2{va.x, va.y};
      s.b[u] = float2{vb.x, vb.y};
    }
  };
  // a conj(b) = (k1 - k3) + i (k1 + k2) with k1 = (ar + ai) br, k2 = -ar (br + bi),
  // k3 = ai (br - bi)
  auto multiply = [&](const GemmSlice& s) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < GK2 / 2; ++u) {
      const float2 a = s.a[u], b = s.b[u];
      k1 = __builtin_amdgcn_mfma_f32_32x32x2f32(__builtin_fmaf(cross, a.y, a.x), b.x, k1, 0, 0, 0);
      k2 = __builtin_amdgcn_mfma_f32_32x32x2f32(a.x, -b.x - b.y, k2, 0, 0, 0);
      k3 = __builtin_amdgcn_mfma_f32_32x32x2f32(a.y, __builtin_fmaf(cross, b.x, -b.y), k3, 0, 0, 0);
    }
  };
  const int slices = g.Kp / GK2;
  const int rangeFirst = blockIdx.y * g.slicesPerSplit;
  const int rangeEnd = min(rangeFirst + g.slicesPerSplit, slices);
  // wave w takes slices w, w + 4, ... of the range: the workgroup reads one front
  const int first = rangeFirst + w;
  ringOfThree<GemmSlice>(first, 4, first < rangeEnd ? (rangeEnd - first + 3) / 4 : 0, fetch,
                         multiply);

  if (w > 0) {
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      red[w - 1][v][lane] = k1[v];
      red[w - 1][16 + v][lane] = k2[v];
      red[w - 1][32 + v][lane] = k3[v];
    }
  }
  __syncthreads();
  if (w > 0) return;
#pragma unroll 1
  for (int u = 0; u < 3; ++u)
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      k1[v] += red[u][v][lane];
      k2[v] += red[u][16 + v][lane];
      k3[v] += red[u][32 + v][lane];
    }
  float2* Cb = g.C + blockIdx.y * g.splitStride + (long)bin * g.I * g.Jp;
  const int j = j0 + r;
  if (j < g.Jp) {
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int i = i0 + 8 * (v / 4) + 4 * h + v % 4;
      if (i < g.I)
        Cb[(long)i * g.Jp + j] =
            pairs ? float2{k1[v], -k3[v]} : float2{k1[v] - k3[v], k1[v] + k2[v]};
    }
  }
}

// The register kernel for products with a short side (up to 32 rows of C per bin; the
// host puts the short side on i): a wave owns 32 rows x 64 columns.  Lane (r, h) loads
// 16 bytes of B per k-pair - columns j0 + 2r and j0 + 2r + 1 at k = 2s + h - which feed two
// MFMA sub-tiles with interleaved columns, and stores the two results of a row side by
// side as 16 bytes: half the memory instructions of two 32 x 32 sub-tiles, 512-byte runs,
// and A (small, shared by every wave of the bin) is read once per 64 columns.  The four
// waves of a workgroup take consecutive column blocks.
struct GemmSliceWide {
  float2 a[GK2 / 2];
  float4 b[GK2 / 2];
};

__global__ __launch_bounds__(kT, 3) void binGemmRegsWide(GemmArgs g) {
  const int t = threadIdx.x;
  const int lane = t % 64, w = __builtin_amdgcn_readfirstlane(t / 64);
  const int r = lane % 32, h = lane / 32;
  // g.IT: 32-row blocks, g.JT: workgroups (4 x 64 columns) along j
  const int total = g.bins * g.IT * g.JT;
  const int per = (total + 7) / 8;
  const int logical = (blockIdx.x % 8) * per + blockIdx.x / 8;
  if (logical >= total) return;
  const int bin = logical / (g.IT * g.JT);
  const int rem = logical % (g.IT * g.JT);
  const int i0 = (rem / g.JT) * 32, j0 = ((rem % g.JT) * 4 + w) * 64;
  if (j0 >= g.Jp) return;
  const bool pairs = bin == 0 || 2 * bin == g.N;  // bins of real pairs: (ar br, ai bi)
  const float cross = pairs ? 0.f : 1.f;

  // operand columns beyond the padded arrays are clamped (they feed accumulators that
  // are never stored); Jp is even and rows of B and C start on 16-byte boundaries
  // (an address: a scalar base - bin, k-rows, column block - plus the lane's fixed offset)
  const unsigned laneA = (unsigned)(h * g.Ip + min(i0 + r, g.Ip - 1)) * (unsigned)sizeof(float2);
  const unsigned laneB = (unsigned)(h * g.Jp + min(2 * r, g.Jp - 2 - j0)) * (unsigned)sizeof(float2);
  const char* const binA = (const char*)(g.A + (long)bin * g.Kp * g.Ip);
  const char* const binB = (const char*)(g.B + (long)bin * g.Kp * g.Jp + j0);
  const long sa = 2L * g.Ip * sizeof(float2), sb = 2L * g.Jp * sizeof(float2);  // two k-rows

  floatx16 k1[2], k2[2], k3[2];
#pragma unroll
  for (int q = 0; q < 2; ++q)
#pragma unroll
    for (int v = 0; v < 16; ++v) k1[q][v] = k2[q][v] = k3[q][v] = 0.f;

  auto fetch = [&](GemmSliceWide& s, int sl) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < GK2 / 2; ++u) {
      const long k2rows = (long)sl * (GK2 / 2) + u;
      const PlainPair va = *(const GlobalPair*)(scalarBase(binA + k2rows * sa) + laneOffset(laneA));
      const PlainQuad vb = *(const GlobalQuad*)(scalarBase(binB + k2rows * sb) + laneOffset(laneB));
      s.a[u] = float2{va.x, va.y};
      s.b[u] = float4{vb.x, vb.y, vb.z, vb.w};
    }
  };
  // a conj(b) = (k1 - k3) + i (k1 + k2) with k1 = (ar + ai) br, k2 = -ar (br + bi),
  // k3 = ai (br - bi)
  auto multiply = [&](const GemmSliceWide& s) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < GK2 / 2; ++u) {
      const float2 a = s.a[u];
      const float as = __builtin_fmaf(cross, a.y, a.x);
      const float4 b = s.b[u];
      k1[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(as, b.x, k1[0], 0, 0, 0);
      k2[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(a.x, -b.x - b.y, k2[0], 0, 0, 0);
      k3[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(a.y, __builtin_fmaf(cross, b.x, -b.y), k3[0], 0, 0, 0);
      k1[1] = __builtin_amdgcn_mfma_f32_32x32x2f32(as, b.z, k1[1], 0, 0, 0);
      k2[1] = __builtin_amdgcn_mfma_f32_32x32x2f32(a.x, -b.z - b.w, k2[1], 0, 0, 0);
      k3[1] = __builtin_amdgcn_mfma_f32_32x32x2f32(a.y, __builtin_fmaf(cross, b.z, -b.w), k3[1], 0, 0, 0);
    }
  };
  const int first = blockIdx.y * g.slicesPerSplit;
  // two register sets instead of three: 153 registers, three waves per SIMD instead of two
  // (the 256 x 256 layer: 294.6 -> 290.1 us per forward pass)
  ringOfTwo<GemmSliceWide>(first, 1, min(first + g.slicesPerSplit, g.Kp / GK2) - first, fetch,
                           multiply);

  float2* Cb = g.C + blockIdx.y * g.splitStride + (long)bin * g.I * g.Jp;
  const int j = j0 + 2 * r;
  if (j < g.Jp) {
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int i = i0 + 8 * (v / 4) + 4 * h + v % 4;
      if (i < g.I) {
        float4 o;
        if (pairs)
          o = float4{k1[0][v], -k3[0][v], k1[1][v], -k3[1][v]};
        else
          o = float4{k1[0][v] - k3[0][v], k1[0][v] + k2[0][v], k1[1][v] - k3[1][v],
                     k1[1][v] + k2[1][v]};
        *reinterpret_cast<float4*>(Cb + (long)i * g.Jp + j) = o;
      }
    }
  }
}

// ... and for up to 16 rows: the same on v_mfma_f32_16x16x4_f32.  A wave owns 16 rows x 64
// columns; lane (c, q) loads 16 bytes of B per four k - columns j0 + 2c and j0 + 2c + 1 at k = q - of
// either half of the columns, and 8 bytes of A.  The matrix work of 16 rows that are not there
// is what bounded the 32-row form: us, 201 x 74 x 17 x 14 images, 9 filters of 8 x 8, named 32 points, weight
// gradient 35.4 -> 16.9; 27 x 4 x 100 x 100, 152 of 9 x 9, weight gradient 109.8 -> 57.6, input gradient
// 105.8 -> 85.8.
struct GemmSliceNarrow {
  float2 a[2];
  float4 b[2][2];
};

__global__ __launch_bounds__(kT, 4) void binGemmRegsNarrow(GemmArgs g) {
  const int t = threadIdx.x;
  const int lane = t % 64, w = __builtin_amdgcn_readfirstlane(t / 64);
  const int c = lane % 16, q = lane / 16;
  const int total = g.bins * g.JT;
  const int per = (total + 7) / 8;
  const int logical = (blockIdx.x % 8) * per + blockIdx.x / 8;
  if (logical >= total) return;
  const int bin = logical / g.JT;
  const int j0 = (logical % g.JT * 4 + w) * 64;
  if (j0 >= g.Jp) return;
  const bool pairs = bin == 0 || 2 * bin == g.N;  // bins of real pairs: (ar br, ai bi)
  const float cross = pairs ? 0.f : 1.f;

  // operand columns beyond the padded arrays are clamped, as above
  const unsigned laneA = (unsigned)(q * g.Ip + min(c, g.Ip - 1)) * (unsigned)sizeof(float2);
  unsigned laneB[2];
#pragma unroll
  for (int u = 0; u < 2; ++u)
    laneB[u] = (unsigned)(q * g.Jp + min(32 * u + 2 * c, g.Jp - 2 - j0)) * (unsigned)sizeof(float2);
  const char* const binA = (const char*)(g.A + (long)bin * g.Kp * g.Ip);
  const char* const binB = (const char*)(g.B + (long)bin * g.Kp * g.Jp + j0);
  const long sa = 4L * g.Ip * sizeof(float2), sb = 4L * g.Jp * sizeof(float2);  // four k-rows

  typedef float floatx4 __attribute__((ext_vector_type(4)));
  floatx4 k1[4], k2[4], k3[4];  // of columns 2c, 2c + 1, 32 + 2c, 33 + 2c
#pragma unroll
  for (int n = 0; n < 4; ++n)
#pragma unroll
    for (int v = 0; v < 4; ++v) k1[n][v] = k2[n][v] = k3[n][v] = 0.f;

  auto fetch = [&](GemmSliceNarrow& s, int sl) __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const long k4 = (long)sl * 2 + h;
      const PlainPair va = *(const GlobalPair*)(scalarBase(binA + k4 * sa) + laneOffset(laneA));
      s.a[h] = float2{va.x, va.y};
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const PlainQuad vb = *(const GlobalQuad*)(scalarBase(binB + k4 * sb) + laneOffset(laneB[u]));
        s.b[h][u] = float4{vb.x, vb.y, vb.z, vb.w};
      }
    }
  };
  auto multiply = [&](const GemmSliceNarrow& s) __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const float2 a = s.a[h];
      const float as = __builtin_fmaf(cross, a.y, a.x);
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        const float4 b = s.b[h][n / 2];
        const float br = n % 2 ? b.z : b.x, bi = n % 2 ? b.w : b.y;
        k1[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(as, br, k1[n], 0, 0, 0);
        k2[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, -br - bi, k2[n], 0, 0, 0);
        k3[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, __builtin_fmaf(cross, br, -bi), k3[n], 0, 0, 0);
      }
    }
  };
  const int first = blockIdx.y * g.slicesPerSplit;
  ringOfThree<GemmSliceNarrow>(first, 1, min(first + g.slicesPerSplit, g.Kp / GK2) - first, fetch, multiply);

  float2* Cb = g.C + blockIdx.y * g.splitStride + (long)bin * g.I * g.Jp;
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int j = j0 + 32 * u + 2 * c;
    if (j >= g.Jp) continue;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int i = 4 * q + v;
      if (i >= g.I) continue;
      auto value = [&](int n) {
        return pairs ? float2{k1[n][v], -k3[n][v]} : float2{k1[n][v] - k3[n][v], k1[n][v] + k2[n][v]};
      };
      const float2 lo = value(2 * u), hi = value(2 * u + 1);
      *reinterpret_cast<float4*>(Cb + (long)i * g.Jp + j) = float4{lo.x, lo.y, hi.x, hi.y};
    }
  }
}

// The same product on the bf16 matrix instructions, for products that outweigh their operands
// (planGemm).  fp32 matrix instructions are what bounds
// binGemmDirect there (155 TFLOP/s); the bf16 ones run at 1600 to 1750 on random operands (the power
// limit; 2400 on zeros).  An fp32 value of 2^-110 or more is the sum of three bf16 values without
// remainder, a = a0 + a1 + a2: the upper half of its bits, the remainder rounded to 8 bits, and what is
// left, which has at most 8.  (Below, the last piece ends at bf16's smallest subnormal, 2^-133: images of
// 2^-100 and 2^-108 2.1e-7 from 64 bits, 2^-116 4.1e-7.  An infinity comes out as NaN.)  Of the nine products of pieces the six largest are formed; the
// three dropped ones are below 2^-23 |a b| each and of either sign, products of pieces
// are exact in fp32, and a sum is rounded once per 16 k and product of pieces where the
// fp32 instructions round every 2 k.  Against 64 bits over random operands: K = 64 1.1e-7, K =
// 1024 4.9e-7 (relative 2-norm); fp32 instructions 1.4e-7 and 5.8e-7.
//
// One workgroup = one bin x a (64 x 64) tile, 4 waves of 32 x 32.  A slice of 16 k passes
// through registers, where each value is split once, into LDS as bf16, [piece][re, im][k
// half][row] of 8 k: what a lane of v_mfma_f32_32x32x16_bf16 supplies is one 16-byte read.
// The next slice's loads fly under this one's products.  114 registers and 24.6 KB of LDS leave
// room for four workgroups per CU.  Four real products per complex one: three (as above) would need a
// third split operand on each side, and LDS reads then take longer than the products saved.
// 128 x 64, 64 x 128 and 128 x 128 tiles and a second LDS buffer measured 1 to 40 % slower
// (fewer workgroups per CU); each wave splitting what it reads, from the stages that
// global_load_lds fills, 25 % slower.
// us per launch, binGemmDirect / this: 128 x 192 x 64 over 512 bins 53.6 / 47.2; 264 x 307 x 273
// over 128 194 / 149 to 161; of 161, 104 are left without its matrix instructions, 156 without its stores,
// 146 without the splits.
typedef __bf16 Bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned Quad __attribute__((ext_vector_type(4)));
typedef unsigned Duo __attribute__((ext_vector_type(2)));
constexpr int GK3 = 16;

// the bf16 pieces of two floats, two to a word.  The first piece is cut off, not rounded: the
// largest finite floats would round to infinity.
__device__ __forceinline__ void split2(float x, float y, unsigned& p0, unsigned& p1, unsigned& p2) {
  typedef float Float2 __attribute__((ext_vector_type(2)));
  typedef __bf16 Bf16x2 __attribute__((ext_vector_type(2)));
  auto bits = [](float f) { return __builtin_bit_cast(unsigned, f); };
  auto real = [](unsigned u) { return __builtin_bit_cast(float, u); };
  auto upper = [&](float a, float b) { return __builtin_amdgcn_perm(bits(b), bits(a), 0x07060302u); };
  p0 = upper(x, y);
  const float rx = x - real(bits(x) & 0xffff0000u), ry = y - real(bits(y) & 0xffff0000u);
  p1 = __builtin_bit_cast(unsigned, __builtin_convertvector(Float2{rx, ry}, Bf16x2));
  p2 = upper(rx - real(p1 << 16), ry - real(p1 & 0xffff0000u));
}

struct SplitOperand {
  Quad v[3][2][2][64];
};

// four k of one row, quarter q of the slice
__device__ __forceinline__ void parkSplit(SplitOperand& s, int row, int q, const PlainPair (&v)[4]) {
  Duo p[3][2];
#pragma unroll
  for (int e = 0; e < 2; ++e)
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      unsigned p0, p1, p2;
      split2(v[2 * e][c], v[2 * e + 1][c], p0, p1, p2);
      p[0][c][e] = p0;
      p[1][c][e] = p1;
      p[2][c][e] = p2;
    }
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int c = 0; c < 2; ++c) reinterpret_cast<Duo*>(&s.v[i][c][q / 2][row])[q % 2] = p[i][c];
}

// Makes LDS writes of the whole workgroup visible to it; global loads stay in flight.
__device__ __forceinline__ void ldsBarrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

__global__ __launch_bounds__(kT, 4) void binGemmSplit(GemmArgs g) {
  __shared__ __align__(16) SplitOperand opA, opB;
  const int t = threadIdx.x;
  const int lane = t % 64;
  const int w = __builtin_amdgcn_readfirstlane(t / 64);
  const int r = lane % 32, h = lane / 32;
  const int total = g.bins * g.IT * g.JT;
  const int per = (total + 7) / 8;
  const int logical = (blockIdx.x % 8) * per + blockIdx.x / 8;
  if (logical >= total) return;
  const int bin = logical / (g.IT * g.JT);
  const int rem = logical % (g.IT * g.JT);
  const int i0 = (rem / g.JT) * 64, j0 = (rem % g.JT) * 64;
  const int rb = w % 2, cb = w / 2;  // this wave's 32-row and 32-column block
  const bool pairs = bin == 0 || 2 * bin == g.N;  // bins of real pairs: (ar br, ai bi)

  // this workgroup's range of the reduction: rows k-rows, a multiple of 8
  const int first = blockIdx.y * g.slicesPerSplit * GK2;
  const int rows = min(g.slicesPerSplit * GK2, g.Kp - first);
  const int slices = (rows + GK3 - 1) / GK3;
  // lane l of wave w loads k-rows 4w .. 4w+3 of row l of each operand, clamped into the padded
  // arrays (what is beyond them feeds accumulators that are never stored)
  const unsigned laneA = (unsigned)min(i0 + lane, g.Ip - 1) * (unsigned)sizeof(float2);
  const unsigned laneB = (unsigned)min(j0 + lane, g.Jp - 1) * (unsigned)sizeof(float2);
  const long rowA = (long)g.Ip * sizeof(float2), rowB = (long)g.Jp * sizeof(float2);
  const char* const baseA = (const char*)(g.A + ((long)bin * g.Kp + first) * g.Ip);
  const char* const baseB = (const char*)(g.B + ((long)bin * g.Kp + first) * g.Jp);
  PlainPair va[4], vb[4];
  auto request = [&](int sl) __attribute__((always_inline)) {
    const int k = min(sl * GK3 + 4 * w, rows - 4);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      va[u] = *(const GlobalPair*)(scalarBase(baseA + (k + u) * rowA) + laneOffset(laneA));
      vb[u] = *(const GlobalPair*)(scalarBase(baseB + (k + u) * rowB) + laneOffset(laneB));
    }
  };

  floatx16 re, im;
#pragma unroll
  for (int v = 0; v < 16; ++v) re[v] = im[v] = 0.f;

  auto loop = [&](auto realPairs) __attribute__((always_inline)) {
    constexpr bool PAIRS = decltype(realPairs)::value;
    for (int sl = 0; sl < slices; ++sl) {
      if (sl * GK3 + 4 * w >= rows) {  // the last slice may be half a slice
#pragma unroll
        for (int u = 0; u < 4; ++u) va[u] = vb[u] = PlainPair{0.f, 0.f};
      }
      parkSplit(opA, lane, w, va);
      parkSplit(opB, lane, w, vb);
      request(min(sl + 1, slices - 1));
      ldsBarrier();
      // products of pieces, the smallest first
      constexpr int PA[6] = {2, 0, 1, 1, 0, 0}, PB[6] = {0, 2, 1, 0, 1, 0};
      const Quad sign = Quad{0x80008000u, 0x80008000u, 0x80008000u, 0x80008000u};
      Quad a[3][2], b[3][2];
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          b[i][c] = opB.v[i][c][h][32 * cb + r];
          a[i][c] = opA.v[i][c][h][32 * rb + r];
        }
      auto multiply = [&](Quad x, Quad y, floatx16& c) __attribute__((always_inline)) {
        c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(Bf16x8, x),
                                                    __builtin_bit_cast(Bf16x8, y), c, 0, 0, 0);
      };
#pragma unroll
      for (int p = 0; p < 6; ++p) {
        const Quad ar = a[PA[p]][0], ai = a[PA[p]][1], br = b[PB[p]][0], bi = b[PB[p]][1];
        multiply(ar, br, re);
        if constexpr (PAIRS) {
          multiply(ai, bi, im);
        } else {
          multiply(ai, br, im);
          multiply(ai, bi, re);
          multiply(ar, bi ^ sign, im);
        }
      }
      ldsBarrier();
    }
  };
  request(0);
  if (pairs)
    loop(std::true_type{});
  else
    loop(std::false_type{});

  float2* Cb = g.C + blockIdx.y * g.splitStride + (long)bin * g.I * g.Jp;
  if (i0 + 32 * rb + 32 <= g.I && j0 + 32 * cb + 32 <= g.Jp) {
    const unsigned laneC = (unsigned)(4 * h * g.Jp + r) * (unsigned)sizeof(float2);
    char* const waveC = (char*)(Cb + (long)(i0 + 32 * rb) * g.Jp + j0 + 32 * cb);
    const long rowC = (long)g.Jp * sizeof(float2);
#pragma unroll
    for (int v = 0; v < 16; ++v)
      *(GlobalPair*)(scalarBase(waveC + (8 * (v / 4) + v % 4) * rowC) + laneOffset(laneC)) =
          PlainPair{re[v], im[v]};
    return;
  }
  const int j = j0 + 32 * cb + r;
  if (j >= g.Jp) return;
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const int i = i0 + 32 * rb + 8 * (v / 4) + 4 * h + v % 4;
    if (i < g.I) Cb[(long)i * g.Jp + j] = float2{re[v], im[v]};
  }
}

inline int roundUp(int a, int b) { return (a + b - 1) / b * b; }

// Which operand takes the 128-wide side of the GEMM tile (and with it the role of i, the
// slow index of C[bin][i][j]).  Results cut into windows of a larger image (outTiled)
// always put the window index on j: the inverse kernel transforms 16 consecutive j per
// workgroup, and 16 neighbouring windows of one output plane store whole stretches of
// image rows where 16 output planes of one window store 24-float pieces 248 floats apart
// (the 256 x 256 layer: 337 -> 308 us per forward pass).  Otherwise: the assignment with fewer
// padded tile elements.
inline bool swapRoles(int I, int J, bool outTiled) {
  if (outTiled) return true;
  if (I <= 32 || J <= 32) return J < I;  // the register kernel takes the short side on i
  return (long)roundUp(J, GI) * roundUp(I, GJ2) < (long)roundUp(I, GI) * roundUp(J, GJ2);
}

// Which contraction kernel runs a product, on which tiles, and into how many ranges the
// reduction is cut (range s writes its partial product to C + s * splitStride and the
// inverse kernel adds the partials in range order, so the result does not depend on
// timing).  A short side (up to 32, which the roles put on i) takes the register kernels:
// the LDS kernels' tiles would be half empty.  64-row tiles when they waste fewer rows,
// or when 128-row tiles would leave the chip with fewer than eight workgroups per CU to
// balance (measured equal or faster there: 84 -> 62 us for 64 x 192 x 128 per bin,
// 77 -> 69 us for 128 x 64 x 192).  Ranges: when the tiles alone leave most of the chip
// idle and the reduction is long - 8- and 16-point transforms have 32 and 128 bins, and a
// weight gradient reduces over every image and window - up to 16 of them, enough for
// about two waves per SIMD in the register kernels and one round of workgroups in the LDS
// kernels, each keeping at least `minSlices` k-slices (weight gradient of the 27 x 27 layer on
// 8-point windows: 423 -> 238 us; 64 x 64 x 512 per bin on 16-point windows: 73 -> 63 us;
// ranges of 8 slices cost 6 % where 16 slices are all there are).  32-point transforms on short sides
// have 512 bins and never split (measured on the weight gradient of the 256 x 256 layer, 32 x 32
// per bin over 1936 windows, 2048 waves: two ranges 337 -> 345 us, four 362: that
// contraction is not short of waves).
struct GemmPlan {
  enum Kind { RegsSplitK, RegsWide, RegsNarrow, Direct64, Direct128, Split } kind;
  int IT, JT;
  int splits, slicesPerSplit;
  long waves;  // of one range
};

// (maxSplits: more ranges than that have no room in the workspace)
inline GemmPlan planGemm(int bins, int I, int Jp, int Kp, int maxSplits) {
  GemmPlan p;
  long waves, target;
  int minSlices;
  if (I <= 32 && Jp <= 32) {
    p.kind = GemmPlan::RegsSplitK;
    p.IT = p.JT = 1;
    waves = 4L * bins;
    target = 2048;
    minSlices = 16;
  } else if (I <= 32) {
    p.kind = GemmPlan::RegsWide;
    p.IT = 1;
    p.JT = ceilDiv(Jp, 256);
    waves = (long)bins * ceilDiv(Jp, 64);
    target = 2048;
    minSlices = 4;
  } else {
    p.JT = ceilDiv(Jp, GJ2);
    const bool small =
        roundUp(I, 64) < roundUp(I, GI) || (long)bins * ceilDiv(I, GI) * p.JT < 8 * 256;
    p.kind = small ? GemmPlan::Direct64 : GemmPlan::Direct128;
    p.IT = ceilDiv(I, small ? 64 : GI);
    waves = 4L * bins * p.IT * p.JT;
    target = 4096;
    minSlices = 16;
  }
  const int slices = Kp / GK2;
  const int want = (int)std::min<long>(maxSplits, ceilDiv(target, waves));
  const int most = std::max(1, slices / minSlices);
  p.slicesPerSplit = ceilDiv(slices, std::min(want, most));
  p.splits = ceilDiv(slices, p.slicesPerSplit);  // no range is empty
  p.waves = waves;
  // A small product on few workgroups is one chain of slices each, on an idle chip:
  // binGemmRegsSplitK's 32 x 32 tiles are two to eight times as many workgroups, and each cuts
  // its chain in four.  us, binGemmRegsWide / 32 x 32 tiles: 192 workgroups 8.4 / 4.8, 384 7.9
  // / 5.7, 768 8.8 / 6.8 (4.7 slices), but 1152 4.8 / 6.9 (1 slice; 6 slices, 1536: 13.2 / 11.1);
  // binGemmDirect<64> / 32 x 32 tiles: 384 (one image, 64 x 27 x 27, 192 of 5 x 5, 8 slices)
  // 7.9 / 7.6, 192 (10) 7.9 / 6.1, 128 (24) 14.6 / 8.0, 768 (21) 13.6 / 12.2, but 512 (5) 6.6 / 7.1.  Whole
  // passes, 300 random products that leave binGemmDirect<64> this way: 0.96 of the time in the middle up to ten
  // slices, 0.90 above, two of 768 tiles 3 % longer.
  // Not for up to 16 rows and three slices, where binGemmRegsNarrow is faster (500 random passes, 32 x 32
  // tiles / it: one slice 1.07 in the middle and always slower, two 1.07, three 1.02; four and five 0.97
  // to 1.10, six to ten 0.94).
  const long tiles = (long)bins * ceilDiv(I, 32) * ceilDiv(Jp, 32) * p.splits;
  if ((p.kind == GemmPlan::RegsWide && (I > 16 || p.slicesPerSplit >= 4) &&
       (tiles <= 768 || (p.slicesPerSplit >= 6 && tiles <= 1536))) ||
      (p.kind == GemmPlan::Direct64 && p.slicesPerSplit >= 8 && tiles <= 768)) {
    p.kind = GemmPlan::RegsSplitK;
    p.IT = ceilDiv(I, 32);
    p.JT = ceilDiv(Jp, 32);
  }
  // up to 16 rows: 91 random products 0.97 to 2.2 times as fast as on 32-row tiles
  if (p.kind == GemmPlan::RegsWide && I <= 16) p.kind = GemmPlan::RegsNarrow;
  // binGemmSplit where the products outweigh the operands by enough: each spectrum value enters
  // I J K / (I J + I K + J K) complex products.  Whole layers, three passes
  // back to back, binGemmDirect / this by that quotient: 93 (66 x 273 x 25 x 26, 307 of 2 x 2)
  // 761 / 708 us; 43 (128 x 128 x 28 x 28, 128 of 5 x 5) 367 / 354; 38 (180 x 65 x 12 x 20, 195 of
  // 10 x 10) 394 / 369; below, the launch waits for memory, splitting has few products to
  // pay for it and the bf16 instructions' power slows the transforms around them on a chip that has
  // been loaded for long: 37 (128 x 64 x 28 x 28, 256 of 5 x 5) 416 / 423, 35 (the 27 x 27 layer) 324 / 332, 28
  // (64 x 64 x 30 x 30, 64 of 4 x 4) 151 / 160.  In runs of a few ms, which do not reach that limit, 230
  // random layers take 0.98 of binGemmDirect's time in the middle at 18 to 24 (0.93 to 1.03), 0.96 at 28
  // to 32, 0.94 at 36 to 40 and 0.89 from 55 up, none above 28 longer: the line lies where
  // neither kind of run loses.  And not with fewer workgroups than two per CU (2 x 178 x 38 x 46, 33 of 5
  // x 5, 128 workgroups: 13.9 / 16.5) or ranges of fewer than 48 k.
  if ((p.kind == GemmPlan::Direct64 || p.kind == GemmPlan::Direct128) && p.slicesPerSplit >= 6 &&
      1.0 / I + 1.0 / Jp + 1.0 / Kp <= 1.0 / 38 &&
      (long)bins * ceilDiv(I, 64) * p.JT * p.splits >= 2 * 256) {
    p.kind = GemmPlan::Split;
    p.IT = ceilDiv(I, 64);
  }
  return p;
}

constexpr int kAnySplits = 16;  // what planGemm cuts a reduction into at most

// What a pass on windows takes: workspace, two estimates of its time, the second for small passes, and
// its contraction.
struct WindowsCost {
  size_t bytes;
  double us, smallUs;
  GemmPlan plan;
};

// The estimate: three launches, every spectrum value written and read once, and the
// contraction's products over whole tiles - at the rate of one wave per SIMD where the waves
// are fewer than that, and of whole rounds of two per SIMD in binGemmRegsWide.  Fitted to 6600
// random layers of 64 and 128 points when only binGemmDirect, binGemmRegsWide and one tile of
// binGemmRegsSplitK ran their contractions; of 4900 random passes of 8 us to 3 ms it is now within 20 % of
// half, and 12 % high in the middle.  It is there to choose between sizes (passSize), whose
// estimates share most of that.
// The second estimate, for three launches of at most a few dozen us: a start each, spectra that
// the caches hold, tiles and chains of slices of the kernel that runs.  Over 2600 random passes it is
// within 10 % of nine in ten.
template <int N>
WindowsCost windowsCost(int I, int J, int K, bool outTiled, int maxSplits) {
  if (swapRoles(I, J, outTiled)) std::swap(I, J);
  const int SL = BMCfg<N>::SLOTS, bins = BMCfg<N>::BINS;
  const int Ip = roundUp(I, SL), Jp = roundUp(J, SL), Kp = roundUp(K, 8);
  const GemmPlan plan = planGemm(bins, I, Jp, Kp, maxSplits);
  WindowsCost c;
  c.plan = plan;
  c.bytes = sizeof(float2) * bins * ((size_t)Kp * Ip + (size_t)Kp * Jp + (size_t)plan.splits * I * Jp);
  const double products = (double)bins * roundUp(I, I <= 32 ? 32 : 64) * roundUp(Jp, 64) * Kp;
  const bool wide = I <= 32 && Jp > 32;  // what binGemmRegsWide runs, its small products apart
  const long waves = plan.waves * plan.splits;
  const double idle = waves < 1024 ? 1024.0 / waves : wide ? (waves + 2047) / 2048 * 2048.0 / waves : 1.0;
  c.us = 15 + 0.14e-6 * 2 * c.bytes + (wide ? 0.055e-6 : 0.04e-6) * products * idle;
  const bool tiles32 = plan.kind == GemmPlan::RegsSplitK;
  const bool narrow = plan.kind == GemmPlan::RegsNarrow;
  const int rows = narrow ? 16 : tiles32 || plan.kind == GemmPlan::RegsWide ? 32 : 64;
  const int chain = tiles32 ? ceilDiv(plan.slicesPerSplit, 4) : plan.slicesPerSplit;
  c.smallUs = (N == 8 ? 8.9 : N == 16 ? 10.7 : 15.3) - (narrow ? 0.5 : 0) + 0.46e-6 * c.bytes +
              0.036e-6 * bins * roundUp(I, rows) * roundUp(Jp, tiles32 ? 32 : 64) * Kp + 0.3 * chain;
  return c;
}

template <int N>
size_t workspaceFloat2(int I, int J, int K, bool outTiled) {
  return windowsCost<N>(I, J, K, outTiled, kAnySplits).bytes / sizeof(float2);
}

// P[i][j] = scale * sum_k X[i][k] * op(Y[j][k]) for planes x(i,k), y(j,k) -> planes out(i,j);
// each PlaneSet names its first index "row" and its second "k".
template <int N>
int runPipeline(PlaneSet x, PlaneSet y, PlaneSet out, bool conjY, float scale, bool accumulate,
                int maxSplits, float2* ws, hipStream_t s) {
  using C = BMCfg<N>;
  const int SL = C::SLOTS, bins = C::BINS;
  float xSign = 1.0f, ySign = conjY ? 1.0f : -1.0f;
  if (swapRoles(x.R, y.R, out.tiled != 0 || out.described != 0)) {
    // G[j][i] = sum_k op(Y[j]) * conj(conj X[i])
    std::swap(x, y);
    xSign = conjY ? -1.0f : 1.0f;
    ySign = -1.0f;
    std::swap(out.sRow, out.sK);
    if (out.tiled) out.tiled = 3 - out.tiled;
    if (out.described) out.described = 3 - out.described;
  }
  const int I = x.R, J = y.R, K = x.K;
  out.R = I;
  out.K = J;
  const int Ip = roundUp(I, SL), Jp = roundUp(J, SL), Kp = roundUp(K, 8);
  // every launch below counts its workgroups in one 31-bit grid index: refuse, before
  // anything runs, a layer whose transforms or contraction tiles outnumber that
  const long gridMax = 0x7fffffffL;
  if ((long)(Ip / SL + Jp / SL) * Kp > gridMax || (long)(Jp / SL) * I > gridMax ||
      (long)bins * ceilDiv(I, 32) * ceilDiv(Jp, 32) > gridMax)
    return FBFFT_UNSUPPORTED_SIZE;
  float2* SA = ws;
  float2* SB = SA + (size_t)bins * Kp * Ip;
  float2* SC = SB + (size_t)bins * Kp * Jp;

  // 1: every window of a set starts on an 8-byte boundary with an even width and pad;
  // 2: the windows are described on the device, each plane decides for itself; 0: 4 bytes
  auto movesAsPairs = [](const PlaneSet& p) {
    if (p.described) return 2;
    return windowMovesAsPairs(p.base, p.sy, p.sx, p.w, p.padL0) && p.sRow % 2 == 0 &&
                   p.sK % 2 == 0 && (!p.tiled || ((p.stepX | p.orgX | p.winW) & 1) == 0)
               ? 1
               : 0;
  };
  // Two runs per workgroup pay once the halved launch still fills every CU several
  // times over (measured: 114.5 -> 109.8 us on 3936 workgroups, 29.9 -> 33.7 us on a
  // launch a quarter of that).
  const bool two = (long)(ceilDiv(Ip / SL, 2) + ceilDiv(Jp / SL, 2)) * Kp >= 3L * 2 * computeUnits();
  // both operands' spectra against half of the 256 MiB last-level cache
  const int stream = (size_t)bins * Kp * ((size_t)Ip + Jp) * sizeof(float2) > (128u << 20);
  const ForwardJob ja{x, SA, Ip, Kp, xSign, two ? ceilDiv(Ip / SL, 2) : Ip / SL, stream},
      jb{y, SB, Jp, Kp, ySign, two ? ceilDiv(Jp / SL, 2) : Jp / SL, stream};
  const dim3 fgrid((unsigned)(ja.rowGroups + jb.rowGroups) * Kp);
  const int pa = movesAsPairs(x), pb = movesAsPairs(y);
  auto launchForward = [&](auto groups) {
    constexpr int G = decltype(groups)::value;
    auto withB = [&](auto modeA) {
      constexpr int A = decltype(modeA)::value;
      if (pb == 2)
        forwardBinMajor<N, A, 2, G><<<fgrid, dim3(kTF), 0, s>>>(ja, jb);
      else if (pb == 1)
        forwardBinMajor<N, A, 1, G><<<fgrid, dim3(kTF), 0, s>>>(ja, jb);
      else
        forwardBinMajor<N, A, 0, G><<<fgrid, dim3(kTF), 0, s>>>(ja, jb);
    };
    if (pa == 2)
      withB(std::integral_constant<int, 2>{});
    else if (pa == 1)
      withB(std::integral_constant<int, 1>{});
    else
      withB(std::integral_constant<int, 0>{});
  };
  if (two)
    launchForward(std::integral_constant<int, 2>{});
  else
    launchForward(std::integral_constant<int, 1>{});
  GemmArgs g;
  g.A = SA;
  g.B = SB;
  g.C = SC;
  g.bins = bins;
  g.N = N;
  g.I = I;
  g.Ip = Ip;
  g.Jp = Jp;
  g.Kp = Kp;
  const GemmPlan plan = planGemm(bins, I, Jp, Kp, maxSplits);
  g.IT = plan.IT;
  g.JT = plan.JT;
  g.splits = plan.splits;
  g.slicesPerSplit = plan.slicesPerSplit;
  g.splitStride = (long)bins * I * Jp;
  const dim3 ggrid(roundUp(bins * g.IT * g.JT, 8), g.splits);
  switch (plan.kind) {
    case GemmPlan::RegsSplitK: binGemmRegsSplitK<<<ggrid, dim3(kT), 0, s>>>(g); break;
    case GemmPlan::RegsWide: binGemmRegsWide<<<ggrid, dim3(kT), 0, s>>>(g); break;
    case GemmPlan::RegsNarrow: binGemmRegsNarrow<<<ggrid, dim3(kT), 0, s>>>(g); break;
    case GemmPlan::Direct64: binGemmDirect<64><<<ggrid, dim3(kT), 0, s>>>(g); break;
    case GemmPlan::Direct128: binGemmDirect<GI><<<ggrid, dim3(kT), 0, s>>>(g); break;
    case GemmPlan::Split: binGemmSplit<<<ggrid, dim3(kT), 0, s>>>(g); break;
  }
  // Two runs per workgroup pay when the paired launch still fills the chip for three
  // rounds or more (two workgroups are resident per CU): 112 -> 108 us at the 256 x 256 layer,
  // 1936 paired workgroups; at the 27 x 27 layer pairing would leave 768 workgroups, one and a
  // half rounds, and costs 35.5 -> 37.1 us.
  const bool pairedRuns = Jp / SL >= 2 && (long)ceilDiv(Jp / SL, 2) * I >= 3L * 2 * computeUnits();
  const int runGroups = pairedRuns ? ceilDiv(Jp / SL, 2) : Jp / SL;
  const dim3 igrid((unsigned)((long)runGroups * I));
  // windows whose rows start on 8-byte boundaries with an even width: a lane stores its
  // two columns of a row as one 8-byte word
  const int po = movesAsPairs(out);
  // the unnormalised transforms' 1 / N^2 (a power of two: exact) rides on the caller's factor
  const float invNorm = 1.0f / (float)(N * N);
  auto launchInverse = [&](auto acc, auto groups, auto pairs) {
    inverseBinMajor<N, decltype(acc)::value, decltype(groups)::value, decltype(pairs)::value>
        <<<igrid, dim3(kTF), 0, s>>>(SC, I, Jp, out, scale * invNorm, g.splits, g.splitStride,
                                     runGroups);
  };
  auto withPairs = [&](auto acc, auto groups) {
    if (po == 2)
      launchInverse(acc, groups, std::integral_constant<int, 2>{});
    else if (po == 1)
      launchInverse(acc, groups, std::integral_constant<int, 1>{});
    else
      launchInverse(acc, groups, std::integral_constant<int, 0>{});
  };
  auto withGroups = [&](auto acc) {
    if (pairedRuns)
      withPairs(acc, std::integral_constant<int, 2>{});
    else
      withPairs(acc, std::integral_constant<int, 1>{});
  };
  if (accumulate)
    withGroups(std::true_type{});
  else
    withGroups(std::false_type{});
  return launchStatus();
}

PlaneSet planes(float* base, const int* stride, const int* size, int rowDim, int kDim) {
  PlaneSet p{};
  p.base = base;
  p.sRow = stride[rowDim];
  p.sK = stride[kDim];
  p.sy = stride[2];
  p.sx = stride[3];
  p.h = size[2];
  p.w = size[3];
  p.R = size[rowDim];
  p.K = size[kDim];
  return p;
}

// Cuts the images of p into tilesY x tilesX windows; the index of dimension 0 (the
// image) - p's row or k - becomes the composite (image, tileY, tileX).
void tile(PlaneSet& p, bool imageIsRow, int tilesY, int tilesX, int stepY, int stepX, int orgY,
          int orgX, int winH, int winW) {
  p.tiled = imageIsRow ? 1 : 2;
  p.tilesY = tilesY;
  p.tilesX = tilesX;
  p.stepY = stepY;
  p.stepX = stepX;
  p.orgY = orgY;
  p.orgX = orgX;
  p.winH = winH;
  p.winW = winW;
  (imageIsRow ? p.R : p.K) *= tilesY * tilesX;
}

template <int N>
int runPass(int pass, const PlaneSet& x, const PlaneSet& y, const PlaneSet& out, float scale,
            bool accumulate, float2* ws, hipStream_t s, int maxSplits = kAnySplits) {
  return runPipeline<N>(x, y, out, /*conjY=*/pass != 1, scale, accumulate, maxSplits, ws, s);
}

}  // namespace

// Tiles per image of a pass: 1 when the image fits the transform.  The forward pass
// and the weight gradient walk the OUTPUT in disjoint (N-kH+1) x (N-kW+1) windows,
// the input gradient walks the INPUT (the tensor it writes) in such windows.
static void tileGrid(int pass, int N, int H, int W, int kH, int kW, int* tilesY, int* tilesX) {
  *tilesY = *tilesX = 1;
  if (H <= N && W <= N) return;
  const int stepY = N - kH + 1, stepX = N - kW + 1;
  const int spanY = pass == 1 ? H : H - kH + 1, spanX = pass == 1 ? W : W - kW + 1;
  *tilesY = ceilDiv(spanY, stepY);
  *tilesX = ceilDiv(spanX, stepX);
}

// (I, J, K) of a pass for batch B (times the tiles per image) and Cin / Cout planes
static void passDims(int pass, int B, int Cin, int Cout, int* I, int* J, int* K) {
  if (pass == 0) { *I = B; *J = Cout; *K = Cin; }
  else if (pass == 1) { *I = B; *J = Cin; *K = Cout; }
  else { *I = Cin; *J = Cout; *K = B; }
}

// a pass on windows of N <= 32 points; no bytes: too many windows
static WindowsCost windowsPass(int pass, int N, int B, int Cin, int Cout, int H, int W, int kH, int kW,
                               int maxSplits) {
  int ty, tx;
  tileGrid(pass, N, H, W, kH, kW, &ty, &tx);
  if ((long)B * ty * tx > (1L << 30)) return {};
  int I, J, K;
  passDims(pass, B * ty * tx, Cin, Cout, &I, &J, &K);
  const bool outTiled = pass != 2 && ty * tx > 1;  // the weight gradient is never tiled
  return N == 8    ? windowsCost<8>(I, J, K, outTiled, maxSplits)
         : N == 16 ? windowsCost<16>(I, J, K, outTiled, maxSplits)
                   : windowsCost<32>(I, J, K, outTiled, maxSplits);
}

size_t convWorkspaceBytes(int pass, int N, int B, int Cin, int Cout, int H, int W, int kH,
                          int kW) {
  if (N > 32) return convSplitWorkspaceBytes(pass, N, B, Cin, Cout);
  return windowsPass(pass, N, B, Cin, Cout, H, W, kH, kW, kAnySplits).bytes;
}

// The same estimate for plane-major spectra of N = 64 or 128 points (conv_split.hip), where
// transposeMM's matrix kernels take 4 k at a time (of 700 random layers it is within 20 % of 63 in 100, 10 % high
// in the middle).
static double planeMajorMicroseconds(int pass, int N, int B, int Cin, int Cout) {
  int I, J, K;
  passDims(pass, B, Cin, Cout, &I, &J, &K);
  const double planes = (double)I * K + (double)J * K + (double)I * J, XY = (N / 2 + 1) * (double)N;
  return 33 + 0.22e-6 * 2 * sizeof(float2) * planes * XY +
         0.033e-6 * XY * roundUp(I, 32) * (double)roundUp(J, 32) * roundUp(K, 4);
}

// The transform size a pass runs on, and how many ranges its reduction may be cut into.  A
// caller's size names the workspace; the same convolution cut into smaller windows - the
// library's own choice for the layer - is faster wherever the windows' spectra are clearly
// the smaller ones: a filter plane costs a quarter or less, and windows end nearer to the
// edge of an image that leaves much of the named transform empty.  That is also what keeps
// the windows within the workspace of the named size.
//
// 64 and 128 points (plane-major spectra of the whole image) give way to windows that hold
// no more spectrum and are not expected to take longer, with as many ranges of the reduction
// as there is room for.  Three passes, plane-major / windows: 32 x 32 x 60 x 60 images, 64
// filters of 5 x 5 216 / 145 us; 24 x 48 x 40 x 40, 96 of 8 x 8 339 / 151 us; 8 x 200 x 50 x
// 58, 300 of 1 x 1 2170 / 273 us; 128 points, 16 x 32 x 100 x 100, 64 of 8 x 8 490 / 207 us.
// Less spectrum alone does not make a weight gradient faster: its windows are longer
// reductions over tiles that many channels or few filters leave partly empty (64 points, 173 x
// 80 x 63 x 64, 362 of 3 x 3 1375 / 2000 us; 162 x 299 x 60 x 60, 115 of 6 x 6 1346 / 1796 us;
// 128 points, 93 x 193 x 122 x 119, 41 of 8 x 8 1360 / 1772 us), and where the planned ranges
// lack a little room (128 points, 153 x 3 x 73 x 70, 33 of 2 x 2: plane-major 308, 1 range 528,
// the 15 that fit 212 us; 64 points, 85 x 32 x 33 x 61, 66 of 7 x 7: 124, 1 range 241, the 3
// that fit 173 us, so plane-major).  Of 6570 random layers whose windows fit, 12 took over 3 %
// longer than plane-major by this rule (at most 18 %), 7 over 10 % longer than on windows; by
// the spectrum alone 59 took over 3 % longer, at most 45 %.  (Times and counts are those of the kernels
// that the estimates were fitted to.  On the present ones 699 of 700 random layers whose windows fit with
// all ranges run on windows, none of them over 3 % longer than plane-major, and the other is 18 % faster
// there; the 85 x 32 x 33 x 61 layer takes 128 / 126, 36 x 18 x 56 x 62, 107 of 8 x 8, 88 / 125.)  Filters larger than 32 or filling
// most of a window stay plane-major.
//
// 16 and 32 points are the same kernels on either side, and a caller who names them may mean
// them (size 0 is there for the fastest): they give way only where most of the named transforms
// would be padding, windows that need at most three fifths of the named size's workspace.  The
// line is drawn for that, not where the gain ends.  One pass, named 32 points / windows of n,
// us at the windows' share of that workspace: 32 x 64 x 27 x 27 images, 192 filters of 5 x 5,
// forward 56.6 / 32.1 (n = 16, 42 %), weight gradient 42.9 / 37.0 (16, 55 %); 64 x 96 x 13 x
// 13, 256 of 3 x 3, forward 91.7 / 34.3 (8, 15 %), input gradient 105.6 / 37.3 (16, 28 %);
// 2030 random layers below it 4 to 88 % faster.  Above it, given up: weight gradient 103.3 /
// 87.6 (61 %), forward 59.2 / 53.3 (84 %), 128 x 64 x 27 x 27, 192 of 5 x 5 99.6 / 91.0 (16, 80
// %); and no gain: weight gradient 16 x 32 x 100 x 100, 64 of 3 x 3 74.9 / 75.4 (16, 79 %),
// 128 x 192 x 27 x 27, 64 of 5 x 5 99.5 / 107.9 (16, 93 %).
//
// From 16 to 8 points the contraction has a quarter of the bins, 32, and small products leave
// most of the chip idle with one chain of slices each, whatever the spectra save (forward 28 x
// 45 x 8 x 9, 15 of 3 x 3, 16 / 8 points 14.8 / 16.6 us; input gradient 2 x 4 x 12 x 12, 50 of
// 1 x 1 14.8 / 16.4; weight gradient 4 x 310 x 25 x 25, 175 of 6 x 6 38.9 / 49.3): there the
// estimates must not differ by more than 5 % to the windows' disadvantage, either.  Of 5790
// random layers below the line 223 took over 3 % longer on 8 points and 66 over 10 %; by both
// tests 92 and 17 (30 x 243 x 14 x 11, 245 of 4 x 4, input gradient 47.2 / 59.0 the most).  With the
// contractions as they are now the second test keeps back more than it should: of 900 random layers below
// the line two take over 3 % longer on 8 points (11 % the most), and of the 127 that it keeps on 16 all would
// be 10 to 40 % faster; but the last of the three passes above takes 39.4 / 50.0.
PassSize passSize(int pass, int N, int B, int Cin, int Cout, int H, int W, int kH, int kW) {
  const PassSize named{N, kAnySplits};
  const int n = fbfft_conv_choose_fft_size(pass, B, Cin, Cout, H, W, kH, kW);
  if (n == 0 || n >= N) return named;
  const size_t room = convWorkspaceBytes(pass, N, B, Cin, Cout, H, W, kH, kW);
  if (N <= 32) {
    const WindowsCost c = windowsPass(pass, n, B, Cin, Cout, H, W, kH, kW, kAnySplits);
    if (c.bytes == 0 || c.bytes > room - room / 100 * 40) return named;
    if (N == 16 && c.us > 1.05 * windowsPass(pass, N, B, Cin, Cout, H, W, kH, kW, kAnySplits).us) return named;
    return {n, kAnySplits};
  }
  for (int maxSplits = kAnySplits; maxSplits > 0; --maxSplits) {
    const WindowsCost c = windowsPass(pass, n, B, Cin, Cout, H, W, kH, kW, maxSplits);
    if (c.bytes != 0 && c.bytes <= room)
      return c.us <= planeMajorMicroseconds(pass, N, B, Cin, Cout) ? PassSize{n, maxSplits} : named;
  }
  return named;
}

// Small layers need no transforms: convSmall (conv_small.hip) sums over the taps in one launch.
// They take the place of the transforms of the library's own choice of size, however a call comes
// to that (size 0, by its name, or in place of a larger named size), so that equal sizes still
// give equal bits; any other size that a call runs on is a transform of that size.
// Both times are estimated: its chain of filter rows on the fullest CU, and the three
// launches as above, less the 3 us by which that estimate is high where they are shortest; it
// has to be 15 % ahead.  us, the three launches / sums: forward 9 x 5 x 8 x 7, 9 filters of 3 x 3 11.2 /
// 3.9; 7 x 4 x 55 x 55, 10 of 2 x 2 19.2 / 6.1; 2 x 24 x 8 x 8, 338 of 2 x 2 13.7 / 4.8; 23 x 80 x 9 x 9, 25 of
// 3 x 3 14.3 / 11.2; input gradient 47 x 11 x 10 x 11, 143 of 1 x 1 26.2 / 6.4.  Not there: 5 x 17 x 9 x 9, 15 of 7 x 7 11.9 / 15; 1 x 64 x 27 x 27, 192 of 5 x 5 16.3 / 23.
// That leaves out a second round of workgroups on some CUs, loads whose lanes are in many images, and
// loads of rows that a wave does not have: 81 x 12 x 6 x 6, 22 of 6 x 6 10.8 / 18.6; 25 x 59 x 5 x 5, 75 of 4 x 4
// 14.4 / 23.8; input gradient 15 x 6 x 112 x 112, 2 of 2 x 9 28.7 / 41.5.
// So a second pair of estimates (convSmallMicroseconds, smallUs) must not see them behind by more than
// its error.  Of 2240 random passes that the first pair sends there 58 are over 10 % slower than on
// transforms; 14 of those are left, the most 38 %, and 8 go back that were over 10 % faster.
bool runsSmall(int pass, int N, int B, int Cin, int Cout, int H, int W, int kH, int kW) {
  const int C = pass == 0 ? Cin : Cout, M = pass == 0 ? Cout : Cin;
  if (pass == 2 || kW > 11 || (long)C * kH * kW > 2048) return false;
  const int OH = pass == 0 ? H - kH + 1 : H, OW = pass == 0 ? W - kW + 1 : W;
  const double full = std::max(1.0, std::ceil((double)B * OH * OW / 64) * ceilDiv(M, 8) / 256);
  if (full > 64) return false;
  const double chain = ceilDiv(C * kH, 8) * kW;
  const double sums = pass == 0 ? 3.1 + 0.88 * full + chain * (0.037 + 0.049 * full)
                                : 3.5 + 0.51 * full + chain * (0.033 + (0.072 + 0.025 / kW) * full);
  if (N != fbfft_conv_choose_fft_size(pass, B, Cin, Cout, H, W, kH, kW)) return false;
  const WindowsCost transforms = windowsPass(pass, N, B, Cin, Cout, H, W, kH, kW, kAnySplits);
  return sums < 0.85 * (transforms.us - 3) &&
         convSmallMicroseconds(pass, B, C, M, OH, OW, kH, kW) < 1.07 * transforms.smallUs;
}

// Whether a pass may take that way: it reads its operands while it writes its result, where the
// pipeline has read all of them before, so the result must not overlap them; a lane's offset
// within the images of its workgroup is counted in 31 bits of bytes.
static bool smallMayRun(const float* x, const int* xStride, const int* xSize, const float* y, const int* yStride,
                        const int* ySize, const float* out, const int* outStride, const int* outSize) {
  const auto last = [](const float* p, const int* stride, const int* size) {
    for (int d = 0; d < 4; ++d) p += (long)stride[d] * (size[d] - 1);
    return p;
  };
  for (int d = 0; d < 4; ++d)
    if (xStride[d] < 0 || yStride[d] < 0 || outStride[d] < 0) return false;
  const float* const end = last(out, outStride, outSize);
  if ((out <= last(x, xStride, xSize) && x <= end) || (out <= last(y, yStride, ySize) && y <= end)) return false;
  const double images = 64.0 / ((double)outSize[2] * outSize[3]) + 2;
  return images * xStride[0] + (double)xSize[2] * xStride[2] + (double)xSize[3] * xStride[3] < (1 << 29);
}

// Filters of 1 x 1 need no transform where the caller leaves the size to the library, or names one that gives
// way to it (64 and 128; 8 to 32 points name the transforms that they run on).  Each pass is one
// product then (conv_point.hip).  us, transforms / product, forward, input gradient, weight gradient: 45 x 79 x 118 x 118,
// 50 filters 283, 306, 326 / 93, 100, 124; 175 x 21 x 186 x 187, 21 723, 723, 852 / 210, 211, 218; 16 x 27 x 120 x 120, 100 91,
// 85, 123 / 31, 27, 39; 11 x 13 x 37 x 37, 298 28, (sums 14), 33 / 9, -, 16.
//
// But where results are few, up to a workgroup of 16 rows x 64 groups of pixels per CU, the product is one chain of loads over all
// contracted planes, 0.045 to 0.061 us each, while the windows' contraction is cut into ranges: there transforms that
// are expected to be faster keep the pass (the estimate is 10 to 50 % high in that range).  us, transforms / product, forward: 1 x 4000 x 4
// x 4, 64 filters 52 / 192; 64 x 1400 x 8 x 8, 256 69 / 83; but 64 x 1000 x 8 x 8, 256 55 / 51, 1 x 4100 x 28 x 28, 400 295 /
// 237; input gradient 64 x 64 x 8 x 8, 1000 28 / 47.
static bool runsPoint(int pass, int N, bool named, PassSize size, int B, int Cin, int Cout, int H, int W, int kH, int kW) {
  if (kH != 1 || kW != 1 || H * W < 4 || (named && N <= 32)) return false;
  if (pass == 2) return true;
  const int planes = pass == 0 ? Cin : Cout, rows = pass == 0 ? Cout : Cin;
  if (std::ceil((double)B * ceilDiv(H * W, 4) / 64) * ceilDiv(rows, 16) > computeUnits()) return true;
  const double transforms = size.N > 32 ? planeMajorMicroseconds(pass, size.N, B, Cin, Cout)
                                        : windowsPass(pass, size.N, B, Cin, Cout, H, W, 1, 1, size.maxSplits).us;
  return 3 + 0.055 * planes <= transforms / 1.2;
}

static_assert(ConvRoute::Windows + GemmPlan::Split + 1 == ConvRoute::Point, "each kind of contraction has a route");

ConvRoute convRoute(int pass, int N, int B, int Cin, int Cout, int H, int W, int kH, int kW) {
  const bool named = N != 0;
  if (!named) N = fbfft_conv_choose_fft_size(pass, B, Cin, Cout, H, W, kH, kW);
  const PassSize size = passSize(pass, N, B, Cin, Cout, H, W, kH, kW);
  if (runsSmall(pass, size.N, B, Cin, Cout, H, W, kH, kW)) return {ConvRoute::Small, size.N, 1};
  if (runsPoint(pass, N, named, size, B, Cin, Cout, H, W, kH, kW)) return {ConvRoute::Point, size.N, 1};
  if (size.N > 32) return {ConvRoute::PlaneMajor, size.N, 1};
  const GemmPlan plan = windowsPass(pass, size.N, B, Cin, Cout, H, W, kH, kW, size.maxSplits).plan;
  return {ConvRoute::Windows + plan.kind, size.N, plan.splits};
}

// pass 0: x = input [B][Cin][H][W], y = weight [Cout][Cin][kH][kW], out = output [B][Cout][oH][oW]
// pass 1: x = gradOutput [B][Cout][oH][oW], y = weight, out = gradInput [B][Cin][H][W]
// pass 2: x = input, y = gradOutput, out = gradWeight [Cout][Cin][kH][kW]
// strides in floats.  Images larger than the transform (N <= 32, by the caller's choice or by
// passSize's) are cut into overlapping windows that ride through the same three kernels as extra rows
// (passes 0 and 1) or extra reduction steps (pass 2).
int launchConvPass(int pass, int N, bool named, float* x, const int* xStride, const int* xSize, float* y,
                   const int* yStride, const int* ySize, float* out, const int* outStride,
                   const int* outSize, float scale, bool accumulate, void* workspace,
                   hipStream_t s) {
  const int* in = pass == 1 ? outSize : xSize;    // the layer's input / gradInput extents
  const int* wt = pass == 2 ? outSize : ySize;    // the filter extents
  const int H = in[2], W = in[3], kH = wt[2], kW = wt[3];
  const PassSize size = passSize(pass, N, in[0], wt[1], wt[0], H, W, kH, kW);
  const int given = N;
  N = size.N;
  if (runsSmall(pass, N, in[0], wt[1], wt[0], H, W, kH, kW) &&
      smallMayRun(x, xStride, xSize, y, yStride, ySize, out, outStride, outSize))
    return launchConvSmall(pass, x, xStride, xSize, y, yStride, ySize, out, outStride, outSize, s);
  if (runsPoint(pass, given, named, size, in[0], wt[1], wt[0], H, W, kH, kW) &&
      pointMayRun(pass, x, xStride, xSize, y, yStride, ySize, out, outStride, outSize))
    return launchConvPoint(pass, x, xStride, xSize, y, yStride, ySize, out, outStride, outSize, scale, accumulate,
                           workspace, pass == 2 ? convWorkspaceBytes(2, given, in[0], wt[1], wt[0], H, W, 1, 1) : 0, s);
  if (N > 32)
    return launchConvSplit(pass, N, x, xStride, xSize, y, yStride, ySize, out, outStride, outSize,
                           scale, accumulate, workspace, s);
  PlaneSet px, py, po;
  if (pass == 0) {
    px = planes(x, xStride, xSize, 0, 1);
    py = planes(y, yStride, ySize, 0, 1);
    po = planes(out, outStride, outSize, 0, 1);
  } else if (pass == 1) {
    px = planes(x, xStride, xSize, 0, 1);
    py = planes(y, yStride, ySize, 1, 0);
    po = planes(out, outStride, outSize, 0, 1);
  } else {
    px = planes(x, xStride, xSize, 1, 0);
    py = planes(y, yStride, ySize, 1, 0);
    po = planes(out, outStride, outSize, 1, 0);
  }
  int ty, tx;
  tileGrid(pass, N, H, W, kH, kW, &ty, &tx);
  if (ty * tx > 1) {
    const int stepY = N - kH + 1, stepX = N - kW + 1;
    if (pass == 0) {
      tile(px, true, ty, tx, stepY, stepX, 0, 0, N, N);
      tile(po, true, ty, tx, stepY, stepX, 0, 0, stepY, stepX);
    } else if (pass == 1) {
      // gradInput rows y0 .. y0+step-1 are a full convolution over gradOutput rows
      // y0-(kH-1) .. y0+step-1; the result for row y0 then sits in plane row kH-1,
      // clear of the circular wrap-around
      tile(px, true, ty, tx, stepY, stepX, -(kH - 1), -(kW - 1), N, N);
      tile(po, true, ty, tx, stepY, stepX, 0, 0, stepY, stepX);
      po.padU0 = kH - 1;
      po.padL0 = kW - 1;
    } else {
      tile(px, false, ty, tx, stepY, stepX, 0, 0, N, N);
      tile(py, false, ty, tx, stepY, stepX, 0, 0, stepY, stepX);
    }
  }
  float2* ws = static_cast<float2*>(workspace);
  switch (N) {
    case 8: return runPass<8>(pass, px, py, po, scale, accumulate, ws, s, size.maxSplits);
    case 16: return runPass<16>(pass, px, py, po, scale, accumulate, ws, s, size.maxSplits);
    case 32: return runPass<32>(pass, px, py, po, scale, accumulate, ws, s, size.maxSplits);
  }
  return FBFFT_UNSUPPORTED_SIZE;
}

// FFTIteratedConvolution's operands - device arrays of tile descriptors - through the
// same three kernels: tile t of ins / outs is a [batch][planes][h][w] view with its own
// strides and pads, the (image, tile) pairs ride as rows (passes 0 and 1) or as
// reduction steps (pass 2).  Roles as in iterated_conv.hip's table: pass 0
// outs[t](n, f) = sum_c ins[t](n, c) * conj(weight(f, c)), pass 1 ins[t](n, c) =
// sum_f outs[t](n, f) * weight(f, c), pass 2 weight(f, c) = scale * sum_(t, n)
// ins[t](n, c) * conj(outs[t](n, f)); results land at (padU, padL) of the destination's
// plane.  The descriptors are only read on the device.
size_t describedWorkspaceBytes(int pass, int N, long rows, int Cin, int Cout) {
  if (rows <= 0 || rows > (1L << 30)) return 0;
  int I, J, K;
  passDims(pass, (int)rows, Cin, Cout, &I, &J, &K);
  const bool outTiled = pass != 2;
  const size_t n = N == 8 ? workspaceFloat2<8>(I, J, K, outTiled)
                          : N == 16 ? workspaceFloat2<16>(I, J, K, outTiled)
                                    : workspaceFloat2<32>(I, J, K, outTiled);
  return n * sizeof(float2);
}

int launchDescribedConv(int pass, int N, const fbfft_tile* ins, const fbfft_tile* outs, float* weight,
                        const int* wStride, const int* wSize, float scale, int batch, int numTiles,
                        void* workspace, hipStream_t s) {
  const int Cout = wSize[0], Cin = wSize[1];
  auto described = [&](const fbfft_tile* tiles, bool compositeIsRow, int planes) {
    PlaneSet p{};
    p.tiles = tiles;
    p.described = compositeIsRow ? 1 : 2;
    p.numTiles = numTiles;
    (compositeIsRow ? p.R : p.K) = numTiles * batch;
    (compositeIsRow ? p.K : p.R) = planes;
    return p;
  };
  float* w = weight;
  PlaneSet px, py, po;
  if (pass == 0) {
    px = described(ins, true, Cin);
    py = planes(w, wStride, wSize, 0, 1);
    po = described(outs, true, Cout);
  } else if (pass == 1) {
    px = described(outs, true, Cout);
    py = planes(w, wStride, wSize, 1, 0);
    po = described(ins, true, Cin);
  } else {
    px = described(ins, false, Cin);
    py = described(outs, false, Cout);
    po = planes(w, wStride, wSize, 1, 0);
  }
  float2* ws = static_cast<float2*>(workspace);
  const float sc = pass == 2 ? scale : 1.0f;
  switch (N) {
    case 8: return runPass<8>(pass, px, py, po, sc, false, ws, s);
    case 16: return runPass<16>(pass, px, py, po, sc, false, ws, s);
    case 32: return runPass<32>(pass, px, py, po, sc, false, ws, s);
  }
  return FBFFT_UNSUPPORTED_SIZE;
}

}  // namespace fbfft_amd
