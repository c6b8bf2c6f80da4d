// Dense and grouped convolution of any window, stride and dilation as an implicit GEMM on the matrix cores, one output
// tile per workgroup, for int8 / uint8, float16 and float32 tensors - vxConvolutionLayer as ovxlib reaches it for those
// (reference: src/tim/vx/internal/src/ops/vsi_nn_op_conv2d.c:35-118, vsi_nn_op_grouped_conv2d.c).
//
// A tile is TW x TH output pixels of one image (whole small images: G of them) times 32 .. 128 output channels of one
// group. The input window behind it - halo included, padding as the input's zero point - is transposed into LDS once as
// [row][column][channel]: a work item loads eight pixels (four of float32) of a 16-byte granule of channels (16 int8, 8 float16 or 4 float32
// planes), all of its loads in flight together, and stores as many 16-byte units, so that a reduction step of the matrix
// core is one 16-byte LDS read per lane at (tap, granule) for every element type. A step's two granules need not belong
// to one tap: a table gives their LDS offsets, and shallow inputs (one granule a pixel) waste half of nothing.
// The weights are packed in fragment order when the operator is created and stream from L2 straight into registers a
// group of steps ahead; they need no LDS, so the whole channel depth of a tile usually fits (else it is walked in chunks).
// Results leave through LDS in runs of a whole tile or row per channel: sixteen bytes a lane straight from the accumulators, each in
// a cache line of its own, wrote 0.5 TB/s (int8 62 -> 144 channels, 3x3 on 73 x 73, batch 48: 100 -> 82 us; float16 29 -> 304 on
// 141 x 141, batch 3: 48 -> 41; float32 3 -> 16 on 132 x 132, batch 10: 15.9 -> 12.5).
// Where several blocks of output channels follow from one window and there are workgroups enough without them, a workgroup takes
// them one after the other over the window it has staged: 8 -> 240 channels 3x3 on 157 x 157, batch 11, 69 -> 49 us; 80 -> 352 on
// 66 x 66, batch 23, 76 -> 62.
// Quantized tensors under a weight zero point need the sum of every window. Where a wavefront has few steps a lane adds up the bytes of the
// fragments it multiplies, four dot products each (kSumsInLoop), and the lanes, halves and shares of a pixel meet in LDS; where it has many
// the staged pixels' channels are summed once and box-filtered per tile (kSumsBox), nothing in the loop.
//
// What bounds it: at the sizes convolutional networks have, a launch is a chain of one memory round trip, the LDS
// transposition (about 70 vector instructions per 64 staged bytes for int8, none for float32) and the steps themselves, and no unit
// is busy for long: int8 3x3 256 -> 256 on 14 x 14, batch 32, 11.2 us under the tracer: matrix cores and vector units 20 % of a CU's cycles each, LDS 28 and
// 10 of bank conflicts, wavefronts waiting 48 % of theirs; float16 5x5 96 -> 256 on 27 x 27, batch 16, 26.5 us: 35, 27, 60 and 32, 31. What a phase needs of the arguments is read when it begins (LateArgs), its first loads' addresses
// come first, and a chunk's odd last step is looked for behind the main loop: int8 80 -> 9 channels, 3x3 on 21 x 21, batch 15, 8.1 -> 6.4 us;
// 288 -> 40, 3x3 at stride 2 on 98 x 65, batch 22, 54 -> 43; float16 3 -> 48, 7x7 on 142 x 142, batch 16, 33 -> 28. The tile is chosen on the
// host so that the chip is filled first and the halo staged per output pixel is small second.
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>

#include "variants.h"

namespace tvx {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));

constexpr int kI8 = 0, kF16 = 1, kF32 = 2;  // element kinds (uint8 runs as int8 with its sign bit flipped)
constexpr int kNoSums = 0, kSumsInLoop = 1, kSumsBox = 2;
constexpr int kMostAhead = 8;  // steps whose weights are on their way to a wavefront at a time, at most (R)

// In the order of their use: what comes before a launch's first loads is fetched together (LateArgs).
struct TileArgs {
  const uint8_t* x;
  int total, per_xcd;
  int oc_wgs, wgs_per_group, loop;  // workgroups that the channel blocks take, of all groups and of one; channel blocks that a workgroup takes one after the other
  int tiles_x, tiles_y;
  uint32_t m_ocb, m_tpg, m_tx, m_ty;  // reciprocals: u / d = mulhi(u, m), exact for the ranges used
  int TW, TH, G;           // tile: columns, rows, images
  int sh, sw, pad_t, pad_l;
  int icg;                 // input channels of a group
  int gpc;                 // granules of a pixel per chunk
  int items;               // work items of a chunk
  int gl, cells, cells4, ncg, IH;  // granules neighbouring lanes take (a divisor of gpc); column groups of all staged rows, fours of them, groups of a row; staged rows per image
  uint32_t m_gl, m_cells4, m_ncg, m_ih;
  int row_step, H, W, batch;  // row_step: input rows between staged rows
  int at_max;              // last place of a plane where a work item's pixels can be read
  uint32_t plane_bytes, image_bytes;
  int IW, pitch;           // staged columns; LDS bytes of a staged pixel: an odd number of granules (bank spread)
  uint32_t xor_mask;
  // ---- under the first loads
  const v4i* wpk;          // [group][32-channel tile][chunk][step][64 lanes]: sixteen bytes of reduction per lane
  const int* tab;          // [half][steps_pad]: LDS byte offset of the granule a lane of that half multiplies at a step
  int steps, steps_pad, odd;  // reduction steps of a chunk, and padded for what is read ahead; the last step's upper half is empty
  int chunks, tiles_per_group;
  int row_stride, NQ, npx;  // staged rows between output rows; pixels of the tile; staged pixels
  uint32_t m_iw, m_tw, m_thtw;
  uint32_t pad_full, pad_last[4];  // a padding granule: full, and the channels' last one
  int last_granule;        // global index of the channels' last granule
  int off_tab, off_sum, off_zt, off_out;  // LDS carve-up behind the staged window; the results (over the window where it is used once)
  int zws;                 // weight zero point in the signed domain (0: no window sums)
  // ---- behind the multiplications
  uint8_t* y;
  const int32_t* biasf;    // quantized: bias with the zero-point terms folded in, per padded output channel
  const float* biasfl;     // floating point: the bias, or null
  const tvx_v4i* rq;
  int OC, OH, OW, ocg;     // ocg: output channels of a group
  int taps_w, taps_h, dil_col, dil_row;  // for the box sum: LDS pixels between taps
  int runs, run_px, run_out, out_pitch;  // copy-out: runs of consecutive outputs of a channel, their pixels and distance; LDS bytes of a channel
  int stack;               // output rows that a tile's row stands for (STACK), the channels of each behind one another
  uint32_t m_ocg, m_th;
  uint32_t m_run4;         // reciprocal of a run's groups of four pixels
  int runs_shift;          // log2 of the threads that a channel's runs take
  uint32_t m_run_wide;     // the same with sixteen bytes a thread
  int wide_shift;
  int pre_ties;            // accumulators' left shift (BuildTieRecords) * 2 + whether ties are possible
  int lo, hi, narrow, out_xor, act;  // quantized: clamp in the signed domain, whether it is narrower than a byte; 0x80808080 for uint8 results
};

// (a sum and not a choice of two: that became a branch per division)
__device__ __forceinline__ int DivM(int u, uint32_t m) {
  const uint32_t one = m ? 0u : ~0u;
  return static_cast<int>(__umulhi(static_cast<uint32_t>(u), m) + (static_cast<uint32_t>(u) & one));
}

template <int DT> struct Kind;
template <> struct Kind<kI8> { using acc = v16i; using elem = int; static constexpr int E = 1; };
template <> struct Kind<kF16> { using acc = v16f; using elem = float; static constexpr int E = 2; };
template <> struct Kind<kF32> { using acc = v16f; using elem = float; static constexpr int E = 4; };

template <int DT>
__device__ __forceinline__ void Multiply(typename Kind<DT>::acc& acc, const v4i& fx, const v4i& fw) {
  if constexpr (DT == kI8) {
    acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(fx, fw, acc, 0, 0, 0);
  } else if constexpr (DT == kF16) {
    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, fx), __builtin_bit_cast(v8h, fw), acc, 0, 0, 0);
  } else {
    const v4f a = __builtin_bit_cast(v4f, fx), b = __builtin_bit_cast(v4f, fw);
#pragma unroll
    for (int j = 0; j < 4; ++j) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[j], b[j], acc, 0, 0, 0);
  }
}

// N bytes at a scalar base and a lane's offset. The base is made anew for every load (sixteen of them kept over a loop are spilled, a lane
// address for each is three instructions) and named global memory: behind the empty assembly the compiler knows no address space and takes
// flat loads, which wait for LDS as well.
typedef const __attribute__((address_space(1))) uint8_t* GlobalBytes;
template <int N>
__device__ __forceinline__ void Fetch(uint32_t* d, const uint8_t*& base, uint32_t at) {
  asm volatile("" : "+s"(base));
  __builtin_memcpy(d, (const void*)((GlobalBytes)base + at), N);
}

// One work item on its way: P consecutive pixels of a row x one granule of channel planes.
template <int DT> struct Item {
  static constexpr int E = Kind<DT>::E;
  static constexpr int N = 16 / E;            // channel planes
  static constexpr int P = DT == kF32 ? 4 : 8;  // pixels: 8 or 16 bytes of a plane
  static constexpr int D = P * E / 4;         // dwords of a plane
  uint32_t d[N * D];

  // FULL: all planes exist; else planes past the last valid one re-read it (masked behind Unit)
  template <bool FULL>
  __device__ __forceinline__ void Load(const uint8_t* base, uint32_t at, uint32_t plane_bytes, int valid) {
    const uint8_t* plane = base;
#pragma unroll
    for (int c = 0; c < N; ++c) {
      if (FULL) {
        Fetch<4 * D>(&d[c * D], plane, at);
        plane += plane_bytes;
      } else {
        __builtin_memcpy(&d[c * D], base + (at + static_cast<uint32_t>(min(c, valid - 1)) * plane_bytes), 4 * D);
      }
    }
  }
  // a granule that holds all the channels there are (uniform): the planes behind them are not loaded but zero
  __device__ __forceinline__ void LoadFew(const uint8_t* base, uint32_t at, uint32_t plane_bytes, int valid) {
    const uint8_t* plane = base;
#pragma unroll
    for (int c = 0; c < N; ++c) {
      if (c < valid) {
        Fetch<4 * D>(&d[c * D], plane, at);
        plane += plane_bytes;
      } else {
#pragma unroll
        for (int i = 0; i < D; ++i) d[c * D + i] = 0;
      }
    }
  }
  // the granules of pixels 4 g .. 4 g + 3
  __device__ __forceinline__ void Units(int g, v4i (&u)[4]) const {
    if constexpr (DT == kI8) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const uint32_t in[4] = {d[4 * q * D + g], d[(4 * q + 1) * D + g], d[(4 * q + 2) * D + g], d[(4 * q + 3) * D + g]};
        uint32_t out[4];
        Transpose4x4(in, out);
#pragma unroll
        for (int i = 0; i < 4; ++i) u[i][q] = static_cast<int>(out[i]);
      }
    } else if constexpr (DT == kF16) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const uint32_t a0 = d[2 * q * D + 2 * g], a1 = d[2 * q * D + 2 * g + 1], b0 = d[(2 * q + 1) * D + 2 * g], b1 = d[(2 * q + 1) * D + 2 * g + 1];
        u[0][q] = static_cast<int>(__builtin_amdgcn_perm(b0, a0, 0x05040100));
        u[1][q] = static_cast<int>(__builtin_amdgcn_perm(b0, a0, 0x07060302));
        u[2][q] = static_cast<int>(__builtin_amdgcn_perm(b1, a1, 0x05040100));
        u[3][q] = static_cast<int>(__builtin_amdgcn_perm(b1, a1, 0x07060302));
      }
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int i = 0; i < 4; ++i) u[i][q] = static_cast<int>(d[q * D + i]);
    }
  }
};

// WM x WN wavefronts share the tile's pixels and channels (MT x NT MFMA tiles each), KS wavefronts a tile's reduction.
// R: steps whose weights are on their way to a wavefront at a time.
// STACK: up to 16 output channels of quantized tensors would leave half of a tile's 32 and more empty. The channels of several output rows
// stand behind one another there instead: a tile's row is `stack` rows of the image, its window as much taller, and each row's weights lie at its
// own taps among the weights' zero point (which drops out with the window sums; a zero of floating point would not under an infinity).
// Three rows of 3x3 take 5 / 9 of the multiplications, LDS reads and weights, two rows of 5x5 3 / 5: int8 144 -> 16 in four groups, 3x3 on 125 x 125, batch 29: 87.7 -> 41.1 us; uint8 160 -> 16, 7x7 on 134 x 134, batch 14, 116.9 -> 87.7.
// (Kernels of their own: the rows' places cost the others .1 to .2 us a launch.)
template <int DT, int SUMS, int WM, int WN, int KS, int MT, int NT, int R, int EU, bool MULTI, bool STACK>
__global__ void __launch_bounds__(64 * WM * WN * KS) __attribute__((amdgpu_waves_per_eu(EU))) ConvTileKernel(TileArgs a) {
  constexpr int kThreads = 64 * WM * WN * KS;
  static_assert(R % 2 == 0 && R <= kMostAhead, "the activations' two buffers alternate with the steps");
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  using acc_t = typename Kind<DT>::acc;
  using elem_t = typename Kind<DT>::elem;
  using item_t = Item<DT>;
  constexpr int E = Kind<DT>::E, P = item_t::P;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // consecutive workgroups of an XCD: the channel blocks of a tile, then the next tile
  const int id = static_cast<int>(blockIdx.x & 7) * a.per_xcd + static_cast<int>(blockIdx.x >> 3);
  if (id >= a.total) return;
  const int tile = DivM(id, a.m_ocb), ocb = id - tile * a.oc_wgs;
  const int group = DivM(ocb, a.m_tpg);
  int ocl = (ocb - group * a.wgs_per_group) * a.loop;  // channel block of the group
  const int tyn = DivM(tile, a.m_tx), tx = tile - tyn * a.tiles_x;
  const int tn = DivM(tyn, a.m_ty), ty = tyn - tn * a.tiles_y;
  const int n0 = tn * a.G;
  const int x0 = tx * a.TW, y0 = ty * a.TH;
  const int ix0 = x0 * a.sw - a.pad_l, iy0 = y0 * a.sh - a.pad_t;
  // window columns inside the image (none where the window lies in padding altogether: the stores' unsigned range needs hi >= lo)
  const int col_lo = max(0, -ix0), col_hi = max(col_lo, min(a.IW, a.W - ix0));

  const int row = lane & 31, half = lane >> 5;
  const int ks = wave % KS, wn = wave / KS % WN, wm = wave / KS / WN;
  uint32_t base[MT];  // LDS byte offset of this lane's pixel in each pixel tile
  acc_t acc[MT][NT];
  int xs[MT];  // kSumsInLoop: sums of the bytes multiplied
  v4i fw[R][NT];

  // A work item's place: an item = (granule, column group, row); lanes take four cells of a plane (contiguous in memory where the rows are
  // whole), then these of gl granules, then the next four cells, then the next gl granules. Four neighbouring lanes are what the L1 looks up
  // at once: with the granules innermost each of the four was a line of its own, and a wavefront's load took 64 clocks of the L1 instead of
  // 16 (int8 3x3 272 -> 64 on 55 x 70, batch 13: 25.0 -> 22.9 us); with cells alone innermost the LDS stores, 128 bytes apart, meet in two banks.
  struct Where { uint32_t at; int to, col, valid; bool inside; };
  auto find = [&](const TileArgs& a, int it, int c0) {
    Where w;
    const bool live = it < a.items;
    const int itc = live ? it : 0, four = itc >> 2;
    const int rest = DivM(four, a.m_gl), gl = four - __mul24(rest, a.gl);
    const int gh = DivM(rest, a.m_cells4), cell = (rest - __mul24(gh, a.cells4)) * 4 + (itc & 3);
    const int gr = __mul24(gh, a.gl) + gl;
    const int r = DivM(cell, a.m_ncg), cg = cell - __mul24(r, a.ncg);
    const int g = DivM(r, a.m_ih), ry = r - __mul24(g, a.IH);
    const int iy = iy0 + __mul24(ry, a.row_step), ixs = ix0 + P * cg;
    w.inside = live && cell < a.cells && static_cast<unsigned>(iy) < static_cast<unsigned>(a.H) && ixs > -P && ixs < a.W && n0 + g < a.batch;
    w.valid = min(a.icg - c0 - gr * (16 / E), 16 / E);  // channels of the granule
    // P pixels from the group's first column inside the image, further in front at the plane's end: what lies outside
    // the row is not stored, what the neighbouring group stores too is the same
    const int px = min(iy * a.W + max(ixs, 0), a.at_max);
    w.col = px - iy * a.W - ix0;  // window column of the first pixel
    w.at = w.inside && w.valid > 0 ? static_cast<uint32_t>(g) * a.image_bytes + static_cast<uint32_t>(gr * (16 / E)) * a.plane_bytes + static_cast<uint32_t>(px) * E : 0u;
    w.to = __mul24(__mul24(r, a.IW) + w.col, a.pitch) + gr * 16;
    return w;
  };
  auto store = [&](const TileArgs& a, const item_t& item, const Where& w, bool all_full) {
    if (!w.inside) return;
    uint8_t* to = lds + w.to;
    v4i mask;
    if (!all_full)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int nb = w.valid * E - 4 * q;
        mask[q] = nb >= 4 ? -1 : nb <= 0 ? 0 : static_cast<int>((1u << (8 * nb)) - 1u);
      }
#pragma unroll
    for (int h = 0; h < P / 4; ++h) {
      v4i u[4];
      item.Units(h, u);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (DT == kI8) u[i] ^= static_cast<int>(a.xor_mask);
        if (!all_full) u[i] &= mask;
        if (static_cast<unsigned>(w.col + 4 * h + i - col_lo) < static_cast<unsigned>(col_hi - col_lo)) *reinterpret_cast<v4i*>(to + (4 * h + i) * a.pitch) = u[i];
      }
    }
  };

  // a wavefront's share of a chunk's steps, and its weights for a block of channels
  struct Steps { int s0, s1; const v4i* wp; uint32_t tile_stride; };
  auto share = [&](const TileArgs& a) {
    Steps w;
    const int per = (a.steps + KS - 1) / KS;
    w.s0 = KS == 1 ? 0 : min(ks * per, a.steps);
    w.s1 = KS == 1 ? a.steps : min(w.s0 + per, a.steps);
    w.tile_stride = static_cast<uint32_t>((MULTI ? a.chunks : 1) * a.steps) * 64;
    w.wp = a.wpk + static_cast<size_t>((group * a.tiles_per_group + ocl) * (WN * NT) + wn * NT) * w.tile_stride + lane;
    return w;
  };
  auto fetch_w = [&](const Steps& w, int first, int s, v4i (&f)[NT]) {
    const uint32_t at = static_cast<uint32_t>(first + max(min(s, w.s1 - 1), 0)) * 64;  // (past the end: the last step once more, not multiplied)
#pragma unroll
    for (int t = 0; t < NT; ++t) f[t] = w.wp[t * w.tile_stride + at];
  };
  // ---- stage a chunk's window. `a`: what the first loads need; `late()`: the rest ----
  // (lanes without an item stay out: reading some valid address instead kept the L1 busy as long as an item does, 0.97 of the time without on 400
  // drawn layers, int8 32 -> 16, 5x5 on 65 x 65, batch 24, 12.3 -> 9.8 us)
  auto load = [&](const TileArgs& a, const uint8_t* xg, bool all_full, item_t& item, const Where& w) {
    if (!w.inside) return;
    if (all_full) item.template Load<true>(xg, w.at, a.plane_bytes, 16 / E);
    else if (a.icg < 16 / E) item.LoadFew(xg, w.at, a.plane_bytes, a.icg);
    else item.template Load<false>(xg, w.at, a.plane_bytes, max(w.valid, 1));
  };
  auto stage = [&](const TileArgs& a, auto late, int chunk) {
    const int c0 = chunk * a.gpc * (16 / E);  // first channel of the chunk
    const uint8_t* xg = a.x + static_cast<size_t>(n0) * a.image_bytes + static_cast<size_t>(group * a.icg + c0) * a.plane_bytes;
    const bool all_full = c0 + a.gpc * (16 / E) <= a.icg;  // uniform: every granule of the chunk has all its channels
    item_t item;
    Where where = find(a, tid, c0);
    load(a, xg, all_full, item, where);
    // under the first loads: the first weights, the table, the lanes' pixels, the padding
    const TileArgs& b = late();
    const int tab_n = 2 * b.steps_pad;
    const int tab_first = b.tab[min(tid, tab_n - 1)];
    if (!MULTI) {
      const Steps w = share(b);
#pragma unroll
      for (int u = 0; u < R; ++u) fetch_w(w, 0, w.s0 + u, fw[u]);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (chunk == 0) {
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const int q = min((wm * MT + m) * 32 + row, b.NQ - 1);  // (pixels past the tile's end repeat its last one and are not stored)
        const int qg = DivM(q, b.m_thtw), rem = q - __mul24(qg, b.TH * b.TW);
        const int qy = DivM(rem, b.m_tw), qx = rem - __mul24(qy, b.TW);
        base[m] = static_cast<uint32_t>(__mul24(__mul24(__mul24(qg, b.IH) + __mul24(qy, b.row_stride), b.IW) + __mul24(qx, b.sw), b.pitch));
      }
    }
    if (ix0 < 0 || ix0 + b.IW > b.W || iy0 < 0 || iy0 + (b.IH - 1) * b.row_step >= b.H) {  // uniform: the window leaves the image
      const int pad_whole = max(0, min(b.last_granule - chunk * b.gpc, b.gpc));
      const int pf = static_cast<int>(b.pad_full);
      const v4i pad_unit = {pf, pf, pf, pf};
      const v4i pad_tail = {static_cast<int>(b.pad_last[0]), static_cast<int>(b.pad_last[1]), static_cast<int>(b.pad_last[2]), static_cast<int>(b.pad_last[3])};
      for (int p = tid; p < b.npx; p += kThreads) {
        const int pr = DivM(p, b.m_iw), cx = p - __mul24(pr, b.IW);
        const int pry = pr - __mul24(DivM(pr, b.m_ih), b.IH);
        const int py = iy0 + __mul24(pry, b.row_step);
        if (static_cast<unsigned>(py) < static_cast<unsigned>(b.H) && cx >= col_lo && cx < col_hi) continue;
        v4i* to = reinterpret_cast<v4i*>(lds + __mul24(p, b.pitch));
        for (int pg = 0; pg < pad_whole; ++pg) to[pg] = pad_unit;
        if (pad_whole < b.gpc) {  // uniform: the chunk holds the channels' last granule (and empty ones)
          to[pad_whole] = pad_tail;
          for (int pg = pad_whole + 1; pg < b.gpc; ++pg) to[pg] = v4i{0, 0, 0, 0};
        }
      }
    }
    if (chunk == 0) {
      int* tab = reinterpret_cast<int*>(lds + b.off_tab);
      if (tid < tab_n) tab[tid] = tab_first;
      for (int i = tid + kThreads; i < tab_n; i += kThreads) tab[i] = b.tab[i];
      if (SUMS == kSumsInLoop && tid < WM * MT * 32) reinterpret_cast<int*>(lds + b.off_zt)[tid] = 0;
    }
    store(b, item, where, all_full);
#pragma unroll 1
    for (int it0 = kThreads; it0 < b.items; it0 += kThreads) {
      where = find(b, it0 + tid, c0);
      load(b, xg, all_full, item, where);
      store(b, item, where, all_full);
    }
    if (MULTI) {  // (beside accumulators, an item's planes and its results the weights would need more registers than two workgroups a CU leave)
      const Steps w = share(b);
#pragma unroll
      for (int u = 0; u < R; ++u) fetch_w(w, chunk * b.steps, w.s0 + u, fw[u]);
      __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();
    if (SUMS == kSumsBox) {  // channel sums of the staged pixels
      int* sum = reinterpret_cast<int*>(lds + b.off_sum);
      for (int p = tid; p < b.npx; p += kThreads) {
        int v = chunk ? sum[p] : 0;
        for (int gr = 0; gr < b.gpc; ++gr) {
          const v4i f = *reinterpret_cast<const v4i*>(lds + __mul24(p, b.pitch) + gr * 16);
#pragma unroll
          for (int q = 0; q < 4; ++q) v = __builtin_amdgcn_sdot4(f[q], 0x01010101, v, false);
        }
        sum[p] = v;
      }
    }
  };

  // MULTI: a pass is a chunk of the channels, the results follow the last. Else: a pass is a block of output channels over the
  // same staged window.
  const int loop = a.loop;
  stage(a, []() -> const TileArgs& { return LateArgs<TileArgs>(); }, 0);
  const TileArgs& b = LateArgs<TileArgs>();
  for (int pass = 0;; ++pass) {
    const int chunk = MULTI ? pass : 0;
    if (MULTI && chunk) {
      __syncthreads();  // the window is free
      stage(b, [&]() -> const TileArgs& { return b; }, chunk);
    }
    const int passes = MULTI ? b.chunks : min(loop, b.tiles_per_group - ocl + pass);
    const Steps w = share(b);
    const int s0 = w.s0, s1 = w.s1;
    if (!MULTI || chunk == 0)
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        xs[m] = 0;
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
          for (int i = 0; i < 16; ++i) acc[m][t][i] = 0;
      }
    // ---- multiply: R steps' weights ahead, two steps' activations, R steps' offsets of those. The order inside a step is kept by hand: left
    // to itself the compiler put an offset and the activations behind it in front of the multiplication that waits for them ----
    const int* tab = reinterpret_cast<const int*>(lds + b.off_tab) + half * b.steps_pad + s0;
    v4i fx[2][MT];
    int off[R];
    auto fetch_x = [&](int o, v4i (&f)[MT]) {
#pragma unroll
      for (int m = 0; m < MT; ++m) f[m] = *reinterpret_cast<const v4i*>(lds + base[m] + o);
    };
    auto multiply = [&](const v4i (&f)[MT], const v4i (&w)[NT]) {
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int t = 0; t < NT; ++t) Multiply<DT>(acc[m][t], f[m], w[t]);
      if (SUMS == kSumsInLoop)
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
          for (int q = 0; q < 4; ++q) xs[m] = __builtin_amdgcn_sdot4(f[m][q], 0x01010101, xs[m], false);
    };
    const v4i* wp = w.wp + static_cast<uint32_t>(chunk * b.steps + s0) * 64;
#pragma unroll
    for (int u = 0; u < 2; ++u) fetch_x(tab[u], fx[u]);
#pragma unroll
    for (int u = 0; u < R; ++u) off[u] = tab[2 + u];  // (the table is padded)
    int s = s0;
#pragma unroll 1
    for (; s + R < s1; s += R) {
      wp += R * 64;
      tab += R;
#pragma unroll
      for (int u = 0; u < R; ++u) {
        __builtin_amdgcn_sched_barrier(0);
        multiply(fx[u & 1], fw[u]);  // (a chunk's last step is below)
#pragma unroll
        for (int t = 0; t < NT; ++t) fw[u][t] = wp[t * w.tile_stride + u * 64];  // (past the share's end: not multiplied; the array is padded)
        fetch_x(off[u], fx[u & 1]);
        if (u & 1) {
          off[u - 1] = tab[2 + u - 1];
          off[u] = tab[2 + u];
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int u = 0; u < R; ++u)
      if (s + u < s1) {  // uniform
        if ((DT != kI8 || SUMS == kSumsInLoop) && b.odd && s + u == b.steps - 1 && half)  // (zero weights, but the data may be an infinity, or is summed up)
#pragma unroll
          for (int m = 0; m < MT; ++m) fx[u & 1][m] = v4i{0, 0, 0, 0};
        multiply(fx[u & 1], fw[u]);
        fetch_x(off[u], fx[u & 1]);
      }
    if (MULTI && pass + 1 < passes) continue;
    if (!MULTI && pass + 1 < passes) {  // the next block's first weights travel under the results
      Steps next = w;
      next.wp += static_cast<uint32_t>(WN * NT) * w.tile_stride;
#pragma unroll
      for (int u = 0; u < R; ++u) fetch_w(next, 0, s0 + u, fw[u]);
    }

    const TileArgs& c = LateArgs<TileArgs>();
    // the epilogue's tables travel while the wavefronts meet
    int bias[NT];
    tvx_v4i rq[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int oc = (ocl * WN + wn) * NT * 32 + t * 32 + row;  // channel of the group
      if constexpr (DT == kI8) {
        const int slot = group * c.tiles_per_group * (WN * NT * 32) + oc;
        rq[t] = c.rq[slot];
        bias[t] = c.biasf[slot];
      } else {
        bias[t] = c.biasfl && oc < c.ocg ? reinterpret_cast<const int*>(c.biasfl)[group * c.ocg + oc] : 0;
      }
    }

    // ---- wavefronts that split a reduction exchange partial sums: an accumulator tile is cut into pieces (pairs of quads
    // that become eight consecutive pixels, or single quads), every wavefront finishes its own ----
    constexpr int kQuads = KS == 1 ? 4 : (2 * MT * NT >= KS ? 2 : 1);  // quads of a piece
    constexpr int kPieces = 4 / kQuads;
    if (SUMS == kSumsInLoop && (MULTI || pass == 0) && wn == 0) {
#pragma unroll
      for (int m = 0; m < MT; ++m) atomicAdd(reinterpret_cast<int*>(lds + c.off_zt) + (wm * MT + m) * 32 + row, -c.zws * xs[m]);
    }
    const bool box = SUMS == kSumsBox && (MULTI || pass == 0);  // the window sums are to be made
    if (KS > 1 || box) {
      __syncthreads();
      v4i* part = reinterpret_cast<v4i*>(lds);  // [wave][tile][quad][lane]
      if (KS > 1)
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
          for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int k = 0; k < 4; ++k)
              if (((m * NT + t) * kPieces + k % kPieces) % KS != ks) {
                const elem_t q[4] = {acc[m][t][4 * k], acc[m][t][4 * k + 1], acc[m][t][4 * k + 2], acc[m][t][4 * k + 3]};
                part[((wave * MT + m) * NT + t) * 256 + k * 64 + lane] = __builtin_bit_cast(v4i, q);
              }
      if (box) {  // the box filter over the channel sums
        const int* sum = reinterpret_cast<const int*>(lds + c.off_sum);
        int* zt = reinterpret_cast<int*>(lds + c.off_zt);
        for (int q = tid; q < c.NQ; q += kThreads) {
          const int g = DivM(q, c.m_thtw), rem = q - g * c.TH * c.TW;
          const int qy = DivM(rem, c.m_tw), qx = rem - qy * c.TW;
          const int* sp = sum + (g * c.IH + qy * c.row_stride) * c.IW + qx * c.sw;
          int v = 0;
          for (int ky = 0; ky < c.taps_h; ++ky)
            for (int kx = 0; kx < c.taps_w; ++kx) v += sp[ky * c.dil_row + kx * c.dil_col];
          zt[q] = -c.zws * v;
        }
      }
      __syncthreads();
      if (KS > 1)
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
          for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int p = 0; p < kPieces; ++p)
              if (((m * NT + t) * kPieces + p) % KS == ks)
#pragma unroll
                for (int k = 1; k < KS; ++k) {
                  const v4i* from = part + (((wave - ks + (ks + k) % KS) * MT + m) * NT + t) * 256 + lane;
#pragma unroll
                  for (int i = p; i < 4; i += kPieces) {
                    struct Quad { elem_t e[4]; };
                    const Quad q = __builtin_bit_cast(Quad, from[i * 64]);
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[m][t][4 * i + e] += q.e[e];
                  }
                }
    }

    // ---- epilogue: a lane holds output channel `row` of each channel tile and, per accumulator quad k, pixels
    // 8 k + 4 half + 0 .. 3 of a pixel tile. The results meet in LDS as [channel][pixel] and leave from there in runs: a tile of
    // whole rows is one run of a channel's plane (per image), else every row is one ----
    if (KS > 1 || !box) __syncthreads();  // the window, the partial sums or the block before are read, the window sums complete
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          if (KS > 1 && ((m * NT + t) * kPieces + k % kPieces) % KS != ks) continue;
          const int q0 = (wm * MT + m) * 32 + 8 * k + 4 * half;
          uint8_t* to = lds + c.off_out + (wn * NT * 32 + t * 32 + row) * c.out_pitch + q0 * E;
          if constexpr (DT == kI8) {
            int v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = acc[m][t][4 * k + e] + bias[t];
            if (SUMS) {
              const v4i z = *reinterpret_cast<const v4i*>(lds + c.off_zt + q0 * 4);
#pragma unroll
              for (int e = 0; e < 4; ++e) v[e] += z[e];
            }
            if (c.pre_ties) {  // (uniform)
#pragma unroll
              for (int e = 0; e < 4; ++e) v[e] <<= c.pre_ties >> 1;
              if (c.pre_ties & 1) LowerOddTies(v, rq[t]);
            }
            const int sh = rq[t][1] & 31;
            const int64_t round = RoundHigh(rq[t][2]);
            *reinterpret_cast<uint32_t*>(to) = (c.narrow ? RequantSaturate4<true>(v, rq[t][0], sh, round, c.lo << sh, ((c.hi + 1) << sh) - 1)
                                                         : RequantSaturate4<false>(v, rq[t][0], sh, round, 0, 0)) ^ c.out_xor;
          } else {
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              v[e] = acc[m][t][4 * k + e] + __builtin_bit_cast(float, bias[t]);
              if (c.act != TVX_ACT_NONE) v[e] = v[e] < 0.f ? 0.f : v[e];
              if (c.act == TVX_ACT_RELU6) v[e] = v[e] > 6.f ? 6.f : v[e];
            }
            if constexpr (DT == kF16) {
              _Float16 h[4];
#pragma unroll
              for (int e = 0; e < 4; ++e) h[e] = static_cast<_Float16>(v[e]);
              *reinterpret_cast<uint2*>(to) = __builtin_bit_cast(uint2, h);
            } else {
              *reinterpret_cast<v4f*>(to) = v4f{v[0], v[1], v[2], v[3]};
            }
          }
        }
    __syncthreads();
    const int stack = STACK ? c.stack : 1;  // (uniform)
    const int ohw = c.OH * c.OW, whole = !STACK && c.TW == c.OW;  // (uniform)
    const int rows_live = min(c.TH, c.OH - y0);
    const int runs_live = whole ? min(c.G, c.batch - n0) : STACK ? c.runs : rows_live, run_live = whole ? rows_live * c.OW : min(c.TW, c.OW - x0);
    const int ocb0 = ocl * (WN * NT * 32), channels = STACK ? stack * c.ocg : min(WN * NT * 32, c.ocg - ocb0);
    uint8_t* yb = c.y + ((static_cast<size_t>(n0) * c.OC + static_cast<size_t>(group) * c.ocg + ocb0) * ohw + y0 * stack * c.OW + x0) * E;
    // a thread keeps its place in the channels' runs and walks the channels: sixteen bytes of one at a time (a run's last begin sixteen
    // bytes before its end), four pixels where runs are shorter. Against four pixels everywhere: f16 44 -> 192, 3x3 on 44 x 44, batch 18,
    // 21.5 -> 18.1 us, 19 -> 432 on 114 x 114, batch 2, 21.4 -> 19.1; int8 1 % on 40 drawn layers, at most 6.
    constexpr int kWide = 16 / E;
    const bool wide = E < 4 && run_live >= kWide;  // (uniform)
    const int shift = wide ? c.wide_shift : c.runs_shift;
    const int place = tid & ((1 << shift) - 1), run = DivM(place, wide ? c.m_run_wide : c.m_run4);
    int px = wide ? (place - run * ((c.run_px + kWide - 1) / kWide)) * kWide : (place - run * ((c.run_px + 3) >> 2)) * 4;
    const int left = run < runs_live ? run_live - px : 0;
    if (wide) px = min(px, run_live - kWide);
    const int ch0 = tid >> shift, ch_step = kThreads >> shift;
    const uint8_t* from = lds + c.off_out + ch0 * c.out_pitch + (run * c.run_px + px) * E;
    uint8_t* to = yb + (static_cast<size_t>(ch0) * ohw + static_cast<size_t>(run) * c.run_out + px) * E;
    const size_t to_step = static_cast<size_t>(ch_step) * ohw * E;
    // stacked rows: where a slot's channel and row begin; false where there is no such row
    const int image = STACK ? DivM(run, c.m_th) : 0, first = (run - image * c.TH) * stack;
    auto find_row = [&](int ch) {
      const int j = DivM(ch, c.m_ocg), r = first + j;
      to = yb + (static_cast<size_t>(image) * c.OC + (ch - j * c.ocg)) * ohw + r * c.OW + px;
      return y0 * stack + r < c.OH && n0 + image < c.batch;
    };
    if (left > 0 && wide) {
      if constexpr (E < 4) {
        const uint32_t by = static_cast<uint32_t>(run * c.run_px + px) * E & 3;
        for (int ch = ch0; ch < channels; ch += ch_step, from += ch_step * c.out_pitch, to += to_step) {
          if (STACK && !find_row(ch)) continue;
          const uint32_t* const w = reinterpret_cast<const uint32_t*>(from - by);  // (the dwords behind a run that begins at any byte)
          uint32_t d[5], out[4];
#pragma unroll
          for (int i = 0; i < 5; ++i) d[i] = w[i];
#pragma unroll
          for (int i = 0; i < 4; ++i) out[i] = __builtin_amdgcn_alignbyte(d[i + 1], d[i], by);
          __builtin_memcpy(to, out, 16);
        }
      }
    } else if (left > 0) {
      for (int ch = ch0; ch < channels; ch += ch_step, from += ch_step * c.out_pitch, to += to_step) {
        if (STACK && !find_row(ch)) continue;
        uint32_t four[E];
        if (left >= 4) {
          if constexpr (E == 1) {  // (a run begins at any byte: the dword out of two)
            const uint32_t at = static_cast<uint32_t>(run * c.run_px), *w = reinterpret_cast<const uint32_t*>(from - (at & 3));
            four[0] = __builtin_amdgcn_alignbyte(w[1], w[0], at & 3);
          } else {
#pragma unroll
            for (int d = 0; d < 4; ++d) {
              if constexpr (E == 2) {
                const uint32_t h = reinterpret_cast<const uint16_t*>(from)[d];
                four[d / 2] = d & 1 ? four[d / 2] | h << 16 : h;
              } else {
                four[d] = reinterpret_cast<const uint32_t*>(from)[d];
              }
            }
          }
          __builtin_memcpy(to, four, 4 * E);
        } else {
#pragma unroll 1
          for (int e = 0; e < left; ++e) {
            if constexpr (E == 1) to[e] = from[e];
            else if constexpr (E == 2) reinterpret_cast<uint16_t*>(to)[e] = reinterpret_cast<const uint16_t*>(from)[e];
            else reinterpret_cast<uint32_t*>(to)[e] = reinterpret_cast<const uint32_t*>(from)[e];
          }
        }
      }
    }
    if (pass + 1 >= passes) break;
    ++ocl;
  }
}

typedef void (*TileFn)(TileArgs);

// The ways a workgroup's wavefronts share a tile.
// fn: int8, float16, float32, int8 with sums in the loop and with sums box-filtered, int8 in stacked rows without and with sums; one chunk of the channels or several
struct Shape { int pixels, channels, ks, waves; double length; TileFn fn[7][2]; };  // length: of its chain, fitted (Cost)
#define TVX_TILE_DT(DT, SUMS, WM, WN, KS, MT, NT, R, EU, STACK) { ConvTileKernel<DT, SUMS, WM, WN, KS, MT, NT, R, EU, false, STACK>, ConvTileKernel<DT, SUMS, WM, WN, KS, MT, NT, R, EU, true, STACK> }
#define TVX_TILE_FNS(WM, WN, KS, MT, NT, R, EU)                                                                   \
  TVX_TILE_DT(kI8, kNoSums, WM, WN, KS, MT, NT, R, EU, false), TVX_TILE_DT(kF16, kNoSums, WM, WN, KS, MT, NT, R, EU, false), \
  TVX_TILE_DT(kF32, kNoSums, WM, WN, KS, MT, NT, R, EU, false), TVX_TILE_DT(kI8, kSumsInLoop, WM, WN, KS, MT, NT, R, EU, false), \
  TVX_TILE_DT(kI8, (MT * NT > 1 ? kSumsBox : kSumsInLoop), WM, WN, KS, MT, NT, R, EU, false)
#define TVX_TILE(WM, WN, KS, MT, NT, R, EU, LENGTH) \
  { WM * MT * 32, WN * NT * 32, KS, WM * WN * KS, LENGTH, { TVX_TILE_FNS(WM, WN, KS, MT, NT, R, EU), { nullptr, nullptr }, { nullptr, nullptr } } }
#define TVX_TILE_32(WM, KS, R, EU, LENGTH) \
  { WM * 32, 32, KS, WM * KS, LENGTH, { TVX_TILE_FNS(WM, 1, KS, 1, 1, R, EU), TVX_TILE_DT(kI8, kNoSums, WM, 1, KS, 1, 1, R, EU, true), TVX_TILE_DT(kI8, kSumsInLoop, WM, 1, KS, 1, 1, R, EU, true) } }
const Shape kShapes[] = {
    TVX_TILE(4, 2, 1, 2, 1, 4, 4, 1.0),   // 0: 256 x 64, eight wavefronts
    TVX_TILE(2, 2, 2, 2, 1, 4, 4, 1.27),  // 1: 128 x 64, eight
    TVX_TILE(2, 2, 1, 2, 1, 4, 4, 0.8),   // 2: 128 x 64, four
    TVX_TILE_32(4, 2, 6, 4, 1.43),        // 3: 128 x 32, eight
    TVX_TILE_32(4, 1, 6, 4, 1.0),         // 4: 128 x 32, four
    TVX_TILE(2, 2, 2, 1, 1, 6, 4, 1.4),   // 5: 64 x 64, eight
    TVX_TILE_32(2, 4, 4, 4, 1.7),         // 6: 64 x 32, eight
    TVX_TILE_32(1, 8, 6, 4, 1.75),        // 7: 32 x 32, eight
};
#undef TVX_TILE_32
#undef TVX_TILE
#undef TVX_TILE_FNS
#undef TVX_TILE_DT
constexpr int kShapeCount = sizeof(kShapes) / sizeof(kShapes[0]);

int RoundUp(int v, int m) { return (v + m - 1) / m * m; }
uint32_t Magic(int d) { return d <= 1 ? 0u : static_cast<uint32_t>(((uint64_t{1} << 32) + d - 1) / d); }

// LDS of a workgroup in front of its tables: the staged window, then the partial sums, then the results - those behind it where
// several blocks of channels read the window
int OutPitch(const Shape& sp, int E) { return (sp.pixels + 4) * E; }  // (four pixels more against bank conflicts)
int64_t OutBytes(const Shape& sp, int E) { return static_cast<int64_t>(sp.channels) * OutPitch(sp, E); }
int64_t WindowBytes(const Shape& sp, int64_t staged, int E, int loop) {
  const int64_t sums = sp.ks > 1 ? static_cast<int64_t>(sp.ks) * sp.pixels * sp.channels * 4 : 0;
  return (std::max({staged, sums, loop > 1 ? 0 : OutBytes(sp, E)}) + 15) / 16 * 16;
}

struct Geometry {
  int shape, TW, TH, G, gpc, chunks, loop;
  int IW, IH, pitch, lds_bytes, sums, stack;
  int64_t wgs;
  double cost;
};

// Microseconds of a launch, to compare tiles by. A workgroup is a chain - staging rounds (an item per thread and round), steps,
// results - which grows longer with every workgroup that shares its CU and counts once per round of workgroups the chip holds; to that
// come the units all of a CU's workgroups share (its memory pipeline, its matrix cores). The constants are a fit to 46000 launches
// measured back to back in a captured graph (900 drawn convolutions x the tiles below). On 900 others the tile chosen takes 3 %
// more than the best measured one on the (geometric) average, a quarter more in one of a hundred, half more at the worst. (Constants
// fitted to launches from a host loop lost 11 % on the same ones, and up to 1.7 times on layers of a few microseconds: int8 14 -> 9
// channels, 3x3 on 43 x 43, batch 14, 11.0 us where a tile of 6.3 was to be had. The host's own time had hidden what those take.)
double Cost(const Shape& sp, const Geometry& g, int dt, int taps, int group_px, bool sums, bool borders, int OW, int cus) {
  const int threads = 64 * sp.waves, steps = (taps * g.gpc + 1) / 2, tiles = sp.pixels * sp.channels / 1024 * sp.ks / sp.waves;
  const double npx = static_cast<double>(g.G) * g.IH * g.IW;
  const double items = static_cast<double>(g.G) * g.IH * ((g.IW + group_px - 1) / group_px) * g.gpc;
  const double runs = g.TW == OW || g.TW % 4 == 0 ? 1.0 : 1.1;  // stores of whole quads
  const double stage = (dt == kI8 ? 1.4 : dt == kF16 ? 0.6 : 0.35) * std::ceil(items / threads) +
                       0.25 * npx * g.gpc / threads * ((sums ? 1.0 : 0.0) + (borders ? 0.5 : 0.0));
  const double multiply = static_cast<double>(steps) / sp.ks * (0.015 + (dt == kF32 ? 0.13 : 0.036) * tiles);
  const double chain = 0.6 + g.chunks * (stage + g.loop * multiply) + g.loop * 1.2 * tiles / sp.ks * runs;
  const double shared = g.chunks * ((dt == kI8 ? 0.12 : dt == kF16 ? 0.24 : 0.033) * items / 64 +
                                    (dt == kF32 ? 0.016 : 0.0025) * g.loop * steps * tiles * sp.waves / sp.ks);
  const double per_cu = static_cast<double>(g.wgs) / cus;
  // (the kernels that walk chunks hold more than 128 registers, but for float32)
  const int waves_cu = g.chunks > 1 && dt != kF32 ? 12 : 16;
  const double resident = std::min<double>(std::max(1, std::min(waves_cu / sp.waves, 160 * 1024 / g.lds_bytes)), std::max(1.0, std::ceil(per_cu)));
  // (eight wavefronts without shares of a sum walk chunks alone on their CU, 1.06 to 1.25 times as long as their length says)
  const double alone = sp.ks == 1 && sp.waves == 8 && waves_cu == 12 ? 1.12 : 1.0;
  const double by_chain = chain * sp.length * alone * (1.0 + 0.48 * (resident - 1.0) * sp.waves / 8);
  return 3.1 + by_chain * (per_cu <= resident ? 1.0 : per_cu / resident + 0.35) + per_cu * shared;
}

// How the window sums are made: in the loop up to 80 multiplications of a wavefront, and always where each of them waits for a weight
// fragment of its own (316 drawn layers, captured: 0.92 of the box filter's time below the line, as low as 0.69; beyond it the dot
// products cost the matrix cores' issue slots, 1.03 on the average and up to 1.17).
int SumsBy(const Shape& sp, int steps) {
  const int tiles = sp.pixels * sp.channels / 1024 * sp.ks / sp.waves;
  return tiles == 1 || steps * tiles / sp.ks <= 80 ? kSumsInLoop : kSumsBox;
}

// By how much less a tile of stacked rows has to promise, and the products of an output that two rows need up to so many outputs: what the results'
// shorter runs take.
// Without these lines the choice was 1.04 to 1.17 of the time of unstacked tiles on four of 132 layers, of 16 channels and few products each (int8
// 8 -> 16, 3x3 / 2 on 50 x 69, batch 37, 7.2 us for 6.1; uint8 3 -> 16, 5x5 on 99 x 99, batch 7, 7.5 for 6.9;
// but int8 20 -> 64 in four groups, 3x3 on 69 x 121, batch 46, 33.0 for 55.3).
constexpr double kStackedMore = 1.06;
constexpr int kStackedProducts = 128, kStackedOutputs = 7812;  // (a compute unit: two million on 256)

struct Plan {
  TileArgs a;
  TileFn fn;
  unsigned grid, threads, lds_bytes;
  int elem;
};

int ConvTileRun(tvx_op* op, const void* in0, const void*, void* out, hipStream_t st) {
  const Plan* plan = reinterpret_cast<const Plan*>(op->host_blob.data());
  if ((reinterpret_cast<uintptr_t>(in0) | reinterpret_cast<uintptr_t>(out)) & (plan->elem - 1))
    return SetError(TVX_E_INVALID, "%s: tensors must be aligned to their elements", op->kernel_name);
  TileArgs a = plan->a;
  a.x = static_cast<const uint8_t*>(in0);
  a.y = static_cast<uint8_t*>(out);
  hipLaunchKernelGGL(plan->fn, dim3(plan->grid), dim3(plan->threads), plan->lds_bytes, st, a);
  TVX_HIP_CHECK(hipGetLastError());
  return TVX_OK;
}

}  // namespace

// Which shapes stay with the kernels asked behind this one (measured back to back in a captured graph on 3900 drawn convolutions;
// what is left slower here than there by more than 3 % is one in twenty-five, at most 1.4 times):
static bool IsBetterChoice(const tvx_conv2d_desc* d, int dt, bool sums) {
  const int groups = d->groups > 1 ? d->groups : 1, ocg = d->out_c / groups;
  const uint64_t reduction = static_cast<uint64_t>(d->in_c / groups) * d->k_w * d->k_h;
  const uint64_t outputs = static_cast<uint64_t>(d->out_c) * d->out_w * d->out_h * d->batch, macs = reduction * outputs;
  const uint64_t cus = ComputeUnits();
  const bool pointwise = d->k_w == 1 && d->k_h == 1;
  // a group of three output channels and fewer fills less than a tenth of a tile's 32 channels: only where each has little to add up
  // (float16 432 -> 12 in four groups, 7x7 on 42 x 42, batch 28: 2495 us with one thread per output, 140 here)
  if (groups > 1 && ocg < 4 && reduction <= 128) return false;
  // a handful of products per output: one thread per output is quicker than staging a window, up to so many outputs. Tiles over it, captured, 1400 layers
  // of seven channels and more, means by outputs in thousands (on 256 compute units):   to 60   140   220   350   600  above
  //                                                     1x1 of one channel                1.49  1.46  1.30  1.14   .90   .61
  //                                                         of two or three               1.29  1.23  1.10   .96   .80   .57
  //                                                         of four                       1.12  1.07  1.01   .82   .65   .49
  //                                                         of five, float16              1.08  1.04   .97   .86   .60   .40
  //                                                         of five, float32               .99  1.02   .85   .75   .60   .42
  //                                                         of six to nine                 .85   .83   .77   .64   .53   .32
  //                                                     larger windows, to five products  1.31  1.25  1.14  1.01   .83   .50
  //                                                         six to eight                  1.10  1.07   .98   .89   .74   .43
  //                                                         nine                          1.06  1.01   .94   .85   .71   .39
  // Fewer channels leave most of a tile's 32 empty: of one the tiles take 1.3 to 2.9 of the time at 20 thousand to 1.8 million outputs, of two or three 1.1 to
  // 1.5, of four to six 1.15 to .87. By these lines all 2097 layers take 1.006 of the time with the better kernel for each.
  const uint64_t few = !pointwise ? (reduction <= 5 ? 1000 : reduction <= 8 ? 700 : reduction == 9 ? 400 : 0)
                                  : reduction == 1 ? 1172 : reduction <= 3 ? 800 : reduction == 4 ? 550 : reduction == 5 && dt == kF16 ? 400 : 0;
  if (dt != kI8 && groups == 1 && 2 * outputs <= few * cus * (d->out_c == 1 ? 64 : d->out_c <= 3 ? 16 : d->out_c <= 6 ? 5 : 2)) return false;
  // (in groups, by products, four millions and one on 256 compute units: 4.3 against 5.7; int8, which has no other kernel for so few: 4 -> 64 in two, 1x1 on
  // 25 x 25, 3.9 against 6.5, but 64 -> 240 in eight on 22 x 22 7.7 against 6.0)
  if (dt != kI8 && groups > 1 && reduction <= 9 && macs <= 15625 * cus) return false;
  if (dt == kI8 && groups > 1 && reduction <= 8 && macs <= (reduction <= 4 ? 15625 : 3906) * cus) return false;
  // int8 1 x 1 in groups that fill less than a tile's channels: conv2d_gemm_i8 (188 -> 60 in four groups on 108 x 108, batch 6: 9.9 against
  // 17.4 us, 240 -> 96 on 74 x 74, batch 49: 36.8 against 52.3); with more than 32 channels in a group the tiles (144 -> 128 in two on
  // 29889 pixels: 9.5 against 16.8)
  if (dt == kI8 && groups > 1 && pointwise && reduction >= 32 && reduction <= 128 && ocg >= 8 && ocg <= 32) return false;
  // float16 1 x 1 that pwconv_reg_f16, asked in front, leaves (strided ones, mostly): conv2d_gemm_f16 has less to set up where channels and results are
  // few (24 -> 16 on 16 x 16 at stride 2, batch 7, 4.1 against 4.8 us; 32 -> 8 on 144 x 144 at stride 2, batch 2, 4.2 against 4.5). It takes eight
  // results and more; fewer would go to a thread per output (32 -> 5 on 9 x 9 at stride 2, batch 3, 14.7 against 4.8). 260 drawn strided layers 1.005 of the
  // time with the better kernel for each, 160 of more than 1024 channels 1.000.
  if (dt == kF16 && groups == 1 && pointwise && d->in_c >= 16 && d->out_c >= 8 && macs <= 16000 * cus && ((d->in_c <= 24 && d->out_c <= 24) || (d->in_c <= 32 && d->out_c <= 8)))
    return false;
  if (dt == kI8 && groups == 1) {
    if (ConvIgemmPersists(d)) return false;
    // a granule of channels under weights with a zero point: up to two million products (on 256 compute units) conv2d_igemm_i8, whose chain is short on small planes and on
    // rows of whole dwords, is within a tenth of the tiles at 5 to 6 us; beyond them its tiles queue up (60 drawn layers .55 of its time, 16 -> 192
    // on 140 x 140, batch 3, 129 us against 15.7). What conv2d_im2col_i8 has left (its short windows) it does not get.
    const bool aligned = d->stride_w == 1 && d->stride_h == 1 && d->in_w % 4 == 0;
    const bool short_window = reduction <= 64 && d->in_c % 16 != 0 && d->out_c <= 128;
    if (sums && d->in_c <= 16 && reduction <= 512 && 2 * macs <= 15625 * cus && !short_window && (aligned || d->in_w * d->in_h <= 256)) return false;
  }
  return true;
}

// Claims dense and grouped convolutions with constant weights on quantized (multipliers of 2^-20 and more), float16 or float32
// tensors whose staged window fits LDS a granule of channels at a time.
int ConvTileSetup(tvx_op* op, const tvx_conv2d_desc* d, const void* w_host, const void* bias_host) {
  if (!w_host || op->fused_add || op->kind != OP_CONV2D || d->multiplier != 0) return TVX_E_UNSUPPORTED;
  int dt;
  if (op->quantized) dt = kI8;
  else if (d->in_dtype == TVX_F16 && d->w_dtype == TVX_F16 && d->out_dtype == TVX_F16) dt = kF16;
  else if (d->in_dtype == TVX_F32 && d->w_dtype == TVX_F32 && d->out_dtype == TVX_F32) dt = kF32;
  else return TVX_E_UNSUPPORTED;
  const int E = dt == kI8 ? 1 : dt == kF16 ? 2 : 4;
  bool forced = false;
  if (const char* f = getenv("TVX_CONV_TILE")) {  // test lever: 0 declines, 1 claims also where another kernel is the better choice
    if (atoi(f) == 0) return TVX_E_UNSUPPORTED;
    forced = true;
  }
  if (!forced && !IsBetterChoice(d, dt, dt == kI8 && op->w_zp != (d->w_dtype == TVX_U8 ? 128 : 0))) return TVX_E_UNSUPPORTED;

  TileArgs a{};
  int W = d->in_w, H = d->in_h, OW = d->out_w, OH = d->out_h;
  int kh = d->k_h;
  const int kw = d->k_w, dh = d->dilation_h, dw = d->dilation_w;
  const bool flat = kh == 1 && kw == 1 && d->stride_w == 1 && d->stride_h == 1 && d->pad_left == 0 && d->pad_top == 0 && OW == W && OH == H;
  if (flat) { W = OW = W * H; H = OH = 1; }  // a 1 x 1 window needs no rows: an image is one
  const int group_px = dt == kF32 ? 4 : 8;
  if (W * H < group_px) return TVX_E_UNSUPPORTED;
  const int groups = d->groups > 1 ? d->groups : 1;
  const int C = d->in_c;
  a.H = H; a.W = W; a.OC = d->out_c; a.OH = OH; a.OW = OW; a.batch = d->batch;
  a.sh = d->stride_h; a.sw = d->stride_w; a.pad_t = d->pad_top; a.pad_l = d->pad_left;
  a.icg = C / groups; a.ocg = a.OC / groups;
  const int granules = (a.icg * E + 15) / 16, real_taps = kh * kw;
  int taps = real_taps;
  if (taps > 1024) return TVX_E_UNSUPPORTED;
  const uint64_t image = static_cast<uint64_t>(C) * H * W * E, out_image = static_cast<uint64_t>(a.OC) * OH * OW;
  a.row_step = kh == 1 ? a.sh : 1;
  a.row_stride = kh == 1 ? 1 : a.sh;

  const int x_u8 = d->in_dtype == TVX_U8, w_u8 = d->w_dtype == TVX_U8;
  const int zxs = dt == kI8 ? d->in_zp - (x_u8 ? 128 : 0) : 0;
  const int zws = dt == kI8 ? op->w_zp - (w_u8 ? 128 : 0) : 0;

  // ---- the tile ----
  const int cus = ComputeUnits();
  int want = -1, want_tw = 0, want_loop = 0;
  if (const char* f = getenv("TVX_CONV_TILE_SHAPE")) want = atoi(f);  // test lever
  if (const char* f = getenv("TVX_CONV_TILE_COLS")) want_tw = atoi(f);  // test lever
  if (const char* f = getenv("TVX_CONV_TILE_LOOP")) want_loop = atoi(f);  // test lever
  int want_stack = 0;
  if (const char* f = getenv("TVX_CONV_TILE_STACK")) want_stack = atoi(f);  // test lever
  const int rows = OH;
  auto stacked = [&](int stack) {
    OH = (rows + stack - 1) / stack;
    kh = d->k_h + (stack - 1) * d->stride_h;
    taps = kh * kw;
    a.sh = stack * d->stride_h;
    if (d->k_h > 1) a.row_stride = a.sh;
  };
  Geometry best{};
  best.shape = -1;
  for (int stack = 1; stack <= 4; ++stack) {
    if (want_stack && stack != want_stack) continue;
    if (stack > 1 && (dt != kI8 || d->k_h == 1 || dh != 1 || stack * a.ocg > 32 || stack > rows)) break;
    if (!want_stack && stack == 2 && real_taps * a.icg < kStackedProducts && out_image * d->batch < static_cast<uint64_t>(kStackedOutputs) * cus) continue;
    stacked(stack);
    if (taps > 1024) break;
    for (int sidx = 0; sidx < kShapeCount; ++sidx) {
      if (want >= 0 && sidx != want) continue;
      const Shape& sp = kShapes[sidx];
      if (stack > 1 && !sp.fn[5][0]) continue;
      const int cand[] = {OW, (OW + 1) / 2, (OW + 2) / 3, 8, 16, 32, 64, 128};
      for (int tw : cand) {
        if (want_tw) tw = want_tw;
        if (tw < 1 || tw > OW || tw > sp.pixels) continue;
        Geometry g{};
        g.shape = sidx;
        g.stack = stack;
        g.TW = tw;
        g.TH = std::min(OH, sp.pixels / tw);
        // rows spread evenly over the tiles of a column
        g.TH = (OH + (OH + g.TH - 1) / g.TH - 1) / ((OH + g.TH - 1) / g.TH);
        g.G = g.TW == OW && g.TH == OH ? std::min<int>(d->batch, sp.pixels / (g.TW * g.TH)) : 1;
        g.IW = (g.TW - 1) * a.sw + (kw - 1) * dw + 1;
        g.IH = (g.TH - 1) * a.row_stride + (kh - 1) * dh + 1;
        const int64_t npx = static_cast<int64_t>(g.G) * g.IH * g.IW;
        if (npx > 40000) continue;
        const int blocks = (a.ocg + sp.channels - 1) / sp.channels;
        for (int loop : {1, 2, 3, 4, 6, 8, 16}) {
          g.loop = loop;
          if (loop > 1 && (loop > blocks || sp.ks > 1)) break;
          if (want_loop && loop != want_loop) continue;
          for (g.chunks = 1; g.chunks <= granules; ++g.chunks) {
            g.gpc = (granules + g.chunks - 1) / g.chunks;
            if (g.chunks > 1 && (granules + g.gpc - 1) / g.gpc != g.chunks) continue;
            g.pitch = (g.gpc | 1) * 16;
            const int steps = (taps * g.gpc + 1) / 2;
            int64_t bytes = WindowBytes(sp, npx * g.pitch, E, loop);
            bytes += 2 * RoundUp(steps + kMostAhead + 4, 4) * 4;
            g.sums = zws ? SumsBy(sp, steps * g.chunks * loop) : kNoSums;
            if (zws) bytes += sp.pixels * 4 + (g.sums == kSumsBox ? npx * 4 : 0);
            if (loop > 1) bytes = RoundUp(bytes, 16) + OutBytes(sp, E);
            g.lds_bytes = static_cast<int>(std::min<int64_t>(bytes, 1 << 30));
            if (g.lds_bytes <= 78 * 1024) break;
          }
          if (g.chunks > granules || (loop > 1 && g.chunks > 1)) continue;
          const int64_t tiles = static_cast<int64_t>((OW + g.TW - 1) / g.TW) * ((OH + g.TH - 1) / g.TH) * ((d->batch + g.G - 1) / g.G);
          g.wgs = tiles * ((blocks + loop - 1) / loop) * groups;
          if (g.wgs > 0x3fffffff) continue;
          g.cost = Cost(sp, g, dt, taps, group_px, zws != 0, (a.pad_l || a.pad_t) && taps > 1, OW, cus);
          if (stack > 1) g.cost *= kStackedMore;
          if (best.shape < 0 || g.cost < best.cost) best = g;
        }
      }
    }
  }
  if (best.shape < 0) return TVX_E_UNSUPPORTED;
  const Geometry& g = best;
  const Shape& sp = kShapes[g.shape];
  stacked(g.stack);
  if (image * g.G >= (1ull << 32) || out_image * g.G >= (1ull << 31)) return TVX_E_UNSUPPORTED;

  a.TW = g.TW; a.TH = g.TH; a.G = g.G; a.NQ = g.TW * g.TH * g.G;
  a.IW = g.IW; a.IH = g.IH; a.pitch = g.pitch; a.gpc = g.gpc; a.chunks = g.chunks;
  a.steps = (taps * g.gpc + 1) / 2;
  a.odd = (taps * g.gpc) & 1;
  a.steps_pad = RoundUp(a.steps + kMostAhead + 4, 4);
  a.taps_w = kw; a.taps_h = kh; a.dil_col = dw; a.dil_row = dh * g.IW;
  a.ncg = (g.IW + group_px - 1) / group_px;
  a.cells = g.G * g.IH * a.ncg;
  a.gl = 1;
  for (int v = 2; v <= 6; ++v) if (a.gpc % v == 0) a.gl = v;
  if (a.gl == 1) a.gl = a.gpc;
  a.tiles_x = (OW + g.TW - 1) / g.TW;
  a.tiles_y = (OH + g.TH - 1) / g.TH;
  a.tiles_per_group = (a.ocg + sp.channels - 1) / sp.channels;
  a.loop = g.loop;
  a.wgs_per_group = (a.tiles_per_group + g.loop - 1) / g.loop;
  a.oc_wgs = a.wgs_per_group * groups;
  a.total = static_cast<int>(g.wgs);
  a.per_xcd = (a.total + 7) / 8;
  a.npx = g.G * g.IH * g.IW;
  a.cells4 = (a.cells + 3) / 4;
  a.items = a.cells4 * 4 * a.gpc;
  a.plane_bytes = static_cast<uint32_t>(H) * W * E;
  a.image_bytes = a.plane_bytes * C;
  a.at_max = H * W - group_px;
  const int64_t npx = static_cast<int64_t>(g.G) * g.IH * g.IW;
  a.off_tab = static_cast<int>(WindowBytes(sp, npx * g.pitch, E, g.loop));
  a.off_sum = a.off_tab + 2 * a.steps_pad * 4;
  a.off_zt = a.off_sum + (g.sums == kSumsBox ? static_cast<int>(npx) * 4 : 0);
  a.off_out = g.loop > 1 ? g.lds_bytes - static_cast<int>(OutBytes(sp, E)) : 0;
  const bool whole = g.stack == 1 && g.TW == OW;
  a.stack = g.stack;
  a.m_ocg = Magic(a.ocg);
  a.m_th = Magic(g.TH);
  a.runs = whole ? g.G : g.G * g.TH;
  a.run_px = whole ? g.TH * OW : g.TW;
  a.run_out = whole ? a.OC * OH * OW : OW;
  a.out_pitch = OutPitch(sp, E);
  a.m_run4 = Magic((a.run_px + 3) / 4);
  while ((1 << a.runs_shift) < a.runs * ((a.run_px + 3) / 4)) ++a.runs_shift;
  const int wide_groups = (a.run_px + 16 / E - 1) / (16 / E);
  a.m_run_wide = Magic(wide_groups);
  while ((1 << a.wide_shift) < a.runs * wide_groups) ++a.wide_shift;
  a.m_gl = Magic(a.gl); a.m_cells4 = Magic(a.cells4); a.m_ncg = Magic(a.ncg); a.m_ih = Magic(a.IH); a.m_iw = Magic(a.IW); a.m_tw = Magic(a.TW); a.m_thtw = Magic(a.TH * a.TW);
  a.m_ocb = Magic(a.oc_wgs); a.m_tpg = Magic(a.wgs_per_group); a.m_tx = Magic(a.tiles_x); a.m_ty = Magic(a.tiles_y);
  if (static_cast<int64_t>(a.IH - 1) * a.row_step >= 1 << 23) return TVX_E_UNSUPPORTED;  // (24-bit products of rows and columns; the others lie within LDS)
  // a reciprocal is exact while dividend * divisor < 2^32
  if (static_cast<uint64_t>(a.total) * std::max({a.oc_wgs, a.tiles_x, a.tiles_y}) >= (1ull << 32)) return TVX_E_UNSUPPORTED;
  if (static_cast<uint64_t>(npx) * a.gpc * std::max({a.gpc, a.cells, a.IH, a.IW}) >= (1ull << 32)) return TVX_E_UNSUPPORTED;
  a.xor_mask = dt == kI8 && x_u8 ? 0x80808080u : 0u;
  a.pad_full = static_cast<uint32_t>(zxs & 0xff) * 0x01010101u;
  a.last_granule = granules - 1;
  for (int q = 0; q < 4; ++q) {
    const int nb = a.icg * E - (granules - 1) * 16 - 4 * q;
    a.pad_last[q] = nb >= 4 ? a.pad_full : nb <= 0 ? 0u : a.pad_full & ((1u << (8 * nb)) - 1u);
  }
  a.zws = zws;
  const int out_flip = dt == kI8 && d->out_dtype == TVX_U8 ? 128 : 0;
  a.lo = op->act_lo - out_flip; a.hi = op->act_hi - out_flip; a.narrow = a.lo > -128 || a.hi < 127;
  a.out_xor = out_flip ? static_cast<int>(0x80808080u) : 0;
  a.act = d->activation;

  // ---- the step table ----
  std::vector<int32_t> tab(2 * static_cast<size_t>(a.steps_pad), 0);
  for (int q = 0; q < taps * a.gpc; ++q) {
    const int t = q / a.gpc, gr = q % a.gpc, ky = t / kw, kx = t % kw;
    tab[static_cast<size_t>(q & 1) * a.steps_pad + q / 2] = (ky * dh * g.IW + kx * dw) * g.pitch + gr * 16;
  }

  // ---- weights [oc][c][ky][kx] -> fragment order; the bias takes the zero points' constants ----
  const size_t alloc_oc = static_cast<size_t>(a.tiles_per_group) * groups * sp.channels;
  const size_t tile_bytes = static_cast<size_t>(a.chunks) * a.steps * 1024;
  std::vector<uint8_t> packed(alloc_oc / 32 * tile_bytes + kMostAhead * 1024, 0);  // (the last steps read ahead)
  std::vector<int32_t> biasf(dt == kI8 ? alloc_oc : 0, 0);
  std::vector<int32_t> mult, shift;
  if (dt == kI8) {
    // (slots past a group's channels: a real channel's record, so that they do not decide the requantization flavour)
    mult.assign(alloc_oc, op->h_mult[0]);
    shift.assign(alloc_oc, op->h_shift[0]);
  }
  const uint8_t* src = static_cast<const uint8_t*>(w_host);
  const int32_t* bi = static_cast<const int32_t*>(bias_host);
  const uint8_t flip = w_u8 ? 0x80 : 0;
  const int epg = 16 / E;  // elements of a granule
  for (int oc = 0; oc < a.OC; ++oc)
  for (int up = 0; up < g.stack; ++up) {
    const int grp = oc / a.ocg, ol = up * a.ocg + oc % a.ocg;
    const size_t slot = static_cast<size_t>(grp) * a.tiles_per_group * sp.channels + ol;
    uint8_t* tile = packed.data() + slot / 32 * tile_bytes + (slot % 32) * 16;
    const uint8_t* ws = src + static_cast<size_t>(oc) * a.icg * real_taps * E;
    int64_t sw = 0;
    // (copies: a byte stored may be any of the fields')
    const int icg = a.icg, gpc = a.gpc;
    const size_t chunk_bytes = static_cast<size_t>(a.steps) * 1024;
    // taps in front of the row's own and behind them: the weights' zero point
    const int before = up * d->stride_h * kw, behind = taps - before - real_taps;
    const uint8_t none = static_cast<uint8_t>(zws & 0xff);
    for (int c = 0; c < icg; ++c) {
      const int gg = c / epg, chunk = gg / gpc;
      uint8_t* cp = tile + static_cast<size_t>(chunk) * chunk_bytes + (c % epg) * E;
      int q = gg % gpc;
      if (E == 1) {
        auto put = [&](uint8_t v) {
          cp[static_cast<size_t>(q >> 1) * 1024 + (q & 1) * 512] = v;
          sw += static_cast<int8_t>(v);
          q += gpc;
        };
        for (int t = 0; t < before; ++t) put(none);
        for (int t = 0; t < real_taps; ++t) put(*ws++ ^ flip);
        for (int t = 0; t < behind; ++t) put(none);
      } else {
        for (int t = 0; t < taps; ++t, q += gpc, ws += E) std::memcpy(cp + static_cast<size_t>(q >> 1) * 1024 + (q & 1) * 512, ws, E);
      }
    }
    if (dt == kI8) {
      const int64_t v = (bi ? bi[oc] : 0) - static_cast<int64_t>(zxs) * sw + static_cast<int64_t>(taps) * a.icg * zxs * zws;
      biasf[slot] = static_cast<int32_t>(static_cast<uint32_t>(v));
      mult[slot] = op->h_mult[oc];
      shift[slot] = op->h_shift[oc];
    }
  }
  int s = op->packed.Upload(packed.data(), packed.size());
  if (s == TVX_OK) s = op->aux3.Upload(tab.data(), tab.size() * 4);
  if (s == TVX_OK && dt == kI8) {
    std::vector<int32_t> rqt;
    const int64_t bound = AccumulatorBound(static_cast<uint64_t>(real_taps) * a.icg, bias_host, d->out_c);
    const int slots = static_cast<int>(alloc_oc);
    int up;
    bool ties;
    if (!BuildTieRecords(mult, shift, slots, slots, d->out_zp - out_flip, bound, &rqt, &up, &ties)) return TVX_E_UNSUPPORTED;
    a.pre_ties = up * 2 + ties;
    s = op->aux.Upload(biasf.data(), biasf.size() * 4);
    if (s == TVX_OK) s = op->aux2.Upload(rqt.data(), rqt.size() * 4);
    a.biasf = op->aux.as<int32_t>();
    a.rq = op->aux2.as<tvx_v4i>();
  } else if (s == TVX_OK && bias_host) {
    s = op->bias.Upload(bias_host, static_cast<size_t>(a.OC) * 4);
    a.biasfl = op->bias.as<float>();
  }
  if (s != TVX_OK) return s;
  a.wpk = op->packed.as<v4i>();
  a.tab = op->aux3.as<int>();

  Plan plan{};
  plan.a = a;
  const int flavour = g.stack > 1 ? (g.sums == kNoSums ? 5 : 6) : g.sums == kNoSums ? dt : g.sums == kSumsInLoop ? 3 : 4;
  plan.fn = sp.fn[flavour][a.chunks > 1];
  plan.lds_bytes = static_cast<unsigned>(g.lds_bytes);
  plan.grid = static_cast<unsigned>(a.per_xcd) * 8;
  plan.threads = 64u * sp.waves;
  plan.elem = E;
  if (plan.lds_bytes > 48 * 1024) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(plan.fn), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(plan.lds_bytes));
    if (e != hipSuccess) return SetError(TVX_E_DEVICE, "hipFuncSetAttribute(dynamic LDS %u): %s", plan.lds_bytes, hipGetErrorString(e));
  }
  op->host_blob.assign(reinterpret_cast<const uint8_t*>(&plan), reinterpret_cast<const uint8_t*>(&plan) + sizeof(plan));
  op->run = ConvTileRun;
  op->kernel_name = dt == kF32 ? "conv2d_tile_f32" : dt == kF16 ? "conv2d_tile_f16" : "conv2d_tile_i8";
  static const char* const kVariants[7] = {nullptr, nullptr, nullptr, "conv2d_tile_i8_sums", "conv2d_tile_i8_box", "conv2d_tile_i8_stacked", "conv2d_tile_i8_stacked_sums"};
  op->variant = kVariants[flavour];
  return TVX_OK;
}

}  // namespace tvx
