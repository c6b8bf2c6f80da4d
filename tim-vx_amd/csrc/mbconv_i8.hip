// pwconv_dwconv3x3_pwconv_i8: an inverted-residual block - 1x1 expansion, depthwise 3x3, 1x1 projection and the
// residual Add behind it - as one kernel, for the small feature maps and batches where three or four
// launches of a few microseconds of work each cost more than the arithmetic. The closed driver fuses such
// chains when it verifies the graph (reference: src/tim/vx/internal/src/vsi_nn_graph.c:1591-1603); the
// operators it fuses are the Conv2d nodes of src/tim/vx/internal/src/ops/vsi_nn_op_conv2d.c:35-118.
//
// The expanded tensor never leaves the CU. A workgroup owns a tile of output pixels of one image and first transposes the input
// pixels behind it - with the halo the 3x3 window needs - into LDS as the MFMA operand [pixel][channel]. The expanded channels are
// then walked in chunks of 32, the wavefronts taking them in turns: expansion of all halo pixels for the chunk
// (v_mfma_i32_32x32x32_i8, requantized), depthwise stencil (signed dot4 over byte windows, requantized and
// transposed into the projection's operand), and the chunk's contribution to every output channel accumulated in
// registers. No barrier inside the walk: a wavefront only reads what it wrote. At the end the partial projections meet in
// LDS by integer atomics and every wavefront requantizes, adds the residual to and stores its share of the outputs.
//
// At stride 1 (MbTileKernel) the expanded chunk stays in a lane's registers, at stride 2 (MbConvKernel) it is a wavefront-private
// [channel][pixel] image in LDS.
#include <algorithm>
#include <climits>
#include <cstdlib>
#include <cstring>

#include "variants.h"

namespace tvx {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

constexpr int kMinWaves = 4;
// (stride 2: two wavefronts a SIMD within 256 registers)
constexpr int MaxWaves(int acc_tiles) { return acc_tiles <= 5 ? 8 : kMinWaves; }
constexpr int kMStride = 48;      // bytes per pixel row of the projection operand (32 channels + 16: bank spread)
constexpr int kMaxCinSteps = 5;   // 32-channel steps of the expansion's reduction (160 input channels)

struct MbArgs {
  const uint8_t* x;    // block input {W, H, Cin, N}
  uint8_t* y;          // block output {OW, OH, Cout, N}
  const uint8_t* res;  // the residual Add's other operand (quantized like y's type), or null
  // expansion: fragments [chunk][cin step][64 lanes], folded bias and requantization records per expanded channel
  const v4i* w1;
  const int32_t* b1;
  const v4i* q1;
  // depthwise: {three tap rows, folded bias} and requantization records per expanded channel
  const v4i* dwk;
  const v4i* q2;
  // projection: fragments [output tile][chunk][64 lanes], folded bias and records per output channel
  const v4i* w2;
  const int32_t* b3;
  const v4i* q3;
  int Cin, H, Cexp, Cout, OH;
  int cin_steps, chunks, nt;
  int R, IR, bands, mh;           // output rows of a band, input rows behind them, bands per image, 32-pixel halo tiles
  int xs;                          // bytes per pixel row of the expansion operand
  int ep;                          // bytes per channel row of the expanded image
  int off_wave, wave_bytes;        // LDS: the wavefronts' private areas (expanded image, then projection operand)
  int off_red;                     // LDS: the projection's sums over all wavefronts, [tile][register][lane] (zeroed at the start)
  // quantization
  int x_xor;                       // 0x80 for uint8 input
  int zp1, neg_zws1_4;             // expansion weights' zero point as a second MFMA
  int e_zp, e_lo, e_hi, e_xor4, e_pad4, ties1;
  int dw_box, dw_zws, m_zp, m_lo, m_hi, m_xor, ties2;
  int zp3, neg_zws3_4;
  int out_zp, lo, hi, ties3;
  // residual Add (mode 0 = none; 1 / 2 = the block's result is the Add's first / second operand)
  double add_ra, add_rb;
  int add_mode, add_signed;
  int add_za, add_zb, add_zo, add_lo, add_hi;
  int aligned4;                    // output planes and bands are whole dwords: dword copy-out
};

// Window of output column J of a depthwise row: W input columns, stride S, SAME padding (one column left at
// stride 1, none at stride 2); byte 0 of `row` is the column under the first output's leftmost tap. Columns past
// the row's end recompute the last one (nobody stores them).
template <int W, int S, int J>
__device__ __forceinline__ int WindowOf(const int (&row)[(W + 5) / 4 + 1]) {
  constexpr int OW = (W + S - 1) / S;
  return Window<S * (J < OW ? J : OW - 1)>(row);
}

template <int W, int S, int J>
__device__ __forceinline__ int DwOne(const MbArgs& a, const int (&rows)[3][(W + 5) / 4 + 1], const v4i& k) {
  const int w0 = WindowOf<W, S, J>(rows[0]), w1 = WindowOf<W, S, J>(rows[1]), w2 = WindowOf<W, S, J>(rows[2]);
  int v = __builtin_amdgcn_sdot4(w0, k[0], k[3], false);
  v = __builtin_amdgcn_sdot4(w1, k[1], v, false);
  v = __builtin_amdgcn_sdot4(w2, k[2], v, false);
  if (a.dw_box) {  // (wave-uniform) weights packed unshifted: their zero point times the window sum
    int sx = __builtin_amdgcn_sdot4(w0, 0x00010101, 0, false);
    sx = __builtin_amdgcn_sdot4(w1, 0x00010101, sx, false);
    sx = __builtin_amdgcn_sdot4(w2, 0x00010101, sx, false);
    v -= a.dw_zws * sx;
  }
  return v;
}

// Four output columns J0 .. J0 + 3 of one channel's depthwise row, requantized.
template <int W, int S, int J0>
__device__ __forceinline__ void DwFour(const MbArgs& a, const int (&rows)[3][(W + 5) / 4 + 1], const v4i& k, const v4i& q,
                                       int (&out)[4]) {
  const int acc[4] = {DwOne<W, S, J0>(a, rows, k), DwOne<W, S, J0 + 1>(a, rows, k), DwOne<W, S, J0 + 2>(a, rows, k),
                      DwOne<W, S, J0 + 3>(a, rows, k)};
  Requant8x4(acc, q, a.m_zp, a.m_lo, a.m_hi, a.ties2, out);
}

template <int W, int S, int J0>
struct DwRow {
  static __device__ __forceinline__ void Run(const MbArgs& a, const int (&rows)[3][(W + 5) / 4 + 1], const v4i& k, const v4i& q,
                                              uint8_t* m_row, int ch_byte, bool ch_live) {
    constexpr int OW = (W + S - 1) / S;
    if constexpr (J0 < OW) {
      int out[4];
      DwFour<W, S, J0>(a, rows, k, q, out);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (J0 + i < OW) m_row[(J0 + i) * kMStride + ch_byte] = ch_live ? static_cast<uint8_t>(out[i] ^ a.m_xor) : uint8_t{0};
      DwRow<W, S, J0 + 4>::Run(a, rows, k, q, m_row, ch_byte, ch_live);
    }
  }
};

// W: columns of the input; S: stride of the depthwise convolution; MO: 32-pixel tiles of a band's output;
// NTMAX: most 32-channel output tiles; ADD: residual Add behind the projection.
// (the register budget follows the accumulators: two wavefronts per SIMD up to five output tiles - three with two
// tiles, 168 registers, spill 36 bytes per lane and measure slower -, one beyond)
template <int W, int S, int MO, int NTMAX, bool ADD>
__global__ void __launch_bounds__(MaxWaves(MO * NTMAX) * 64) MbConvKernel(MbArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  constexpr int PL = S == 1 ? 1 : 0;               // left (and top) padding of the depthwise convolution
  constexpr int OW = (W + S - 1) / S;
  constexpr int NW = (W + 5) / 4;                  // dwords of a normalized input row: bytes 0 .. W + PL
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), threads = blockDim.x, waves = threads >> 6;
  const int n = blockIdx.x / a.bands, band = blockIdx.x - n * a.bands;
  const int or0 = band * a.R;
  const int rows_out = min(a.R, a.OH - or0);
  const int po = rows_out * OW;                    // live output pixels of the band
  const int ir0 = or0 * S - PL;                    // image row of the band's first halo row (may be -1)
  const int hp = a.IR * W;                         // halo pixels
  uint8_t* xin = lds;
  uint8_t* e_w = lds + a.off_wave + wave * a.wave_bytes + 4;  // (+ 4: the byte in front of row 0 is read)
  uint8_t* m_w = lds + a.off_wave + wave * a.wave_bytes + 16 + 32 * a.ep;

  const int frow = lane & 31, fh = lane >> 5;
  // The expansion's operands of the next chunk (fragments, the lane's bias and requantization record) are fetched
  // while this one is computed; what the later phases need is fetched at the chunk's start and has arrived by then.
  struct ExpandOperands {
    v4i wf[kMaxCinSteps];
    int bias1;
    v4i rq1;
  };
  auto fetch = [&](int chunk, ExpandOperands& o) {
    const int c = min(chunk, a.chunks - 1);
#pragma unroll
    for (int k = 0; k < kMaxCinSteps; ++k) o.wf[k] = a.w1[(c * a.cin_steps + min(k, a.cin_steps - 1)) * 64 + lane];
    o.bias1 = a.b1[c * 32 + frow];
    o.rq1 = a.q1[c * 32 + frow];
  };
  ExpandOperands next;
  fetch(wave, next);  // (on its way while the input rows are loaded)

  // ---- the band's input rows as the expansion's operand: xin[halo pixel][channel], signed bytes ----
  // A channel's halo rows are consecutive bytes of its plane. A thread takes four of them for four channels (dwords
  // at any byte offset where all sixteen bytes exist, else byte by byte with zeros for what lies outside the image,
  // the band or the channels), transposes, and stores four pixels' channel quads.
  {
    const int quads = a.mh * 8;                        // pixel quads of the halo tiles
    const int units = a.cin_steps * 8 * quads;         // x channel quads
    const int plane = a.H * W;
    const uint8_t* xn = a.x + static_cast<size_t>(n) * a.Cin * plane;
    const int live_lo = max(0, -ir0) * W, live_hi = min(a.IR, a.H - ir0) * W;  // the live bytes of a channel's halo rows
    const uint32_t xor4 = static_cast<uint32_t>(a.x_xor) * 0x01010101u;
    for (int unit = tid; unit < units; unit += threads) {
      const int c4 = unit / quads, p0 = (unit - c4 * quads) * 4;
      const int c = c4 * 4;
      const int at = ir0 * W + p0;                     // byte offset in the plane (negative above the image)
      uint32_t d[4];
      if (p0 >= live_lo && p0 + 4 <= live_hi && c + 4 <= a.Cin) {
#pragma unroll
        for (int j = 0; j < 4; ++j) __builtin_memcpy(&d[j], xn + (c + j) * plane + at, 4);
#pragma unroll
        for (int j = 0; j < 4; ++j) d[j] ^= xor4;
      } else {
        uint8_t b[4][4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const bool live = p0 + e >= live_lo && p0 + e < live_hi && c + j < a.Cin;
            b[j][e] = live ? static_cast<uint8_t>(xn[(c + j) * plane + at + e] ^ a.x_xor) : uint8_t{0};
          }
#pragma unroll
        for (int j = 0; j < 4; ++j) d[j] = b[j][0] | b[j][1] << 8 | b[j][2] << 16 | static_cast<uint32_t>(b[j][3]) << 24;
      }
      uint32_t px[4];
      Transpose4x4(d, px);
#pragma unroll
      for (int i = 0; i < 4; ++i) *reinterpret_cast<uint32_t*>(xin + (p0 + i) * a.xs + c) = px[i];
    }
  }
  for (int i = tid; i < a.nt * MO * 256; i += threads) reinterpret_cast<v4i*>(lds + a.off_red)[i] = v4i{0, 0, 0, 0};
  __syncthreads();

  v16i acc_out[MO][NTMAX];
#pragma unroll
  for (int mo = 0; mo < MO; ++mo)
#pragma unroll
    for (int t = 0; t < NTMAX; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc_out[mo][t][r] = 0;
  const v4i fz1 = {a.neg_zws1_4, a.neg_zws1_4, a.neg_zws1_4, a.neg_zws1_4};
  const v4i fz3 = {a.neg_zws3_4, a.neg_zws3_4, a.neg_zws3_4, a.neg_zws3_4};

  // one halo tile of the chunk: accumulate, requantize, store as [channel][halo pixel]
  auto expand_finish = [&](const v16i& acc, int mt, const v4i& rq1) {
#pragma unroll
    for (int gq = 0; gq < 4; ++gq) {
      const int av[4] = {acc[gq * 4], acc[gq * 4 + 1], acc[gq * 4 + 2], acc[gq * 4 + 3]};
      *reinterpret_cast<uint32_t*>(e_w + frow * a.ep + mt * 32 + 8 * gq + 4 * fh) =
          Requant8x4Pack(av, rq1, a.e_zp, a.e_lo, a.e_hi, a.ties1) ^ static_cast<uint32_t>(a.e_xor4);
    }
  };
  for (int chunk = wave; chunk < a.chunks; chunk += waves) {
    const int ch = chunk * 32 + frow;  // this lane's expanded channel, in all three phases
    const ExpandOperands cur = next;
    fetch(chunk + waves, next);
    const v4i dk = a.dwk[ch];
    const v4i rq2 = a.q2[ch];
    v4i w2f[NTMAX];
#pragma unroll
    for (int t = 0; t < NTMAX; ++t) w2f[t] = a.w2[(min(t, a.nt - 1) * a.chunks + chunk) * 64 + lane];

    // ---- expansion of every halo pixel for this chunk: e_w[channel][halo pixel], signed bytes; two halo tiles
    // at a time, so that one tile's MFMA chain runs under the other's ----
    for (int mt = 0; mt < a.mh; mt += 2) {
      const bool two = mt + 1 < a.mh;  // (wave-uniform)
      const int mt1 = two ? mt + 1 : mt;
      v16i acc0, acc1;
#pragma unroll
      for (int r = 0; r < 16; ++r) acc0[r] = acc1[r] = cur.bias1;
      const uint8_t* xa0 = xin + (mt * 32 + frow) * a.xs + fh * 16;
      const uint8_t* xa1 = xin + (mt1 * 32 + frow) * a.xs + fh * 16;
#pragma unroll
      for (int k = 0; k < kMaxCinSteps; ++k) {
        if (k < a.cin_steps) {
          const v4i fx0 = *reinterpret_cast<const v4i*>(xa0 + k * 32);
          const v4i fx1 = *reinterpret_cast<const v4i*>(xa1 + k * 32);
          acc0 = __builtin_amdgcn_mfma_i32_32x32x32_i8(fx0, cur.wf[k], acc0, 0, 0, 0);
          if (two) acc1 = __builtin_amdgcn_mfma_i32_32x32x32_i8(fx1, cur.wf[k], acc1, 0, 0, 0);
          if (a.zp1) {
            acc0 = __builtin_amdgcn_mfma_i32_32x32x32_i8(fx0, fz1, acc0, 0, 0, 0);
            if (two) acc1 = __builtin_amdgcn_mfma_i32_32x32x32_i8(fx1, fz1, acc1, 0, 0, 0);
          }
        }
      }
      expand_finish(acc0, mt, cur.rq1);
      if (two) expand_finish(acc1, mt1, cur.rq1);
    }
    __builtin_amdgcn_wave_barrier();

    // ---- depthwise 3x3: lane = (channel, every second output row) -> m_w[output pixel][channel] ----
    for (int orr = fh; orr < rows_out; orr += 2) {
      int rows[3][NW + 1];
#pragma unroll
      for (int t = 0; t < 3; ++t) {
        const int irr = orr * S + t;                 // halo row
        const int ih = ir0 + irr;
        const bool row_ok = ih >= 0 && ih < a.H;
        const int o = frow * a.ep + irr * W - PL;    // byte 0 of the normalized row (>= -1: e_w has room in front)
        const int shift = (o + 4) & 3;
        const uint32_t* src = reinterpret_cast<const uint32_t*>(e_w + ((o + 4) & ~3) - 4);
        uint32_t raw[NW + 1];
#pragma unroll
        for (int i = 0; i <= NW; ++i) raw[i] = src[i];
#pragma unroll
        for (int i = 0; i < NW; ++i)
          rows[t][i] = row_ok ? static_cast<int>(__builtin_amdgcn_alignbyte(raw[i + 1], raw[i], shift)) : a.e_pad4;
        rows[t][NW] = a.e_pad4;
        // the padding columns: byte 0 at stride 1 (column -1), byte W + PL (column W)
        if (PL) rows[t][0] = (rows[t][0] & ~0xff) | (a.e_pad4 & 0xff);
        constexpr int rb = W + PL;
        rows[t][rb / 4] = (rows[t][rb / 4] & ~(0xff << (8 * (rb % 4)))) | (a.e_pad4 & (0xff << (8 * (rb % 4))));
      }
      DwRow<W, S, 0>::Run(a, rows, dk, rq2, m_w + orr * OW * kMStride, frow, ch < a.Cexp);
    }
    __builtin_amdgcn_wave_barrier();

    // ---- this chunk's contribution to every output tile ----
#pragma unroll
    for (int mo = 0; mo < MO; ++mo) {
      const v4i fx = *reinterpret_cast<const v4i*>(m_w + (mo * 32 + frow) * kMStride + fh * 16);
#pragma unroll
      for (int t = 0; t < NTMAX; ++t) {
        if (t < a.nt) {
          acc_out[mo][t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fx, w2f[t], acc_out[mo][t], 0, 0, 0);
          if (a.zp3) acc_out[mo][t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fx, fz3, acc_out[mo][t], 0, 0, 0);
        }
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
  // ---- the wavefronts' partial projections meet in LDS (integer atomics on a zeroed image laid out like the
  // accumulators: [tile][register][lane]); then every wavefront finishes its share of the (output tile, pixel tile,
  // register quad) units: requantize, add the residual, store. A unit is four pixels of each of 32 channels.
  int* red = reinterpret_cast<int*>(lds + a.off_red);
  const size_t out_plane = static_cast<size_t>(a.OH) * OW;
  const int units = a.nt * MO * 4;
  constexpr int kMaxUnits = (NTMAX * MO * 4 + kMinWaves - 1) / kMinWaves;
  // what the units need from memory is requested first: the sums then form under these loads
  int bias3[kMaxUnits];
  v4i rq3[kMaxUnits];
  uint32_t resv[kMaxUnits];
  size_t at[kMaxUnits];
  int px0[kMaxUnits];
#pragma unroll
  for (int i = 0; i < kMaxUnits; ++i) {
    const int u = wave + i * waves;
    if (u >= units) break;
    const int t = u / (MO * 4), mo = (u >> 2) % MO, gq = u & 3;
    const int oc = t * 32 + frow;
    bias3[i] = a.b3[oc];
    rq3[i] = a.q3[oc];
    px0[i] = mo * 32 + 8 * gq + 4 * fh;
    at[i] = (static_cast<size_t>(n) * a.Cout + oc) * out_plane + static_cast<size_t>(or0) * OW + px0[i];
    resv[i] = 0;
    if (ADD && oc < a.Cout) {
      if (a.aligned4) {
        if (px0[i] < po) resv[i] = *reinterpret_cast<const uint32_t*>(a.res + at[i]);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (px0[i] + e < po) resv[i] |= static_cast<uint32_t>(a.res[at[i] + e]) << (8 * e);
      }
    }
  }
  if (wave < a.chunks) {  // (a wavefront that walked no chunk has nothing to add)
#pragma unroll
    for (int t = 0; t < NTMAX; ++t)
      if (t < a.nt) {
#pragma unroll
        for (int mo = 0; mo < MO; ++mo)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            __hip_atomic_fetch_add(red + ((t * MO + mo) * 16 + r) * 64 + lane, acc_out[mo][t][r], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kMaxUnits; ++i) {
    const int u = wave + i * waves;
    if (u >= units) break;
    const int t = u / (MO * 4), gq = u & 3;
    const int oc = t * 32 + frow;
    int av[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) av[e] = red[((u >> 2) * 16 + gq * 4 + e) * 64 + lane] + bias3[i];
    const uint32_t codes = Requant8x4Pack(av, rq3[i], a.out_zp, a.lo, a.hi, a.ties3);
    if (oc >= a.Cout) continue;
    if (a.aligned4) {
      if (px0[i] < po) {
        uint32_t o = codes;
        if (ADD) o = AddResidual4(a, o, resv[i]);
        *reinterpret_cast<uint32_t*>(a.y + at[i]) = o;
      }
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (px0[i] + e < po) {
          int o = static_cast<int>((codes >> (8 * e)) & 0xff);
          if (ADD) o = AddResidual1(a, o, static_cast<int>((resv[i] >> (8 * e)) & 0xff));
          a.y[at[i] + e] = static_cast<uint8_t>(o);
        }
    }
  }
}

// ---- stride 1: a lane keeps its halo rows in registers ----
//
// Tile rows of the expansion's matrix product come in fours to a lane (rows 8 i + 4 f .. + 3 to lane half f), so four neighbouring
// halo columns are one requantized dword of a lane, and the halo can be dealt out such that a lane half finds the whole halo of
// the outputs it computes in its own accumulators: the expanded tensor passes through registers only. Of the two splits
//   WIDE   64 halo pixels, four rows x eight columns a half, 2 x 7 outputs a half (the ninth halo column is padding): the halves
//          are the two column halves of 14 columns, or two pairs of rows of 7;
//   narrow 32 halo pixels, four rows x four columns a half (two of them in both), 2 x 2 outputs a half: 2 x 4 outputs a workgroup,
// the first computes an output for fewer expanded pixels (2.3 against 4), the second makes four times the workgroups. Bound by
// the vector ALU (390 instructions and 2200 cycles a chunk in the wide form, a third of them dot products) where a batch fills the
// chip, by the chain load - expansion - stencil - projection - sum - store in small ones. Before, one kernel served both strides: the
// expanded image went through LDS, every window was cut from it and every code requantized by itself. uint8, before and
// now, microseconds: 14 columns, 64 to 384 to 64: batch 1 9.0 / 4.8, batch 64 15.8 / 10.6; 96 to 576 to 96: 12.9 / 6.3, 26.3 / 16.6.
struct MbTileArgs : MbArgs {
  int W, batch;
  int tiles_per_image, col_tiles, tile_rows;
  uint32_t m_tiles, m_cols;        // reciprocals
  int half_rows, half_cols, half_halo;  // the second half's outputs: rows and columns behind the first's, and its halo's columns
  int last1, last3;                // channels of the last reduction step of the expansion and of the projection
  int dw_nzws3;                    // minus the depthwise weights' zero point in three bytes (0: folded)
  int pre1, pre2, pre3;            // as RequantCodes4 takes them (clamps in the signed domain)
  int out_xor4;
};

constexpr int TileWaves(bool wide, int steps) { return wide || steps > 3 ? 8 : 12; }  // (two wavefronts a SIMD within 256 registers, three within 168)

template <bool WIDE, int KS, int NT, bool ADD, bool PLAIN>
__global__ void __launch_bounds__(TileWaves(WIDE, KS) * 64) MbTileKernel(MbTileArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  constexpr int MT = WIDE ? 2 : 1;    // 32-pixel halo tiles = dwords of a lane's halo row
  constexpr int kWin = WIDE ? 4 : 1;  // window dwords of a halo row: two outputs each
  const int tid = threadIdx.x, lane = tid & 63, col = lane & 31, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), threads = blockDim.x, waves = threads >> 6;
  int wg = blockIdx.x;  // an XCD gets a contiguous run of tiles: neighbours share halo rows in its L2
  {
    const int per = gridDim.x >> 3, rem = gridDim.x & 7, xcd = wg & 7;
    wg = xcd * per + min(xcd, rem) + (wg >> 3);
  }
  const auto over = [](int v, uint32_t m) { return static_cast<int>(__umulhi(static_cast<uint32_t>(v), m) + (static_cast<uint32_t>(v) & (m ? 0u : ~0u))); };
  const int n = over(wg, a.m_tiles), tile = wg - n * a.tiles_per_image;
  const int band = over(tile, a.m_cols);
  const int r0 = band * a.tile_rows, c0 = (tile - band * a.col_tiles) * 4;  // (WIDE: one tile of columns)

  // what the first chunk needs is requested before the input
  struct ExpandOperands {
    v4i wf[KS];
    int bias;
    v4i q;
  } next;
  v4i taps4, q2, w2[WIDE ? NT : 2 * NT];
  const auto fetch = [&](int chunk) {
#pragma unroll
    for (int k = 0; k < KS; ++k) next.wf[k] = a.w1[(chunk * a.cin_steps + min(k, a.cin_steps - 1)) * 64 + lane];
    next.bias = a.b1[chunk * 32 + col];
    next.q = a.q1[chunk * 32 + col];
  };
  const auto fetch_depthwise = [&](int chunk) {
    taps4 = a.dwk[chunk * 32 + col];
    q2 = a.q2[chunk * 32 + col];
  };
  const auto fetch_projection = [&](int chunk) {
    if constexpr (WIDE) {
#pragma unroll
      for (int t = 0; t < NT; ++t) w2[t] = a.w2[(min(t, a.nt - 1) * a.chunks + chunk) * 64 + lane];
    } else {  // sixteen output channels a product, the upper half of whose reduction meets zeros
#pragma unroll
      for (int t = 0; t < 2 * NT; ++t) w2[t] = a.w2[(min(t >> 1, a.nt - 1) * a.chunks + chunk) * 64 + (lane & 16) * 2 + (t & 1) * 16 + (lane & 15)];
    }
  };
  if (wave < a.chunks) {
    fetch(wave);
    fetch_depthwise(wave);
  }

  // ---- the halo as the expansion's operand: xin[slot][channel], signed bytes; slots 4 s .. 4 s + 3 are dword s >> 1 of half s & 1.
  // What lies outside the image holds anything: its expanded codes are replaced. ----
  const int items = a.cin_steps * 64 * MT;
  struct Item {
    uint32_t d[4];
    int by[4];
  };
  const auto slots = [&](int u) { return u & (8 * MT - 1); };
  const auto channel = [&](int u) { return u / (8 * MT) * 4; };
  const auto load = [&](int u) {
    Item it;
    const int plane = a.H * a.W, image = a.Cin * plane;
    const uint8_t* xn = a.x + static_cast<size_t>(n) * image;
    const int lowest = n == 0 ? 0 : -4, highest = n == a.batch - 1 ? image - 4 : INT_MAX;  // (inside the tensor)
    const int s = slots(u), c = channel(u), f = s & 1, i = s >> 1;
    const int row = r0 + f * a.half_rows - 1 + (WIDE ? i >> 1 : i);
    const int x = WIDE ? f * a.half_halo + 4 * (i & 1) : c0 - 1 + 2 * f;
    const int at = min(max(row, 0), a.H - 1) * a.W + x;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int o = min(c + j, a.Cin - 1) * plane + at, in = min(max(o, lowest), highest);
      it.by[j] = in - o;
      __builtin_memcpy(&it.d[j], xn + in, 4);
    }
    return it;
  };
  const auto store = [&](int u, const Item& it) {
    uint32_t d[4], px[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)  // a dword at an end of the tensor was read from inside it
      d[j] = (it.d[j] << (8 * max(it.by[j], 0)) >> (8 * min(max(-it.by[j], 0), 3))) ^ (a.x_xor * 0x01010101u);
    Transpose4x4(d, px);
#pragma unroll
    for (int e = 0; e < 4; ++e) *reinterpret_cast<uint32_t*>(lds + (4 * slots(u) + e) * a.xs + channel(u)) = px[e];
  };
  Item first;
  if (tid < items) first = load(tid);

  // ---- under these loads: the constants of the later phases ----
  const MbTileArgs& b = LateArgs<MbTileArgs>();
  constexpr int kQuads = WIDE ? 4 : 1;  // of output pixels of a lane and 32-channel tile
  int* red = reinterpret_cast<int*>(lds + b.off_red);
  for (int i = tid; i < b.nt * kQuads * 64; i += threads) reinterpret_cast<v4i*>(red)[i] = v4i{0, 0, 0, 0};
  const auto constant = [&](int value4, int live, int group) {  // a fragment of `value` for `live` channels
    v4i f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int left = live - 16 * group - 4 * i;
      f[i] = left >= 4 ? value4 : left <= 0 ? 0 : value4 & static_cast<int>((1u << (8 * left)) - 1u);
    }
    return f;
  };
  const v4i z1_last = constant(b.neg_zws1_4, b.last1, half);
  const v4i z1 = {b.neg_zws1_4, b.neg_zws1_4, b.neg_zws1_4, b.neg_zws1_4};
  // bytes of a lane's halo dwords that are columns of the image, and which of its four halo rows are none
  uint32_t keep[MT], fill[MT];
  int outside = 0;
#pragma unroll
  for (int j = 0; j < MT; ++j) {
    const int x = WIDE ? half * b.half_halo + 4 * j : c0 - 1 + 2 * half;
    keep[j] = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (static_cast<unsigned>(x + e) < static_cast<unsigned>(b.W)) keep[j] |= 0xffu << (8 * e);
    fill[j] = static_cast<uint32_t>(b.e_pad4) & ~keep[j];
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int row = r0 + half * b.half_rows - 1 + r;
    if (static_cast<unsigned>(row) >= static_cast<unsigned>(b.H)) outside |= 1 << r;
  }
  const bool edge = r0 == 0 || r0 + b.tile_rows >= b.H;
  const uint32_t order = WIDE && half && b.half_halo ? 0x07060504u : 0x06050403u;  // left padding in front of the halo's columns, or right behind
  const int cin_steps = b.cin_steps, xs = b.xs, e_pad4 = b.e_pad4, chunks = b.chunks, nt = b.nt, zp1 = b.zp1, zp3 = b.zp3, neg_zws3_4 = b.neg_zws3_4,
            dw_box = b.dw_box, dw_nzws3 = b.dw_nzws3, last3 = b.last3, H = b.H, W = b.W, Cout = b.Cout, half_rows = b.half_rows, half_cols = b.half_cols;
  const int32_t* const b3 = b.b3;
  const v4i* const q3 = b.q3;
  const uint8_t* const other = b.res;
  uint8_t* const y = b.y;  // (read through the reference behind a store, each would be loaded again)

  if (tid < items) store(tid, first);
  for (int u = tid + threads; u < items; u += threads) store(u, load(u));
  __syncthreads();

  // the zero-point term of uint8 expansion weights depends on the pixel alone
  const uint8_t* xa = lds + col * xs + half * 16;
  v16i xsum[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int r = 0; r < 16; ++r) xsum[mt][r] = 0;
  if (zp1) {  // (uniform)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int k = 0; k < KS; ++k)
        if (k < cin_steps)
          xsum[mt] = __builtin_amdgcn_mfma_i32_32x32x32_i8(*reinterpret_cast<const v4i*>(xa + mt * 32 * xs + k * 32), k + 1 < cin_steps ? z1 : z1_last, xsum[mt], 0, 0, 0);
  }

  constexpr bool kResident = WIDE ? KS <= 3 : NT <= 5;  // the operand stays in registers (with more steps it would not fit)
  v4i fx[MT][KS];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int k = 0; k < (kResident ? KS : 0); ++k) fx[mt][k] = *reinterpret_cast<const v4i*>(xa + mt * 32 * xs + min(k, cin_steps - 1) * 32);
  uint8_t* m_w = lds + b.off_wave + wave * b.wave_bytes;
  v16i acc_w[WIDE ? NT : 1], zp_w;
  v4i acc_n[WIDE ? 1 : 2 * NT], zp_n = {0, 0, 0, 0};
#pragma unroll
  for (int r = 0; r < 16; ++r) zp_w[r] = 0;
#pragma unroll
  for (int t = 0; t < (WIDE ? NT : 1); ++t) acc_w[t] = zp_w;
#pragma unroll
  for (int t = 0; t < (WIDE ? 1 : 2 * NT); ++t) acc_n[t] = zp_n;

  // a chunk's contribution to every output tile
  v4i fm = {0, 0, 0, 0};
#pragma unroll
  for (int t = 0; t < (WIDE ? NT : 2 * NT); ++t) w2[t] = fm;
  const auto project = [&](int live3) {
    if constexpr (!WIDE) fm = half ? v4i{0, 0, 0, 0} : fm;
    if constexpr (WIDE) {
#pragma unroll
      for (int t = 0; t < NT; ++t)
        if (t < nt) acc_w[t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fm, w2[t], acc_w[t], 0, 0, 0);
      if (zp3) zp_w = __builtin_amdgcn_mfma_i32_32x32x32_i8(fm, constant(neg_zws3_4, live3, half), zp_w, 0, 0, 0);
    } else {
#pragma unroll
      for (int t = 0; t < 2 * NT; ++t)
        if (t < 2 * nt) acc_n[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fm, w2[t], acc_n[t], 0, 0, 0);
      if (zp3) zp_n = __builtin_amdgcn_mfma_i32_16x16x64_i8(fm, constant(neg_zws3_4, live3, lane >> 4 & 1), zp_n, 0, 0, 0);
    }
  };
  for (int chunk = wave; chunk < chunks; chunk += waves) {
    // ---- expansion of the halo for this chunk's 32 channels: a lane's is `col` ----
    const uint8_t* xc = xa;
    if (!kResident) asm volatile("" : "+v"(xc));  // (or the compiler takes the reads out of the loop)
    v16i acc[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[mt][r] = xsum[mt][r] + next.bias;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int k = 0; k < KS; ++k)
        if (k < cin_steps) acc[mt] = __builtin_amdgcn_mfma_i32_32x32x32_i8(kResident ? fx[mt][k] : *reinterpret_cast<const v4i*>(xc + mt * 32 * xs + k * 32), next.wf[k], acc[mt], 0, 0, 0);
    project(32);
    fetch_projection(chunk);
    uint32_t e[4][MT];
    {
      const int64_t round = RoundHigh(next.q[2]);
#pragma unroll
      for (int i = 0; i < 4 * MT; ++i) {
        int v[4] = {acc[i / 4][4 * (i % 4)], acc[i / 4][4 * (i % 4) + 1], acc[i / 4][4 * (i % 4) + 2], acc[i / 4][4 * (i % 4) + 3]};
        e[i / MT][i % MT] = (RequantCodes4<PLAIN>(v, next.q, round, b.pre1, b.e_lo, b.e_hi) & keep[i % MT]) | fill[i % MT];
      }
    }
    if (edge) {  // (uniform)
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int j = 0; j < MT; ++j) e[r][j] = outside >> r & 1 ? static_cast<uint32_t>(e_pad4) : e[r][j];
    }
    const bool more = chunk + waves < chunks;
    if (more) fetch(chunk + waves);

    // ---- depthwise 3x3: two rows of outputs; a window dword serves two outputs, the second by taps a byte further up ----
    int win[4][kWin];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if constexpr (WIDE) {
        const uint32_t pad = static_cast<uint32_t>(e_pad4);
        const uint32_t w0 = __builtin_amdgcn_perm(e[r][0], pad, order), w1 = __builtin_amdgcn_perm(e[r][1], e[r][0], order), w2 = __builtin_amdgcn_perm(pad, e[r][1], order);
        win[r][0] = static_cast<int>(w0);
        win[r][1] = static_cast<int>(__builtin_amdgcn_alignbyte(w1, w0, 2));
        win[r][2] = static_cast<int>(w1);
        win[r][3] = static_cast<int>(__builtin_amdgcn_alignbyte(w2, w1, 2));
      } else {
        win[r][0] = static_cast<int>(e[r][0]);
      }
    }
    int sums[2][2 * kWin];  // [row][column]
    {
      int taps[2][3];
#pragma unroll
      for (int t = 0; t < 3; ++t) {
        taps[0][t] = taps4[t];
        taps[1][t] = taps4[t] << 8;
      }
#pragma unroll
      for (int o = 0; o < 2; ++o)
#pragma unroll
        for (int c = 0; c < 2 * kWin; ++c) {
          int v = __builtin_amdgcn_sdot4(win[o][c / 2], taps[c % 2][0], taps4[3], false);
          v = __builtin_amdgcn_sdot4(win[o + 1][c / 2], taps[c % 2][1], v, false);
          sums[o][c] = __builtin_amdgcn_sdot4(win[o + 2][c / 2], taps[c % 2][2], v, false);
        }
      if (dw_box) {  // (uniform) weights packed unshifted: their zero point times the window sum
#pragma unroll
        for (int o = 0; o < 2; ++o)
#pragma unroll
          for (int c = 0; c < 2 * kWin; ++c)
#pragma unroll
            for (int t = 0; t < 3; ++t) {
              if (PLAIN) sums[o][c] = __builtin_amdgcn_sdot4(win[o + t][c / 2], dw_nzws3 << (c % 2 * 8), sums[o][c], false);
              else sums[o][c] -= b.dw_zws * __builtin_amdgcn_sdot4(win[o + t][c / 2], 0x00010101 << (c % 2 * 8), 0, false);
            }
      }
    }
    {
      const int64_t round = RoundHigh(q2[2]);
      const auto codes = [&](int v0, int v1, int v2, int v3) {
        int v[4] = {v0, v1, v2, v3};
        return RequantCodes4<PLAIN>(v, q2, round, b.pre2, b.m_lo, b.m_hi);
      };
      if constexpr (WIDE) {  // the projection's operand [pixel][channel]: pixel 16 half + 8 row + column
#pragma unroll
        for (int o = 0; o < 2; ++o)
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const uint32_t c = codes(sums[o][4 * h], sums[o][4 * h + 1], sums[o][4 * h + 2], sums[o][4 * h + 3]);
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (4 * h + i < 7) m_w[(16 * half + 8 * o + 4 * h + i) * kMStride + col] = static_cast<uint8_t>(c >> (8 * i));
          }
      } else {  // pixel 4 row + column
        const uint32_t c = codes(sums[0][0], sums[0][1], sums[1][0], sums[1][1]);
#pragma unroll
        for (int i = 0; i < 4; ++i) m_w[(4 * (i / 2) + 2 * half + i % 2) * kMStride + col] = static_cast<uint8_t>(c >> (8 * i));
      }
    }
    __builtin_amdgcn_wave_barrier();  // (a wavefront reads what it wrote)

    // its contribution to the output tiles is added behind the next chunk's expansion
    fm = *reinterpret_cast<const v4i*>(m_w + (WIDE ? col * kMStride + half * 16 : (lane & 7) * kMStride + (lane & 16)));
    if (chunk + waves < chunks) fetch_depthwise(chunk + waves);
    __builtin_amdgcn_wave_barrier();
  }

  project((chunks - 1) % waves == wave ? last3 : 32);  // (a wavefront that walked no chunk adds nothing)
  // ---- the wavefronts' partial projections meet in LDS, laid out [32-channel tile][pixel quad][pixel][lane half = quad of the eight
  // pixels, channel]; every wavefront finishes its share of the quads. What a unit needs from memory is requested first. ----
  const int units = nt * kQuads;
  constexpr int kUnits = (NT * kQuads + kMinWaves - 1) / kMinWaves;
  const size_t plane = static_cast<size_t>(H) * W, lane_at = col * plane + (WIDE ? 4 : W) * half;
  int bias[kUnits], live[kUnits];
  v4i q[kUnits];
  uint32_t res[kUnits];
  size_t at[kUnits];
#pragma unroll
  for (int i = 0; i < kUnits; ++i) {
    const int u = wave + i * waves;
    if (u >= units) break;
    const int t = u / kQuads, quad = u % kQuads, oc = t * 32 + col;  // (u, t and quad are uniform)
    const int row = r0 + (WIDE ? (quad >> 1) * half_rows + (quad & 1) : 0), x = c0 + (WIDE ? (quad >> 1) * half_cols : 0);
    live[i] = row + (WIDE ? 0 : half) < H && oc < Cout ? (WIDE ? 4 - half : min(4, W - x)) : 0;
    at[i] = (static_cast<size_t>(n) * Cout + t * 32) * plane + static_cast<size_t>(row) * W + x + lane_at;
    bias[i] = b3[oc];
    q[i] = q3[oc];
    res[i] = 0;
    if (ADD) {
      if (live[i] == 4) {
        __builtin_memcpy(&res[i], other + at[i], 4);
      } else {
        uint16_t lo = 0;
        if (live[i] & 2) __builtin_memcpy(&lo, other + at[i], 2);
        res[i] = lo;
        if (live[i] & 1) res[i] |= static_cast<uint32_t>(other[at[i] + (live[i] & 2)]) << (8 * (live[i] & 2));
      }
    }
  }
  if (wave < chunks) {  // (a wavefront that walked no chunk has nothing to add)
    if constexpr (WIDE) {
#pragma unroll
      for (int t = 0; t < NT; ++t)
        if (t < nt)
#pragma unroll
          for (int r = 0; r < 16; ++r) __hip_atomic_fetch_add(red + (t * 16 + r) * 64 + lane, acc_w[t][r] + zp_w[r], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    } else if (half == 0) {  // (rows 8 to 15 of a product hold no pixel)
#pragma unroll
      for (int t = 0; t < 2 * NT; ++t)
        if (t < 2 * nt)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            __hip_atomic_fetch_add(red + ((t >> 1) * 4 + r) * 64 + (lane & 16) * 2 + (t & 1) * 16 + (lane & 15), acc_n[t][r] + zp_n[r], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kUnits; ++i) {
    const int u = wave + i * waves;
    if (u >= units) break;
    int v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = red[(u * 4 + e) * 64 + lane] + bias[i];
    uint32_t codes = RequantCodes4<PLAIN>(v, q[i], RoundHigh(q[i][2]), b.pre3, b.lo, b.hi) ^ static_cast<uint32_t>(b.out_xor4);
    if (ADD) codes = AddResidual4(b, codes, res[i]);
    if (live[i] == 4) {
      __builtin_memcpy(y + at[i], &codes, 4);
    } else {
      if (live[i] & 2) __builtin_memcpy(y + at[i], &codes, 2);
      if (live[i] & 1) y[at[i] + (live[i] & 2)] = static_cast<uint8_t>(codes >> (8 * (live[i] & 2)));
    }
  }
}

typedef void (*MbFn)(MbArgs);
typedef void (*MbTileFn)(MbTileArgs);

template <bool WIDE, bool ADD, bool PLAIN>
MbTileFn TileKernelOf(int widest) {  // (in 32-channel steps: the block's input and output)
  if (widest <= 2) return MbTileKernel<WIDE, 2, 2, ADD, PLAIN>;
  if (widest <= 3) return MbTileKernel<WIDE, 3, 3, ADD, PLAIN>;
  if (widest <= 5) return MbTileKernel<WIDE, 5, 5, ADD, PLAIN>;
  if constexpr (!WIDE) return MbTileKernel<false, 5, 10, ADD, PLAIN>;
  return nullptr;
}
template <bool WIDE>
MbTileFn TileKernelOf(int widest, bool add, bool plain) {
  return add ? (plain ? TileKernelOf<WIDE, true, true>(widest) : TileKernelOf<WIDE, true, false>(widest))
             : (plain ? TileKernelOf<WIDE, false, true>(widest) : TileKernelOf<WIDE, false, false>(widest));
}

template <int W, bool ADD>
MbFn KernelNt(int nt) {
  if (nt <= 2) return MbConvKernel<W, 2, 1, 2, ADD>;
  if (nt <= 5) return MbConvKernel<W, 2, 1, 5, ADD>;
  if (nt <= 10) return MbConvKernel<W, 2, 1, 10, ADD>;
  return nullptr;
}

template <bool ADD>
MbFn KernelOf(int w, int nt) {
  return w == 28 ? KernelNt<28, ADD>(nt) : w == 14 ? KernelNt<14, ADD>(nt) : nullptr;
}

struct Plan {
  MbTileArgs a;
  MbFn fn;            // stride 2
  MbTileFn tile_fn;   // stride 1
  int lds_bytes;
  unsigned grid, block;
};

int MbConvRun(tvx_op* op, const void* in0, const void* in1, void* out, hipStream_t st) {
  const Plan* plan = reinterpret_cast<const Plan*>(op->host_blob.data());
  MbTileArgs a = plan->a;
  a.x = static_cast<const uint8_t*>(in0);
  a.y = static_cast<uint8_t*>(out);
  a.res = static_cast<const uint8_t*>(in1);
  if (a.add_mode && !in1) return SetError(TVX_E_INVALID, "pwconv_dwconv3x3_pwconv_i8: the fused Add needs its second operand as in1");
  if (a.aligned4 && ((reinterpret_cast<uintptr_t>(out) | (a.add_mode ? reinterpret_cast<uintptr_t>(in1) : 0)) & 3))
    a.aligned4 = 0;
  if (plan->tile_fn) hipLaunchKernelGGL(plan->tile_fn, dim3(plan->grid), dim3(plan->block), plan->lds_bytes, st, a);
  else hipLaunchKernelGGL(plan->fn, dim3(plan->grid), dim3(plan->block), plan->lds_bytes, st, static_cast<const MbArgs&>(a));
  TVX_HIP_CHECK(hipGetLastError());
  return TVX_OK;
}

int RoundUp(int v, int m) { return (v + m - 1) / m * m; }

// weights [oc][c] (uint8 re-biased to int8) -> MFMA fragments [oc tile][32-channel step][64 lanes][16 bytes];
// sums[oc] = sum of the signed weights
void PackPointwise(const void* w_host, bool w_u8, int OC, int C, std::vector<int8_t>* packed, std::vector<int64_t>* sums) {
  const int tiles = (OC + 31) / 32, steps = (C + 31) / 32;
  packed->assign(static_cast<size_t>(tiles) * steps * 1024, 0);
  sums->assign(static_cast<size_t>(tiles) * 32, 0);
  const uint8_t* src = static_cast<const uint8_t*>(w_host);
  for (int oc = 0; oc < OC; ++oc)
    for (int c = 0; c < C; ++c) {
      const uint8_t raw = src[static_cast<size_t>(oc) * C + c];
      const int8_t v = static_cast<int8_t>(w_u8 ? raw ^ 0x80 : raw);
      const int ks = c / 32, half = (c % 32) / 16, j = c % 16;
      (*packed)[((static_cast<size_t>(oc / 32) * steps + ks) * 64 + half * 32 + oc % 32) * 16 + j] = v;
      (*sums)[oc] += v;
    }
}

bool IsPointwise(const tvx_conv2d_desc* d) {
  return d->multiplier == 0 && d->groups <= 1 && d->k_w == 1 && d->k_h == 1 && d->stride_w == 1 && d->stride_h == 1 &&
         d->dilation_w == 1 && d->dilation_h == 1 && d->pad_left == 0 && d->pad_top == 0 && d->out_w == d->in_w &&
         d->out_h == d->in_h;
}

bool Feeds(const tvx_conv2d_desc* a, const tvx_conv2d_desc* b) {
  return b->in_w == a->out_w && b->in_h == a->out_h && b->in_c == a->out_c && b->batch == a->batch &&
         b->in_dtype == a->out_dtype && b->in_scale == a->out_scale && b->in_zp == a->out_zp;
}

}  // namespace

// `op` carries the projection (op->conv, its requantization tables in h_mult / h_shift, clamp, fused Add);
// the expansion and the depthwise convolution come with their own tables. Declines (TVX_E_UNSUPPORTED) what
// the kernel does not cover; the caller then creates the operators one by one.
int MbConvSetup(tvx_op* op, const MbStage& ex, const MbStage& dw, const tvx_conv2d_desc* pr, const void* pr_w, const void* pr_b) {
  const tvx_conv2d_desc *e = ex.desc, *d = dw.desc;
  if (!IsPointwise(e) || !IsPointwise(pr) || !Feeds(e, d) || !Feeds(d, pr)) return TVX_E_UNSUPPORTED;
  if (d->multiplier != 1 || d->k_w != 3 || d->k_h != 3 || d->dilation_w != 1 || d->dilation_h != 1) return TVX_E_UNSUPPORTED;
  const int S = d->stride_w, W = d->in_w, H = d->in_h;
  if (d->stride_h != d->stride_w || (S != 1 && S != 2)) return TVX_E_UNSUPPORTED;
  const int PL = S == 1 ? 1 : 0;
  if (static_cast<int>(d->pad_left) != PL || static_cast<int>(d->pad_top) != PL) return TVX_E_UNSUPPORTED;
  const int OW = (W + S - 1) / S;
  if (static_cast<int>(d->out_w) != OW || static_cast<int>(d->out_h) != (H + S - 1) / S) return TVX_E_UNSUPPORTED;
  if (S == 2 && ((W | H) & 1)) return TVX_E_UNSUPPORTED;
  const int Cin = e->in_c, Cexp = e->out_c, Cout = pr->out_c;
  const int cin_steps = (Cin + 31) / 32, chunks = (Cexp + 31) / 32, nt = (Cout + 31) / 32;
  if (cin_steps > kMaxCinSteps) return TVX_E_UNSUPPORTED;
  const bool two_forms = W == 7 || W == 14;
  if (S == 1 ? W < 3 || static_cast<uint64_t>(Cin) * H * W < 4 || nt > (two_forms ? 10 : 5) : (W != 14 && W != 28) || nt > 10) return TVX_E_UNSUPPORTED;
  Plan plan{};
  MbTileArgs& a = plan.a;
  a.nt = nt;
  a.add_mode = op->fused_add;
  if (const char* f = getenv("TVX_NO_MBCONV"))  // tuning aid: leaves blocks to the single operators
    if (atoi(f)) return TVX_E_UNSUPPORTED;
  if (static_cast<uint64_t>(e->in_c) * H * W >= (1ull << 31)) return TVX_E_UNSUPPORTED;
  const char* const every = getenv("TVX_MBCONV_ALL");  // takes blocks also where the single operators are faster
  const bool all = every && atoi(every);
  if (S == 2 && !all) return TVX_E_UNSUPPORTED;  // (28 columns, 32 to 192 to 64: batch 1 8.5 us against 7.5, batch 64 15.0 against 15.7; 14 columns: twice their time)
  a.Cin = Cin; a.H = H; a.Cexp = Cexp; a.Cout = Cout; a.OH = d->out_h;
  a.cin_steps = cin_steps; a.chunks = chunks;
  a.xs = cin_steps * 32 + 16;
  uint64_t wgs;
  int waves;
  bool wide = false;
  if (S == 1) {
    // Microseconds, uint8 (a network of single operators: "apart"), by batch:
    //                                             1    4    8    16    32    64
    //   14 columns, 64 to 384 to 64    narrow   4.8  5.1  5.4   6.8   9.6  15.3    (the better of four and twelve wavefronts)
    //                                  wide     6.4  6.5  6.6   6.9   7.4  10.8    (of four and eight)
    //   14 columns, 96 to 576 to 96    narrow   6.4  6.7  6.9   9.6  15.2  25.9    wide 8.8  8.8  9.1  9.4  10.3  16.7
    //   28 columns, 32 to 192 to 32    narrow   4.2  5.3  6.7  10.2  16.3  29.5    apart 9.2  9.4  9.7  11.0  13.9  20.5
    //   7 columns, 160 to 960 to 160   narrow   9.7  9.9  9.9  10.3  11.0  18.0    apart 10.4  11.6  12.2  14.3  16.6  20.2    wide - 16.6
    //   7 columns, 160 to 960 to 320   narrow  33.6  ...             36.0  61.8    apart 10.3  11.4  12.0  14.3  16.8  20.5
    //  14 columns, 160 to 960 to 320   narrow  19.3  20.1       35.1       108.6   apart 10.1  13.6       20.5        46.6
    // Taken: up to 160 results; of 28 columns only while workgroups are few (batch 13, here and as two or three launches: 32 to 192 to 32 9.2 and 9.9,
    // 64 to 384 to 64 13.1 and 14.2, 96 to 576 to 96 20.9 and 22.8; batch 14 10.1 and 10.2, 14.7 and 14.8; 160 to 160 to 160 batch 5 8.2 and 10.1, 6
    // 13.0 and 10.1; 128 to 768 to 128 14.5 and 16.6, 21.3 and 18.2). Narrow as long as each of its workgroups finds a CU of its own.
    // The narrow form cares for no width, and what counts is the workgroups: 3 to 56 columns, batch 1 to 64, 480 blocks of the sizes above in front of
    // the same line take .62 of the time apart on the average (24 to 144 to 24 on 56 columns, batch 1, 5.5 and 9.1; 64 to 384 to 64 on 12, batch 16, 7.2
    // and 9.8; 96 to 576 to 96 on 5, batch 8, 7.1 and 10.4; 160 to 160 on 10, batch 16, 11.2 and 15.4); behind it .78 to 1.41. Fewer
    // chunks than the four wavefronts that walk them leave wavefronts idle: those stay apart but on the widths above.
    // In front of the line the parts are ahead in blocks of more than three steps (96 channels) and many chunks only, measured on 1600 of them:
    //  - a second workgroup of a CU has just begun, and the rows are those that dwconv3x3_i8 is best at: 160 to 960 to 160 on 8 columns, 264 to 288 workgroups,
    //    1.06 to 1.10 of the time apart (320 and more below 1), on 24 to 56 (wholes of eight), 288 to 400, 1.03 to 1.18 (448 and more below .95);
    //    of 20 to 24 chunks on 24 and 48 columns, 288, 1.00 to 1.13. Rows of 12, 20, 36: .82 to .99.
    //  - one small image whose rows are no whole dwords but whose planes are: 6 x 6 1.08 to 1.11, 10 x 10 1.05 to 1.07, 12 x 9 1.04 to 1.06 with 30 chunks
    //    (25 .95 to 1.01; 7 x 6, planes of no whole dwords, .95 to .99; 18 x 18 .95).
    const uint64_t narrow_wgs = static_cast<uint64_t>(e->batch) * ((H + 1) / 2) * ((W + 3) / 4), cus = ComputeUnits();
    wide = two_forms && nt <= 5 && narrow_wgs > cus;
    if (const char* f = getenv("TVX_MBCONV_WIDE")) wide = two_forms && nt <= 5 && atoi(f);  // test lever
    if (!all && W != 28 && !two_forms && chunks < kMinWaves) return TVX_E_UNSUPPORTED;
    const bool deep = std::max(cin_steps, nt) > 3, eights = W % 8 == 0;
    if (!all && deep && !two_forms && eights && narrow_wgs > cus &&
        ((5 * narrow_wgs <= 6 * cus && (chunks > 24 || (chunks >= 20 && W >= 24))) || (5 * narrow_wgs <= 8 * cus && chunks > 24 && W >= 24)))
      return TVX_E_UNSUPPORTED;
    if (!all && deep && !two_forms && chunks > 25 && e->batch == 1 && W % 4 && H * W % 4 == 0 && H * W <= 128) return TVX_E_UNSUPPORTED;
    if (!all && (nt > 5 || (!two_forms && narrow_wgs > (std::max(cin_steps, nt) <= 3 ? 5 : 2) * cus))) return TVX_E_UNSUPPORTED;
    a.W = W; a.batch = e->batch;
    a.half_rows = wide && W == 7 ? 2 : 0;
    a.half_cols = wide && W == 14 ? 7 : 0;
    a.half_halo = wide && W == 14 ? 6 : 0;
    a.tile_rows = 2 + a.half_rows;
    a.col_tiles = wide ? 1 : (W + 3) / 4;
    a.tiles_per_image = (H + a.tile_rows - 1) / a.tile_rows * a.col_tiles;
    const auto reciprocal = [](int v) { return v > 1 ? static_cast<uint32_t>(((1ull << 32) + v - 1) / v) : 0u; };
    a.m_tiles = reciprocal(a.tiles_per_image);
    a.m_cols = reciprocal(a.col_tiles);
    wgs = static_cast<uint64_t>(e->batch) * a.tiles_per_image;
    if (wgs * a.tiles_per_image >= (1ull << 32)) return TVX_E_UNSUPPORTED;
    a.last1 = Cin - (cin_steps - 1) * 32;
    a.last3 = Cexp - (chunks - 1) * 32;
    a.off_wave = (wide ? 64 : 32) * a.xs;
    a.wave_bytes = (wide ? 32 : 8) * kMStride;
    const int most = TileWaves(wide, std::max(cin_steps, nt));
    // as many wavefronts as share the chunks evenly; four where a CU holds several workgroups (others leave SIMDs empty: 28 columns,
    // batch 64, 29.5 us with four, 49 with five, 46 with six)
    const int rounds = (chunks + most - 1) / most;
    waves = wgs > cus ? kMinWaves : std::max(kMinWaves, wide ? most : (chunks + rounds - 1) / rounds);
    if (const char* f = getenv("TVX_MBCONV_WAVES")) waves = std::min(std::max(kMinWaves, atoi(f)), most);  // test lever
    a.off_red = a.off_wave + waves * a.wave_bytes;
    plan.lds_bytes = a.off_red + nt * (wide ? 4096 : 1024);
  } else {
    // rows of a band: what fills the output tile
    const int R = std::min<int>(32 / OW, d->out_h);
    if (R < 1) return TVX_E_UNSUPPORTED;
    const int IR = (R - 1) * S + 3, mh = (IR * W + 31) / 32;
    a.R = R; a.IR = IR; a.bands = (d->out_h + R - 1) / R; a.mh = mh;
    a.ep = mh * 32 + 4;
    a.off_wave = RoundUp(mh * 32 * a.xs, 16);
    a.wave_bytes = RoundUp(16 + 32 * a.ep + 32 * kMStride, 16);
    wgs = static_cast<uint64_t>(e->batch) * a.bands;
    // with at most one workgroup a CU eight wavefronts walk the chunks in half the rounds; with more, four and a second workgroup are better
    const int most = MaxWaves(nt <= 2 ? 2 : nt <= 5 ? 5 : 10);
    waves = wgs <= static_cast<uint64_t>(ComputeUnits()) ? most : kMinWaves;
    if (const char* f = getenv("TVX_MBCONV_WAVES")) waves = std::max(kMinWaves, atoi(f));  // tuning aid
    waves = std::min(waves, most);
    while (waves > kMinWaves && a.off_wave + waves * a.wave_bytes + nt * 4096 > 160 * 1024) --waves;
    a.off_red = a.off_wave + waves * a.wave_bytes;
    plan.lds_bytes = a.off_red + nt * 4096;
    a.aligned4 = static_cast<uint64_t>(d->out_h) * OW % 4 == 0 && (R * OW) % 4 == 0 && (static_cast<int>(d->out_h) % R * OW) % 4 == 0;
  }
  plan.block = 64 * waves;
  if (plan.lds_bytes > 160 * 1024) return TVX_E_UNSUPPORTED;
  if (!LaunchFits(wgs, plan.block)) return TVX_E_UNSUPPORTED;
  plan.grid = static_cast<unsigned>(wgs);

  // ---- expansion ----
  const bool x_u8 = e->in_dtype == TVX_U8, w1_u8 = e->w_dtype == TVX_U8;
  const int zxs = e->in_zp - (x_u8 ? 128 : 0);
  const int zws1 = (e->w_scales ? 0 : e->w_zp) - (w1_u8 ? 128 : 0);
  if (zxs < -128 || zxs > 127 || zws1 < -127 || zws1 > 127) return TVX_E_UNSUPPORTED;
  std::vector<int8_t> pk1, pk3;
  std::vector<int64_t> sw1, sw3;
  PackPointwise(ex.w, w1_u8, Cexp, Cin, &pk1, &sw1);
  const int exp_alloc = chunks * 32;
  std::vector<int32_t> b1(exp_alloc, 0), rq1, rq2, rq3;
  const int32_t* eb = static_cast<const int32_t*>(ex.b);
  for (int c = 0; c < Cexp; ++c) {
    const int64_t v = (eb ? eb[c] : 0) - static_cast<int64_t>(zxs) * sw1[c] + static_cast<int64_t>(Cin) * zxs * zws1;
    b1[c] = static_cast<int32_t>(static_cast<uint32_t>(v));
  }
  const int f1 = BuildRequantRecords(*ex.mult, *ex.shift, Cexp, exp_alloc, e->out_zp, &rq1, AccumulatorBound(Cin, ex.b, Cexp));
  if (f1 == kRqGeneric) return TVX_E_UNSUPPORTED;
  a.x_xor = x_u8 ? 0x80 : 0;
  a.zp1 = zws1 != 0;
  a.neg_zws1_4 = static_cast<int>(static_cast<uint32_t>((-zws1) & 0xff) * 0x01010101u);
  const bool e_u8 = e->out_dtype == TVX_U8;
  a.e_zp = e->out_zp; a.e_lo = ex.lo; a.e_hi = ex.hi; a.ties1 = f1 == kRqFast;
  a.e_xor4 = e_u8 ? static_cast<int>(0x80808080u) : 0;
  const int zes = e->out_zp - (e_u8 ? 128 : 0);
  a.e_pad4 = static_cast<int>(static_cast<uint32_t>(zes & 0xff) * 0x01010101u);

  // ---- depthwise ----
  const bool wd_u8 = d->w_dtype == TVX_U8;
  const int zwd = (d->w_scales ? 0 : d->w_zp) - (wd_u8 ? 128 : 0);
  std::vector<int32_t> dwpk, dbias;
  a.dw_box = PackDepthwise3x3(Cexp, dw.w, wd_u8, dw.b, zes, zwd, true, &dwpk, &dbias);
  a.dw_zws = zwd;
  std::vector<int32_t> dwk(static_cast<size_t>(exp_alloc) * 4, 0);
  for (int c = 0; c < Cexp; ++c) {
    for (int t = 0; t < 3; ++t) dwk[4 * c + t] = dwpk[4 * c + t];
    dwk[4 * c + 3] = dbias[c];
  }
  const int f2 = BuildRequantRecords(*dw.mult, *dw.shift, Cexp, exp_alloc, d->out_zp, &rq2, AccumulatorBound(9, dw.b, Cexp));
  if (f2 == kRqGeneric) return TVX_E_UNSUPPORTED;
  const bool m_u8 = d->out_dtype == TVX_U8;
  a.m_zp = d->out_zp; a.m_lo = dw.lo; a.m_hi = dw.hi; a.ties2 = f2 == kRqFast;
  a.m_xor = m_u8 ? 0x80 : 0;
  const int zms = d->out_zp - (m_u8 ? 128 : 0);

  // ---- projection ----
  const bool w3_u8 = pr->w_dtype == TVX_U8;
  const int zws3 = op->w_zp - (w3_u8 ? 128 : 0);
  if (zms < -128 || zms > 127 || zws3 < -127 || zws3 > 127) return TVX_E_UNSUPPORTED;
  PackPointwise(pr_w, w3_u8, Cout, Cexp, &pk3, &sw3);
  const int out_alloc = nt * 32;
  std::vector<int32_t> b3(out_alloc, 0);
  const int32_t* pb = static_cast<const int32_t*>(pr_b);
  for (int c = 0; c < Cout; ++c) {
    const int64_t v = (pb ? pb[c] : 0) - static_cast<int64_t>(zms) * sw3[c] + static_cast<int64_t>(Cexp) * zms * zws3;
    b3[c] = static_cast<int32_t>(static_cast<uint32_t>(v));
  }
  const int f3 = BuildRequantRecords(op->h_mult, op->h_shift, Cout, out_alloc, pr->out_zp, &rq3, AccumulatorBound(Cexp, pr_b, Cout));
  if (f3 == kRqGeneric) return TVX_E_UNSUPPORTED;
  a.zp3 = zws3 != 0;
  a.neg_zws3_4 = static_cast<int>(static_cast<uint32_t>((-zws3) & 0xff) * 0x01010101u);
  a.out_zp = pr->out_zp; a.lo = op->act_lo; a.hi = op->act_hi; a.ties3 = f3 == kRqFast;
  if (op->fused_add) {
    const tvx_eltwise_desc& el = op->elt;
    const double ra = static_cast<double>(el.a_scale) / static_cast<double>(el.out_scale);
    const double rb = static_cast<double>(el.b_scale) / static_cast<double>(el.out_scale);
    if (!(ra < 1048576.0) || !(rb < 1048576.0)) return TVX_E_UNSUPPORTED;
    a.add_signed = pr->out_dtype == TVX_I8;
    a.add_ra = ra; a.add_rb = rb;
    a.add_za = el.a_zp; a.add_zb = el.b_zp; a.add_zo = el.out_zp;
    ActRange(pr->out_dtype, el.out_scale, el.out_zp, TVX_ACT_NONE, &a.add_lo, &a.add_hi);
  }
  if (S == 1) {
    // codes in the signed domain, records for the packed requantization
    const int e_flip = e_u8 ? 128 : 0, m_flip = m_u8 ? 128 : 0, out_flip = pr->out_dtype == TVX_U8 ? 128 : 0;
    int up[3];
    bool ties[3];
    const auto capped = [](int64_t bound) { return std::min<int64_t>(bound, INT32_MAX); };
    if (!BuildTieRecords(*ex.mult, *ex.shift, Cexp, exp_alloc, e->out_zp - e_flip, capped(AccumulatorBound(Cin, ex.b, Cexp)), &rq1, &up[0], &ties[0]) ||
        !BuildTieRecords(*dw.mult, *dw.shift, Cexp, exp_alloc, d->out_zp - m_flip, capped(AccumulatorBound(9, dw.b, Cexp)), &rq2, &up[1], &ties[1]) ||
        !BuildTieRecords(op->h_mult, op->h_shift, Cout, out_alloc, pr->out_zp - out_flip, capped(AccumulatorBound(Cexp, pr_b, Cout)), &rq3, &up[2], &ties[2]))
      return TVX_E_UNSUPPORTED;
    a.pre1 = up[0] * 2 + ties[0]; a.pre2 = up[1] * 2 + ties[1]; a.pre3 = up[2] * 2 + ties[2];
    a.e_lo -= e_flip; a.e_hi -= e_flip;
    a.m_lo -= m_flip; a.m_hi -= m_flip;
    a.lo -= out_flip; a.hi -= out_flip;
    const auto narrow = [](int lo, int hi) { return lo > -128 || hi < 127; };
    a.out_xor4 = out_flip ? static_cast<int>(0x80808080u) : 0;
    a.dw_nzws3 = (-zwd & 0xff) * 0x010101;
    const bool plain = !(a.pre1 | a.pre2 | a.pre3 | narrow(a.e_lo, a.e_hi) | narrow(a.m_lo, a.m_hi) | narrow(a.lo, a.hi)) && !(a.dw_box && zwd == -128);
    const int widest = std::max(cin_steps, nt);
    plan.tile_fn = wide ? TileKernelOf<true>(widest, a.add_mode, plain) : TileKernelOf<false>(widest, a.add_mode, plain);
  } else {
    plan.fn = a.add_mode ? KernelOf<true>(W, nt) : KernelOf<false>(W, nt);
  }

  // ---- one device image: [w1 | w2 | b1 | q1 | dwk | q2 | b3 | q3], every part 16-byte aligned ----
  std::vector<uint8_t> blob;
  auto append = [&](const void* p, size_t n) {
    const size_t at = blob.size();
    blob.resize(at + (n + 15) / 16 * 16, 0);
    std::memcpy(blob.data() + at, p, n);
    return at;
  };
  // the projection's fragments are read [output tile][chunk]: PackPointwise's order
  const size_t o_w1 = append(pk1.data(), pk1.size()), o_w2 = append(pk3.data(), pk3.size());
  const size_t o_b1 = append(b1.data(), b1.size() * 4), o_q1 = append(rq1.data(), rq1.size() * 4);
  const size_t o_dk = append(dwk.data(), dwk.size() * 4), o_q2 = append(rq2.data(), rq2.size() * 4);
  const size_t o_b3 = append(b3.data(), b3.size() * 4), o_q3 = append(rq3.data(), rq3.size() * 4);
  int s = op->packed.Upload(blob.data(), blob.size());
  if (s != TVX_OK) return s;
  const uint8_t* base = op->packed.as<uint8_t>();
  a.w1 = reinterpret_cast<const v4i*>(base + o_w1);
  a.w2 = reinterpret_cast<const v4i*>(base + o_w2);
  a.b1 = reinterpret_cast<const int32_t*>(base + o_b1);
  a.q1 = reinterpret_cast<const v4i*>(base + o_q1);
  a.dwk = reinterpret_cast<const v4i*>(base + o_dk);
  a.q2 = reinterpret_cast<const v4i*>(base + o_q2);
  a.b3 = reinterpret_cast<const int32_t*>(base + o_b3);
  a.q3 = reinterpret_cast<const v4i*>(base + o_q3);

  const hipError_t err = hipFuncSetAttribute(plan.tile_fn ? reinterpret_cast<const void*>(plan.tile_fn) : reinterpret_cast<const void*>(plan.fn),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, plan.lds_bytes);
  if (err != hipSuccess) return SetError(TVX_E_DEVICE, "hipFuncSetAttribute(dynamic LDS %d): %s", plan.lds_bytes, hipGetErrorString(err));
  op->host_blob.resize(sizeof(Plan));
  std::memcpy(op->host_blob.data(), &plan, sizeof(Plan));
  op->run = MbConvRun;
  op->kernel_name = op->fused_add ? "pwconv_dwconv3x3_pwconv_add_i8" : "pwconv_dwconv3x3_pwconv_i8";
  return TVX_OK;
}

}  // namespace tvx
