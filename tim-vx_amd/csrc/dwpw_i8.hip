// Depthwise 3x3 convolution and the pointwise (1x1) convolution it only feeds, as one kernel: the tensor
// between them - in a MobileNet block the widest of the block - never leaves the CU. In the reference the
// two are separate vxConvolutionLayer nodes that the closed driver merges when it verifies the graph
// (src/tim/vx/internal/src/vsi_nn_graph.c:1591-1603); here the runtime asks for the merged operator when
// the depthwise result has no other reader. Bit for bit the two operators one after the other: the
// depthwise result is requantized to its own tensor's scale and zero point (and clamped by its fused
// ReLU / ReLU6) before the pointwise convolution reads it.
//
// A workgroup owns RPT whole output rows of one image for every channel:
//   1. depthwise phase - a thread holds four columns x RPT rows of four channel planes. A row behind four outputs is loaded as it
//      lies, from the column in front of them on; windows are cut with v_alignbyte and multiplied with v_dot4. Four requantized
//      dwords (four pixels of a channel each) are transposed in registers and go straight to the operand tile of the matrix cores,
//      [pixel slot][channel]; no copy of the tensor in its own order, one barrier;
//   2. pointwise phase - a wavefront takes 32 pixels x 32 output channels at a time. A tile's pixels are permuted: pixel 4 i + e lies in
//      slot 8 e + i. The depthwise stores of neighbouring lanes then spread over four times the banks, and a lane finds the sixteen
//      consecutive pixels of a channel in its accumulators: results are stored from there, sixteen bytes a lane. The zero-point term of
//      uint8 weights is a second MFMA against a constant fragment; a residual Add behind the pointwise convolution rides on the
//      results. A last channel tile of at most 16 takes two pixel tiles at once: the second one's weights stand in the
//      columns that hold no channel, so that no lane requantizes nothing.
// Bound by the vector ALU in large batches (about 15 instructions a depthwise result, 11 a pointwise one) and by the chain load -
// windows - barrier - MFMA - store in small ones. uint8, before (codes staged in the tensor's order, the operand tile built from them
// behind a second barrier, results staged per wavefront) and now, microseconds: 112 x 112, 32 to 16: batch 1 5.0 / 4.6, batch 64 32.9 / 24.6;
// 56 x 56, 144 to 24: 8.1 / 6.9, 36.1 / 30.3; 28 x 28, 144 to 32, stride 2: 9.2 / 5.0, 15.2 / 13.5; 28 x 28, 192 to 32: 9.3 / 6.4, 15.6 / 14.6;
// int8 112 x 112, 32 to 64, batch 32: 22.5 / 20.0. (Two pixel tiles at once: 25.7 -> 24.6 in the first of these.)
#include <algorithm>
#include <cstdlib>

#include "variants.h"

namespace tvx {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

constexpr int kWaves = 4, kMaxWaves = 8;  // of a workgroup: many tiles, few tiles
constexpr int kMaxSlots = 512;            // most pixels of a tile
constexpr int kWeightBytes = 64 * 1024;   // most weights that are copied to LDS

struct DwPwArgs {
  const uint8_t* x;      // depthwise input {W, H, C, N}
  // ---- depthwise part
  const v4i* dw;         // per channel: {three rows of taps, folded bias}, {multiplier, shift and tie bit, rounding constant, -}
  int C, H, W, OW, batch;
  int pad_t, ow4, lpr_shift, quads;  // quads: channels in fours
  int tiles_per_image;
  uint32_t m_tiles;      // reciprocal
  int dw_xor_mask, dw_pad_fill;
  int dw_nzws3, dw_rest3;  // minus the weights' zero point where they are packed unshifted (the window sum carries it), else 0, in three bytes; of 128 a half each
  int dw_pre_ties, dw_lo, dw_hi;
  // ---- pointwise part
  const v4i* wpk;        // [32-channel tile][step][64 lanes]
  const int32_t* biasf;
  const v4i* rq;
  int cp, ksteps, pix_stride, oc_tiles, ptiles;
  int paired;            // the last 32-channel tile holds at most 16 channels: it takes two pixel tiles at a time
  int off_w, off_rq, off_bias;  // LDS behind the operand tile
  int neg_zws4, zp, last_channels;  // last_channels: of the last reduction step
  int P;                 // pixels of a tile: RPT * OW
  uint8_t* y;            // pointwise output {OW, OH, OC, N}
  int OC, hw;
  int pre_ties, lo, hi, out_xor;
  // ---- fused residual Add behind the pointwise convolution (0 = off), as in pwconv_i8
  const uint8_t* res;
  double add_ra, add_rb;
  int add_mode, add_signed;
  int add_za, add_zb, add_zo, add_lo, add_hi;
};

// FLAVOUR: window sums, clamps narrower than a byte, what BuildTieRecords asks for (and such clamps), window sums times 128
constexpr int kBox = 1, kClamp = 2, kTies = 4, kTwice = 8;

// N x 4 accumulators of one channel -> codes, four to a dword; `pre_ties`, the records and the clamp (signed domain) as RequantCodes4 takes
// them. Ties are looked for in all of them at once: with a branch for each four, and one around the clamp, 112 x 112 x 32 -> 64 under a
// narrow ReLU6 took 38 us against 18 without one.
template <int FLAVOUR, int N, class Emit>
__device__ __forceinline__ void Codes(int (&v)[N][4], const v4i& q, int pre_ties, int lo, int hi, Emit emit) {
  const int sh = q[1] & 31;
  const int64_t round = RoundHigh(q[2]);
  if (FLAVOUR & kTies) {
#pragma unroll
    for (int o = 0; o < N; ++o)
#pragma unroll
      for (int i = 0; i < 4; ++i) v[o][i] <<= pre_ties >> 1;
    if (pre_ties & 1) LowerOddTies(reinterpret_cast<int (&)[4 * N]>(v), q);  // (uniform)
  }
  const int lo_t = lo << sh, hi_t = ((hi + 1) << sh) - 1;
#pragma unroll
  for (int o = 0; o < N; ++o) emit(o, RequantSaturate4<(FLAVOUR & (kClamp | kTies)) != 0>(v[o], q[0], sh, round, lo_t, hi_t));
}

// S: stride of the depthwise convolution (left padding 1 at stride 1, 0 at stride 2: SAME); RPT: output rows of a tile;
// WLDS: the pointwise weights are copied to LDS; FLAVOUR: above.
template <int S, int RPT, bool ADD, bool WLDS, int FLAVOUR>
__global__ void __launch_bounds__(kMaxWaves * 64) __attribute__((amdgpu_waves_per_eu(4))) DwPwKernel(DwPwArgs a) {
  extern __shared__ __attribute__((aligned(16))) int8_t lds[];
  constexpr int kRows = S * (RPT - 1) + 3;  // input rows behind a thread's output rows; its dwords of each: S
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), threads = blockDim.x, waves = threads >> 6;
  // an XCD gets a contiguous run of tiles: vertically neighbouring tiles share input rows in its L2
  int wg = blockIdx.x;
  {
    const int per = gridDim.x >> 3, rem = gridDim.x & 7, xcd = wg & 7;
    wg = xcd * per + min(xcd, rem) + (wg >> 3);
  }
  const uint32_t one = a.m_tiles ? 0u : ~0u;
  const int n = static_cast<int>(__umulhi(static_cast<uint32_t>(wg), a.m_tiles) + (static_cast<uint32_t>(wg) & one));
  const int g = wg - n * a.tiles_per_image;
  const int oh0 = g * RPT, ih0 = oh0 * S - a.pad_t;

  // ---- the pointwise weights and the epilogue's tables: global -> LDS by DMA, under the depthwise phase ----
  {
    typedef const __attribute__((address_space(1))) void* gptr;
    typedef __attribute__((address_space(3))) void* lptr;
    const int oc_alloc = a.oc_tiles * 32, chunks = oc_alloc * a.cp >> 4;
    if (WLDS)
      for (int i = wave * 64; i < chunks; i += threads)
        if (i + lane < chunks) __builtin_amdgcn_global_load_lds((gptr)(a.wpk + i + lane), (lptr)(lds + a.off_w + i * 16), 16, 0, 0);
    for (int i = wave * 64; i < oc_alloc; i += threads)
      if (i + lane < oc_alloc) {
        __builtin_amdgcn_global_load_lds((gptr)(a.rq + i + lane), (lptr)(lds + a.off_rq + i * 16), 16, 0, 0);
        __builtin_amdgcn_global_load_lds((gptr)(a.biasf + i + lane), (lptr)(lds + a.off_bias + i * 4), 4, 0, 0);
      }
  }

  // ---- 1. depthwise: (four channels, four columns) per thread and pass, RPT rows. A row behind four outputs is the bytes from the
  // column in front of them on (stride 1: eight; stride 2 needs none in front: twelve), loaded as they lie: what is no column of the row is
  // masked. (x & keep) ^ flip is that and the move to the signed domain in one instruction. ----
  {
    constexpr int kDw = S + 1;
    const int w4 = tid & ((1 << a.lpr_shift) - 1);
    const uint32_t plane = static_cast<uint32_t>(a.H) * static_cast<uint32_t>(a.W);
    const uint8_t* xn = a.x + static_cast<size_t>(n) * a.C * plane - 4;  // (offsets inside an image fit 32 bits)
    const uint32_t image = static_cast<uint32_t>(a.C) * plane;
    const int col = 4 * S * min(w4, a.ow4 - 1) - (S == 1 ? 1 : 0);
    int keep[kDw], flip[kDw];
#pragma unroll
    for (int i = 0; i < kDw; ++i) {
      uint32_t k = ~0u;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (static_cast<unsigned>(col + 4 * i + e) >= static_cast<unsigned>(a.W)) k &= ~(0xffu << (8 * e));
      keep[i] = static_cast<int>(k);
      flip[i] = (a.dw_xor_mask & keep[i]) | (a.dw_pad_fill & ~keep[i]);
    }
    // a run that would leave the tensor, at its first and its last bytes, is read from inside it
    const uint32_t lowest = n == 0 ? 4u : 0u, highest = n == a.batch - 1 ? image + 4u - 4u * kDw : ~0u;
    for (int c4 = tid >> a.lpr_shift; c4 < a.quads; c4 += threads >> a.lpr_shift) {
      int raw[4][kRows][kDw];
      int moved = 0;
      v4i taps[4], q[4];
#pragma unroll
      for (int r = 0; r < kRows; ++r) {
        const int ih = ih0 + r;
        if (ih >= 0 && ih < a.H) {  // (uniform)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const uint32_t at = static_cast<uint32_t>(min(4 * c4 + j, a.C - 1)) * plane + static_cast<uint32_t>(ih) * static_cast<uint32_t>(a.W) + static_cast<uint32_t>(col + 4);
            const uint32_t in = min(max(at, lowest), highest);
            moved |= static_cast<int>(in - at);
            __builtin_memcpy(raw[j][r], xn + in, 4 * kDw);
          }
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int i = 0; i < kDw; ++i) raw[j][r][i] = a.dw_pad_fill ^ a.dw_xor_mask;
        }
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int c = min(4 * c4 + j, a.C - 1);
        taps[j] = a.dw[2 * c];
        q[j] = a.dw[2 * c + 1];
      }
      if (__ballot(moved)) {  // (the first and the last workgroup)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int r = 0; r < kRows; ++r) {
            const int ih = ih0 + r;
            if (ih < 0 || ih >= a.H) continue;
            const uint32_t at = static_cast<uint32_t>(min(4 * c4 + j, a.C - 1)) * plane + static_cast<uint32_t>(ih) * static_cast<uint32_t>(a.W) + static_cast<uint32_t>(col + 4);
            const int by = static_cast<int>(min(max(at, lowest), highest) - at);
            if constexpr (S == 1) {  // one byte up or three down
              const uint64_t v = static_cast<uint64_t>(static_cast<uint32_t>(raw[j][r][1])) << 32 | static_cast<uint32_t>(raw[j][r][0]);
              const uint64_t w = by > 0 ? v << 8 : by < 0 ? v >> 24 : v;
              raw[j][r][0] = static_cast<int>(w);
              raw[j][r][1] = static_cast<int>(w >> 32);
            } else {  // a dword down
              const int down = by ? ~0 : 0;
              raw[j][r][0] = (raw[j][r][1] & down) | (raw[j][r][0] & ~down);
              raw[j][r][1] = (raw[j][r][2] & down) | (raw[j][r][1] & ~down);
            }
          }
      }
      uint32_t codes[RPT][4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        int acc[RPT][4];
#pragma unroll
        for (int r = 0; r < kRows; ++r) {
          int d[kDw + 1];
          d[kDw] = 0;
#pragma unroll
          for (int i = 0; i < kDw; ++i) d[i] = S == 2 && i < 2 ? raw[j][r][i] ^ a.dw_xor_mask : (raw[j][r][i] & keep[i]) ^ flip[i];
          // (at stride 1 a window dword serves two outputs, the second by taps a byte further up)
          int win[4];
          win[0] = Window<0>(d);
          win[1] = S == 1 ? win[0] : Window<S>(d);
          win[2] = Window<2 * S>(d);
          win[3] = S == 1 ? win[2] : Window<3 * S>(d);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
#pragma unroll
            for (int o = 0; o < RPT; ++o) {
              const int ky = r - S * o;
              if (ky < 0 || ky > 2) continue;
              const int up = S == 1 ? i % 2 * 8 : 0;
              acc[o][i] = __builtin_amdgcn_sdot4(win[i], taps[j][ky] << up, ky == 0 ? taps[j][3] : acc[o][i], false);
              if (FLAVOUR & kBox) acc[o][i] = __builtin_amdgcn_sdot4(win[i], a.dw_nzws3 << up, acc[o][i], false);
              if (FLAVOUR & kTwice) acc[o][i] = __builtin_amdgcn_sdot4(win[i], a.dw_rest3 << up, acc[o][i], false);
            }
          }
        }
        Codes<FLAVOUR>(acc, q[j], a.dw_pre_ties, a.dw_lo, a.dw_hi, [&](int o, uint32_t c) { codes[o][j] = c; });
      }
      if (w4 < a.ow4) {
#pragma unroll
        for (int o = 0; o < RPT; ++o) {
          uint32_t t[4];
          Transpose4x4(codes[o], t);
          const int p4 = o * a.ow4 + w4;
          int8_t* to = lds + __mul24((p4 >> 3) * 32 + (p4 & 7), a.pix_stride) + 4 * c4;
#pragma unroll
          for (int e = 0; e < 4; ++e) *reinterpret_cast<uint32_t*>(to + 8 * e * a.pix_stride) = t[e];
        }
      }
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (the DMA above)
  __syncthreads();

  // ---- 2. pointwise: a wavefront takes 32 pixel slots x 32 output channels at a time ----
  const DwPwArgs& b = LateArgs<DwPwArgs>();
  const int row = lane & 31, half = lane >> 5;
  const v4i fz = {b.neg_zws4, b.neg_zws4, b.neg_zws4, b.neg_zws4};
  v4i fz_last;  // (what lies behind the channels in their last step counts for no sum)
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int left = b.last_channels - 16 * half - 4 * i;
    fz_last[i] = left >= 4 ? fz[i] : left <= 0 ? 0 : fz[i] & static_cast<int>((1u << (8 * left)) - 1u);
  }
  int ot = 0, pair = b.oc_tiles == 1 ? b.paired : 0, tasks = b.ptiles;
  if (pair) tasks = (b.ptiles + 1) >> 1;
  for (int task = wave; ; task += waves) {
    while (task >= tasks) {
      task -= tasks;
      if (++ot == b.oc_tiles - 1 && b.paired) { pair = 1; tasks = (b.ptiles + 1) >> 1; }
    }
    if (ot >= b.oc_tiles) break;
    const int pt = task << pair, second = pair ? row & 16 : 0;
    const int oc = ot * 32 + row - second, p0 = (pt + (second >> 4)) * 32 + 16 * half;
    const bool live = oc < b.OC && p0 < b.P, whole = p0 + 16 <= b.P;
    const size_t at = (static_cast<size_t>(n) * b.OC + oc) * b.hw + static_cast<size_t>(g) * b.P + p0;
    uint32_t res[4] = {0, 0, 0, 0};
    if (ADD && live) {
      if (whole) __builtin_memcpy(res, b.res + at, 16);
      else
#pragma unroll
        for (int e = 0; e < 3; ++e)
          if (p0 + 4 * e < b.P) __builtin_memcpy(&res[e], b.res + at + 4 * e, 4);
    }
    const v4i q = *reinterpret_cast<const v4i*>(lds + b.off_rq + oc * 16);
    const int bias = *reinterpret_cast<const int*>(lds + b.off_bias + oc * 4);
    v16i acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = bias;
    const int8_t* xa = lds + (pt * 32 + row) * b.pix_stride + half * 16;
    const int8_t* wl = lds + b.off_w + (ot * b.ksteps * 64 + lane) * 16;
    const v4i* wg4 = b.wpk + static_cast<size_t>(ot) * b.ksteps * 64 + lane;
    auto weights = [&](int k) { return WLDS ? *reinterpret_cast<const v4i*>(wl + k * 1024) : wg4[k * 64]; };
    // at most 16 channels: two pixel tiles at once, the second one's results in the columns that hold no channel
    const int8_t* xb = xa + (pt + 1 < b.ptiles ? 32 * b.pix_stride : 0);
    auto weights2 = [&](int k) { return WLDS ? *reinterpret_cast<const v4i*>(wl + k * 1024 + (second ? -256 : 256)) : wg4[k * 64 + (second ? -16 : 16)]; };
    const int upper = second ? ~0 : 0, lower = ~upper;
    v4i fw = weights(0), fx = *reinterpret_cast<const v4i*>(xa);
    for (int k = 0; k < b.ksteps; ++k) {
      const int kn = min(k + 1, b.ksteps - 1);
      const v4i fw1 = weights(kn);
      const v4i fx1 = *reinterpret_cast<const v4i*>(xa + kn * 32);
      acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(fx, fw, acc, 0, 0, 0);
      if (b.zp) acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(fx, (k + 1 < b.ksteps ? fz : fz_last) & lower, acc, 0, 0, 0);
      if (pair) {  // (uniform)
        const v4i fx2 = *reinterpret_cast<const v4i*>(xb + k * 32);
        acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(fx2, weights2(k), acc, 0, 0, 0);
        if (b.zp) acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(fx2, (k + 1 < b.ksteps ? fz : fz_last) & upper, acc, 0, 0, 0);
      }
      fw = fw1; fx = fx1;
    }
    // accumulator 4 e + i is slot 8 e + 4 half + i: pixel 16 half + 4 i + e of the tile
    uint32_t out[4];
    int v[4][4];
#pragma unroll
    for (int r = 0; r < 16; ++r) v[r & 3][r >> 2] = acc[r];
    Codes<FLAVOUR>(v, q, b.pre_ties, b.lo, b.hi, [&](int i, uint32_t c) {
      out[i] = c ^ static_cast<uint32_t>(b.out_xor);
      if (ADD) out[i] = AddResidual4(b, out[i], res[i]);
    });
    if (!live) continue;
    if (whole) __builtin_memcpy(b.y + at, out, 16);
    else
#pragma unroll
      for (int e = 0; e < 3; ++e)
        if (p0 + 4 * e < b.P) __builtin_memcpy(b.y + at + 4 * e, &out[e], 4);
  }
}

struct Plan {
  DwPwArgs a;
  void (*fn)(DwPwArgs);
  int lds_bytes, block;
  dim3 grid;
};

typedef void (*DwPwFn)(DwPwArgs);

template <bool ADD, bool WLDS, int FLAVOUR>
DwPwFn KernelOf(int stride, int rpt) {
  if (stride == 1) return rpt == 4 ? DwPwKernel<1, 4, ADD, WLDS, FLAVOUR> : (rpt == 2 ? DwPwKernel<1, 2, ADD, WLDS, FLAVOUR> : DwPwKernel<1, 1, ADD, WLDS, FLAVOUR>);
  return rpt == 2 ? DwPwKernel<2, 2, ADD, WLDS, FLAVOUR> : DwPwKernel<2, 1, ADD, WLDS, FLAVOUR>;
}
template <bool ADD>
DwPwFn KernelOf(int stride, int rpt, bool wlds, int flavour) {
  if (!wlds) return flavour & kBox ? KernelOf<ADD, false, kBox | kTies | kTwice>(stride, rpt) : KernelOf<ADD, false, kTies>(stride, rpt);
  switch (flavour) {
    case 0: return KernelOf<ADD, true, 0>(stride, rpt);
    case kBox: return KernelOf<ADD, true, kBox>(stride, rpt);
    case kClamp: return KernelOf<ADD, true, kClamp>(stride, rpt);
    case kBox | kClamp: return KernelOf<ADD, true, kBox | kClamp>(stride, rpt);
    case kTies: return KernelOf<ADD, true, kTies>(stride, rpt);
    case kBox | kTies: return KernelOf<ADD, true, kBox | kTies>(stride, rpt);
    default: return KernelOf<ADD, true, kBox | kTies | kTwice>(stride, rpt);
  }
}

int DwPwRun(tvx_op* op, const void* in0, const void* in1, void* out, hipStream_t st) {
  const Plan* plan = reinterpret_cast<const Plan*>(op->host_blob.data());
  DwPwArgs a = plan->a;
  a.x = static_cast<const uint8_t*>(in0);
  a.y = static_cast<uint8_t*>(out);
  a.res = static_cast<const uint8_t*>(in1);
  if (a.add_mode && !in1) return SetError(TVX_E_INVALID, "dwpw_i8: the fused Add needs its second operand as in1");
  if ((reinterpret_cast<uintptr_t>(in0) & 3) | ((reinterpret_cast<uintptr_t>(out) | (a.add_mode ? reinterpret_cast<uintptr_t>(in1) : 0)) & 15))
    return SetError(TVX_E_INVALID, "dwpw_i8: the input must be 4-byte, the output (and the Add's operand) 16-byte aligned");
  hipLaunchKernelGGL(plan->fn, plan->grid, dim3(plan->block), plan->lds_bytes, st, a);
  TVX_HIP_CHECK(hipGetLastError());
  return TVX_OK;
}

int RoundUp(int v, int m) { return (v + m - 1) / m * m; }

}  // namespace

// `op` carries the pointwise convolution (op->conv, requantization tables, clamp, fused Add); `dw` and its
// tables describe the depthwise convolution in front of it. Declines (TVX_E_UNSUPPORTED) what the kernel does
// not cover; the caller then creates the two operators.
int DwPwSetup(tvx_op* op, const tvx_conv2d_desc* dw, const void* dw_w, const void* dw_b,
              const std::vector<int32_t>& dw_mult, const std::vector<int32_t>& dw_shift, int dw_lo, int dw_hi,
              const tvx_conv2d_desc* pw, const void* pw_w, const void* pw_b) {
  if (!dw_w || !pw_w) return TVX_E_UNSUPPORTED;
  // ---- depthwise: 3x3, multiplier 1, SAME at stride 1 or 2, rows of whole dwords ----
  if (dw->multiplier != 1 || dw->k_w != 3 || dw->k_h != 3 || dw->dilation_w != 1 || dw->dilation_h != 1) return TVX_E_UNSUPPORTED;
  if (dw->stride_w != dw->stride_h || (dw->stride_w != 1 && dw->stride_w != 2)) return TVX_E_UNSUPPORTED;
  const int S = dw->stride_w;
  if (dw->pad_left != (S == 1 ? 1u : 0u) || dw->pad_top > 1 || (dw->in_w & 3) || (dw->out_w & 3)) return TVX_E_UNSUPPORTED;
  const int ow4 = dw->out_w / 4, in_dw = dw->in_w / 4;
  int lpr_shift = 0;
  while ((1 << lpr_shift) < ow4 || S * (1 << lpr_shift) < in_dw) ++lpr_shift;
  if (lpr_shift > 6) return TVX_E_UNSUPPORTED;
  if (static_cast<uint32_t>((dw->out_w - 1) * S + 2) >= dw->in_w + dw->pad_left + 4) return TVX_E_UNSUPPORTED;
  // ---- pointwise: 1x1, stride 1, unpadded, on the depthwise result ----
  if (pw->multiplier != 0 || pw->groups > 1 || pw->k_w != 1 || pw->k_h != 1 || pw->stride_w != 1 || pw->stride_h != 1 ||
      pw->pad_left != 0 || pw->pad_top != 0)
    return TVX_E_UNSUPPORTED;
  if (pw->in_w != dw->out_w || pw->in_h != dw->out_h || pw->in_c != dw->out_c || pw->batch != dw->batch ||
      pw->out_w != pw->in_w || pw->out_h != pw->in_h || pw->in_dtype != dw->out_dtype ||
      pw->in_scale != dw->out_scale || pw->in_zp != dw->out_zp)
    return TVX_E_UNSUPPORTED;
  // ---- which pairs: those with whole rows of at most kMaxSlots pixels that make 16-byte chunks, up to this much LDS (larger ones: two
  // kernels) ----
  const int cp_ = RoundUp(static_cast<int>(dw->in_c), 32);
  const int oc_alloc_ = RoundUp(static_cast<int>(pw->out_c), 32);
  int fewest = 0;
  for (int r : {4, 2, 1})
    if (r * dw->out_w <= static_cast<uint32_t>(kMaxSlots) && dw->out_h % r == 0 && (r * dw->out_w) % 16 == 0) fewest = r;
  const int slots_ = RoundUp(fewest * static_cast<int>(dw->out_w), 128);
  if (!fewest || cp_ * (slots_ + 4) + slots_ * (cp_ + 16) + 5120 + oc_alloc_ * (cp_ + 20) > 160 * 1024) return TVX_E_UNSUPPORTED;
  // ---- tile: more rows share more of the loads and the requantization tables, fewer fill more CUs. Microseconds with (rows, wavefronts),
  // uint8, by output rows in the batch per CU:
  //   0.9  28 x 28, 144 to 32, stride 2    (1,8) 5.1, (2,8) 6.4      28 x 28, 192 to 32            (1,8) 6.7, (2,8) 7.3, (4,8) 9.3
  //   1.8  112 x 112, 32 to 16             (1,8) 5.7, (2,8) 5.3      28 x 28, 144 to 32, stride 2  (1,8) 6.0, (2,8) 6.3
  //   3.5  56 x 56, 144 to 24              (1,4) 15.4, (2,8) 12.2, (4,8) 12.3, (2,4) 13.8      28 x 28, 192 to 32  (2,8) 10.5, (4,8) 9.7
  //   7    28 x 28, 192 to 32              (1,4) 18.5, (2,4) 15.0, (4,8) 14.4, (4,4) 16.0
  //   14   56 x 56, 96 to 24, stride 2     (1,4) 27.7, (2,4) 24.4, (2,8) 25.9
  //   28   112 x 112, 32 to 16             (1,4) 36.6, (2,4) 28.8, (4,4) 25.7, (4,8) 29.2
  // Never more than fit LDS: of the pairs taken at all one row always does (int8, batch 8, four rows too many: 128 x 128, 288 to 64 (1,8) 40.6, (2,8)
  // 34.8; 112 x 112, 224 to 256 58.2, 41.0; 128 x 128, 256 to 96 39.1, 36.1. As two kernels these are 28.3, 34.3 and 28.5: callers who need the
  // fused operator get it, callers who have the choice lose by it.) ----
  const int cus = ComputeUnits();
  const uint64_t rows = static_cast<uint64_t>(dw->batch) * dw->out_h, cu = cus;
  const int oc_bytes = oc_alloc_ * cp_;
  const bool wlds = oc_bytes <= kWeightBytes;
  const auto weights_at = [&](int r) { return RoundUp(r * static_cast<int>(dw->out_w), 32) * (cp_ + 16); };  // behind the operand tile
  const auto lds_of = [&](int r) { return weights_at(r) + (wlds ? oc_bytes : 0) + oc_alloc_ * 20; };
  const auto fits = [&](int r) { return dw->out_h % r == 0 && (r < 4 || S == 1) && r * dw->out_w <= static_cast<uint32_t>(kMaxSlots) && lds_of(r) <= 160 * 1024; };
  int rpt = 1;
  for (int r : {2, 4})
    if (rows > (r == 4 ? 3 * cu : S * cu) && fits(r)) rpt = r;
  if (const char* f = getenv("TVX_DWPW_ROWS")) {  // test lever
    const int r = atoi(f);
    if ((r == 1 || r == 2 || r == 4) && fits(r)) rpt = r;
  }
  const uint64_t tiles = static_cast<uint64_t>(dw->batch) * (dw->out_h / rpt);
  if (tiles > 0x7fffffffull || static_cast<uint64_t>(dw->in_h) * dw->in_w * dw->in_c >= (1ull << 32) - 16 || dw->in_h >= (1u << 24)) return TVX_E_UNSUPPORTED;  // (32-bit offsets inside an image)

  DwPwArgs a{};
  const int C = dw->in_c;
  a.C = C; a.H = dw->in_h; a.W = dw->in_w; a.OW = dw->out_w; a.batch = dw->batch;
  a.pad_t = dw->pad_top;
  a.ow4 = ow4; a.lpr_shift = lpr_shift; a.quads = (C + 3) / 4;
  const bool x_u8 = dw->in_dtype == TVX_U8, dww_u8 = dw->w_dtype == TVX_U8;
  const int dzxs = dw->in_zp - (x_u8 ? 128 : 0);
  const int dzws = (dw->w_scales ? 0 : dw->w_zp) - (dww_u8 ? 128 : 0);
  if (dzxs < -128 || dzxs > 127) return TVX_E_UNSUPPORTED;
  std::vector<int32_t> dwpk, dbiasf, drq;
  const bool box = PackDepthwise3x3(C, dw_w, dww_u8, dw_b, dzxs, dzws, true, &dwpk, &dbiasf);
  // (the 32-bit record forms decide which pairs are taken; accumulators are 32 bits, whatever the bias would make of their bound)
  if (BuildRequantRecords(dw_mult, dw_shift, C, C, dw->out_zp, &drq, AccumulatorBound(9, dw_b, C)) == kRqGeneric) return TVX_E_UNSUPPORTED;
  const bool mid_u8 = pw->in_dtype == TVX_U8;
  const int mid_flip = mid_u8 ? 128 : 0;
  int up;
  bool ties;
  if (!BuildTieRecords(dw_mult, dw_shift, C, C, dw->out_zp - mid_flip, std::min<int64_t>(AccumulatorBound(9, dw_b, C), INT32_MAX), &drq, &up, &ties)) return TVX_E_UNSUPPORTED;
  a.dw_pre_ties = up * 2 + ties;
  a.dw_lo = dw_lo - mid_flip; a.dw_hi = dw_hi - mid_flip;
  a.dw_xor_mask = x_u8 ? static_cast<int>(0x80808080u) : 0;
  a.dw_pad_fill = static_cast<int>(static_cast<uint32_t>(dzxs & 0xff) * 0x01010101u);
  const int nzws = box ? -dzws : 0, rest = nzws == 128 ? 64 : 0;
  a.dw_nzws3 = ((nzws - rest) & 0xff) * 0x010101;
  a.dw_rest3 = rest * 0x010101;
  std::vector<int32_t> dw_tab(static_cast<size_t>(C) * 8);
  for (int c = 0; c < C; ++c) {
    for (int i = 0; i < 3; ++i) dw_tab[c * 8 + i] = dwpk[c * 4 + i];
    dw_tab[c * 8 + 3] = dbiasf[c];
    for (int i = 0; i < 4; ++i) dw_tab[c * 8 + 4 + i] = drq[c * 4 + i];
  }

  a.OC = pw->out_c;
  a.hw = static_cast<int>(dw->out_w) * static_cast<int>(dw->out_h);
  a.cp = RoundUp(C, 32);
  a.ksteps = a.cp / 32;
  a.last_channels = C - (a.ksteps - 1) * 32;
  a.pix_stride = a.cp + 16;
  a.oc_tiles = (a.OC + 31) / 32;
  a.paired = a.oc_tiles * 32 - a.OC >= 16;
  a.P = rpt * dw->out_w;
  a.ptiles = (a.P + 31) / 32;
  a.tiles_per_image = dw->out_h / rpt;
  a.m_tiles = a.tiles_per_image > 1 ? static_cast<uint32_t>(((1ull << 32) + a.tiles_per_image - 1) / a.tiles_per_image) : 0u;
  if (tiles * a.tiles_per_image >= (1ull << 32)) return TVX_E_UNSUPPORTED;
  const bool pww_u8 = pw->w_dtype == TVX_U8;
  const int zxs = pw->in_zp - mid_flip;
  const int zws = op->w_zp - (pww_u8 ? 128 : 0);
  if (zxs < -128 || zxs > 127 || zws < -127 || zws > 127) return TVX_E_UNSUPPORTED;
  a.neg_zws4 = static_cast<int>(static_cast<uint32_t>((-zws) & 0xff) * 0x01010101u);
  a.zp = zws != 0;
  const int out_flip = pw->out_dtype == TVX_U8 ? 128 : 0;
  a.lo = op->act_lo - out_flip; a.hi = op->act_hi - out_flip;
  a.out_xor = out_flip ? static_cast<int>(0x80808080u) : 0;
  if (op->fused_add) {
    const tvx_eltwise_desc& e = op->elt;
    const double ra = static_cast<double>(e.a_scale) / static_cast<double>(e.out_scale);
    const double rb = static_cast<double>(e.b_scale) / static_cast<double>(e.out_scale);
    if (!(ra < 1048576.0) || !(rb < 1048576.0)) return TVX_E_UNSUPPORTED;
    a.add_mode = op->fused_add;
    a.add_signed = pw->out_dtype == TVX_I8;
    a.add_ra = ra; a.add_rb = rb;
    a.add_za = e.a_zp; a.add_zb = e.b_zp; a.add_zo = e.out_zp;
    ActRange(pw->out_dtype, e.out_scale, e.out_zp, TVX_ACT_NONE, &a.add_lo, &a.add_hi);
  }
  a.off_w = weights_at(rpt);
  a.off_rq = a.off_w + (wlds ? oc_bytes : 0);
  a.off_bias = a.off_rq + oc_alloc_ * 16;
  const int lds_bytes = lds_of(rpt);
  if (lds_bytes > 160 * 1024) return TVX_E_UNSUPPORTED;
  // (where a CU holds one workgroup, eight: 80 x 80, 352 to 128, batch 16 63.7 us, 95.4 with four)
  int waves = tiles <= 2ull * cus || lds_bytes > 80 * 1024 || (rpt == 4 && (a.quads << lpr_shift) > 64 * kWaves) ? kMaxWaves : kWaves;
  // stride 2, a depthwise pass of at most 128 threads: half of four wavefronts would only wait for the other half (batch 64: 112 x 112, 32 to 16
  // 11.6 -> 9.9 us, 16 to 32 10.7 -> 8.9, 56 x 56, 32 to 64 6.3 -> 6.2; at stride 1 four are ahead: 28 x 28, 32 to 64 6.4 against 7.7)
  if (S == 2 && tiles > 2ull * cus && (a.quads << lpr_shift) <= 128) waves = 2;
  if (!LaunchFits(tiles, 64 * waves)) waves = kWaves;
  if (const char* f = getenv("TVX_DWPW_WAVES")) waves = std::max(1, std::min(atoi(f), kMaxWaves));  // test lever
  // pointwise weights in fragment order, constants folded into the bias (as PwConvSetup packs them)
  const int oc_alloc = a.oc_tiles * 32;
  std::vector<int8_t> packed(static_cast<size_t>(a.oc_tiles) * a.ksteps * 1024, 0);
  std::vector<int32_t> biasf(oc_alloc, 0);
  const uint8_t* src = static_cast<const uint8_t*>(pw_w);
  const int32_t* b = static_cast<const int32_t*>(pw_b);
  for (int oc = 0; oc < a.OC; ++oc) {
    int64_t sw = 0;
    for (int c = 0; c < C; ++c) {
      const uint8_t raw = src[static_cast<size_t>(oc) * C + c];
      const int8_t v = static_cast<int8_t>(pww_u8 ? raw ^ 0x80 : raw);
      const int ks = c / 32, half = (c % 32) / 16, j = c % 16;
      packed[((static_cast<size_t>(oc / 32) * a.ksteps + ks) * 64 + half * 32 + oc % 32) * 16 + j] = v;
      sw += v;
    }
    const int64_t v = (b ? b[oc] : 0) - static_cast<int64_t>(zxs) * sw + static_cast<int64_t>(C) * zxs * zws;
    biasf[oc] = static_cast<int32_t>(static_cast<uint32_t>(v));
  }
  std::vector<int32_t> rqt;
  const int64_t bound = AccumulatorBound(C, pw_b, a.OC);
  if (BuildRequantRecords(op->h_mult, op->h_shift, a.OC, oc_alloc, pw->out_zp, &rqt, bound) == kRqGeneric) return TVX_E_UNSUPPORTED;
  if (!BuildTieRecords(op->h_mult, op->h_shift, a.OC, oc_alloc, pw->out_zp - out_flip, std::min<int64_t>(bound, INT32_MAX), &rqt, &up, &ties)) return TVX_E_UNSUPPORTED;
  a.pre_ties = up * 2 + ties;
  int s = op->packed.Upload(packed.data(), packed.size());
  if (s == TVX_OK) s = op->aux.Upload(biasf.data(), biasf.size() * 4);
  if (s == TVX_OK) s = op->aux2.Upload(rqt.data(), rqt.size() * 4);
  if (s == TVX_OK) s = op->aux3.Upload(dw_tab.data(), dw_tab.size() * 4);
  if (s != TVX_OK) return s;
  a.wpk = op->packed.as<v4i>();
  a.biasf = op->aux.as<int32_t>();
  a.rq = op->aux2.as<v4i>();
  a.dw = op->aux3.as<v4i>();
  Plan plan{};
  plan.a = a;
  const bool clamp = std::max(a.dw_lo, a.lo) > -128 || std::min(a.dw_hi, a.hi) < 127;
  const int flavour = a.dw_rest3 ? kBox | kTies | kTwice : (a.dw_nzws3 ? kBox : 0) | (a.dw_pre_ties || a.pre_ties ? kTies : clamp ? kClamp : 0);
  plan.fn = a.add_mode ? KernelOf<true>(S, rpt, wlds, flavour) : KernelOf<false>(S, rpt, wlds, flavour);
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(plan.fn), hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
  if (e != hipSuccess) return SetError(TVX_E_DEVICE, "hipFuncSetAttribute(dynamic LDS %d): %s", lds_bytes, hipGetErrorString(e));
  plan.lds_bytes = lds_bytes;
  plan.block = 64 * waves;
  plan.grid = dim3(static_cast<unsigned>(tiles));
  op->host_blob.assign(reinterpret_cast<const uint8_t*>(&plan), reinterpret_cast<const uint8_t*>(&plan) + sizeof(plan));
  op->run = DwPwRun;
  op->kernel_name = op->fused_add ? "dwconv3x3_pwconv_add_i8" : "dwconv3x3_pwconv_i8";
  return TVX_OK;
}

}  // namespace tvx
