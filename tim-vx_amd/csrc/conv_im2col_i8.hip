// Quantized Conv2d with a short reduction (C * Kh * Kw <= 64) on the int8 matrix cores: the first
// layers of image networks (3 x 3 x 3 = 27, 1 x 5 x 5 = 25). The implicit-GEMM kernel pads the
// channels of every tap to 16 and would multiply mostly zeros there; here the whole window of an
// output pixel - its (c, ky, kx) bytes, padded to 32 or 64 - is one row of the MFMA A operand.
//
// Windows three or five taps wide are gathered into registers (ConvIm2colRegKernel, below), any others through LDS: a
// workgroup = 256 output pixels of one image x all output channels (<= 128). Each thread
// gathers the window of one pixel with byte loads (16 in flight, no branches: out-of-image taps
// read a safe address and are replaced by the input zero point), keeps the window sum for the
// zero-point expansion
//   sum (x - zx)(w - zw) = sum xs ws - zws * Sx - zxs * Sw + K zxs zws
// and stores the row to LDS. One or two v_mfma_i32_32x32x32_i8 steps per (pixel tile, channel
// tile) follow; the epilogue is the implicit-GEMM kernel's: requantize, pack four pixels per
// dword, stage [oc][pixel] in LDS, copy out as contiguous runs of the WHCN output.
#include <algorithm>
#include <type_traits>

#include "variants.h"

namespace tvx {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

constexpr int kThreads = 256;
constexpr int kPixels = 256;  // per workgroup: eight 32-pixel MFMA tiles, two per wavefront

struct ImArgs {
  const uint8_t* x;
  const int8_t* w;       // packed [oct][row_stride] (the LDS image), reduction order (c, ky, kx), zero padded
  uint8_t* y;
  const int32_t* biasf;  // bias + per-channel zero-point terms
  const v4i* rq;         // per channel {mult, shift | t, half, lowmask}
  int C, H, W, OC, OH, OW;
  int sh, sw, pad_t, pad_l;
  int kp;                // reduction length padded to 32 or 64
  int row_stride;        // bytes per LDS row of A and of the weights: kp + 16 (an odd number of 16-byte chunks)
  int oct;               // output channels padded to 32
  int xor_mask;          // 0x80 for uint8 activations, else 0
  int pad_fill;          // input zero point in the int8 domain (one byte)
  int zws, out_zp, lo, hi;
  int out_stride;        // epilogue staging row stride in bytes (odd number of dwords)
  int off_a, off_w, off_sx, off_rq, off_bias;  // LDS carve-up
  // The window, per reduction index: dy | dx << 8 | 1 << 16 (zero past the end) and the input offset
  // c * H * W + dy * W + dx. They travel in the kernel arguments so that the (wavefront-uniform) reads
  // are scalar loads of memory nothing can write; a table in global memory is read per lane, one round
  // trip a tap.
  int taps[64];
  int offs[64];
  int pool;              // 1: a 2 x 2 / stride-2 max pooling rides on the epilogue (the result has OH / 2 x OW / 2 pixels)
};

// any window, one byte load per tap
// (two wavefronts per SIMD at least: within 256 registers the compiler keeps MFMA accumulators in ordinary vector
// registers, where the epilogue reads them, instead of moving every value out of the accumulation registers first)
template <int OT, int RQ>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2))) ConvIm2colKernel(ImArgs a) {
  extern __shared__ __attribute__((aligned(16))) int8_t lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int n = blockIdx.y;
  const int hw = a.OH * a.OW;
  const int p0 = blockIdx.x * kPixels;
  const int valid = min(kPixels, hw - p0);

  int8_t* a_lds = lds + a.off_a;
  int8_t* w_lds = lds + a.off_w;
  int* sx_lds = reinterpret_cast<int*>(lds + a.off_sx);
  v4i* rq_lds = reinterpret_cast<v4i*>(lds + a.off_rq);
  int* bias_lds = reinterpret_cast<int*>(lds + a.off_bias);

  // weights (already laid out as their LDS image) and the epilogue's tables: global -> LDS by DMA,
  // waited for together with the window loads
  {
    typedef const __attribute__((address_space(1))) void* gptr;
    typedef __attribute__((address_space(3))) void* lptr;
    const int chunks = a.oct * a.row_stride >> 4;
    for (int i = wave * 64; i < chunks; i += kThreads)
      if (i + lane < chunks)
        __builtin_amdgcn_global_load_lds((gptr)(a.w + static_cast<size_t>(i + lane) * 16), (lptr)(w_lds + i * 16), 16, 0, 0);
    for (int i = wave * 64; i < a.oct; i += kThreads)
      if (i + lane < a.oct) {
        __builtin_amdgcn_global_load_lds((gptr)(a.rq + i + lane), (lptr)(rq_lds + i), 16, 0, 0);
        __builtin_amdgcn_global_load_lds((gptr)(a.biasf + i + lane), (lptr)(bias_lds + i), 4, 0, 0);
      }
  }

  // ---- the window of this thread's pixel ------------------------------------------------
  int sx = 0;
  {
    const int p = min(p0 + tid, hw - 1);  // threads past the end redo the last pixel; nobody reads their row
    int oh = p / a.OW, ow = p - oh * a.OW;
    if (a.pool) {
      // pixels in pooling order: four consecutive ones are a 2 x 2 window (row-major), windows row-major over
      // the pooled image - the four accumulators a lane holds per quad then are one pooled pixel's candidates
      const int q = p >> 2, e = p & 3, pw = a.OW >> 1;
      const int qh = q / pw, qw = q - qh * pw;
      oh = 2 * qh + (e >> 1);
      ow = 2 * qw + (e & 1);
    }
    const int ih0 = oh * a.sh - a.pad_t, iw0 = ow * a.sw - a.pad_l;
    const uint8_t* img = a.x + static_cast<size_t>(n) * a.C * a.H * a.W;
    const int origin = ih0 * a.W + iw0;  // may be negative; only added to offsets of taps inside the image
    // Which window rows / columns (offsets 0..31 from the window's origin) lie inside the image, as bit
    // masks: a tap's validity is then two shifts and an AND instead of two additions and two compares.
    auto span_mask = [](int first, int extent) {  // bits d with 0 <= first + d < extent, d in 0..31
      const int lo = max(0, -first), hi = min(32, extent - first);
      const int n = hi - lo;
      return n <= 0 ? 0u : ((n >= 32 ? 0xffffffffu : ((1u << n) - 1u)) << lo);
    };
    const uint32_t row_ok = span_mask(ih0, a.H), col_ok = span_mask(iw0, a.W);
    for (int k0 = 0; k0 < a.kp; k0 += 16) {
      int b[16];
      bool inside[16];
      int fill[16];
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const int t = a.taps[k0 + j];  // scalar: dy | dx << 8 | real << 16
        const int dy = t & 0xff, dx = (t >> 8) & 0xff;
        const uint32_t real = 0u - static_cast<uint32_t>(t >> 16);  // all ones or zero
        fill[j] = a.pad_fill & static_cast<int>(real);
        // bitwise, not short-circuit: no branch may stand between the loads
        inside[j] = ((row_ok >> dy) & (col_ok >> dx) & real & 1u) != 0;
        b[j] = img[static_cast<uint32_t>(inside[j] ? origin + a.offs[k0 + j] : 0)];  // uniform base + 32-bit lane offset
      }
      __builtin_amdgcn_sched_barrier(0);  // all sixteen loads travel together
      int dw[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        int v = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int j = q * 4 + e;
          const int byte = inside[j] ? (b[j] ^ a.xor_mask) : fill[j];  // both below 256
          v |= byte << (8 * e);
        }
        dw[q] = v;
        sx = __builtin_amdgcn_sdot4(v, 0x01010101, sx, false);
      }
      *reinterpret_cast<v4i*>(a_lds + tid * a.row_stride + k0) = v4i{dw[0], dw[1], dw[2], dw[3]};
    }
  }
  sx_lds[tid] = a.zws * sx;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the table DMA has landed
  __syncthreads();

  // ---- MFMA: wave w owns pixel tiles w and w + 4, all channel tiles ---------------------------
  const int frag_row = lane & 31, frag_half = lane >> 5;
  v16i acc[2][OT];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < OT; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0;
  for (int ks = 0; ks < a.kp; ks += 32) {
    v4i fa[2], fb[OT];
#pragma unroll
    for (int i = 0; i < 2; ++i)
      fa[i] = *reinterpret_cast<const v4i*>(a_lds + ((wave + 4 * i) * 32 + frag_row) * a.row_stride + ks + frag_half * 16);
#pragma unroll
    for (int j = 0; j < OT; ++j)
      fb[j] = *reinterpret_cast<const v4i*>(w_lds + (j * 32 + frag_row) * a.row_stride + ks + frag_half * 16);
#pragma unroll
    for (int j = 0; j < OT; ++j)
#pragma unroll
      for (int i = 0; i < 2; ++i) acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[i], fb[j], acc[i][j], 0, 0, 0);
  }
  __syncthreads();  // everyone is done with the A rows and the weights: the staging tile takes their place

  // ---- epilogue ---------------------------------------------------------------------------
  int8_t* out_tile = lds + a.off_a;  // [oct][out_stride]
  const int lo = a.lo, hi = a.hi;
#pragma unroll
  for (int j = 0; j < OT; ++j) {
    const int ocl = j * 32 + frag_row;
    const v4i q = rq_lds[ocl];
    const int bias = bias_lds[ocl];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int pt = wave + 4 * i;
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int pl = pt * 32 + 8 * g + 4 * frag_half;
        const v4i s4 = *reinterpret_cast<const v4i*>(sx_lds + pl);
        if (a.pool) {
          // requantization is monotone: the window's largest accumulator gives its largest code
          const int m = max(max(acc[i][j][g * 4] - s4[0], acc[i][j][g * 4 + 1] - s4[1]),
                            max(acc[i][j][g * 4 + 2] - s4[2], acc[i][j][g * 4 + 3] - s4[3]));
          out_tile[ocl * a.out_stride + (pl >> 2)] = static_cast<int8_t>(Requant8<RQ>(m + bias, q, a.out_zp, lo, hi));
          continue;
        }
        int r4[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) r4[e] = acc[i][j][g * 4 + e] + (bias - s4[e]);
        *reinterpret_cast<uint32_t*>(out_tile + ocl * a.out_stride + pl) = RequantPack4<RQ>(r4, q, a.out_zp, lo, hi);
      }
    }
  }
  __syncthreads();
  // what leaves: the tile's pixels, or its pooled pixels (a quarter as many)
  const int hw_y = a.pool ? hw >> 2 : hw, valid_y = a.pool ? valid >> 2 : valid;
  uint8_t* ybase = a.y + static_cast<size_t>(n) * a.OC * hw_y + (a.pool ? p0 >> 2 : p0);
  if ((hw_y & 3) == 0) {
    const int per_row = valid_y >> 2;  // the tile's first pixel and the plane are multiples of 4: whole dwords
    for (int o = wave; o < a.OC; o += 4)
      for (int dwi = lane; dwi < per_row; dwi += 64)
        *reinterpret_cast<uint32_t*>(ybase + static_cast<size_t>(o) * hw_y + dwi * 4) =
            *reinterpret_cast<const uint32_t*>(out_tile + o * a.out_stride + dwi * 4);
  } else {
    for (int o = wave; o < a.OC; o += 4)
      for (int pi = lane; pi < valid_y; pi += 64)
        ybase[static_cast<size_t>(o) * hw_y + pi] = static_cast<uint8_t>(out_tile[o * a.out_stride + pi]);
  }
}

// ---- windows three or five taps wide, undilated along the row: the operand in registers ----
//
// A reduction step of the matrix product takes 32 bytes of a window, sixteen from either lane half; a half is given five (three) whole
// kernel rows of three (five) taps, and the weights are packed in the same order. A lane thus gathers its own fragment - an unaligned
// load a row - and nothing passes through LDS: no barrier, every wavefront goes its own way through a run of 32-pixel tiles, with
// the next tile's loads in flight. Pixel 4 i + e of a tile stands in row 8 e + i of the product, so that a lane finds sixteen
// consecutive pixels of a channel (or the candidates of four consecutive pooled ones) in its accumulators and stores them from there. The
// window sums of the zero-point expansion are a product with a constant fragment.
// Bound by the latency of the chain in small layers, by the vector ALU (6.5 of the 14 us below) and by stores of 32 bytes a channel and tile in
// large ones. Before (every pixel's window through LDS, results staged there, three barriers) and now, microseconds, uint8: 3 x 3 at
// stride 2 on 224 x 224, 3 to 32: batch 1 6.0 / 2.7, batch 64 18.3 / 14.3; 5 x 5 on 28 x 28, 1 to 20, pooled: batch 1 5.6 / 2.4, batch 207 6.8 / 3.8.
struct ImRegArgs {
  const uint8_t* x;
  const v4i* w;          // [channel tile][step][64 lanes], then the constant fragments [step][64 lanes]
  const int32_t* biasf;
  const v4i* rq;
  int offs[2][16];       // per lane half and kernel row: c * H * W + dy * W
  int dys[2][16];
  int image, W, H, OW, hw, sh, sw, pad_t, pad_l;
  int tiles_per_image, tiles, run;  // run: tiles of a wavefront
  uint32_t m_tiles, m_ow;           // reciprocals (of the pooled width under a pooling)
  int last, max_off;     // highest index a load may start at; highest of the offsets
  int max_dy;            // lowest window row
  uint32_t flip_in, flip_out;  // a window byte inside the image is moved to the signed domain, one outside is the zero point: all four bytes
  int ztwice;            // the constant fragment holds half of minus the weights' zero point, 128, and is taken twice
  uint8_t* y;
  int OC, pre, lo, hi, out_xor4, out_zp, generic;
};

// PLAIN: no ties, narrow clamps, 64-bit products or second constant, factors below 2^23, and biases that leave sums within 32 bits.
template <int KW, int KS, int OT, bool PLAIN, bool POOL>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2))) ConvIm2colRegKernel(ImRegArgs a) {
  constexpr int kRows = KW == 3 ? 5 : 3, kDw = KW == 3 ? 1 : 2;  // kernel rows of a lane half and step; dwords of each
  const int lane = threadIdx.x & 63, col = lane & 31, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int wg = blockIdx.x;  // an XCD gets a contiguous run of tiles: neighbours share input rows in its L2
  {
    const int per = gridDim.x >> 3, rem = gridDim.x & 7, xcd = wg & 7;
    wg = xcd * per + min(xcd, rem) + (wg >> 3);
  }
  int t = (wg * static_cast<int>(blockDim.x >> 6) + wave) * a.run;
  const int t_end = min(t + a.run, a.tiles);
  if (t >= t_end) return;
  // v / d by the reciprocal rounded up, which is never too small and at most one too large (m = 0: d = 1)
  const auto times = [](int v, int w) { return PLAIN ? __mul24(v, w) : v * w; };
  const auto over = [&](int v, uint32_t m, int d) {
    const int q = static_cast<int>(__umulhi(static_cast<uint32_t>(v), m) + (static_cast<uint32_t>(v) & (m ? 0u : ~0u)));
    return q - (times(q, d) > v ? 1 : 0);
  };

  const auto image = [](int tile, uint32_t m, int d) {  // (uniform)
    const int q = static_cast<int>(__umulhi(static_cast<uint32_t>(tile), m) + (static_cast<uint32_t>(tile) & (m ? 0u : ~0u)));
    return q - (static_cast<uint32_t>(q) * static_cast<uint32_t>(d) > static_cast<uint32_t>(tile) ? 1 : 0);
  };

  int off[KS * kRows];
#pragma unroll
  for (int j = 0; j < KS * kRows; ++j) off[j] = half ? a.offs[1][j] : a.offs[0][j];
  struct Raw {
    uint32_t v[KS * kRows][kDw];
    int at, iw0;        // of the window's origin
    int ih0;
  };
  const int slot = 4 * (col & 7) + (col >> 3);  // the pixel of this lane's row of a product
  const auto load = [&](int tile) {
    Raw r;
    const int n = image(tile, a.m_tiles, a.tiles_per_image);
    const int p = min((tile - n * a.tiles_per_image) * 32 + slot, a.hw - 1);  // (past the end the last pixel again: nobody stores it)
    int oh, ow;
    if constexpr (POOL) {  // four consecutive pixels are a 2 x 2 window, windows row-major over the pooled image
      const int pw = a.OW >> 1, qh = over(p >> 2, a.m_ow, pw);
      oh = 2 * qh + (p >> 1 & 1);
      ow = 2 * ((p >> 2) - times(qh, pw)) + (p & 1);
    } else {
      oh = over(p, a.m_ow, a.OW);
      ow = p - times(oh, a.OW);
    }
    r.ih0 = times(oh, a.sh) - a.pad_t;
    r.iw0 = times(ow, a.sw) - a.pad_l;
    r.at = n * a.image + times(r.ih0, a.W) + r.iw0;
#pragma unroll
    for (int j = 0; j < KS * kRows; ++j) __builtin_memcpy(r.v[j], a.x + static_cast<uint32_t>(Med3(r.at + off[j], 0, a.last)), 4 * kDw);
    return r;
  };
  Raw cur = load(t);

  // ---- under these loads: weights, tables ----
  const ImRegArgs& b = LateArgs<ImRegArgs>();
  v4i fw[OT][KS], fz[KS], q[OT];
  int bias[OT];
#pragma unroll
  for (int j = 0; j < OT; ++j) {
#pragma unroll
    for (int k = 0; k < KS; ++k) fw[j][k] = b.w[(j * KS + k) * 64 + lane];
    q[j] = b.rq[j * 32 + col];
    bias[j] = b.biasf[j * 32 + col];
  }
#pragma unroll
  for (int k = 0; k < KS; ++k) fz[k] = b.w[(OT * KS + k) * 64 + lane];
  const int W = b.W, last = b.last, max_off = b.max_off, ztwice = b.ztwice, OC = b.OC, tiles_per_image = b.tiles_per_image, hw = b.hw;
  const int hw_y = POOL ? hw >> 2 : hw;
  const int H = b.H, below = H - 1 - b.max_dy;
  const uint32_t m_tiles = b.m_tiles, flip_in = b.flip_in, flip_out = b.flip_out, out_xor4 = static_cast<uint32_t>(b.out_xor4);
  uint8_t* const y = b.y;
  const size_t lane_y = static_cast<size_t>(col) * hw_y;
  int dy[KS * kRows];
#pragma unroll
  for (int j = 0; j < KS * kRows; ++j) dy[j] = half ? b.dys[1][j] : b.dys[0][j];

  // (a plain requantization takes the bias in its rounding constant: mult * (acc + bias) + round)
  int64_t rounds[OT];
#pragma unroll
  for (int j = 0; j < OT; ++j) rounds[j] = static_cast<int64_t>(static_cast<uint64_t>(static_cast<uint32_t>(q[j][2])) << 32) + static_cast<int64_t>(q[j][0]) * bias[j];

  for (;;) {
    const bool more = t + 1 < t_end;
    Raw next = cur;
    if (more) next = load(t + 1);
    if (__builtin_amdgcn_ballot_w64(cur.at < 0 || cur.at > last - max_off)) {  // a load at the tensor's ends was moved inside
#pragma unroll
      for (int j = 0; j < KS * kRows; ++j) {
        const int at = cur.at + off[j], by = min(max(min(max(at, 0), last) - at, -4 * kDw), 4 * kDw);
        uint64_t v = cur.v[j][0];
        if (kDw == 2) v |= static_cast<uint64_t>(cur.v[j][kDw - 1]) << 32;
        v = by > 4 * kDw - 1 || by < 1 - 4 * kDw ? 0 : by > 0 ? v << (8 * by) : v >> (-8 * by);
        cur.v[j][0] = static_cast<uint32_t>(v);
        if (kDw == 2) cur.v[j][kDw - 1] = static_cast<uint32_t>(v >> 32);
      }
    }
    // window columns outside the image, the same in each row: (byte & keep) ^ flip
    uint32_t keep[kDw], flip[kDw];
    {
      typedef std::conditional_t<KW == 3, uint32_t, uint64_t> Bytes;
      constexpr Bytes kAll = static_cast<Bytes>((1ull << (8 * KW)) - 1);
      const int left = min(max(-cur.iw0, 0), KW), right = KW - min(max(W - cur.iw0, 0), KW);
      const Bytes k = (kAll << (8 * left)) & (kAll >> (8 * right));
#pragma unroll
      for (int i = 0; i < kDw; ++i) {
        keep[i] = static_cast<uint32_t>(static_cast<uint64_t>(k) >> (32 * i));
        flip[i] = ((flip_in ^ flip_out) & keep[i]) ^ (flip_out & static_cast<uint32_t>(static_cast<uint64_t>(kAll) >> (32 * i)));
      }
    }
    if (__builtin_amdgcn_ballot_w64(cur.ih0 < 0 || cur.ih0 > below) == 0) {  // every window row lies inside the image
#pragma unroll
      for (int j = 0; j < KS * kRows; ++j)
#pragma unroll
        for (int i = 0; i < kDw; ++i) cur.v[j][i] = (cur.v[j][i] & keep[i]) ^ flip[i];
    } else {
#pragma unroll
      for (int j = 0; j < KS * kRows; ++j) {
        const uint32_t in = static_cast<unsigned>(cur.ih0 + dy[j]) < static_cast<unsigned>(H) ? ~0u : 0u;
#pragma unroll
        for (int i = 0; i < kDw; ++i) {
          const uint32_t all = KW == 3 ? 0xffffffu : i ? 0xffu : ~0u;
          cur.v[j][i] = (((cur.v[j][i] & keep[i]) ^ flip[i]) & in) | (flip_out & all & ~in);
        }
      }
    }
    v4i fx[KS];
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      const uint32_t (*v)[kDw] = cur.v + k * kRows;
      uint32_t d[4];
      if constexpr (KW == 3) {
        d[0] = v[0][0] | v[1][0] << 24;
        d[1] = __builtin_amdgcn_perm(v[2][0], v[1][0], 0x05040201);
        d[2] = v[2][0] >> 16 | v[3][0] << 8;
        d[3] = v[4][0];
      } else {
        d[0] = v[0][0];
        d[1] = v[0][kDw - 1] | v[1][0] << 8;
        d[2] = __builtin_amdgcn_perm(v[1][kDw - 1], v[1][0], 0x0c0c0403) | v[2][0] << 16;
        d[3] = v[2][0] >> 16 | v[2][kDw - 1] << 16;
      }
      fx[k] = v4i{static_cast<int>(d[0]), static_cast<int>(d[1]), static_cast<int>(d[2]), static_cast<int>(d[3])};
    }
    const int n = image(t, m_tiles, tiles_per_image), p0 = (t - n * tiles_per_image) * 32;
    // what of this lane's sixteen pixels (four pooled ones) exists
    const int first = POOL ? (p0 >> 2) + 4 * half : p0 + 16 * half;
    const int live = hw_y - first;
    v16i zsum;  // the window sums' part
#pragma unroll
    for (int r = 0; r < 16; ++r) zsum[r] = 0;
#pragma unroll
    for (int k = 0; k < KS; ++k) zsum = __builtin_amdgcn_mfma_i32_32x32x32_i8(fx[k], fz[k], zsum, 0, 0, 0);
    if constexpr (!PLAIN)
      if (ztwice)  // (uniform)
#pragma unroll
        for (int k = 0; k < KS; ++k) zsum = __builtin_amdgcn_mfma_i32_32x32x32_i8(fx[k], fz[k], zsum, 0, 0, 0);
    uint8_t* const tile_y = y + static_cast<size_t>(n) * OC * hw_y + first;
#pragma unroll
    for (int j = 0; j < OT; ++j) {
      v16i acc = zsum;
#pragma unroll
      for (int k = 0; k < KS; ++k) acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(fx[k], fw[j][k], acc, 0, 0, 0);
      if constexpr (!PLAIN)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[r] += bias[j];
      const int oc = j * 32 + col;
      const int64_t round = PLAIN ? rounds[j] : RoundHigh(q[j][2]);
      const auto codes = [&](int (&v)[4]) {
        if constexpr (!PLAIN)
          if (b.generic) return RequantPack4<kRqGeneric>(v, q[j], b.out_zp, b.lo, b.hi);
        return RequantCodes4<PLAIN>(v, q[j], round, b.pre, b.lo, b.hi) ^ out_xor4;
      };
      uint8_t* const to = tile_y + lane_y + static_cast<size_t>(j * 32) * hw_y;
      constexpr int kOut = POOL ? 1 : 4;
      uint32_t out[kOut];
      // accumulator 4 e + i is row 8 e + 4 half + i of the product: pixel 16 half + 4 i + e
      if constexpr (POOL) {  // requantization is monotone: a window's largest accumulator gives its largest code
        int v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = max(max(acc[i], acc[4 + i]), max(acc[8 + i], acc[12 + i]));
        out[0] = codes(v);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          int v[4] = {acc[i], acc[4 + i], acc[8 + i], acc[12 + i]};
          out[i] = codes(v);
        }
      }
      if (oc >= OC || live <= 0) continue;
      if (live >= 4 * kOut) {
        __builtin_memcpy(to, out, 4 * kOut);
      } else {
#pragma unroll
        for (int i = 0; i < kOut; ++i) {
          if (live >= 4 * i + 4) {
            __builtin_memcpy(to + 4 * i, &out[i], 4);
          } else {
#pragma unroll
            for (int e = 0; e < 3; ++e)
              if (live > 4 * i + e) to[4 * i + e] = static_cast<uint8_t>(out[i] >> (8 * e));
          }
        }
      }
    }
    if (!more) break;
    ++t;
    cur = next;
  }
}

struct RegPlan {
  ImRegArgs a;
  void (*fn)(ImRegArgs);
  unsigned grid, block;
};

struct Plan {
  ImArgs a;
  int lds_bytes;
  int ot, rq;
  dim3 grid;
};

template <int OT>
void Launch(const Plan* plan, const ImArgs& a, hipStream_t st) {
  const dim3 block(kThreads);
  if (plan->rq == kRqFastNoTie)
    hipLaunchKernelGGL((ConvIm2colKernel<OT, kRqFastNoTie>), plan->grid, block, plan->lds_bytes, st, a);
  else if (plan->rq == kRqFast)
    hipLaunchKernelGGL((ConvIm2colKernel<OT, kRqFast>), plan->grid, block, plan->lds_bytes, st, a);
  else
    hipLaunchKernelGGL((ConvIm2colKernel<OT, kRqGeneric>), plan->grid, block, plan->lds_bytes, st, a);
}

int ConvIm2colRun(tvx_op* op, const void* in0, const void*, void* out, hipStream_t st) {
  const Plan* plan = reinterpret_cast<const Plan*>(op->host_blob.data());
  ImArgs a = plan->a;
  a.x = static_cast<const uint8_t*>(in0);
  a.y = static_cast<uint8_t*>(out);
  if (plan->ot == 1) Launch<1>(plan, a, st);
  else if (plan->ot == 2) Launch<2>(plan, a, st);
  else Launch<4>(plan, a, st);
  TVX_HIP_CHECK(hipGetLastError());
  return TVX_OK;
}

typedef void (*RegFn)(ImRegArgs);

template <int KW, int KS, bool PLAIN, bool POOL>
RegFn RegKernel(int ot) {
  return ot == 1 ? ConvIm2colRegKernel<KW, KS, 1, PLAIN, POOL> : ot == 2 ? ConvIm2colRegKernel<KW, KS, 2, PLAIN, POOL> : ConvIm2colRegKernel<KW, KS, 4, PLAIN, POOL>;
}
template <bool PLAIN, bool POOL>
RegFn RegKernel(int kw, int ks, int ot) {
  if (kw == 5) return ks == 1 ? RegKernel<5, 1, PLAIN, POOL>(ot) : RegKernel<5, 2, PLAIN, POOL>(ot);
  return ks == 1 ? RegKernel<3, 1, PLAIN, POOL>(ot) : ks == 2 ? RegKernel<3, 2, PLAIN, POOL>(ot) : RegKernel<3, 3, PLAIN, POOL>(ot);
}

int ConvIm2colRegRun(tvx_op* op, const void* in0, const void*, void* out, hipStream_t st) {
  const RegPlan* plan = reinterpret_cast<const RegPlan*>(op->host_blob.data());
  ImRegArgs a = plan->a;
  a.x = static_cast<const uint8_t*>(in0);
  a.y = static_cast<uint8_t*>(out);
  hipLaunchKernelGGL(plan->fn, dim3(plan->grid), dim3(plan->block), 0, st, a);
  TVX_HIP_CHECK(hipGetLastError());
  return TVX_OK;
}

// The register form: windows three or five taps wide, undilated along the row.
int RegSetup(tvx_op* op, const tvx_conv2d_desc* d, const void* w_host, const void* bias_host, int zxs, int zws) {
  const int kw = static_cast<int>(d->k_w), C = d->in_c, kh = d->k_h, rows = C * kh;
  const uint64_t total = static_cast<uint64_t>(d->batch) * d->in_c * d->in_h * d->in_w;
  const uint64_t out_pixels = static_cast<uint64_t>(d->out_h) * d->out_w, tpi = (out_pixels + 31) / 32, tiles = tpi * d->batch;
  if ((kw != 3 && kw != 5) || d->dilation_w != 1 || total < 8 || total >= (1ull << 31) - 64 || !LaunchFits((tiles + 7) / 8, 64)) return TVX_E_UNSUPPORTED;
  if (const char* f = getenv("TVX_IM2COL_ROWS"))  // tuning aid
    if (!atoi(f)) return TVX_E_UNSUPPORTED;
  const int per = kw == 3 ? 5 : 3, ks = (rows + 2 * per - 1) / (2 * per), K = rows * kw;
  if (ks > (kw == 3 ? 3 : 2)) return TVX_E_UNSUPPORTED;
  const bool x_u8 = d->in_dtype == TVX_U8, w_u8 = d->w_dtype == TVX_U8;
  RegPlan plan{};
  ImRegArgs& a = plan.a;
  const int pool = op->fused_pool;
  a.image = C * static_cast<int>(d->in_h) * static_cast<int>(d->in_w);
  a.W = d->in_w; a.H = d->in_h; a.OW = d->out_w; a.hw = static_cast<int>(out_pixels);
  a.sh = d->stride_h; a.sw = d->stride_w; a.pad_t = d->pad_top; a.pad_l = d->pad_left;
  const auto reciprocal = [](uint64_t v) { return v > 1 ? static_cast<uint32_t>(((1ull << 32) + v - 1) / v) : 0u; };
  a.tiles_per_image = static_cast<int>(tpi); a.tiles = static_cast<int>(tiles);
  a.m_tiles = reciprocal(tpi);
  a.m_ow = reciprocal(pool ? d->out_w / 2 : d->out_w);
  a.last = static_cast<int>(total) - (kw == 3 ? 4 : 8);
  a.flip_in = x_u8 ? 0x80808080u : 0u;
  a.flip_out = static_cast<uint32_t>(zxs & 0xff) * 0x01010101u;
  a.OC = d->out_c;
  for (int r = 0; r < rows; ++r) {
    const int dy = r % kh * static_cast<int>(d->dilation_h), group = r / per;
    a.offs[group & 1][group / 2 * per + r % per] = (r / kh * a.H + dy) * a.W;
    a.dys[group & 1][group / 2 * per + r % per] = dy;
    a.max_dy = std::max(a.max_dy, dy);
    a.max_off = std::max(a.max_off, (r / kh * a.H + dy) * a.W);
  }
  a.ztwice = zws == -128;
  const int ot = d->out_c <= 32 ? 1 : d->out_c <= 64 ? 2 : 4, alloc = 32 * ot;
  std::vector<int8_t> packed(static_cast<size_t>(ot + 1) * ks * 1024, 0);
  std::vector<int32_t> biasf(alloc, 0);
  const uint8_t* src = static_cast<const uint8_t*>(w_host);
  const int32_t* b = static_cast<const int32_t*>(bias_host);
  // byte k of a window -> [step][half][16 bytes]
  const auto place = [&](int tile, int column, int k) {
    const int r = k / kw, group = r / per;
    return ((static_cast<size_t>(tile) * ks + group / 2) * 64 + (group & 1) * 32 + column) * 16 + r % per * kw + k % kw;
  };
  for (int oc = 0; oc < a.OC; ++oc) {
    int64_t sum = 0;
    for (int k = 0; k < K; ++k) {
      const uint8_t raw = src[static_cast<size_t>(oc) * K + k];
      const int8_t v = static_cast<int8_t>(w_u8 ? raw ^ 0x80 : raw);
      packed[place(oc / 32, oc % 32, k)] = v;
      sum += v;
    }
    const int64_t v = (b ? b[oc] : 0) - static_cast<int64_t>(zxs) * sum + static_cast<int64_t>(K) * zxs * zws;
    biasf[oc] = static_cast<int32_t>(static_cast<uint32_t>(v));
  }
  for (int column = 0; column < 32; ++column)
    for (int k = 0; k < K; ++k) packed[place(ot, column, k)] = static_cast<int8_t>(a.ztwice ? 64 : -zws);
  const int64_t bound = AccumulatorBound(static_cast<uint64_t>(K), bias_host, a.OC);
  const int flip = d->out_dtype == TVX_U8 ? 128 : 0;
  std::vector<int32_t> rqt;
  int up = 0;
  bool ties = false;
  a.out_zp = d->out_zp; a.lo = op->act_lo; a.hi = op->act_hi;
  a.generic = BuildRequantRecords(op->h_mult, op->h_shift, a.OC, alloc, d->out_zp, &rqt, bound) == kRqGeneric;
  if (!a.generic) {
    if (!BuildTieRecords(op->h_mult, op->h_shift, a.OC, alloc, d->out_zp - flip, std::min<int64_t>(bound, INT32_MAX), &rqt, &up, &ties)) return TVX_E_UNSUPPORTED;
    a.lo -= flip; a.hi -= flip;
    a.pre = up * 2 + ties;
    a.out_xor4 = flip ? static_cast<int>(0x80808080u) : 0;
  }
  int s = op->packed.Upload(packed.data(), packed.size());
  if (s == TVX_OK) s = op->aux.Upload(biasf.data(), biasf.size() * 4);
  if (s == TVX_OK) s = op->aux2.Upload(rqt.data(), rqt.size() * 4);
  if (s != TVX_OK) return s;
  a.w = op->packed.as<v4i>();
  a.biasf = op->aux.as<int32_t>();
  a.rq = op->aux2.as<v4i>();
  const bool small = out_pixels < (1u << 23) && d->in_h < (1u << 23) && d->in_w < (1u << 23) && d->stride_h < (1u << 23) && d->stride_w < (1u << 23) && d->pad_top < (1u << 22);
  // (the plain form multiplies sum and bias apart, in 64 bits: a bias whose folded constants wrap around has to meet the sum in 32)
  const bool plain = !a.generic && a.lo == -128 && a.hi == 127 && !a.pre && !a.ztwice && small && bound <= INT32_MAX;
  plan.fn = pool ? (plain ? RegKernel<true, true>(kw, ks, ot) : RegKernel<false, true>(kw, ks, ot)) : plain ? RegKernel<true, false>(kw, ks, ot) : RegKernel<false, false>(kw, ks, ot);
  // a wavefront's run: one tile until every SIMD has a few wavefronts (the first of the layers above at batch 64, 98 tiles a CU: 16.1 us with
  // runs of one, 14.6 two, 14.2 three, 14.8 four, 15.6 six; at batch 1, 1.5 a CU: 2.7, 3.3, 3.8, 4.7, 5.0)
  const int cus = ComputeUnits();
  a.run = static_cast<int>(std::min<uint64_t>(8, std::max<uint64_t>(1, tiles / (32ull * cus))));
  if (const char* f = getenv("TVX_IM2COL_RUN")) a.run = std::max(1, atoi(f));  // test lever
  const uint64_t waves = (tiles + a.run - 1) / a.run;
  const int per_wg = waves <= 2ull * cus ? 1 : kThreads / 64;
  plan.block = 64 * per_wg;
  plan.grid = static_cast<unsigned>((waves + per_wg - 1) / per_wg);
  op->host_blob.assign(reinterpret_cast<const uint8_t*>(&plan), reinterpret_cast<const uint8_t*>(&plan) + sizeof(plan));
  op->run = ConvIm2colRegRun;
  op->kernel_name = pool ? "conv2d_im2col_maxpool_i8" : "conv2d_im2col_i8";
  op->variant = pool ? "conv2d_im2col_reg_maxpool_i8" : "conv2d_im2col_reg_i8";
  return TVX_OK;
}

int RoundUp(int v, int m) { return (v + m - 1) / m * m; }

}  // namespace

// Claims dense quantized convolutions with constant weights whose whole window is at most 64
// bytes and whose channel count the implicit-GEMM kernel would have to pad (C % 16 != 0).
static int Im2colSetup(tvx_op* op, const tvx_conv2d_desc* d, const void* w_host, const void* bias_host, bool rest) {
  if (!op->quantized || !w_host || d->multiplier != 0 || d->groups > 1) return TVX_E_UNSUPPORTED;
  const int taps = static_cast<int>(d->k_w * d->k_h);
  const uint64_t k_real = static_cast<uint64_t>(d->in_c) * taps;
  if (k_real > 64 || d->in_c % 16 == 0 || d->out_c > 128) return TVX_E_UNSUPPORTED;
  if (static_cast<uint64_t>(d->in_c) * d->in_h * d->in_w >= (1ull << 31) || d->batch > 65535) return TVX_E_UNSUPPORTED;
  ImArgs a{};
  a.C = d->in_c; a.H = d->in_h; a.W = d->in_w; a.OC = d->out_c; a.OH = d->out_h; a.OW = d->out_w;
  a.sh = d->stride_h; a.sw = d->stride_w; a.pad_t = d->pad_top; a.pad_l = d->pad_left;
  const int K = static_cast<int>(k_real);
  a.kp = K <= 32 ? 32 : 64;
  a.row_stride = a.kp + 16;
  const int ot = d->out_c <= 32 ? 1 : (d->out_c <= 64 ? 2 : 4);
  a.oct = 32 * ot;
  const bool x_u8 = d->in_dtype == TVX_U8, w_u8 = d->w_dtype == TVX_U8;
  const int zxs = d->in_zp - (x_u8 ? 128 : 0);
  const int zws = op->w_zp - (w_u8 ? 128 : 0);
  if (zxs < -128 || zxs > 127) return TVX_E_UNSUPPORTED;  // zero point outside the tensor's range
  if ((d->k_h - 1) * d->dilation_h > 31 || (d->k_w - 1) * d->dilation_w > 31) return TVX_E_UNSUPPORTED;  // window offsets index 32-bit masks
  if (!rest) {
    const int reg = RegSetup(op, d, w_host, bias_host, zxs, zws);
    if (reg != TVX_E_UNSUPPORTED) return reg;
  }
  // What does not fit registers is asked for twice, in front of the tiles (conv_tile.hip) and behind them, which take what lies between a handful of
  // pixels (windows of several taps: a few thousand) and eighty thousand on 256 compute units: 0.64 of the time on 80 drawn layers (int8 12 -> 115, 1x1 / 2 on 13 x 13, batch 2, 11.9 -> 5.1 us; uint8 43 -> 80,
  // 1x1 / 2 on 17 x 17, batch 10, 15.9 -> 5.5). With more pixels a pass of this kernel is the shorter one (8 -> 64, 1x1 / 2 on 126 x 160, batch 64,
  // 16.6 against 26.8; 1 -> 80 on 79 x 153, batch 33, 13.0 against 15.9; 1 -> 128, 7x7 on 120 x 120, batch 30, 47.6 against 67.3).
  const uint64_t pixels = static_cast<uint64_t>(d->batch) * d->out_h * d->out_w, cus = ComputeUnits();
  if (!rest && !op->fused_pool && 2 * pixels < 625 * cus && 2 * pixels > (taps == 1 ? 1 : 32) * cus) return TVX_E_UNSUPPORTED;
  a.xor_mask = x_u8 ? 0x80 : 0;
  a.pad_fill = zxs & 0xff;
  a.zws = zws;
  a.out_zp = d->out_zp; a.lo = op->act_lo; a.hi = op->act_hi;
  a.pool = op->fused_pool;  // (the caller has checked the pooling: 2 x 2, stride 2, even output extents)
  a.out_stride = ((kPixels / 4) | 1) * 4;
  // LDS: window sums and tables first; A rows + weights behind them are reused as the staging tile
  a.off_sx = 0;
  a.off_rq = kPixels * 4;
  a.off_bias = a.off_rq + a.oct * 16;
  a.off_a = a.off_bias + a.oct * 4;
  a.off_w = a.off_a + kPixels * a.row_stride;
  const int lds_bytes = a.off_a + std::max(kPixels * a.row_stride + a.oct * a.row_stride, a.oct * a.out_stride);

  // ---- pack weights [oc][(c, ky, kx)] int8 with zero padding, fold constants ---------------
  std::vector<int8_t> packed(static_cast<size_t>(a.oct) * a.row_stride, 0);
  std::vector<int32_t> biasf(a.oct, 0);
  const uint8_t* src = static_cast<const uint8_t*>(w_host);
  const int32_t* b = static_cast<const int32_t*>(bias_host);
  for (int oc = 0; oc < a.OC; ++oc) {
    int64_t sw = 0;
    for (int k = 0; k < K; ++k) {  // the weight tensor's own order: [oc][c][ky][kx]
      const uint8_t raw = src[static_cast<size_t>(oc) * K + k];
      const int8_t v = static_cast<int8_t>(w_u8 ? raw ^ 0x80 : raw);
      packed[static_cast<size_t>(oc) * a.row_stride + k] = v;
      sw += v;
    }
    const int64_t v = (b ? b[oc] : 0) - static_cast<int64_t>(zxs) * sw + static_cast<int64_t>(K) * zxs * zws;
    biasf[oc] = static_cast<int32_t>(static_cast<uint32_t>(v));
  }
  std::vector<int32_t> rqt;
  const int rq = BuildRequantRecords(op->h_mult, op->h_shift, a.OC, a.oct, d->out_zp, &rqt,
                                     AccumulatorBound(static_cast<uint64_t>(K), bias_host, a.OC));
  for (int k = 0; k < K; ++k) {
    const int c = k / taps, t = k % taps;
    const int dy = (t / static_cast<int>(d->k_w)) * static_cast<int>(d->dilation_h);
    const int dx = (t % static_cast<int>(d->k_w)) * static_cast<int>(d->dilation_w);
    a.taps[k] = dy | dx << 8 | 1 << 16;
    a.offs[k] = c * a.H * a.W + dy * a.W + dx;
  }
  int s = op->packed.Upload(packed.data(), packed.size());
  if (s == TVX_OK) s = op->aux.Upload(biasf.data(), biasf.size() * 4);
  if (s == TVX_OK) s = op->aux2.Upload(rqt.data(), rqt.size() * 4);
  if (s != TVX_OK) return s;
  a.w = op->packed.as<int8_t>();
  a.biasf = op->aux.as<int32_t>();
  a.rq = op->aux2.as<v4i>();

  Plan plan;
  plan.a = a;
  plan.lds_bytes = lds_bytes;
  plan.ot = ot;
  plan.rq = rq;
  const int hw = a.OH * a.OW;
  plan.grid = dim3(static_cast<unsigned>((hw + kPixels - 1) / kPixels), static_cast<unsigned>(d->batch));
  op->host_blob.assign(reinterpret_cast<const uint8_t*>(&plan), reinterpret_cast<const uint8_t*>(&plan) + sizeof(plan));
  op->run = ConvIm2colRun;
  op->kernel_name = op->fused_pool ? "conv2d_im2col_maxpool_i8" : "conv2d_im2col_i8";
  return TVX_OK;
}

int ConvIm2colSetup(tvx_op* op, const tvx_conv2d_desc* d, const void* w_host, const void* bias_host) { return Im2colSetup(op, d, w_host, bias_host, false); }
int ConvIm2colRestSetup(tvx_op* op, const tvx_conv2d_desc* d, const void* w_host, const void* bias_host) { return Im2colSetup(op, d, w_host, bias_host, true); }

}  // namespace tvx
