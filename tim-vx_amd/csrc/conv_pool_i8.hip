// Dense quantized Conv2d and the 2 x 2 / stride-2 MAX pooling behind it on small planes (LeNet's second layer: 12 x 12, 20 to 50
// channels), the whole input image in LDS. What bounds such a layer is not its arithmetic but the chain a workgroup walks - load,
// transpose, multiply, sum, store - and how many wavefronts share it.
//
// Workgroup = (image, 32 output channels, all or some of the 32-pixel tiles). Its wavefronts are (tile, part of the reduction) pairs, eight
// where the layer has that many: weights come straight from L2 into registers, the first ones requested before the input; the rows behind its
// tiles are transposed into LDS as [pixel][channel], each tap's operand is read from there; partial sums meet in LDS by integer atomics where the reduction is
// split. Pixels run in pooling order, and pixel 4 i + e of a tile stands in row 8 e + i of the product: a lane finds the four candidates
// of four consecutive pooled pixels in its accumulators. Requantization is monotone, so a window's largest accumulator is
// requantized once. The zero-point term of uint8 weights is a second product with a constant fragment.
// Channels behind the real ones hold anything: their weights and constants are zero.
// 12 x 12, 20 to 50, 5 x 5, before (conv2d_igemm_i8's tile, weights through LDS, results staged there) and now,
// microseconds: batch 1 7.9 / 4.8, batch 90 9.4 / 5.2, batch 207 9.6 / 6.7.
#include <algorithm>
#include <cmath>
#include <cstdlib>

#include "variants.h"

namespace tvx {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

constexpr int kMaxWaves = 8, kAhead = 8;   // wavefronts of a workgroup; reduction steps whose weights are requested together
constexpr int kMaxImage = 64 * 1024;       // bytes of LDS for the image

struct PoolConvArgs {
  const uint8_t* x;
  const v4i* w;          // [32-channel tile][step][64 lanes]; steps run over (ky, kx, 32 channels)
  const int32_t* biasf;
  const v4i* rq;
  int C, H, W, oc_tiles, groups;  // groups: workgroups that share an image's tiles
  uint32_t m_octiles, m_groups;   // reciprocals
  int chan_quads, col_quads;  // of the input in fours
  uint32_t m_units, m_cols;
  int pix_stride, row_stride, pad_t, pad_l;
  uint32_t xor4;
  int tiles, per_group;       // 32-pixel tiles, of a workgroup
  int pooled, pw, tile_rows;  // input rows behind two rows of outputs
  uint32_t m_pw;
  int sh;
  // ---- later
  int steps, per_tap, kw;     // reduction steps; of a tap; taps of a kernel row
  int tap_x, tap_y;           // bytes from a tap to the next one, from a kernel row's start to the next's
  int parts, per_part;        // parts of the reduction, steps of a part
  uint32_t m_parts;
  int sw, OH, OW;
  int halo_rows, halo_cols, pad_fill4, padded;
  int z4, z4_last, ztwice;    // constant fragment: minus the weights' zero point in four bytes
  int last_channels;
  int off_red;
  int OC, pre, lo, hi, out_xor4, out_zp, generic;
  uint8_t* y;
};

__global__ void __launch_bounds__(kMaxWaves * 64) ConvPoolKernel(PoolConvArgs a) {
  extern __shared__ __attribute__((aligned(16))) int8_t lds[];
  const int tid = threadIdx.x, lane = tid & 63, col = lane & 31, half = lane >> 5, threads = blockDim.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), waves = threads >> 6;
  const auto over = [](int v, uint32_t m) { return static_cast<int>(__umulhi(static_cast<uint32_t>(v), m) + (static_cast<uint32_t>(v) & (m ? 0u : ~0u))); };
  const int pair = over(blockIdx.x, a.m_groups), group = blockIdx.x - pair * a.groups;
  const int n = over(pair, a.m_octiles), ot = pair - n * a.oc_tiles;
  const int tile0 = group * a.per_group, tiles = min(a.per_group, a.tiles - tile0);

  // ---- the first weights, then the input: [row][column][channel] ----
  const int first_tile = over(wave, a.m_parts), part = wave - first_tile * a.parts;
  const int k0 = part * a.per_part, k1 = min(k0 + a.per_part, a.steps);
  const v4i* const wt = a.w + static_cast<size_t>(ot) * a.steps * 64 + lane;
  v4i fw[kAhead];
  const auto fetch = [&](int k) {
#pragma unroll
    for (int i = 0; i < kAhead; ++i) fw[i] = wt[min(k + i, a.steps - 1) * 64];
  };
  fetch(k0);
  const int oc = ot * 32 + col;
  const v4i q = a.rq[oc];
  const int bias = a.biasf[oc];
  {
    // the rows behind the workgroup's tiles
    const int top = 2 * a.sh * over(8 * tile0, a.m_pw) - a.pad_t, bottom = 2 * a.sh * over(min(8 * (tile0 + tiles), a.pooled) - 1, a.m_pw) - a.pad_t + a.tile_rows;
    const int plane = a.H * a.W, units = a.H * a.col_quads * a.chan_quads;
    const uint8_t* const xn = a.x + static_cast<size_t>(n) * a.C * plane;
    for (int u = tid; u < units; u += threads) {
      const int c4 = over(u, a.m_units), at = u - c4 * (a.H * a.col_quads);
      const int r = over(at, a.m_cols), x = min((at - r * a.col_quads) * 4, a.W - 4);  // (the last four columns of a row may overlap the ones before)
      if (r < top || r >= bottom) continue;
      uint32_t d[4], px[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) __builtin_memcpy(&d[j], xn + static_cast<uint32_t>(min(4 * c4 + j, a.C - 1) * plane + r * a.W + x), 4);
#pragma unroll
      for (int j = 0; j < 4; ++j) d[j] ^= a.xor4;
      Transpose4x4(d, px);
      int8_t* to = lds + (r + a.pad_t) * a.row_stride + (x + a.pad_l) * a.pix_stride + 4 * c4;
#pragma unroll
      for (int e = 0; e < 4; ++e) *reinterpret_cast<uint32_t*>(to + e * a.pix_stride) = px[e];
    }
  }
  const PoolConvArgs& b = LateArgs<PoolConvArgs>();
  const int parts = b.parts, steps = b.steps;
  if (b.padded) {  // (uniform) the cells around the image
    const int quads = b.chan_quads, cells = b.halo_rows * b.halo_cols;
    for (int u = tid; u < cells; u += threads) {
      const int r = u / b.halo_cols, x = u - r * b.halo_cols;
      if (static_cast<unsigned>(r - b.pad_t) < static_cast<unsigned>(b.H) && static_cast<unsigned>(x - b.pad_l) < static_cast<unsigned>(b.W)) continue;
      for (int c = 0; c < quads; ++c) *reinterpret_cast<int*>(lds + r * b.row_stride + x * b.pix_stride + 4 * c) = b.pad_fill4;
    }
  }
  int* const red = reinterpret_cast<int*>(lds + b.off_red);
  if (parts > 1)
    for (int i = tid; i < tiles * 256; i += threads) reinterpret_cast<v4i*>(red)[i] = v4i{0, 0, 0, 0};
  __syncthreads();

  v4i z, z_last;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int left = b.last_channels - 16 * half - 4 * i;
    z[i] = b.z4;
    z_last[i] = left >= 4 ? b.z4 : left <= 0 ? 0 : b.z4 & static_cast<int>((1u << (8 * left)) - 1u);
  }
  const int per_tap = b.per_tap, kw = b.kw, tap_x = b.tap_x, tap_y = b.tap_y, zp = b.z4, ztwice = b.ztwice, pooled = b.pooled;
  const auto finish = [&](int tile, const v16i& acc) {
    int v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = max(max(acc[i], acc[4 + i]), max(acc[8 + i], acc[12 + i])) + bias;
    const int p = (tile0 + tile) * 8 + 4 * half, live = pooled - p;
    if (oc >= b.OC || live <= 0) return;
    const uint32_t codes = b.generic ? RequantPack4<kRqGeneric>(v, q, b.out_zp, b.lo, b.hi)
                                     : RequantCodes4<false>(v, q, RoundHigh(q[2]), b.pre, b.lo, b.hi) ^ static_cast<uint32_t>(b.out_xor4);
    uint8_t* const to = b.y + (static_cast<size_t>(n) * b.OC + oc) * pooled + p;
    if (live >= 4) {
      __builtin_memcpy(to, &codes, 4);
    } else {
#pragma unroll
      for (int e = 0; e < 3; ++e)
        if (live > e) to[e] = static_cast<uint8_t>(codes >> (8 * e));
    }
  };
  for (int tile = first_tile; tile < tiles; tile += parts > 1 ? tiles : waves) {  // (a split reduction: one tile a wavefront)
    const int slot = min((tile0 + tile) * 32 + 4 * (col & 7) + (col >> 3), 4 * pooled - 1);
    const int qh = over(slot >> 2, b.m_pw), oh = 2 * qh + (slot >> 1 & 1), ow = 2 * ((slot >> 2) - qh * b.pw) + (slot & 1);
    const int8_t* const window = lds + oh * b.sh * b.row_stride + ow * b.sw * b.pix_stride + 16 * half;
    // the step k0 stands at: channels, column and row of its tap
    int chan = 0, kx = 0, row = 0, at = 0;
    {
      const int tap = k0 / per_tap;
      chan = k0 - tap * per_tap;
      row = tap / kw;
      kx = tap - row * kw;
      at = row * tap_y + kx * tap_x + chan * 32;
    }
    v16i acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0;
    if (tile != first_tile) fetch(k0);
    for (int k = k0; k < k1; k += kAhead) {
      if (k != k0) fetch(k);
      v4i fx[kAhead];
      uint32_t ends = 0;  // steps that are their tap's last
#pragma unroll
      for (int i = 0; i < kAhead; ++i) {  // (behind the part's end the last operand again)
        fx[i] = *reinterpret_cast<const v4i*>(window + at);
        ends |= chan + 1 == per_tap ? 1u << i : 0u;
        if (k + i + 1 < k1) {  // (uniform)
          at += 32;
          if (++chan == per_tap) {
            chan = 0;
            at += tap_x - 32 * per_tap;
            if (++kx == kw) {
              kx = 0;
              at += tap_y - kw * tap_x;
            }
          }
        }
      }
#pragma unroll
      for (int i = 0; i < kAhead; ++i)
        if (k + i < k1) {  // (uniform)
          acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(fx[i], fw[i], acc, 0, 0, 0);
          if (zp) {
            const v4i f = ends >> i & 1 ? z_last : z;
            acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(fx[i], f, acc, 0, 0, 0);
            if (ztwice) acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(fx[i], f, acc, 0, 0, 0);
          }
        }
    }
    if (parts == 1) {
      finish(tile, acc);
      continue;
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) __hip_atomic_fetch_add(red + (tile * 16 + r) * 64 + lane, acc[r], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  }
  if (parts == 1) return;  // (uniform)
  __syncthreads();
  for (int tile = wave; tile < tiles; tile += waves) {
    v16i acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = red[(tile * 16 + r) * 64 + lane];
    finish(tile, acc);
  }
}

struct Plan {
  PoolConvArgs a;
  int lds_bytes, block;
  unsigned grid;
};

int ConvPoolRun(tvx_op* op, const void* in0, const void*, void* out, hipStream_t st) {
  const Plan* plan = reinterpret_cast<const Plan*>(op->host_blob.data());
  PoolConvArgs a = plan->a;
  a.x = static_cast<const uint8_t*>(in0);
  a.y = static_cast<uint8_t*>(out);
  hipLaunchKernelGGL(ConvPoolKernel, dim3(plan->grid), dim3(plan->block), plan->lds_bytes, st, a);
  TVX_HIP_CHECK(hipGetLastError());
  return TVX_OK;
}

}  // namespace

int ConvPoolSetup(tvx_op* op, const tvx_conv2d_desc* d, const void* w_host, const void* bias_host) {
  if (!op->quantized || !op->fused_pool || !w_host || d->multiplier != 0 || d->groups > 1 || d->in_w < 4) return TVX_E_UNSUPPORTED;
  if (const char* f = getenv("TVX_CONV_POOL")) if (!atoi(f)) return TVX_E_UNSUPPORTED;  // test lever: leaves the pair to the implicit GEMM
  const uint64_t plane = static_cast<uint64_t>(d->in_h) * d->in_w;
  if (plane > kMaxImage || d->in_c > 4096 || d->out_h > 4096 || d->out_w > 4096 || d->pad_top > 64 || d->pad_left > 64) return TVX_E_UNSUPPORTED;
  const int cp = (static_cast<int>(d->in_c) + 31) / 32 * 32, taps = static_cast<int>(d->k_w * d->k_h);
  PoolConvArgs a{};
  a.C = d->in_c; a.H = d->in_h; a.W = d->in_w; a.OC = d->out_c; a.OH = d->out_h; a.OW = d->out_w;
  a.sh = d->stride_h; a.sw = d->stride_w; a.pad_t = d->pad_top; a.pad_l = d->pad_left;
  // the cells that windows touch
  const uint64_t rows = static_cast<uint64_t>(a.OH - 1) * a.sh + static_cast<uint64_t>(d->k_h - 1) * d->dilation_h + 1;
  const uint64_t cols = static_cast<uint64_t>(a.OW - 1) * a.sw + static_cast<uint64_t>(d->k_w - 1) * d->dilation_w + 1;
  a.pix_stride = cp + 16;  // (an odd number of 16-byte chunks: a fragment's pixels spread over the banks)
  if (rows > 4096 || cols > 4096) return TVX_E_UNSUPPORTED;
  a.halo_rows = std::max<int>(static_cast<int>(rows), a.H + a.pad_t);
  a.halo_cols = std::max<int>(static_cast<int>(cols), a.W + a.pad_l);
  a.row_stride = a.halo_cols * a.pix_stride;
  const uint64_t image = static_cast<uint64_t>(a.halo_rows) * a.row_stride;
  if (image > static_cast<uint64_t>(kMaxImage) || static_cast<uint64_t>(d->batch) * ((a.OC + 31) / 32) > 0x3fffffffull) return TVX_E_UNSUPPORTED;
  a.padded = a.halo_rows != a.H || a.halo_cols != a.W;
  const auto reciprocal = [](uint64_t v) { return v > 1 ? static_cast<uint32_t>(((1ull << 32) + v - 1) / v) : 0u; };
  a.oc_tiles = (a.OC + 31) / 32;
  const uint64_t pairs = static_cast<uint64_t>(d->batch) * a.oc_tiles;  // of an image and 32 channels
  if (pairs * a.oc_tiles >= (1ull << 32)) return TVX_E_UNSUPPORTED;
  a.m_octiles = reciprocal(a.oc_tiles);
  a.chan_quads = (a.C + 3) / 4; a.col_quads = (a.W + 3) / 4;
  const uint64_t row_units = static_cast<uint64_t>(a.H) * a.col_quads;
  if (row_units * row_units * a.chan_quads >= (1ull << 32)) return TVX_E_UNSUPPORTED;  // (exact reciprocals)
  a.m_units = reciprocal(row_units); a.m_cols = reciprocal(a.col_quads);
  const bool x_u8 = d->in_dtype == TVX_U8, w_u8 = d->w_dtype == TVX_U8;
  const int zxs = d->in_zp - (x_u8 ? 128 : 0), zws = op->w_zp - (w_u8 ? 128 : 0);
  if (zxs < -128 || zxs > 127) return TVX_E_UNSUPPORTED;
  a.xor4 = x_u8 ? 0x80808080u : 0u;
  a.pad_fill4 = static_cast<int>(static_cast<uint32_t>(zxs & 0xff) * 0x01010101u);
  a.per_tap = cp / 32; a.kw = d->k_w;
  a.steps = taps * a.per_tap;
  a.tap_x = static_cast<int>(d->dilation_w) * a.pix_stride;
  a.tap_y = static_cast<int>(d->dilation_h) * a.row_stride;
  a.pw = a.OW / 2; a.pooled = a.pw * (a.OH / 2);
  a.m_pw = reciprocal(a.pw);
  if (static_cast<uint64_t>(a.pooled) * a.pw >= (1ull << 32)) return TVX_E_UNSUPPORTED;
  a.tiles = (4 * a.pooled + 31) / 32;
  a.tile_rows = a.sh + (static_cast<int>(d->k_h) - 1) * static_cast<int>(d->dilation_h) + 1;
  // While there are CUs without one, more workgroups share an image: a wavefront's chain is then shorter. Microseconds, from 3254 launches on
  // 865 drawn layers: per reduction step of a wavefront, per pass over the input's units and per unit loaded. int8, 5 x 5, 32 x 32, before
  // this kernel, with a workgroup an image and here: 3 to 16, batch 2 6.6, 18.9 and 7.3; 16 to 64, batch 31 10.2, 20.4 and 12.4. Of those layers
  // 24 are slower than the implicit GEMM's by more than 3 %, 163 with a workgroup an image; the mean is 0.57 of its time (0.71). What is left are
  // long chains on about as many workgroups as CUs (12 to 21, 32 x 32, batch 150: 11.4 and 19.6), among which more gain, up to six times.
  a.per_group = a.tiles; a.groups = 1;
  {
    const int cus = ComputeUnits();
    double least = 0;
    for (int groups = 1; groups <= a.tiles && (groups == 1 || pairs * groups <= static_cast<uint64_t>(cus)); ++groups) {
      const int per_group = (a.tiles + groups - 1) / groups;
      if (groups > 1 && per_group == (a.tiles + groups - 2) / (groups - 1)) continue;
      const int share = pairs * groups <= static_cast<uint64_t>(cus) ? kMaxWaves : kMaxWaves / 2;
      const int parts = std::max(1, std::min(share / per_group, a.steps)), waves = parts > 1 ? parts * per_group : std::min(kMaxWaves, per_group);
      const double chain = static_cast<double>((a.steps + parts - 1) / parts) * (parts > 1 ? 1 : (per_group + waves - 1) / waves);
      const double units = static_cast<double>(row_units) * a.chan_quads / (64 * waves);
      const double loaded = std::min(1.0, (2.0 * a.sh * (8 * per_group / a.pw + 2) + a.tile_rows) / a.H);
      const double cost = 4.0 + 0.13 * chain + 0.2 * std::ceil(units) + 0.14 * units * loaded;
      if (groups > 1 && cost >= least) continue;
      least = groups > 1 ? cost : 0.95 * cost;
      a.per_group = per_group;
      a.groups = (a.tiles + per_group - 1) / per_group;
    }
  }
  if (const char* f = getenv("TVX_CONV_POOL_GROUPS")) {  // test lever
    a.per_group = (a.tiles + std::max(1, atoi(f)) - 1) / std::max(1, atoi(f));
    a.groups = (a.tiles + a.per_group - 1) / a.per_group;
  }
  const uint64_t wgs = pairs * a.groups;
  if (wgs * a.groups >= (1ull << 32)) return TVX_E_UNSUPPORTED;  // (exact reciprocals)
  a.m_groups = reciprocal(a.groups);
  // few tiles: the reduction is split, so that eight wavefronts share the chain, four where a CU gets more than one workgroup
  // (the layer above: batch 1 6.3 us with one part, 5.3 with two, 4.8 with four; batch 207 8.3, 6.7, 8.4)
  const int share = wgs <= static_cast<uint64_t>(ComputeUnits()) ? kMaxWaves : kMaxWaves / 2;
  a.parts = std::max(1, std::min(share / a.per_group, a.steps));
  if (const char* f = getenv("TVX_CONV_POOL_PARTS")) a.parts = std::max(1, std::min(std::min(atoi(f), kMaxWaves / a.per_group), a.steps));  // test lever
  a.per_part = (a.steps + a.parts - 1) / a.parts;
  a.parts = (a.steps + a.per_part - 1) / a.per_part;
  a.m_parts = reciprocal(a.parts);
  const int waves = a.parts > 1 ? a.parts * a.per_group : std::min(kMaxWaves, a.per_group);
  if (!LaunchFits(wgs, 64 * waves)) return TVX_E_UNSUPPORTED;
  a.z4 = static_cast<int>(static_cast<uint32_t>((zws == -128 ? 64 : -zws) & 0xff) * 0x01010101u);
  a.ztwice = zws == -128;
  a.last_channels = a.C - (a.per_tap - 1) * 32;
  a.off_red = (static_cast<int>(image) + 15) / 16 * 16;
  const int lds_bytes = a.off_red + (a.parts > 1 ? a.per_group * 4096 : 0);
  // ---- weights in fragment order, constants folded into the bias ----
  const int alloc = a.oc_tiles * 32;
  std::vector<int8_t> packed(static_cast<size_t>(a.oc_tiles) * a.steps * 1024, 0);
  std::vector<int32_t> biasf(alloc, 0), rqt;
  const uint8_t* src = static_cast<const uint8_t*>(w_host);
  const int32_t* b = static_cast<const int32_t*>(bias_host);
  for (int oc = 0; oc < a.OC; ++oc) {
    int64_t sum = 0;
    for (int c = 0; c < a.C; ++c)
      for (int t = 0; t < taps; ++t) {
        const uint8_t raw = src[(static_cast<size_t>(oc) * a.C + c) * taps + t];
        const int8_t v = static_cast<int8_t>(w_u8 ? raw ^ 0x80 : raw);
        const int step = t * a.per_tap + c / 32, half = c % 32 / 16;
        packed[((static_cast<size_t>(oc / 32) * a.steps + step) * 64 + half * 32 + oc % 32) * 16 + c % 16] = v;
        sum += v;
      }
    const int64_t v = (b ? b[oc] : 0) - static_cast<int64_t>(zxs) * sum + static_cast<int64_t>(taps) * a.C * zxs * zws;
    biasf[oc] = static_cast<int32_t>(static_cast<uint32_t>(v));
  }
  const int64_t bound = AccumulatorBound(static_cast<uint64_t>(taps) * a.C, bias_host, a.OC);
  const int flip = d->out_dtype == TVX_U8 ? 128 : 0;
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
  Plan plan{};
  plan.a = a;
  plan.lds_bytes = lds_bytes;
  plan.block = 64 * waves;
  plan.grid = static_cast<unsigned>(wgs);
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(ConvPoolKernel), hipFuncAttributeMaxDynamicSharedMemorySize, kMaxImage + 8 * 4096 + 16);
  if (e != hipSuccess) return SetError(TVX_E_DEVICE, "hipFuncSetAttribute(dynamic LDS %d): %s", lds_bytes, hipGetErrorString(e));
  op->host_blob.assign(reinterpret_cast<const uint8_t*>(&plan), reinterpret_cast<const uint8_t*>(&plan) + sizeof(plan));
  op->run = ConvPoolRun;
  op->kernel_name = "conv2d_igemm_maxpool_i8";
  op->variant = "conv2d_pool_i8";
  return TVX_OK;
}

}  // namespace tvx
