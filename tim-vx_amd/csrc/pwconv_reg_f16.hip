// Pointwise (1x1, stride 1, unpadded) float16 Conv2d without a window in LDS: a wavefront keeps all channels of its pixels in registers, as
// pwconv_reg_i8.hip does for bytes.
//
// The float16 MFMA 16x16x32 takes eight consecutive reduction elements per lane. A lane loads PW neighbouring pixels of its eight channels straight
// from their rows (sixteen lanes: one run of 32 * PW bytes per channel), pairs the channels with byte permutes, and the wavefront walks the
// 16-channel output tiles over its pixels with the weights streaming in fragment order (L1 / L2): the input is read once, there is no barrier, and
// results leave as PW neighbouring pixels of four channels a lane, runs of 32 * PW bytes again.
//  - Pixel groups never straddle images: the last group of an image begins at HW - PW and computes some pixels a second time.
//  - KS = 4: inputs of more than 128 channels share the reduction between the four wavefronts of a workgroup, which exchange partial sums through LDS.
//  - Channels that do not exist are zero (their weights are too, but a channel read in their place may hold an infinity).
// Bound by memory where results are many, by the chain load - pair - multiply - store where few. Against the window in LDS (conv_tile.hip) and the
// gathered windows (conv_gemm.hip): 70 drawn layers .63 of the time, none slower: 20 -> 144 on 73 x 128, batch 40, 39.0 -> 21.4 us (122 MB, floor
// 24.5 at a copy's rate), 464 -> 156 on 77 x 110, batch 15, 84 -> 40, 416 -> 48 on 39 x 39, batch 24, 17.6 -> 9.8. 191 layers of at most 576 pixels .59 (56 ->
// 382 on 6 x 6 7.2 -> 2.5; the slowest 848 -> 8 on 12 pixels, batch 13, 5.7 -> 5.8), 110 of at most 16 results from at most 64 channels on planes of
// whole 16 pixels .42 (16 -> 8 on 88 x 88, batch 8, 3.9 -> 3.1; 64 -> 6 on 15200 pixels, batch 20, 162 by a thread per output, 8.4).
// Reference: src/tim/vx/ops/conv2d.cc (1x1 kernels).
#include <algorithm>
#include <cstdlib>
#include <cstring>

#include "variants.h"

namespace tvx {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));

constexpr int kStep = 32;  // channels of a reduction step, eight a lane

struct PwfArgs {
  const _Float16* x;
  _Float16* y;
  const v4i* wpk;        // [16-channel tile][step][lane]: eight channels of output channel tile * 16 + lane % 16
  const float* bias;     // per padded output channel
  uint32_t C, OC, HW;
  uint32_t groups;       // batch * groups per image
  uint32_t per_image, m_per_image;
  int ksteps;
  int tiles, tiles_per_wave;  // 16-channel output tiles
  uint32_t tile_groups, m_tile_groups, units;  // pixel tiles x tile groups
  int act;
};

__device__ __forceinline__ uint32_t DivM(uint32_t u, uint32_t m) { return m ? __umulhi(u, m) : u; }

// PW: pixels of a lane (8: 128 pixels a wavefront; 4: 64). KR: steps of a wavefront. KS: wavefronts that share a reduction (4), or 1.
template <int PW, int KR, int KS>
__global__ void __launch_bounds__(256, 2) PwRegF16Kernel(PwfArgs a) {
  constexpr int kDw = PW / 2;  // dwords of a lane's pixels
  __shared__ v4f part[KS > 1 ? 4 * 4 * 64 : 1];
  const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // each XCD a contiguous run of units: neighbouring pixel tiles share cache lines, tile groups of a pixel tile their input
  uint32_t wg = blockIdx.x;
  {
    const uint32_t per = gridDim.x >> 3, rem = gridDim.x & 7, xcd = wg & 7;
    wg = xcd * per + min(xcd, rem) + (wg >> 3);
  }
  const uint32_t unit = KS > 1 ? wg : wg * (blockDim.x >> 6) + wave;
  if (unit >= a.units) return;
  const uint32_t pix_tile = DivM(unit, a.m_tile_groups);
  const int t0 = static_cast<int>(unit - pix_tile * a.tile_groups) * a.tiles_per_wave;
  const int t1 = min(t0 + a.tiles_per_wave, a.tiles);
  const int k0 = KS > 1 ? wave * KR : 0;

  // ---- weights and bias of the first output tile; pixels ----
  auto frag = [&](int t, int k) { return a.wpk[(static_cast<uint32_t>(t) * a.ksteps + (k0 + k)) * 64 + lane]; };
  v4i w[KR];
#pragma unroll
  for (int k = 0; k < KR; ++k) w[k] = frag(t0, k);
  // (four consecutive channels, or the one this wavefront finishes)
  auto bias_of = [&](int t) { return KS == 1 ? *reinterpret_cast<const v4f*>(a.bias + t * 16 + g * 4) : v4f{a.bias[t * 16 + g * 4 + wave], 0.f, 0.f, 0.f}; };
  v4f bias = bias_of(t0);
  const uint32_t grp = min(pix_tile * 16 + n, a.groups - 1);
  const uint32_t image = DivM(grp, a.m_per_image), gi = grp - image * a.per_image;
  const uint32_t p = min(gi * PW, a.HW - PW);
  v4i b[KR][PW];
  {
    const int channel0 = k0 * kStep + g * 8;  // this lane's first channel; its steps are 32 apart
    const uint32_t at = (image * a.C + channel0) * a.HW + p;
    uint32_t raw[KR][8][kDw];
#pragma unroll
    for (int k = 0; k < KR; ++k) {
      const int left = static_cast<int>(a.C) - (channel0 + k * kStep);  // channels of this lane that exist
#pragma unroll
      for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int d = 0; d < kDw; ++d) raw[k][j][d] = 0;
      if (left > 0) {
        const uint32_t first = at + static_cast<uint32_t>(k * kStep) * a.HW, last = first + static_cast<uint32_t>(left - 1) * a.HW;
#pragma unroll
        for (int j = 0; j < 8; ++j) __builtin_memcpy(raw[k][j], a.x + min(first + static_cast<uint32_t>(j) * a.HW, last), 2 * PW);
      }
    }
    __builtin_amdgcn_sched_barrier(0);  // all of them in flight before the first is used
    if (a.C & 7)  // uniform: a lane's eight channels may end among them
#pragma unroll
      for (int k = 0; k < KR; ++k) {
        const int left = static_cast<int>(a.C) - (channel0 + k * kStep);
#pragma unroll
        for (int j = 0; j < 8; ++j)
#pragma unroll
          for (int d = 0; d < kDw; ++d) raw[k][j][d] = j < left ? raw[k][j][d] : 0u;
      }
#pragma unroll
    for (int k = 0; k < KR; ++k)
#pragma unroll
      for (int j = 0; j < PW; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          b[k][j][q] = static_cast<int>(__builtin_amdgcn_perm(raw[k][2 * q + 1][j / 2], raw[k][2 * q][j / 2], j & 1 ? 0x07060302 : 0x05040100));
  }

  const uint32_t out_at = (image * a.OC + g * 4) * a.HW + p;
  auto emit = [&](const float (&v)[PW], int t, int i) {  // PW pixels of channel 4 g + i of a tile
    if (t * 16 + g * 4 + i >= static_cast<int>(a.OC)) return;
    _Float16 h[PW];
#pragma unroll
    for (int j = 0; j < PW; ++j) {
      float r = v[j];
      if (a.act != TVX_ACT_NONE) r = r < 0.f ? 0.f : r;  // uniform
      if (a.act == TVX_ACT_RELU6) r = r > 6.f ? 6.f : r;
      h[j] = static_cast<_Float16>(r);
    }
    __builtin_memcpy(a.y + (out_at + static_cast<uint32_t>(t * 16 + i) * a.HW), h, 2 * PW);
  };
  for (int t = t0; t < t1; ++t) {
    v4f acc[PW];
#pragma unroll
    for (int j = 0; j < PW; ++j) acc[j] = KS > 1 ? v4f{0.f, 0.f, 0.f, 0.f} : bias;
#pragma unroll
    for (int k = 0; k < KR; ++k)
#pragma unroll
      for (int j = 0; j < PW; ++j)
        acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, w[k]), __builtin_bit_cast(v8h, b[k][j]), acc[j], 0, 0, 0);
    // the next tile's weights travel while this one's results are stored
    const int tn = min(t + 1, t1 - 1);
#pragma unroll
    for (int k = 0; k < KR; ++k) w[k] = frag(tn, k);
    const float mine = bias[0];
    bias = bias_of(tn);
    if constexpr (KS == 1) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float v[PW];
#pragma unroll
        for (int j = 0; j < PW; ++j) v[j] = acc[j][i];
        emit(v, t, i);
      }
    } else {
      static_assert(KS == 1 || PW == 4, "the exchange moves four pixels");
      if (t > t0) __syncthreads();
#pragma unroll
      for (int i = 0; i < 4; ++i) part[(wave * 4 + i) * 64 + lane] = v4f{acc[0][i], acc[1][i], acc[2][i], acc[3][i]};
      __syncthreads();
      v4f s = part[wave * 64 + lane];  // this wavefront finishes channels 4 g + wave
#pragma unroll
      for (int o = 1; o < 4; ++o) s += part[(o * 4 + wave) * 64 + lane];
      float v[PW];
#pragma unroll
      for (int j = 0; j < PW; ++j) v[j] = s[j & 3] + mine;
      emit(v, t, wave);
    }
  }
}

typedef void (*PwfFn)(PwfArgs);
struct Plan {
  PwfArgs a;
  PwfFn fn;
  unsigned grid, block;
};

int PwRegF16Run(tvx_op* op, const void* in0, const void*, void* out, hipStream_t st) {
  const Plan& p = *reinterpret_cast<const Plan*>(op->host_blob.data());
  if ((reinterpret_cast<uintptr_t>(in0) | reinterpret_cast<uintptr_t>(out)) & 1) return SetError(TVX_E_INVALID, "pwconv_reg_f16: tensors must be aligned to their elements");
  PwfArgs a = p.a;
  a.x = static_cast<const _Float16*>(in0);
  a.y = static_cast<_Float16*>(out);
  hipLaunchKernelGGL(p.fn, dim3(p.grid), dim3(p.block), 0, st, a);
  TVX_HIP_CHECK(hipGetLastError());
  return TVX_OK;
}

uint32_t Magic(uint64_t d) { return d <= 1 ? 0u : static_cast<uint32_t>(((uint64_t{1} << 32) + d - 1) / d); }

}  // namespace

// Claims dense float16 1x1 convolutions with unit stride, no padding and constant weights of up to 1024 channels on planes of eight pixels and more.
int PwRegF16Setup(tvx_op* op, const tvx_conv2d_desc* d, const void* w_host, const void* bias_host) {
  if (op->kind != OP_CONV2D || !w_host || d->multiplier != 0 || d->groups > 1 || op->fused_add || op->fused_pool) return TVX_E_UNSUPPORTED;
  if (d->in_dtype != TVX_F16 || d->w_dtype != TVX_F16 || d->out_dtype != TVX_F16) return TVX_E_UNSUPPORTED;
  if (d->k_w != 1 || d->k_h != 1 || d->stride_w != 1 || d->stride_h != 1 || d->pad_left != 0 || d->pad_top != 0 || d->out_w != d->in_w || d->out_h != d->in_h)
    return TVX_E_UNSUPPORTED;
  const uint64_t hw = static_cast<uint64_t>(d->in_w) * d->in_h, pixels = hw * d->batch;
  if (hw < 8 || pixels * d->in_c + (hw << 11) >= (1ull << 32) || pixels * d->out_c + (hw << 6) >= (1ull << 32)) return TVX_E_UNSUPPORTED;  // 32-bit offsets
  const uint32_t C = d->in_c, OC = d->out_c;
  const int tiles = static_cast<int>((OC + 15) / 16), ksteps = static_cast<int>((C + kStep - 1) / kStep);
  // Up to 128 channels (128 registers) in one wavefront. Four share the reduction of more, and of as many where the results are few: their loads are
  // most of such a launch, and half as many pixels each. In pieces of 64 pixels x 16 results the two cross at about 900 for every step: 64 -> 32 on
  // 42 x 42, batch 12, 660 pieces, 3.7 us shared and 4.0 not; 8 -> 48 on 90 x 90, batch 5, 1900, 4.8 and 4.2; 128 -> 400 on 45 x 83, batch 2, 2900, 7.8
  // and 8.6; 64 -> 96 on 29 x 29, batch 61, 4800, 8.9 and 7.8.
  const uint64_t cus = ComputeUnits(), pieces = (pixels + 63) / 64 * tiles;
  int ks = ksteps <= 4 && 2 * pieces > 7 * cus * ksteps ? 1 : 4;
  if (const char* f = getenv("TVX_PWCONV_F16")) {  // test lever: wavefronts that share a reduction; 0 declines
    ks = atoi(f);
    if ((ks != 1 && ks != 4) || (ks == 1 && ksteps > 4)) return TVX_E_UNSUPPORTED;
  }
  const int pw = ks == 1 ? 8 : 4;
  int kr = (ksteps + ks - 1) / ks;
  if (kr > 8) return TVX_E_UNSUPPORTED;
  if (kr > 4) kr = kr <= 6 ? 6 : 8;
  Plan plan{};
  PwfArgs& a = plan.a;
  if (ks == 1) plan.fn = kr == 1 ? PwRegF16Kernel<8, 1, 1> : kr == 2 ? PwRegF16Kernel<8, 2, 1> : kr == 3 ? PwRegF16Kernel<8, 3, 1> : PwRegF16Kernel<8, 4, 1>;
  else plan.fn = kr == 1 ? PwRegF16Kernel<4, 1, 4> : kr == 2 ? PwRegF16Kernel<4, 2, 4> : kr == 3 ? PwRegF16Kernel<4, 3, 4> : kr == 4 ? PwRegF16Kernel<4, 4, 4>
                 : kr == 6 ? PwRegF16Kernel<4, 6, 4> : PwRegF16Kernel<4, 8, 4>;
  a.C = C; a.OC = OC; a.HW = static_cast<uint32_t>(hw);
  const uint64_t per_image = (hw + pw - 1) / pw, groups = per_image * d->batch;
  if (groups * per_image >= (1ull << 32)) return TVX_E_UNSUPPORTED;
  a.per_image = static_cast<uint32_t>(per_image);
  a.m_per_image = Magic(per_image);
  a.groups = static_cast<uint32_t>(groups);
  a.ksteps = kr * ks;  // (steps past the last channel: zero weights)
  a.tiles = tiles;
  a.act = d->activation;
  // pixel tiles fill the chip, or the output tiles of each are spread over wavefronts: two a SIMD, four where that reads at most 32 channels again
  // (16 -> 160 on 57 x 85, batch 36: 18.1 us and 14.5; 64 -> 96 on 29 x 29, batch 61: 7.6 and 8.5). Four as well of up to 96 channels
  // where two would leave the SIMDs with one, if there are four output tiles to spread: 16 drawn layers of 1050 to 1841 pixel tiles .88 of the time, none
  // slower (64 -> 344 on 139 x 139, batch 8, 33.4 us and 25.5; 92 -> 64 on 105 x 160, batch 8, 12.4 and 11.3); of 512 to 1024 pixel tiles .91 to 1.16
  // (64 -> 160 on 147 x 147, batch 6, 13.5 and 15.7), of fewer output tiles to 1.2 (80 -> 48 on 99 x 99, batch 14, 9.8 and 11.7).
  const uint64_t pix_tiles = (groups + 15) / 16;
  const bool four = kr == 1 || (kr <= 3 && tiles >= 4 && pix_tiles > 4 * cus);
  uint64_t want = cus * (ks > 1 ? (kr > 4 ? 1 : kr > 2 ? 2 : 4) : four ? 16 : 8);
  if (const char* f = getenv("TVX_PWCONV_F16_WAVES")) want = std::max(1, atoi(f));  // test lever
  const uint64_t split = std::min<uint64_t>(tiles, std::max<uint64_t>(1, want / pix_tiles));
  a.tiles_per_wave = static_cast<int>((tiles + split - 1) / split);
  a.tile_groups = static_cast<uint32_t>((tiles + a.tiles_per_wave - 1) / a.tiles_per_wave);
  a.m_tile_groups = Magic(a.tile_groups);
  const uint64_t units = pix_tiles * a.tile_groups;
  if (units * a.tile_groups >= (1ull << 32)) return TVX_E_UNSUPPORTED;
  a.units = static_cast<uint32_t>(units);
  const unsigned waves = ks > 1 ? 1 : units >= 4096 ? 4 : 1;
  plan.block = ks > 1 ? 256 : 64 * waves;
  plan.grid = static_cast<unsigned>((units + waves - 1) / waves);
  if (!LaunchFits(plan.grid, plan.block)) return TVX_E_UNSUPPORTED;

  // ---- weights in fragment order ----
  std::vector<uint16_t> packed(static_cast<size_t>(tiles) * a.ksteps * 64 * 8, 0);
  std::vector<float> bias(static_cast<size_t>(tiles) * 16, 0.f);
  const uint16_t* src = static_cast<const uint16_t*>(w_host);
  for (uint32_t oc = 0; oc < OC; ++oc)
    for (uint32_t c = 0; c < C; ++c)
      packed[((static_cast<size_t>(oc / 16) * a.ksteps + c / kStep) * 64 + c / 8 % 4 * 16 + oc % 16) * 8 + c % 8] = src[static_cast<size_t>(oc) * C + c];
  if (bias_host) std::memcpy(bias.data(), bias_host, static_cast<size_t>(OC) * 4);
  int s = op->packed.Upload(packed.data(), packed.size() * 2);
  if (s == TVX_OK) s = op->aux.Upload(bias.data(), bias.size() * 4);
  if (s != TVX_OK) return s;
  a.wpk = op->packed.as<v4i>();
  a.bias = op->aux.as<float>();
  op->host_blob.assign(reinterpret_cast<const uint8_t*>(&plan), reinterpret_cast<const uint8_t*>(&plan) + sizeof(plan));
  op->run = PwRegF16Run;
  op->kernel_name = "pwconv_reg_f16";
  return TVX_OK;
}

}  // namespace tvx
