// Pointwise (1x1, stride 1, unpadded) quantized Conv2d without LDS: a wavefront keeps all channels of its pixels in registers.
//
// The int8 MFMA 16x16x64 takes sixteen consecutive reduction bytes per lane. A lane loads PW neighbouring pixels of its sixteen
// channels straight from their rows (sixteen lanes: one run of 16 * PW bytes per channel), turns them into PW operands with byte
// permutes, and that is the whole input side: the wavefront walks the 16-channel output tiles over them with the weights streaming
// in fragment order (L1 / L2), so the input is read once and there is no barrier. Results come out as PW neighbouring pixels of
// four channels a lane and are stored as they are, again runs of 16 * PW bytes.
//  - Pixel groups never straddle images: the last group of an image begins at HW - PW and computes some pixels a second time
//    (the same values to the same addresses; with an Add, stored once), so that there are no partial groups at any HW >= PW.
//  - KS = 4: inputs that are deep (or whose pixels are few) share the reduction between the four wavefronts of a workgroup, which
//    exchange partial sums through LDS.
//  - Lanes load the channels that exist and no others; inputs of at most 32 take steps of 32 channels instead of 64. All lanes
//    loading 64 channels fetched the next image's rows with these: 32 x 32 x 112 x 112 -> 64 channels 15.5 -> 13.5 us, 64 x 32 x 112 x
//    112 -> 16 12.8 -> 10.9, 64 x 32 x 28 x 28 -> 192 7.5 -> 6.6, 12 x 12 x 150 x 150 -> 12 5.7 -> 4.6 (buffers in rotation).
//  - Zero points: sum (x - zx)(w - zw) = sum xs ws - zws Sx - zxs Sw + C zxs zws with xs, ws moved to the signed domain; Sx is one
//    more MFMA against a constant fragment per pixel tile, the per-channel constants are folded into the bias.
// Bound by memory; what is left above it is the launch, whose wavefronts load, compute and store at about the same time. Against
// the form that stages pixels in LDS (pwconv_i8.hip): 36 x 80 x 117 x 132 -> 40 channels 31.4 -> 17.0 us (66.7 MB, floor 13),
// 32 x 256 x 28 x 28 -> 256 10.4 -> 7.8 us, 2 x 48 x 114 x 114 -> 352 9.7 -> 6.1 us, 960 x 7 x 7 -> 320 7.7 -> 4.4 us.
// Reference: src/tim/vx/ops/conv2d.cc (1x1 kernels).
#include <algorithm>
#include <cstdlib>
#include <type_traits>

#include "variants.h"

namespace tvx {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v2i __attribute__((ext_vector_type(2)));

struct PwrArgs {
  const uint8_t* x;
  uint8_t* y;
  const uint8_t* wpk;    // [16-channel tile][step of 4 KL channels][lane]: KL reduction bytes of channel tile * 16 + lane % 16
  const v4i* rec;        // per channel {multiplier, shift, rounding constant, folded bias}
  uint32_t C, OC, HW;
  uint32_t groups;       // batch * groups per image
  uint32_t per_image, m_per_image;  // pixel groups of an image, and their reciprocal
  int ksteps;
  int tiles, tiles_per_wave;  // 16-channel output tiles
  uint32_t tile_groups, m_tile_groups, units;  // pixel tiles x tile groups
  int xor_mask;          // 0x80808080 for uint8 activations
  int neg_zws4;          // -(weight zero point, int8 domain) in all four bytes
  int lo, hi;            // output clamp in the signed domain
  int plain_tiles;       // the first so many output tiles need no masks, clamps or ties
  int out_xor;           // 0x80808080 for uint8 results
  int pre_ties;          // accumulators' left shift (BuildTieRecords) * 2 + whether ties are possible
};
struct PwrAdd {          // the quantized Add behind it (AddResidual4)
  const uint8_t* res;
  double add_ra, add_rb;
  int add_mode, add_signed, add_za, add_zb, add_zo, add_lo, add_hi;
};
struct PwrNoAdd {};

__device__ __forceinline__ uint32_t DivM(uint32_t u, uint32_t m) { return m ? __umulhi(u, m) : u; }

__device__ __forceinline__ v4i Multiply(const v4i& w, const v4i& x, const v4i& acc) { return __builtin_amdgcn_mfma_i32_16x16x64_i8(w, x, acc, 0, 0, 0); }
__device__ __forceinline__ v4i Multiply(const v2i& w, const v2i& x, const v4i& acc) {
  return __builtin_amdgcn_mfma_i32_16x16x32_i8(__builtin_bit_cast(long, w), __builtin_bit_cast(long, x), acc, 0, 0, 0);
}

// PW: pixels of a lane (8: 128 pixels a wavefront; 4: 64, for deep inputs and few pixels). KL: channels of a lane and step (16; 8 for
// inputs of at most 32 channels, half the bytes and half the transposition). KR: steps of a wavefront (4 KL channels each).
// KS: wavefronts that share a reduction (4), or 1.
template <int PW, int KL, int KR, int KS, class ADD>
__global__ void __launch_bounds__(256, 2) PwRegKernel(PwrArgs a, ADD add) {
  constexpr int kDw = PW / 4;  // dwords of a lane's pixels
  using frag_t = std::conditional_t<KL == 16, v4i, v2i>;
  __shared__ v4i part[KS > 1 ? 4 * 4 * 64 : 1];
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

  // ---- weights and tables of the first output tile; pixels ----
  auto frag = [&](int t, int k) { return reinterpret_cast<const frag_t*>(a.wpk)[(static_cast<uint32_t>(t) * a.ksteps + (k0 + k)) * 64 + lane]; };
  frag_t w[KR];
  v4i q[4];
#pragma unroll
  for (int k = 0; k < KR; ++k) w[k] = frag(t0, k);
  auto records = [&](int t) {
#pragma unroll
    for (int i = 0; i < 4; ++i) q[i] = a.rec[t * 16 + g * 4 + i];
  };
  if (KS == 1) records(t0);
  else q[0] = a.rec[t0 * 16 + g * 4 + wave];
  const uint32_t grp = min(pix_tile * 16 + n, a.groups - 1);
  const uint32_t image = DivM(grp, a.m_per_image), gi = grp - image * a.per_image;
  const uint32_t p = min(gi * PW, a.HW - PW);
  const uint32_t twice = gi * PW - p;  // pixels that the group before it computes too
  uint32_t raw[KR][KL][kDw];
  const int channel0 = k0 * 4 * KL + g * KL;  // this lane's first channel; its steps are 4 KL apart
  {
    // lanes whose channels do not exist load nothing; past the input's last channel it is read again. Both meet zero weights.
    const uint32_t at = (image * a.C + channel0) * a.HW + p;
#pragma unroll
    for (int k = 0; k < KR; ++k) {
      const int left = static_cast<int>(a.C) - (channel0 + k * 4 * KL);
#pragma unroll
      for (int j = 0; j < KL; ++j)
#pragma unroll
        for (int d = 0; d < kDw; ++d) raw[k][j][d] = 0;
      if (left > 0) {
        const uint32_t first = at + static_cast<uint32_t>(k * 4 * KL) * a.HW, last = first + static_cast<uint32_t>(left - 1) * a.HW;
#pragma unroll
        for (int j = 0; j < KL; ++j) __builtin_memcpy(raw[k][j], a.x + min(first + static_cast<uint32_t>(j) * a.HW, last), PW);
      }
    }
  }
  __builtin_amdgcn_sched_barrier(0);  // all of them in flight before the first is used
  frag_t b[KR][PW];
#pragma unroll
  for (int k = 0; k < KR; ++k)
#pragma unroll
    for (int d = 0; d < kDw; ++d)
#pragma unroll
      for (int c = 0; c < KL / 4; ++c) {
        uint32_t in[4], t[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) in[j] = raw[k][c * 4 + j][d] ^ a.xor_mask;
        Transpose4x4(in, t);
#pragma unroll
        for (int e = 0; e < 4; ++e) b[k][d * 4 + e][c] = static_cast<int>(t[e]);
      }
  // -zws * (sum over the channels), the same for every output channel: one register a pixel tile
  int z[PW];
#pragma unroll
  for (int j = 0; j < PW; ++j) z[j] = 0;
  if (a.neg_zws4) {
#pragma unroll
    for (int j = 0; j < PW; ++j) {
      v4i acc = {0, 0, 0, 0};
#pragma unroll
      for (int k = 0; k < KR; ++k) {
        const int left = static_cast<int>(a.C) - (channel0 + k * 4 * KL);  // channels of this lane that exist
        frag_t f;
#pragma unroll
        for (int c = 0; c < KL / 4; ++c) {
          const int bytes = min(max(left - c * 4, 0), 4);
          f[c] = bytes == 4 ? a.neg_zws4 : a.neg_zws4 & ((1 << (8 * bytes)) - 1);
        }
        acc = Multiply(f, b[k][j], acc);
      }
      z[j] = acc[0];
    }
  }

  const uint32_t out_at = (image * a.OC + g * 4) * a.HW + p;
  // A tile of output channels. Plain: all of them exist, no accumulator can land on a tie, the clamp is a byte's: straight code.
  auto tile = [&](const int t, auto plain) {
    constexpr bool kPlain = decltype(plain)::value;
    v4i acc[PW];
    const v4i bias = {q[0][3], q[1][3], q[2][3], q[3][3]};
#pragma unroll
    for (int j = 0; j < PW; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[j][i] = KS > 1 ? z[j] : bias[i] + z[j];
#pragma unroll
    for (int k = 0; k < KR; ++k)
#pragma unroll
      for (int j = 0; j < PW; ++j) acc[j] = Multiply(w[k], b[k][j], acc[j]);
    // the next tile's weights and records travel during this one's requantization
    const int tn = min(t + 1, t1 - 1);
    v4i r[4] = {q[0], q[1], q[2], q[3]};
#pragma unroll
    for (int k = 0; k < KR; ++k) w[k] = frag(tn, k);
    if (KS == 1) records(tn);
    else q[0] = a.rec[tn * 16 + g * 4 + wave];
    const uint32_t row0 = out_at + static_cast<uint32_t>(t) * 16 * a.HW;
    // codes of channel 4 g + i: PW accumulators -> kDw dwords -> memory
    auto emit = [&](int (&v)[PW], const v4i& rq, int i) {
      if (!kPlain && a.pre_ties) {
#pragma unroll
        for (int j = 0; j < PW; ++j) v[j] <<= a.pre_ties >> 1;
        if (a.pre_ties & 1) LowerOddTies(v, rq);
      }
      const int sh = rq[1] & 31;
      const int64_t round = RoundHigh(rq[2]);
      const int lo_t = a.lo << sh, hi_t = ((a.hi + 1) << sh) - 1;
      uint32_t o[kDw];
      const uint32_t at = row0 + static_cast<uint32_t>(i) * a.HW;
#pragma unroll
      for (int d = 0; d < kDw; ++d) {
        const int v4[4] = {v[d * 4], v[d * 4 + 1], v[d * 4 + 2], v[d * 4 + 3]};
        o[d] = RequantSaturate4<!kPlain>(v4, rq[0], sh, round, lo_t, hi_t) ^ a.out_xor;
      }
      if (!kPlain && t * 16 + g * 4 + i >= static_cast<int>(a.OC)) return;
      if constexpr (!std::is_same<ADD, PwrNoAdd>::value) {
        uint32_t res[kDw];
        __builtin_memcpy(res, add.res + at, PW);
#pragma unroll
        for (int d = 0; d < kDw; ++d) o[d] = AddResidual4(add, o[d], res[d]);
      }
      if constexpr (!std::is_same<ADD, PwrNoAdd>::value) {
        if (twice) {  // (the result may be written over the Add's other operand: a pixel is stored once)
          for (int e = static_cast<int>(twice); e < PW; ++e) a.y[at + e] = static_cast<uint8_t>(o[e / 4] >> (8 * (e & 3)));
          return;
        }
      }
      __builtin_memcpy(a.y + at, o, PW);
    };
    if constexpr (KS == 1) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        int v[PW];
#pragma unroll
        for (int j = 0; j < PW; ++j) v[j] = acc[j][i];
        emit(v, r[i], i);
      }
    } else {
      static_assert(KS == 1 || PW == 4, "the exchange moves four pixels");
      if (t > t0) __syncthreads();
#pragma unroll
      for (int i = 0; i < 4; ++i) part[(wave * 4 + i) * 64 + lane] = v4i{acc[0][i], acc[1][i], acc[2][i], acc[3][i]};
      __syncthreads();
      v4i s = part[wave * 64 + lane];  // this wavefront finishes channels 4 g + wave
#pragma unroll
      for (int o = 1; o < 4; ++o) s += part[(o * 4 + wave) * 64 + lane];
      int v[PW];
#pragma unroll
      for (int j = 0; j < PW; ++j) v[j] = s[j & 3] + r[0][3];
      emit(v, r[0], wave);
    }
  };
  const int straight = min(t1, a.plain_tiles);
  int t = t0;
  for (; t < straight; ++t) tile(t, std::true_type{});
  for (; t < t1; ++t) tile(t, std::false_type{});
}

struct Plan {
  PwrArgs a;
  PwrAdd add;
  int kl, kr, ks;
  unsigned grid, block;
};

template <int PW, int KL, int KR, int KS>
void Launch(const Plan& p, const PwrArgs& a, const void* res, hipStream_t st) {
  if (p.add.add_mode) {
    PwrAdd add = p.add;
    add.res = static_cast<const uint8_t*>(res);
    hipLaunchKernelGGL((PwRegKernel<PW, KL, KR, KS, PwrAdd>), dim3(p.grid), dim3(p.block), 0, st, a, add);
  } else {
    hipLaunchKernelGGL((PwRegKernel<PW, KL, KR, KS, PwrNoAdd>), dim3(p.grid), dim3(p.block), 0, st, a, PwrNoAdd{});
  }
}

int PwRegRun(tvx_op* op, const void* in0, const void* in1, void* out, hipStream_t st) {
  const Plan& p = *reinterpret_cast<const Plan*>(op->host_blob.data());
  if (p.add.add_mode && !in1) return SetError(TVX_E_INVALID, "pwconv_reg_add_i8: the fused Add needs its second operand as in1");
  PwrArgs a = p.a;
  a.x = static_cast<const uint8_t*>(in0);
  a.y = static_cast<uint8_t*>(out);
  switch (p.kl == 8 ? 0 : p.ks * 10 + p.kr) {
    case 0: Launch<8, 8, 1, 1>(p, a, in1, st); break;
    case 11: Launch<8, 16, 1, 1>(p, a, in1, st); break;
    case 12: Launch<8, 16, 2, 1>(p, a, in1, st); break;
    case 13: Launch<8, 16, 3, 1>(p, a, in1, st); break;
    case 14: Launch<8, 16, 4, 1>(p, a, in1, st); break;
    case 41: Launch<4, 16, 1, 4>(p, a, in1, st); break;
    case 42: Launch<4, 16, 2, 4>(p, a, in1, st); break;
    case 43: Launch<4, 16, 3, 4>(p, a, in1, st); break;
    case 44: Launch<4, 16, 4, 4>(p, a, in1, st); break;
    case 46: Launch<4, 16, 6, 4>(p, a, in1, st); break;
    default: Launch<4, 16, 8, 4>(p, a, in1, st);
  }
  TVX_HIP_CHECK(hipGetLastError());
  return TVX_OK;
}

uint32_t Magic(uint64_t d) { return d <= 1 ? 0u : static_cast<uint32_t>(((uint64_t{1} << 32) + d - 1) / d); }

}  // namespace

// Claims dense quantized 1x1 convolutions with unit stride, no padding and constant weights.
int PwRegSetup(tvx_op* op, const tvx_conv2d_desc* d, const void* w_host, const void* bias_host) {
  if (!op->quantized || !w_host || d->multiplier != 0 || d->groups > 1 || op->out_blocked || op->fused_pool) return TVX_E_UNSUPPORTED;
  if (d->k_w != 1 || d->k_h != 1 || d->stride_w != 1 || d->stride_h != 1 || d->pad_left != 0 || d->pad_top != 0 || d->out_w != d->in_w ||
      d->out_h != d->in_h)
    return TVX_E_UNSUPPORTED;
  const uint64_t hw = static_cast<uint64_t>(d->in_w) * d->in_h;
  const uint64_t in_bytes = hw * d->in_c * d->batch, out_bytes = hw * d->out_c * d->batch;
  if (hw < 4 || in_bytes + (hw << 11) >= (1ull << 32) || out_bytes + (hw << 6) >= (1ull << 32)) return TVX_E_UNSUPPORTED;  // 32-bit offsets
  const bool x_u8 = d->in_dtype == TVX_U8, w_u8 = d->w_dtype == TVX_U8;
  const int zxs = d->in_zp - (x_u8 ? 128 : 0), zws = op->w_zp - (w_u8 ? 128 : 0);
  if (zxs < -128 || zxs > 127 || zws < -127 || zws > 127) return TVX_E_UNSUPPORTED;
  const uint32_t C = d->in_c, OC = d->out_c;
  const int out_flip = d->out_dtype == TVX_U8 ? 128 : 0;
  std::vector<int32_t> rqt;
  const int tiles = static_cast<int>((OC + 15) / 16), ksteps = static_cast<int>((C + 63) / 64);
  int pre;
  bool ties;
  if (!BuildTieRecords(op->h_mult, op->h_shift, OC, tiles * 16, d->out_zp - out_flip, AccumulatorBound(C, bias_host, OC), &rqt, &pre, &ties)) return TVX_E_UNSUPPORTED;

  Plan plan{};
  PwrArgs& a = plan.a;
  // up to 256 channels (128 registers) in one wavefront; deeper inputs would leave too few wavefronts in flight: 16 x 14 x 14 pixels,
  // 512 -> 512 channels, 9.4 us with the reduction in one, 6.0 us shared by four (old form 6.8)
  int ks = hw >= 8 && ksteps <= 4 ? 1 : 4;
  // ... and so do inputs of 65 to 256 channels where the results are few: a wavefront's loads, one step after the other, are most of such
  // a launch. 7 x 19 x 19 pixels, 224 -> 256 channels: 5.6 us in one wavefront, 4.2 shared (5.2 staged in LDS); 4 x 18 x 18, 246 -> 24: 4.3,
  // 3.0 (4.1); 64 x 7 x 7, 160 -> 960: 7.8, 7.3 (7.4). With more, the four wavefronts' exchange costs more than the shorter chain gives: over
  // 200 drawn layers the two cross at about 1600 pieces of 64 pixels x 16 results for two steps and as many again for every further one
  // (17 x 29 x 29, 65 -> 186, 2700 pieces: 3 % slower shared; 13 x 52 x 52, 208 -> 80, 2750 pieces: 10 % faster).
  const uint64_t cus = ComputeUnits(), pieces = (((hw + 3) / 4) * d->batch + 15) / 16 * tiles;
  if (ksteps > 1 && ksteps <= 4 && 4 * pieces <= 25 * cus * (ksteps - 1)) ks = 4;
  if (const char* f = getenv("TVX_PWCONV_REG")) {  // tuning / test aid: wavefronts that share a reduction; 0 = off
    ks = atoi(f);
    if ((ks != 1 && ks != 4) || (ks == 1 && (hw < 8 || ksteps > 4))) return TVX_E_UNSUPPORTED;
  }
  const int pw = ks == 1 ? 8 : 4;
  int kr = (ksteps + ks - 1) / ks;
  if (kr > 8) return TVX_E_UNSUPPORTED;
  if (kr > 4) kr = kr <= 6 ? 6 : 8;
  const int kl = ks == 1 && C <= 32 ? 8 : 16;
  plan.kl = kl;
  plan.ks = ks;
  plan.kr = kr;
  a.C = C;
  a.OC = OC;
  a.HW = static_cast<uint32_t>(hw);
  const uint64_t per_image = (hw + pw - 1) / pw, groups = per_image * d->batch;
  if (groups * per_image >= (1ull << 32)) return TVX_E_UNSUPPORTED;
  a.per_image = static_cast<uint32_t>(per_image);
  a.m_per_image = Magic(per_image);
  a.groups = static_cast<uint32_t>(groups);
  const int ksteps_alloc = kr * ks;  // (steps past the last channel: zero weights)
  a.ksteps = ksteps_alloc;
  a.tiles = tiles;
  // pixel tiles fill the chip, or the output tiles of each are spread over wavefronts: two wavefronts a SIMD, or one where every
  // further one reads more than 64 channels again (64 x 7 x 7 pixels, 960 -> 320 channels: 512 workgroups 9.2 us, 256 7.2 us), four
  // where that is at most 32 (64 x 56 x 56 pixels, 32 -> 128 channels: 1568 wavefronts 13.7 us, 3136 12.8, 6272 14.2) - short of four, since
  // pixel tiles that make two wavefronts a SIMD as they are stay whole (19 x 116 x 116, 14 -> 80: 1998 wavefronts 10.8 us, 3996 11.5)
  const uint64_t pix_tiles = (groups + 15) / 16;
  uint64_t want = cus * (ks > 1 ? (ksteps > 8 ? 1 : ksteps > 4 ? 2 : 4) : (ksteps > 1 ? 4 : kl == 16 ? 8 : 14));
  if (const char* f = getenv("TVX_PWCONV_REG_WAVES")) want = std::max(1, atoi(f));  // tuning aid
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
  a.xor_mask = x_u8 ? static_cast<int>(0x80808080u) : 0;
  a.neg_zws4 = static_cast<int>(static_cast<uint32_t>((-zws) & 0xff) * 0x01010101u);
  a.lo = op->act_lo - out_flip;
  a.hi = op->act_hi - out_flip;
  a.out_xor = out_flip ? static_cast<int>(0x80808080u) : 0;
  a.pre_ties = pre * 2 + ties;
  a.plain_tiles = a.pre_ties || a.lo > -128 || a.hi < 127 ? 0 : static_cast<int>(OC / 16);
  if (op->fused_add) {
    const tvx_eltwise_desc& e = op->elt;  // a_* / b_* are the Add's first / second operand
    const double ra = static_cast<double>(e.a_scale) / static_cast<double>(e.out_scale);
    const double rb = static_cast<double>(e.b_scale) / static_cast<double>(e.out_scale);
    // as for the stand-alone 16-element Add: the sum must stay far below 2^31 for the 32-bit conversion
    if (!(ra < 1048576.0) || !(rb < 1048576.0)) return TVX_E_UNSUPPORTED;
    plan.add = PwrAdd{nullptr, ra, rb, op->fused_add, d->out_dtype == TVX_I8, e.a_zp, e.b_zp, e.out_zp, 0, 0};
    ActRange(d->out_dtype, e.out_scale, e.out_zp, TVX_ACT_NONE, &plan.add.add_lo, &plan.add.add_hi);
  }

  // ---- weights in fragment order, constants folded into the bias ----
  std::vector<int8_t> packed(static_cast<size_t>(tiles) * ksteps_alloc * 64 * kl, 0);
  const uint8_t* src = static_cast<const uint8_t*>(w_host);
  const int32_t* bias = static_cast<const int32_t*>(bias_host);
  for (uint32_t oc = 0; oc < OC; ++oc) {
    int64_t sw = 0;
    for (uint32_t c = 0; c < C; ++c) {
      const uint8_t r = src[static_cast<size_t>(oc) * C + c];
      const int8_t v = static_cast<int8_t>(w_u8 ? r ^ 0x80 : r);
      const uint32_t step = c / (4 * kl), lane = c / kl % 4 * 16 + oc % 16;
      packed[((static_cast<size_t>(oc / 16) * ksteps_alloc + step) * 64 + lane) * kl + c % kl] = v;
      sw += v;
    }
    const int64_t v = (bias ? bias[oc] : 0) - static_cast<int64_t>(zxs) * sw + static_cast<int64_t>(C) * zxs * zws;
    rqt[static_cast<size_t>(oc) * 4 + 3] = static_cast<int32_t>(static_cast<uint32_t>(v));
  }
  int s = op->packed.Upload(packed.data(), packed.size());
  if (s == TVX_OK) s = op->aux.Upload(rqt.data(), rqt.size() * 4);
  if (s != TVX_OK) return s;
  a.wpk = op->packed.as<uint8_t>();
  a.rec = op->aux.as<v4i>();
  op->host_blob.assign(reinterpret_cast<const uint8_t*>(&plan), reinterpret_cast<const uint8_t*>(&plan) + sizeof(plan));
  op->run = PwRegRun;
  op->kernel_name = op->fused_add ? "pwconv_reg_add_i8" : "pwconv_reg_i8";
  return TVX_OK;
}

}  // namespace tvx
