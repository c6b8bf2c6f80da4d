// Depthwise convolution (multiplier 1) as a register stencil on planes of any width: float16 and float32 windows of 3x3 and
// 5x5, int8 / uint8 windows of 5x5 and, where BetterAt3x3 finds this ahead, of 3x3, at stride 1 or 2 (vxConvolutionLayer's depthwise form;
// reference: src/tim/vx/internal/src/ops/vsi_nn_op_conv2d.c:35-118).
//
// A thread computes one, two or four output rows x eight neighbouring outputs (four of float32, and at stride 2) of one plane from rows held in
// registers (plane_rows.h).
// A plane's channel is uniform where its threads fill whole wavefronts (weights then are scalar operands); small planes share
// wavefronts and keep their weights in vector registers.
//
// What bounds it: vector instructions and bytes, about even. One thread per output took (us, back to back; here) 125 (15.5: 49 MB at 3.2
// TB/s) for float16 3x3 on 92 channels of 105 x 160, batch 8; 186 (34: 131 MB at 3.9 TB/s) for float32 3x3 on 400 of 39 x 39, batch 27;
// 166 (27.8) for float16 5x5 at stride 2 on 352 of 46 x 46, batch 42. Planes in LDS with a byte load a tap took 34 (4.4) for int8 5x5 on
// 48 of 114 x 114, batch 2, and 43 (15.5) for uint8 on 208 of 38 x 38, batch 26.
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>

#include "plane_rows.h"
#include "variants.h"

namespace tvx {
namespace {

struct DwrArgs : PlaneArgs {
  const float* wf;        // floating point: [channel][K * K, padded to whole fours], then the bias at place K * K
  const int* wi;          // quantized: [channel][K rows of two dwords, folded bias, pad]
  const tvx_v4i* rq;
  int C;
  uint32_t m_c;
  int act;
  int nzws4, nzws1, sum_shift;  // minus the weights' zero point (its half, where that is 128) in the bytes of a row's two windows; twice the sum then
  int lo, hi, narrow, out_xor, pre_ties;
};

// DT: TVX_I8 (uint8 too), TVX_F16 or TVX_F32
template <int DT, int K, int S, int R> struct Tile {
  static constexpr int E = DT == TVX_F32 ? 4 : DT == TVX_F16 ? 2 : 1;
  static constexpr int PX = S == 1 && DT != TVX_F32 ? 8 : 4;
  static constexpr int L = (PX - 1) * S + K;          // elements of a row behind PX outputs
  static constexpr int NR = (R - 1) * S + K;          // rows behind R outputs
  static constexpr int WS = DT == TVX_I8 ? 2 * K + 2 : (K * K + 4) / 4 * 4;  // words of a channel's table: weights, bias
  using Rows = PlaneRows<E, L, NR>;
};

// Place of a thread: its plane, channel and first output.
struct Place { int plane, c, oy, ox; bool live; };
template <bool UNIFORM, int R, int PX>
__device__ __forceinline__ Place Find(const DwrArgs& a) {
  Place p;
  int t;
  if (UNIFORM) {  // a grid of (channel, part of the plane, image)
    p.c = blockIdx.x;
    p.plane = static_cast<int>(blockIdx.z) * a.C + p.c;
    t = static_cast<int>(blockIdx.y * blockDim.x + threadIdx.x);
    p.live = t < a.tpp;
    t = min(t, a.tpp - 1);
  } else {
    int plane0;
    p.plane = SharedPlane(a, &plane0, &t, &p.live);
    const int c0 = __builtin_amdgcn_readfirstlane(static_cast<int>(static_cast<uint32_t>(plane0) % static_cast<uint32_t>(a.C)));
    const int c = c0 + p.plane - plane0;
    p.c = c - DivReciprocal(c, a.m_c) * a.C;
  }
  FirstOutput<R, PX>(a, t, &p.oy, &p.ox);
  return p;
}

template <int DT, int K, int S, int R, bool UNIFORM>
__global__ void __launch_bounds__(256) DwRegFloatKernel(DwrArgs a) {
  using T = Tile<DT, K, S, R>;
  constexpr int PX = T::PX;
  const Place p = Find<UNIFORM, R, PX>(a);
  const float* w = a.wf + p.c * T::WS;
  typename T::Rows rows;
  rows.Load(a, p.plane, p.oy * S - a.pad_t, p.ox * S - a.pad_l);
  float acc[R][PX];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int q = 0; q < PX; ++q) acc[r][q] = 0.f;
#pragma unroll
  for (int i = 0; i < T::NR; ++i) {
    float v[T::L];
#pragma unroll
    for (int j = 0; j < T::L; ++j) {
      if constexpr (DT == TVX_F16) v[j] = static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(rows.d[i][j / 2] >> (16 * (j & 1)))));
      else v[j] = __builtin_bit_cast(float, rows.d[i][j]);
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int ky = i - r * S;
      if (ky < 0 || ky >= K) continue;
#pragma unroll
      for (int kx = 0; kx < K; ++kx)
#pragma unroll
        for (int q = 0; q < PX; ++q) acc[r][q] = __builtin_fmaf(v[q * S + kx], w[ky * K + kx], acc[r][q]);
    }
  }
  if (!p.live) return;
  const float bias = w[K * K];
  const size_t to0 = static_cast<size_t>(p.plane) * (a.OH * a.OW) + p.oy * a.OW + p.ox;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (p.oy + r >= a.OH) continue;
    uint32_t out[PX * T::E / 4];
#pragma unroll
    for (int q = 0; q < PX; ++q) {
      float v = acc[r][q] + bias;
      if (a.act != TVX_ACT_NONE) v = v < 0.f ? 0.f : v;
      if (a.act == TVX_ACT_RELU6) v = v > 6.f ? 6.f : v;
      if constexpr (DT == TVX_F16) {
        const uint32_t h = __builtin_bit_cast(uint16_t, static_cast<_Float16>(v));
        out[q / 2] = q & 1 ? out[q / 2] | h << 16 : h;
      } else {
        out[q] = __builtin_bit_cast(uint32_t, v);
      }
    }
    StoreRow<T::E>(a.y + (to0 + static_cast<size_t>(r) * a.OW) * T::E, out, a.OW);
  }
}

// bytes o .. o + 3 of a row; what lies behind its last dword meets zero weights
template <int N>
__device__ __forceinline__ int Cut(const uint32_t (&d)[N], int o) {
  const uint32_t lo = d[o / 4], hi = o / 4 + 1 < N ? d[o / 4 + 1] : 0u;
  return static_cast<int>(o % 4 ? __builtin_amdgcn_alignbyte(hi, lo, o % 4) : lo);
}

// Accumulators start from the folded bias. A row's window is two dot products (weights 0 .. 3, and the fifth alone); under a weight zero point (SUMS)
// the rows' window sums are made once per input row, times minus that (times minus its half, and doubled, where that is 128), and added up per
// output row. The first dot product of a sum is the form that saturates, which none does (the bound of BuildTieRecords): it has a destination of its
// own, where the other adds in place and what it starts from is copied in front of it. Bound by vector instructions (93 % of the busy cycles).
// Layer and pointwise one behind it against a sum of plain windows times the zero point at the end, with choices in place of plane_rows.h's masks:
// uint8 3x3 on 72 of 138 x 138, batch 10, 25.3 -> 24.6 us, 5x5 on 64 of 74 x 74, batch 14, 14.6 -> 14.3; int8 3x3 on 336 of 54 x 54, batch 17, 20.2 -> 19.7.
template <int K, int S, int R, bool UNIFORM, bool SUMS>
__global__ void __launch_bounds__(256) DwRegI8Kernel(DwrArgs a) {
  using T = Tile<TVX_I8, K, S, R>;
  constexpr int PX = T::PX;
  const Place p = Find<UNIFORM, R, PX>(a);
  const int* w = a.wi + p.c * T::WS;
  const tvx_v4i rq = a.rq[p.c];
  typename T::Rows rows;
  rows.Load(a, p.plane, p.oy * S - a.pad_t, p.ox * S - a.pad_l);
  const int bias = w[2 * K];
  int acc[R][PX], sum[R][PX];
#pragma unroll
  for (int i = 0; i < T::NR; ++i) {
#pragma unroll
    for (int q = 0; q < PX; ++q) {
      const int w0 = Cut(rows.d[i], q * S), w1 = K > 4 ? Cut(rows.d[i], q * S + 4) : 0;
      int box = 0;
      if (SUMS) {
        box = __builtin_amdgcn_sdot4(w0, a.nzws4, 0, true);
        if (K > 4) box = __builtin_amdgcn_sdot4(w1, a.nzws1, box, true);
      }
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int ky = i - r * S;
        if (ky < 0 || ky >= K) continue;
        acc[r][q] = ky == 0 ? __builtin_amdgcn_sdot4(w0, w[2 * ky], bias, true) : __builtin_amdgcn_sdot4(w0, w[2 * ky], acc[r][q], false);
        if (K > 4) acc[r][q] = __builtin_amdgcn_sdot4(w1, w[2 * ky + 1], acc[r][q], false);
        if (SUMS) sum[r][q] = ky == 0 ? box : sum[r][q] + box;
      }
    }
  }
  if (!p.live) return;
  const int sh = rq[1] & 31;
  const int64_t round = RoundHigh(rq[2]);
  const size_t to0 = static_cast<size_t>(p.plane) * (a.OH * a.OW) + p.oy * a.OW + p.ox;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (p.oy + r >= a.OH) continue;
    uint32_t out[PX / 4];
#pragma unroll
    for (int h = 0; h < PX / 4; ++h) {
      int v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = SUMS ? (sum[r][4 * h + e] << a.sum_shift) + acc[r][4 * h + e] : acc[r][4 * h + e];
      if (a.pre_ties) {  // (uniform)
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] <<= a.pre_ties >> 1;
        if (a.pre_ties & 1) LowerOddTies(v, rq);
      }
      out[h] = (a.narrow ? RequantSaturate4<true>(v, rq[0], sh, round, a.lo << sh, ((a.hi + 1) << sh) - 1) : RequantSaturate4<false>(v, rq[0], sh, round, 0, 0)) ^ static_cast<uint32_t>(a.out_xor);
    }
    StoreRow<1>(a.y + to0 + static_cast<size_t>(r) * a.OW, out, a.OW);
  }
}

typedef void (*DwRegFn)(DwrArgs);
template <int DT, int K, int S, int R>
DwRegFn Pick(bool uniform, bool sums) {
  if constexpr (DT == TVX_I8) {
    if (sums) return uniform ? DwRegI8Kernel<K, S, R, true, true> : DwRegI8Kernel<K, S, R, false, true>;
    return uniform ? DwRegI8Kernel<K, S, R, true, false> : DwRegI8Kernel<K, S, R, false, false>;
  } else {
    return uniform ? DwRegFloatKernel<DT, K, S, R, true> : DwRegFloatKernel<DT, K, S, R, false>;
  }
}
template <int DT, int K, int S>
DwRegFn PickRows(int r, bool uniform, bool sums) {
  return r == 4 ? Pick<DT, K, S, 4>(uniform, sums) : r == 2 ? Pick<DT, K, S, 2>(uniform, sums) : Pick<DT, K, S, 1>(uniform, sums);
}
template <int DT>
DwRegFn PickKernel(int k, int s, int r, bool uniform, bool sums) {
  if (k == 3) return s == 1 ? PickRows<DT, 3, 1>(r, uniform, sums) : PickRows<DT, 3, 2>(r, uniform, sums);
  return s == 1 ? PickRows<DT, 5, 1>(r, uniform, sums) : PickRows<DT, 5, 2>(r, uniform, sums);
}

struct Plan {
  DwrArgs a;
  DwRegFn fn;
  dim3 grid;
  unsigned threads;
};

int DwRegRun(tvx_op* op, const void* in0, const void*, void* out, hipStream_t st) {
  const Plan* p = reinterpret_cast<const Plan*>(op->host_blob.data());
  DwrArgs a = p->a;
  a.x = static_cast<const uint8_t*>(in0);
  a.y = static_cast<uint8_t*>(out);
  hipLaunchKernelGGL(p->fn, p->grid, dim3(p->threads), 0, st, a);
  TVX_HIP_CHECK(hipGetLastError());
  return TVX_OK;
}

// dwconv3x3_i8's layers: rows of whole dwords, shared between lanes
bool WholeDwordRows(const tvx_conv2d_desc* d) { return d->in_w % 4 == 0 && d->out_w % 4 == 0 && d->pad_left <= 1 && d->out_w <= 256; }

// Which quantized 3x3 layers come here. The stencil for rows of whole dwords gives a row a power of two of lanes: where its outputs fill
// less than 0.6 of them (132 columns: 33 of 64) it takes 41.8 us against 33.0 (80 channels, 117 x 132, batch 36), else it is ahead (52
// columns: 12.6 against 14.3). The one that stages planes in LDS is behind on all others (25 channels of 14 x 14, batch 2: 3.1 against
// 2.8 here; 240 of 57 x 57 at stride 2, batch 44, 26.1 against 13.7; 64 of 93 x 93, batch 43, 29.8 against 21.2).
bool BetterAt3x3(const tvx_conv2d_desc* d) {
  if (WholeDwordRows(d)) {
    if (d->stride_w == 1 && d->in_w % 8 == 0 && d->out_w % 8 == 0) return false;  // (eight columns a lane there)
    const int patches = d->out_w / 4;
    int lanes = 1;
    while (lanes < patches) lanes *= 2;
    return patches * 10 < lanes * 6;
  }
  return true;
}

float HalfToFloat(uint16_t h) {
  _Float16 v;
  std::memcpy(&v, &h, 2);
  return static_cast<float>(v);
}

}  // namespace

// Claims depthwise 3x3 and 5x5 convolutions of stride 1 or 2 with constant weights: float16, float32, and int8 / uint8.
int DwRegSetup(tvx_op* op, const tvx_conv2d_desc* d, const void* w_host, const void* bias_host) {
  if (!w_host || op->kind != OP_CONV2D || d->multiplier != 1 || op->fused_add || op->out_blocked) return TVX_E_UNSUPPORTED;
  const int K = d->k_w, S = d->stride_w;
  if (d->k_h != d->k_w || (K != 3 && K != 5) || d->stride_h != d->stride_w || (S != 1 && S != 2) || d->dilation_w != 1 || d->dilation_h != 1)
    return TVX_E_UNSUPPORTED;
  const bool q = op->quantized;
  if (!q && (d->in_dtype != d->w_dtype || d->in_dtype != d->out_dtype || (d->in_dtype != TVX_F16 && d->in_dtype != TVX_F32))) return TVX_E_UNSUPPORTED;
  const int dt = q ? TVX_I8 : d->in_dtype;
  const char* lever = getenv("TVX_DWCONV_REG");  // test lever: 0 declines, 1 claims quantized 3x3 windows too
  if (lever && atoi(lever) == 0) return TVX_E_UNSUPPORTED;
  if (q && K == 3 && !lever && !BetterAt3x3(d)) return TVX_E_UNSUPPORTED;

  DwrArgs a{};
  a.C = d->in_c;
  a.act = d->activation;
  const uint64_t planes = static_cast<uint64_t>(d->batch) * d->in_c;
  if (d->in_c > 60000) return TVX_E_UNSUPPORTED;

  // Output rows of a thread: four in registers read a row 1.5 times (3x3) or twice (5x5, stride 1) instead of three or five times, but are a
  // long chain for few wavefronts. One up to 300000 threads, 1172 a CU (16 channels of 23 x 25, 3x3: 2.8 us, 3.5 with two, 4.4 with four; 20 x 24 of 48 x
  // 32 in float32 3.4, 3.9, 4.6), two up to four times as many (60 K planes of 7 x 7: 6.4, 6.0, 6.2), four from there on (5 x 288 of 125 x 125 23.1,
  // 19.3, 17.9; 5x5 on 37 x 341 of 34 x 34 32.6, 29.3, 25.6).
  const int px = S == 1 && dt != TVX_F32 ? 8 : 4;
  const uint64_t row_threads = planes * ((d->out_w + px - 1) / px) * d->out_h;
  const uint64_t few = 1172ull * ComputeUnits();
  int R = row_threads < few ? 1 : row_threads < 4 * few ? 2 : 4;
  if (const char* f = getenv("TVX_DWCONV_REG_ROWS")) R = atoi(f) == 4 ? 4 : atoi(f) == 2 ? 2 : 1;  // test lever
  if (!PlanPlaneRows(&a, planes, d->in_h, d->in_w, d->out_h, d->out_w, d->pad_top, d->pad_left, px, R)) return TVX_E_UNSUPPORTED;
  if (a.total < 12) return TVX_E_UNSUPPORTED;  // (a run of at most twelve elements fits the tensor)
  // whole wavefronts per plane where at most a quarter of their lanes is idle
  const int waves = (a.tpp + 63) / 64;
  const bool uniform = a.tpp * 4 >= waves * 64 * 3;
  unsigned block = 256, parts = 1;
  if (uniform) {
    parts = static_cast<unsigned>((waves + 3) / 4);
    block = static_cast<unsigned>((waves + parts - 1) / parts) * 64;
    if (d->batch > 65535 || parts > 65535) return TVX_E_UNSUPPORTED;
  }
  a.m_c = Reciprocal(a.C);

  int s = TVX_OK;
  bool sums = false;  // window sums are needed
  if (q) {
    const bool w_u8 = d->w_dtype == TVX_U8, x_u8 = d->in_dtype == TVX_U8;
    const int zxs = d->in_zp - (x_u8 ? 128 : 0), zws = op->w_zp - (w_u8 ? 128 : 0);
    const int words = 2 * K + 2;
    std::vector<int32_t> tab(static_cast<size_t>(a.C) * words, 0);
    const uint8_t* src = static_cast<const uint8_t*>(w_host);
    const int32_t* bi = static_cast<const int32_t*>(bias_host);
    for (int c = 0; c < a.C; ++c) {
      int64_t sw = 0;
      int32_t* t = &tab[static_cast<size_t>(c) * words];
      for (int i = 0; i < K * K; ++i) {
        const uint8_t v = src[static_cast<size_t>(c) * K * K + i] ^ (w_u8 ? 0x80 : 0);
        sw += static_cast<int8_t>(v);
        const int ky = i / K, kx = i % K;
        t[2 * ky + kx / 4] |= static_cast<int32_t>(static_cast<uint32_t>(v) << (8 * (kx & 3)));
      }
      const int64_t v = (bi ? bi[c] : 0) - static_cast<int64_t>(zxs) * sw + static_cast<int64_t>(K) * K * zxs * zws;
      t[2 * K] = static_cast<int32_t>(static_cast<uint32_t>(v));
    }
    const int out_flip = d->out_dtype == TVX_U8 ? 128 : 0;
    std::vector<int32_t> rqt;
    int up;
    bool ties;
    if (!BuildTieRecords(op->h_mult, op->h_shift, a.C, a.C, d->out_zp - out_flip, AccumulatorBound(K * K, bias_host, a.C), &rqt, &up, &ties)) return TVX_E_UNSUPPORTED;
    a.pre_ties = up * 2 + ties;
    a.fill = static_cast<int>(static_cast<uint32_t>(zxs & 0xff) * 0x01010101u);
    a.xor_in = x_u8 ? static_cast<int>(0x80808080u) : 0;
    a.sum_shift = zws == -128;
    const uint32_t nzws = static_cast<uint32_t>(zws == -128 ? 64 : -zws) & 0xff;
    a.nzws4 = static_cast<int>(nzws * (K > 3 ? 0x01010101u : 0x00010101u));
    a.nzws1 = static_cast<int>(nzws);
    sums = zws != 0;
    a.lo = op->act_lo - out_flip; a.hi = op->act_hi - out_flip; a.narrow = a.lo > -128 || a.hi < 127;
    a.out_xor = out_flip ? static_cast<int>(0x80808080u) : 0;
    s = op->packed.Upload(tab.data(), tab.size() * 4);
    if (s == TVX_OK) s = op->aux2.Upload(rqt.data(), rqt.size() * 4);
    a.wi = op->packed.as<int>();
    a.rq = op->aux2.as<tvx_v4i>();
  } else {
    const int words = (K * K + 4) / 4 * 4;
    std::vector<float> tab(static_cast<size_t>(a.C) * words, 0.f);
    for (int c = 0; c < a.C; ++c) {
      float* t = &tab[static_cast<size_t>(c) * words];
      for (int i = 0; i < K * K; ++i) {
        const size_t at = static_cast<size_t>(c) * K * K + i;
        t[i] = dt == TVX_F16 ? HalfToFloat(static_cast<const uint16_t*>(w_host)[at]) : static_cast<const float*>(w_host)[at];
        if (!std::isfinite(t[i])) return TVX_E_UNSUPPORTED;  // (padding multiplies its zeros by the weights)
      }
      t[K * K] = bias_host ? static_cast<const float*>(bias_host)[c] : 0.f;
    }
    s = op->packed.Upload(tab.data(), tab.size() * 4);
    a.wf = op->packed.as<float>();
  }
  if (s != TVX_OK) return s;
  Plan plan{a, nullptr, dim3(1), block};
  plan.fn = dt == TVX_I8 ? PickKernel<TVX_I8>(K, S, R, uniform, sums) : dt == TVX_F16 ? PickKernel<TVX_F16>(K, S, R, uniform, false) : PickKernel<TVX_F32>(K, S, R, uniform, false);
  plan.grid = uniform ? dim3(a.C, parts, d->batch) : dim3(static_cast<unsigned>((planes * a.tpp + 255) / 256));
  op->host_blob.assign(reinterpret_cast<const uint8_t*>(&plan), reinterpret_cast<const uint8_t*>(&plan) + sizeof(plan));
  op->run = DwRegRun;
  op->kernel_name = dt == TVX_I8 ? "dwconv_planes_i8" : dt == TVX_F16 ? "dwconv_reg_f16" : "dwconv_reg_f32";
  if (dt == TVX_I8) op->variant = "dwconv_reg_i8";
  return TVX_OK;
}

}  // namespace tvx
