// Pooling as a register stencil on planes of any width: MAX, AVG and AVG_ANDROID over 2x2 and 3x3 windows at stride 1 or 2 and over
// 7x7 windows that lie side by side, for uint8 / int8, float16 and float32 (vxPoolingLayer2 as
// src/tim/vx/internal/src/ops/vsi_nn_op_pool.c:144-150 calls it).
//
// A thread computes R output rows x PX neighbouring outputs from rows held in registers (plane_rows.h). 8-bit codes are unsigned there
// (int8 with the sign bit flipped). Their maxima are taken two at a time on 16-bit halves, even and odd bytes apart, down the rows first;
// their sums are dot products of a row's window with ones. An average between equal scales is rounded in integers: with v = sum over the
// window + 256 * count (no negative, the parity kept) it is floor((2 v + count) / (2 count)), an exact half downwards where that is odd;
// between other scales, and for the maximum, the generic kernel's arithmetic. Floating point windows are walked in that kernel's order.
//
// What bounds it: the bytes for large planes, the launch for small ones. Back to back, from one thread per output or rows staged in LDS, to
// here: float16 maximum 7x7 on 288 channels of 63 x 82, batch 41, 92 -> 26 us; int8 maximum 2x2 / 2 on 96 of 141 x 141, batch 64, 115 -> 29;
// float32 maximum 3x3 / 2 on 56 of 116 x 116, batch 23, 37 -> 14.6; uint8 average 3x3 on 32 of 119 x 119 16.8 -> 2.8.
#include <algorithm>
#include <cmath>
#include <cstdlib>

#include "plane_rows.h"
#include "variants.h"

namespace tvx {
namespace {

struct PoolRegArgs : PlaneArgs {
  int android;                     // averages count the taps inside the image
  int in_zp, out_zp, flip;         // of unsigned codes; the bits that make them int8 again
  int mult, shift;
  double ratio;
};

template <int DT, int K, int S, int ROWS> struct Tile {
  static constexpr int E = DT == TVX_F32 ? 4 : DT == TVX_F16 ? 2 : 1;
  static constexpr int PX = S == 7 ? 1 : DT == TVX_F32 ? 4 : DT == TVX_F16 && S == 2 ? 4 : 8;
  static constexpr int R = ROWS;
  static constexpr int L = (PX - 1) * S + K;
  static constexpr int NR = (R - 1) * S + K;
  using Rows = PlaneRows<E, L, NR>;
};

__device__ __forceinline__ uint32_t PkMax(uint32_t x, uint32_t y) {
  uint32_t r;
  asm("v_pk_max_u16 %0, %1, %2" : "=v"(r) : "v"(x), "v"(y));
  return r;
}
template <int N>
__device__ __forceinline__ uint32_t Cut(const uint32_t (&d)[N], int o) {  // bytes o .. o + 3 of a row (zeros behind it)
  const uint32_t lo = d[o / 4], hi = o / 4 + 1 < N ? d[o / 4 + 1 < N ? o / 4 + 1 : 0] : 0u;
  return o % 4 ? __builtin_amdgcn_alignbyte(hi, lo, o % 4) : lo;
}

// (sum or maximum) - zero points -> code, between different scales
__device__ __forceinline__ int Rescaled(const PoolRegArgs& a, int v, int div, bool max) {
  const int64_t r = max ? RequantRne(v, a.mult, a.shift) : static_cast<int64_t>(rint(static_cast<double>(v) * a.ratio / static_cast<double>(div)));
  const int64_t c = r + a.out_zp;
  return static_cast<int>(c < 0 ? 0 : c > 255 ? 255 : c);
}

// SAME: equal scales (the other arithmetic, thirty-two times in line, is a code of its own: its fetch cost launches of few workgroups 2 us)
template <int K, int S, int ROWS, bool MAX, bool SAME>
__global__ void __launch_bounds__(256) PoolRegI8Kernel(PoolRegArgs a) {
  using T = Tile<TVX_I8, K, S, ROWS>;
  constexpr int PX = T::PX, R = T::R, LD = T::Rows::LD;
  int first, t, oy, ox;
  bool live;
  const int plane = SharedPlane(a, &first, &t, &live);
  FirstOutput<R, PX>(a, t, &oy, &ox);
  const int iy = oy * S - a.pad_t, ix = ox * S - a.pad_l;
  typename T::Rows rows;
  rows.Load(a, plane, iy, ix);
  uint32_t out[R][(PX + 3) / 4];
  if constexpr (MAX) {
    uint32_t ev[T::NR][LD], od[T::NR][LD];
#pragma unroll
    for (int i = 0; i < T::NR; ++i)
#pragma unroll
      for (int q = 0; q < LD; ++q) {
        ev[i][q] = rows.d[i][q] & 0x00ff00ffu;
        od[i][q] = (rows.d[i][q] >> 8) & 0x00ff00ffu;
      }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      uint32_t e[LD + 1], o[LD + 1];
      e[LD] = o[LD] = 0;
#pragma unroll
      for (int q = 0; q < LD; ++q) {
        e[q] = ev[r * S][q];
        o[q] = od[r * S][q];
#pragma unroll
        for (int k = 1; k < K; ++k) {
          e[q] = PkMax(e[q], ev[r * S + k][q]);
          o[q] = PkMax(o[q], od[r * S + k][q]);
        }
      }
      if constexpr (S == 7) {  // (bytes 0, 2, 4, 6 and 1, 3, 5 of a row)
        const uint32_t m = PkMax(PkMax(e[0], e[1]), PkMax(o[0], o[1] & 0xffffu));
        out[r][0] = max(m & 0xffffu, m >> 16);
      } else if constexpr (S == 1) {
#pragma unroll
        for (int q = 0; q < PX / 4; ++q) {  // columns 4 q and 4 q + 2, 4 q + 1 and 4 q + 3
          const uint32_t e2 = __builtin_amdgcn_alignbit(e[q + 1], e[q], 16), o2 = __builtin_amdgcn_alignbit(o[q + 1], o[q], 16);
          uint32_t m = PkMax(e[q], o[q]), n = PkMax(o[q], e2);
          if (K == 3) { m = PkMax(m, e2); n = PkMax(n, o2); }
          out[r][q] = m | n << 8;
        }
      } else {
        uint32_t m[PX / 2];
#pragma unroll
        for (int q = 0; q < PX / 2; ++q) {  // outputs 2 q and 2 q + 1
          m[q] = PkMax(e[q], o[q]);
          if (K == 3) m[q] = PkMax(m[q], __builtin_amdgcn_alignbit(e[q + 1], e[q], 16));
        }
#pragma unroll
        for (int q = 0; q < PX / 4; ++q) out[r][q] = __builtin_amdgcn_perm(m[2 * q + 1], m[2 * q], 0x06040200);
      }
      if (!SAME || a.in_zp != a.out_zp) {  // (uniform)
#pragma unroll
        for (int q = 0; q < (PX + 3) / 4; ++q) {
          uint32_t c = 0;
#pragma unroll
          for (int b = 0; b < min(PX, 4); ++b) {
            const int v = static_cast<int>((out[r][q] >> (8 * b)) & 0xff) - a.in_zp;
            c |= static_cast<uint32_t>(SAME ? Med3(v + a.out_zp, 0, 255) : Rescaled(a, v, 1, true)) << (8 * b);
          }
          out[r][q] = c;
        }
      }
    }
  } else {
    // taps of a window inside the image, per column and per row: all of them, but for averages that count them at the edges
    int nx[PX], ny[R];
    float rx[PX], ry[R];
    const bool count = a.android && __ballot(ix < 0 || ix + T::L > a.W || iy < 0 || iy + T::NR > a.H);
#pragma unroll
    for (int p = 0; p < PX; ++p) {
      nx[p] = K;
      if (count) nx[p] = max(min(ix + p * S + K, a.W) - max(ix + p * S, 0), 1);  // (the columns past a row's last output: not stored)
      rx[p] = __builtin_amdgcn_rcpf(static_cast<float>(nx[p]));
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      ny[r] = K;
      if (count) ny[r] = max(min(iy + r * S + K, a.H) - max(iy + r * S, 0), 1);
      ry[r] = 0.5f * __builtin_amdgcn_rcpf(static_cast<float>(ny[r]));
    }
    int sum[R][PX];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int p = 0; p < PX; ++p) sum[r][p] = -K * K * a.in_zp;
#pragma unroll
    for (int i = 0; i < T::NR; ++i)
#pragma unroll
      for (int p = 0; p < PX; ++p) {
        const uint32_t w = Cut(rows.d[i], p * S);
        int part = static_cast<int>(__builtin_amdgcn_udot4(w, K == 2 ? 0x00000101u : K == 3 ? 0x00010101u : 0x01010101u, 0u, false));
        if (K > 4) part = static_cast<int>(__builtin_amdgcn_udot4(Cut(rows.d[i], p * S + 4), 0x00010101u, static_cast<uint32_t>(part), false));
#pragma unroll
        for (int r = 0; r < R; ++r)
          if (i - r * S >= 0 && i - r * S < K) sum[r][p] += part;
      }
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int p = 0; p < PX; ++p) {
        const int div = __mul24(nx[p], ny[r]);
        int c;
        if constexpr (SAME) {
          const int u = 2 * sum[r][p] + __mul24(513, div);
          // (u + .5, at most 50128, lies half a step or more from a multiple of 2 div, and the factor is good to 2^-21)
          int w = static_cast<int>((static_cast<float>(u) + .5f) * (rx[p] * ry[r]));
          if (u == 2 * __mul24(w, div)) w -= w & 1;
          c = Med3(w - 256 + a.out_zp, 0, 255);
        } else {
          c = Rescaled(a, sum[r][p], div, false);
        }
        out[r][p / 4] = p % 4 ? out[r][p / 4] | static_cast<uint32_t>(c) << (8 * (p % 4)) : static_cast<uint32_t>(c);
      }
  }
  if (!live) return;
  uint8_t* to = a.y + static_cast<size_t>(plane) * (a.OH * a.OW) + oy * a.OW + ox;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (oy + r >= a.OH) continue;
#pragma unroll
    for (int q = 0; q < (PX + 3) / 4; ++q) out[r][q] ^= static_cast<uint32_t>(a.flip);
    if constexpr (PX == 1) *to = static_cast<uint8_t>(out[0][0]);
    else StoreRow<1>(to + static_cast<size_t>(r) * a.OW, out[r], a.OW);
  }
}

template <int DT, int K, int S, int ROWS, bool MAX>
__global__ void __launch_bounds__(256) PoolRegFloatKernel(PoolRegArgs a) {
  using T = Tile<DT, K, S, ROWS>;
  constexpr int PX = T::PX, R = T::R;
  int first, t, oy, ox;
  bool live;
  const int plane = SharedPlane(a, &first, &t, &live);
  FirstOutput<R, PX>(a, t, &oy, &ox);
  const int iy = oy * S - a.pad_t, ix = ox * S - a.pad_l;
  typename T::Rows rows;
  rows.Load(a, plane, iy, ix);
  float acc[R][PX];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int p = 0; p < PX; ++p) acc[r][p] = MAX ? -INFINITY : 0.f;
#pragma unroll
  for (int i = 0; i < T::NR; ++i) {
    float v[T::L];
#pragma unroll
    for (int j = 0; j < T::L; ++j) {
      if constexpr (DT == TVX_F16) v[j] = static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(rows.d[i][j / 2] >> (16 * (j & 1)))));
      else v[j] = __builtin_bit_cast(float, rows.d[i][j]);
    }
    float m[PX];  // a row's part of the maximum: the output rows share it (no sum does: sums keep their order)
    if (MAX)
#pragma unroll
      for (int p = 0; p < PX; ++p) {
        m[p] = -INFINITY;
#pragma unroll
        for (int k = 0; k < K; ++k) m[p] = v[p * S + k] > m[p] ? v[p * S + k] : m[p];
      }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (i - r * S < 0 || i - r * S >= K) continue;
#pragma unroll
      for (int p = 0; p < PX; ++p) {
        if (MAX) acc[r][p] = m[p] > acc[r][p] ? m[p] : acc[r][p];
        else
#pragma unroll
          for (int k = 0; k < K; ++k) acc[r][p] += v[p * S + k];
      }
    }
  }
  if (!MAX) {
    const bool count = a.android && __ballot(ix < 0 || ix + T::L > a.W || iy < 0 || iy + T::NR > a.H);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int ny = count ? max(min(iy + r * S + K, a.H) - max(iy + r * S, 0), 1) : K;
#pragma unroll
      for (int p = 0; p < PX; ++p) {
        const int nx = count ? max(min(ix + p * S + K, a.W) - max(ix + p * S, 0), 1) : K;
        acc[r][p] /= static_cast<float>(nx * ny);
      }
    }
  }
  if (!live) return;
  uint8_t* to = a.y + (static_cast<size_t>(plane) * (a.OH * a.OW) + oy * a.OW + ox) * T::E;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (oy + r >= a.OH) continue;
    uint32_t out[(PX * T::E + 3) / 4];
#pragma unroll
    for (int p = 0; p < PX; ++p) {
      if constexpr (DT == TVX_F16) {
        const uint32_t h = __builtin_bit_cast(uint16_t, static_cast<_Float16>(acc[r][p]));
        out[p / 2] = p & 1 ? out[p / 2] | h << 16 : h;
      } else {
        out[p] = __builtin_bit_cast(uint32_t, acc[r][p]);
      }
    }
    if constexpr (PX * T::E < 4) *reinterpret_cast<uint16_t*>(to) = static_cast<uint16_t>(out[0]);
    else StoreRow<T::E>(to + static_cast<size_t>(r) * a.OW * T::E, out, a.OW);
  }
}

typedef void (*PoolRegFn)(PoolRegArgs);
template <int DT, int K, int S, int ROWS>
PoolRegFn Pick(bool max, bool same) {
  if constexpr (DT == TVX_I8) {
    if (same) return max ? PoolRegI8Kernel<K, S, ROWS, true, true> : PoolRegI8Kernel<K, S, ROWS, false, true>;
    return max ? PoolRegI8Kernel<K, S, ROWS, true, false> : PoolRegI8Kernel<K, S, ROWS, false, false>;
  } else {
    return max ? PoolRegFloatKernel<DT, K, S, ROWS, true> : PoolRegFloatKernel<DT, K, S, ROWS, false>;
  }
}
template <int DT>
int Columns(int s) { return s == 7 ? Tile<DT, 7, 7, 1>::PX : s == 1 ? Tile<DT, 3, 1, 1>::PX : Tile<DT, 3, 2, 1>::PX; }
template <int DT>
PoolRegFn PickKernel(int k, int s, int rows, bool max, bool same) {
  if (k == 7) return Pick<DT, 7, 7, 1>(max, same);
  if (k == 2) {
    if (s == 2) return Pick<DT, 2, 2, 1>(max, same);
    return rows == 4 ? Pick<DT, 2, 1, 4>(max, same) : Pick<DT, 2, 1, 1>(max, same);
  }
  if (s == 2) return Pick<DT, 3, 2, 1>(max, same);
  return rows == 4 ? Pick<DT, 3, 1, 4>(max, same) : Pick<DT, 3, 1, 1>(max, same);
}

struct Plan {
  PoolRegArgs a;
  PoolRegFn fn;
  unsigned grid, align_in, align_out;  // address bits of the tensors that must not be set
};

int PoolRegRun(tvx_op* op, const void* in0, const void*, void* out, hipStream_t st) {
  const Plan* p = reinterpret_cast<const Plan*>(op->host_blob.data());
  if ((reinterpret_cast<uintptr_t>(in0) & p->align_in) || (reinterpret_cast<uintptr_t>(out) & p->align_out))
    return SetError(TVX_E_INVALID, "%s: the input must be %u-byte aligned, the output %u-byte", op->kernel_name, p->align_in + 1, p->align_out + 1);
  PoolRegArgs a = p->a;
  a.x = static_cast<const uint8_t*>(in0);
  a.y = static_cast<uint8_t*>(out);
  hipLaunchKernelGGL(p->fn, dim3(p->grid), dim3(256), 0, st, a);
  TVX_HIP_CHECK(hipGetLastError());
  return TVX_OK;
}

}  // namespace

int PoolRegSetup(tvx_op* op) { return PoolRegPlan(op, 0, 0, nullptr); }

// Claims the windows above. `name`, align_in, align_out: those of the kernel whose layer it is otherwise (null: windows of two and three
// quantized taps are not claimed).
int PoolRegPlan(tvx_op* op, unsigned align_in, unsigned align_out, const char* name) {
  const tvx_pool2d_desc& d = op->pool;
  if (d.pool_type != TVX_POOL_MAX && d.pool_type != TVX_POOL_AVG && d.pool_type != TVX_POOL_AVG_ANDROID) return TVX_E_UNSUPPORTED;
  const int K = d.k_w, S = d.stride_w;
  if (d.k_h != d.k_w || d.stride_h != d.stride_w || d.pad_left >= d.k_w || d.pad_top >= d.k_h) return TVX_E_UNSUPPORTED;
  if (!(K == 7 && S == 7) && !((K == 2 || K == 3) && (S == 1 || S == 2))) return TVX_E_UNSUPPORTED;
  const bool max = d.pool_type == TVX_POOL_MAX;
  if (!max && d.out_w == 1 && d.out_h == 1 && d.k_w == d.in_w && d.k_h == d.in_h) return TVX_E_UNSUPPORTED;  // (the average of a plane)
  // every window holds a tap of the image
  if (static_cast<uint64_t>(d.out_w - 1) * S >= static_cast<uint64_t>(d.in_w) + d.pad_left || static_cast<uint64_t>(d.out_h - 1) * S >= static_cast<uint64_t>(d.in_h) + d.pad_top)
    return TVX_E_UNSUPPORTED;
  if (const char* f = getenv("TVX_POOL_STENCIL")) if (atoi(f) == 0) return TVX_E_UNSUPPORTED;  // test lever: no register stencils
  if (op->quantized && K != 7 && !name) return TVX_E_UNSUPPORTED;
  const int px = op->quantized ? Columns<TVX_I8>(S) : d.dtype == TVX_F16 ? Columns<TVX_F16>(S) : Columns<TVX_F32>(S);
  const uint64_t planes = static_cast<uint64_t>(d.channels) * d.batch;
  // Output rows of a thread: one - four in registers read a row 1.5 times instead of three times, but are a long chain for few wavefronts (int8
  // average 3x3 on 480 channels of 15 x 15: 2.6 against 4.9 us) - until there are two wavefronts a SIMD at four (336 of 32 x 32, batch 18: 6.8
  // against 5.2), and at stride 2, where rows are read 1.5 times at the most, always.
  int rows = S == 1 && planes * ((d.out_w + px - 1) / px) * ((d.out_h + 3) / 4) >= 512ull * ComputeUnits() ? 4 : 1;
  if (const char* f = getenv("TVX_POOL_REG_ROWS")) rows = S == 1 && atoi(f) == 4 ? 4 : 1;  // test lever
  Plan plan{};
  PoolRegArgs& a = plan.a;
  if (!PlanPlaneRows(&a, planes, d.in_h, d.in_w, d.out_h, d.out_w, d.pad_top, d.pad_left, px, rows)) return TVX_E_UNSUPPORTED;
  if (a.total < 20) return TVX_E_UNSUPPORTED;  // (a run of at most twenty elements fits the tensor)
  a.android = d.pool_type == TVX_POOL_AVG_ANDROID;
  bool same = true;
  if (op->quantized) {
    const int flip = d.dtype == TVX_I8 ? 128 : 0;
    std::vector<int32_t> mult, shift;
    const int s = BuildRequantTables(1, d.in_scale, 1.0f, nullptr, d.out_scale, &mult, &shift);
    if (s != TVX_OK) return s;
    a.mult = mult[0]; a.shift = shift[0];
    same = max ? mult[0] == (1 << 30) && shift[0] == 30 : d.in_scale == d.out_scale;
    a.ratio = static_cast<double>(d.in_scale) / static_cast<double>(d.out_scale);
    a.in_zp = d.in_zp + flip; a.out_zp = d.out_zp + flip;
    a.flip = a.xor_in = flip ? static_cast<int>(0x80808080u) : 0;
    a.fill = max ? 0 : static_cast<int>(static_cast<uint32_t>(a.in_zp & 0xff) * 0x01010101u);
  } else if (max) {
    a.fill = static_cast<int>(d.dtype == TVX_F16 ? 0xfc00fc00u : 0xff800000u);  // (minus infinity)
  }
  plan.fn = op->quantized ? PickKernel<TVX_I8>(K, S, rows, max, same) : d.dtype == TVX_F16 ? PickKernel<TVX_F16>(K, S, rows, max, true) : PickKernel<TVX_F32>(K, S, rows, max, true);
  plan.grid = static_cast<unsigned>((static_cast<uint64_t>(a.planes) * a.tpp + 255) / 256);
  plan.align_in = align_in;
  plan.align_out = align_out;
  op->host_blob.assign(reinterpret_cast<const uint8_t*>(&plan), reinterpret_cast<const uint8_t*>(&plan) + sizeof(plan));
  op->run = PoolRegRun;
  op->variant = op->quantized ? "pool2d_reg_i8" : nullptr;
  op->kernel_name = name ? name : op->quantized ? "pool2d_reg_i8" : d.dtype == TVX_F16 ? "pool2d_reg_f16" : "pool2d_reg_f32";
  return TVX_OK;
}

}  // namespace tvx
