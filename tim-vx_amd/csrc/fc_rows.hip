// FullyConnected for few rows, few outputs or element types the large tiles do not take: int8 / uint8, float16 and
// float32 with constant weights, any K - vxFullyConnectedLayer as ovxlib reaches it for such layers (reference:
// src/tim/vx/internal/src/ops/vsi_nn_op_fullconnect2.c:118-126).
//
// A workgroup owns a small tile of outputs (16 x 16 up to 64 x 64), its wavefronts split the reduction: each streams a
// contiguous run of the weights - packed in fragment order at creation, one kilobyte of consecutive memory per load -
// and the matching sixteen bytes per lane of the activation rows straight into registers, R steps in flight, with no LDS and
// no barrier on the way; the partial sums meet in LDS once, and every wavefront finishes its share of the outputs.
// Weights are the A operand, so a lane ends up with one activation row and four consecutive features.
//
// Many rows and outputs: tiles of up to 128 x 128 with the rows and weights of a stage in LDS (FcTileKernel).
//
// What bounds it: at the few rows of a classifier or a small batch every weight is used once per row tile, so the launch is
// the time to read them; what a CU has in flight (wavefronts x R x 1 KiB) has to cover the memory's latency, which is why a
// tile's reduction is cut over up to four wavefronts before tiles grow.
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

struct RowsArgs {
  const uint8_t* x;
  uint8_t* y;
  const v4i* wpk;        // [feature tile][step][64 lanes]
  const int32_t* bias;   // per padded feature: int32 with the zero-point terms folded in, or float bits
  const tvx_v4i* rq;
  int M, N, row_bytes;   // bytes of an activation row
  int64_t x_bytes;
  int steps;
  int tiles_m, total, per_xcd;
  uint32_t m_tiles_m;    // reciprocal of tiles_m
  uint32_t xor_mask;
  int zws;               // weight zero point in the signed domain
  int out_zp, lo, hi, rq_mode, act;
};

template <int DT, int TS> struct Mfma;
template <> struct Mfma<kI8, 32> {
  using acc = v16i;
  static __device__ __forceinline__ void Step(acc& c, const v4i& w, const v4i& x) { c = __builtin_amdgcn_mfma_i32_32x32x32_i8(w, x, c, 0, 0, 0); }
};
template <> struct Mfma<kI8, 16> {
  using acc = v4i;
  static __device__ __forceinline__ void Step(acc& c, const v4i& w, const v4i& x) { c = __builtin_amdgcn_mfma_i32_16x16x64_i8(w, x, c, 0, 0, 0); }
};
template <> struct Mfma<kF16, 32> {
  using acc = v16f;
  static __device__ __forceinline__ void Step(acc& c, const v4i& w, const v4i& x) {
    c = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, w), __builtin_bit_cast(v8h, x), c, 0, 0, 0);
  }
};
template <> struct Mfma<kF16, 16> {
  using acc = v4f;
  static __device__ __forceinline__ void Step(acc& c, const v4i& w, const v4i& x) {
    c = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, w), __builtin_bit_cast(v8h, x), c, 0, 0, 0);
  }
};
// (four float32 products per step: lane part p's j-th element is reduction index 4 p + j on both sides)
template <> struct Mfma<kF32, 32> {
  using acc = v16f;
  static __device__ __forceinline__ void Step(acc& c, const v4i& w, const v4i& x) {
    const v4f a = __builtin_bit_cast(v4f, w), b = __builtin_bit_cast(v4f, x);
#pragma unroll
    for (int j = 0; j < 4; ++j) c = __builtin_amdgcn_mfma_f32_32x32x2f32(a[j], b[j], c, 0, 0, 0);
  }
};
template <> struct Mfma<kF32, 16> {
  using acc = v4f;
  static __device__ __forceinline__ void Step(acc& c, const v4i& w, const v4i& x) {
    const v4f a = __builtin_bit_cast(v4f, w), b = __builtin_bit_cast(v4f, x);
#pragma unroll
    for (int j = 0; j < 4; ++j) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], b[j], c, 0, 0, 0);
  }
};

typedef int Dwords4 __attribute__((ext_vector_type(4), aligned(4)));

__device__ __forceinline__ int DivM(int u, uint32_t m) { return m ? static_cast<int>(__umulhi(static_cast<uint32_t>(u), m)) : u; }

// TS: extent of an MFMA tile (16 or 32); WM x WN wavefronts share the rows and features (MT x NT tiles each), KS a tile's
// reduction; R: steps in flight. SPLIT: rows that do not begin on whole dwords: sixteen bytes out of five dwords - a load at any
// byte takes several times as long (int8 29 x 2501 -> 46: 6.7 -> 5.3 us,
// 512 x 2501 -> 512 9.0 -> 7.0; at 2500 bytes 4.0 and 5.3)
template <int DT, int TS, int WM, int WN, int KS, int MT, int NT, int R, bool SPLIT>
__global__ void __launch_bounds__(64 * WM * WN * KS) __attribute__((amdgpu_waves_per_eu(4))) FcRowsKernel(RowsArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  using mfma = Mfma<DT, TS>;
  constexpr int E = DT == kI8 ? 1 : DT == kF16 ? 2 : 4;
  constexpr int kParts = 64 / TS, kStep = 16 * kParts;  // lane parts of a step, bytes of a row a step covers
  constexpr int kQuads = TS * TS / 256;                 // accumulator quads of a lane
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // consecutive workgroups of an XCD: the row tiles of a feature tile, which share its weights
  const int id = static_cast<int>(blockIdx.x & 7) * a.per_xcd + static_cast<int>(blockIdx.x >> 3);
  if (id >= a.total) return;
  const int tn = DivM(id, a.m_tiles_m), tm = id - tn * a.tiles_m;
  const int ks = wave % KS, wn = wave / KS % WN, wm = wave / KS / WN;
  const int row = lane & (TS - 1), part = lane / TS;
  const int per = (a.steps + KS - 1) / KS;
  const int s0 = min(ks * per, a.steps), s1 = min(s0 + per, a.steps);

  const v4i* wp = a.wpk + static_cast<size_t>((tn * WN + wn) * NT) * a.steps * 64 + lane;
  const uint8_t* xp[MT];
  int m[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    m[t] = ((tm * WM + wm) * MT + t) * TS + row;
    xp[t] = a.x + static_cast<int64_t>(min(m[t], a.M - 1)) * a.row_bytes + part * 16;  // (rows past the end repeat the last and are not stored)
  }
  v4i fw[R][NT], fx[R][MT];
  int fifth[R][MT];
  auto fetch = [&](int s, v4i (&w)[NT], v4i (&x)[MT], int (&x5)[MT]) {
    s = max(min(s, s1 - 1), 0);  // (past the end: the last step once more, not multiplied)
#pragma unroll
    for (int t = 0; t < NT; ++t) w[t] = wp[static_cast<uint32_t>(t * a.steps + s) * 64];
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      // a step that ends behind the row: from where sixteen bytes of the tensor can be read, put right in `multiply`
      const uint8_t* p = xp[t] + static_cast<size_t>(s) * kStep;
      const uint8_t* last = a.x + (a.x_bytes - 16);
      p = p < last ? p : last;
      if (SPLIT) {  // the dwords with the first and the last of the sixteen bytes, and what lies between (at the tensor's ends up to three
                    // bytes beside it, in a dword that holds bytes of it; they are shifted out)
        const uintptr_t at = reinterpret_cast<uintptr_t>(p);
        x[t] = *reinterpret_cast<const Dwords4*>(at & ~uintptr_t{3});
        x5[t] = *reinterpret_cast<const int*>((at + 15) & ~uintptr_t{3});
      } else {
        __builtin_memcpy(&x[t], p, 16);
      }
    }
  };
  typename mfma::acc acc[MT][NT];
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int i = 0; i < 4 * kQuads; ++i) acc[t][n][i] = 0;
  int rs[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) rs[t] = 0;
  const bool ragged = a.row_bytes % kStep != 0;
  uint32_t by_row[MT], by_last[MT];  // SPLIT: bytes behind a dword; of the last step, whose load may have been moved
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const uint8_t *p = xp[t] + static_cast<size_t>(a.steps - 1) * kStep, *last = a.x + (a.x_bytes - 16);
    by_row[t] = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(xp[t])) & 3;
    by_last[t] = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(p < last ? p : last)) & 3;
  }
  auto multiply = [&](int s, const v4i (&w)[NT], v4i (&x)[MT], const int (&x5)[MT]) {
    if (SPLIT)
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        const uint32_t by = s == a.steps - 1 ? by_last[t] : by_row[t];  // (the condition is uniform)
        const v4i v = x[t];
#pragma unroll
        for (int q = 0; q < 4; ++q) x[t][q] = static_cast<int>(__builtin_amdgcn_alignbyte(q < 3 ? v[q + 1] : x5[t], v[q], by));
      }
    if (DT == kI8)
#pragma unroll
      for (int t = 0; t < MT; ++t) x[t] ^= static_cast<int>(a.xor_mask);
    if (ragged && s == a.steps - 1) {  // uniform: the row ends inside this step
      const int valid = a.row_bytes - (s * kStep + part * 16);  // bytes of this lane's granule inside the row
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        const int64_t over = (xp[t] + static_cast<size_t>(s) * kStep) - (a.x + (a.x_bytes - 16));  // bytes the load was moved to the front
        unsigned __int128 v = __builtin_bit_cast(unsigned __int128, x[t]);
        if (over > 0) v = over < 16 ? v >> (8 * static_cast<int>(over)) : 0;
        if (valid < 16) v = valid > 0 ? v & ((static_cast<unsigned __int128>(1) << (8 * valid)) - 1) : 0;
        x[t] = __builtin_bit_cast(v4i, v);
      }
    }
    if (DT == kI8 && a.zws)  // uniform
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int q = 0; q < 4; ++q) rs[t] = __builtin_amdgcn_sdot4(x[t][q], 0x01010101, rs[t], false);
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int n = 0; n < NT; ++n) mfma::Step(acc[t][n], w[n], x[t]);
  };
#pragma unroll
  for (int u = 0; u < R; ++u) fetch(s0 + u, fw[u], fx[u], fifth[u]);
  int s = s0;
#pragma unroll 1
  for (; s + R < s1; s += R) {
#pragma unroll
    for (int u = 0; u < R; ++u) {
      multiply(s + u, fw[u], fx[u], fifth[u]);
      fetch(s + u + R, fw[u], fx[u], fifth[u]);
    }
  }
#pragma unroll
  for (int u = 0; u < R; ++u)
    if (s + u < s1) multiply(s + u, fw[u], fx[u], fifth[u]);  // uniform

  // ---- the wavefronts of a tile meet: partial sums by quads, [wave][tile][quad][lane]; quad i is finished by wavefront i % KS ----
  v4i* red = reinterpret_cast<v4i*>(lds);
  int* red_rs = reinterpret_cast<int*>(lds + WM * WN * KS * MT * NT * kQuads * 1024);
  if (KS > 1) {
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int k = 0; k < kQuads; ++k) {
          v4i q;
          if constexpr (DT == kI8) q = v4i{acc[t][n][4 * k], acc[t][n][4 * k + 1], acc[t][n][4 * k + 2], acc[t][n][4 * k + 3]};
          else q = __builtin_bit_cast(v4i, v4f{acc[t][n][4 * k], acc[t][n][4 * k + 1], acc[t][n][4 * k + 2], acc[t][n][4 * k + 3]});
          red[((wave * MT + t) * NT + n) * kQuads * 64 + k * 64 + lane] = q;
        }
  }
  if (DT == kI8 && a.zws) {
#pragma unroll
    for (int t = 0; t < MT; ++t) {
#pragma unroll
      for (int o = TS; o < 64; o <<= 1) rs[t] += __shfl_xor(rs[t], o);
      if (KS > 1 && part == 0) red_rs[(wave * MT + t) * TS + row] = rs[t];
    }
  }
  if (KS > 1) __syncthreads();
  const int wave0 = wave - ks;  // the tile's first wavefront
  if (KS > 1 && DT == kI8 && a.zws)
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      rs[t] = 0;
#pragma unroll
      for (int k = 0; k < KS; ++k) rs[t] += red_rs[((wave0 + k) * MT + t) * TS + row];
    }
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int k = 0; k < kQuads; ++k) {
        if (KS > 1 && ((t * NT + n) * kQuads + k) % KS != ks) continue;  // uniform
        const int f = ((tn * WN + wn) * NT + n) * TS + (TS == 32 ? 8 * k : 0) + 4 * part;  // first of four features
        const v4i b = *reinterpret_cast<const v4i*>(a.bias + f);
        if constexpr (DT == kI8) {
          v4i v = {acc[t][n][4 * k], acc[t][n][4 * k + 1], acc[t][n][4 * k + 2], acc[t][n][4 * k + 3]};
          if (KS > 1) {
            v = red[((wave0 * MT + t) * NT + n) * kQuads * 64 + k * 64 + lane];
#pragma unroll
            for (int w = 1; w < KS; ++w) v += red[(((wave0 + w) * MT + t) * NT + n) * kQuads * 64 + k * 64 + lane];
          }
          v += b - a.zws * rs[t];
          uint32_t r = 0;
          if (a.rq_mode == kRqFastNoTie) {  // uniform
#pragma unroll
            for (int e = 0; e < 4; ++e) r |= (static_cast<uint32_t>(Requant8<kRqFastNoTie>(v[e], a.rq[f + e], a.out_zp, a.lo, a.hi)) & 0xff) << (8 * e);
          } else {  // (rare: a loop keeps the 64-bit form out of the common path's instruction stream)
#pragma unroll 1
            for (int e = 0; e < 4; ++e) {
              const int c = a.rq_mode == kRqFast ? Requant8<kRqFast>(v[e], a.rq[f + e], a.out_zp, a.lo, a.hi)
                                                 : Requant8<kRqGeneric>(v[e], a.rq[f + e], a.out_zp, a.lo, a.hi);
              r |= (static_cast<uint32_t>(c) & 0xff) << (8 * e);
            }
          }
          if (m[t] >= a.M) continue;
          uint8_t* yp = a.y + static_cast<int64_t>(m[t]) * a.N + f;
          if (f + 3 < a.N) __builtin_memcpy(yp, &r, 4);
          else
#pragma unroll
            for (int e = 0; e < 3; ++e)
              if (f + e < a.N) yp[e] = static_cast<uint8_t>(r >> (8 * e));
        } else {
          v4f v = {acc[t][n][4 * k], acc[t][n][4 * k + 1], acc[t][n][4 * k + 2], acc[t][n][4 * k + 3]};
          if (KS > 1) {
            v = __builtin_bit_cast(v4f, red[((wave0 * MT + t) * NT + n) * kQuads * 64 + k * 64 + lane]);
#pragma unroll
            for (int w = 1; w < KS; ++w) v += __builtin_bit_cast(v4f, red[(((wave0 + w) * MT + t) * NT + n) * kQuads * 64 + k * 64 + lane]);
          }
          v += __builtin_bit_cast(v4f, b);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            if (a.act != TVX_ACT_NONE) v[e] = v[e] < 0.f ? 0.f : v[e];
            if (a.act == TVX_ACT_RELU6) v[e] = v[e] > 6.f ? 6.f : v[e];
          }
          if (m[t] >= a.M) continue;
          uint8_t* yp = a.y + (static_cast<int64_t>(m[t]) * a.N + f) * E;
          if constexpr (DT == kF16) {
            _Float16 h[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) h[e] = static_cast<_Float16>(v[e]);
            if (f + 3 < a.N) __builtin_memcpy(yp, h, 8);
            else
#pragma unroll
              for (int e = 0; e < 3; ++e)
                if (f + e < a.N) reinterpret_cast<_Float16*>(yp)[e] = h[e];
          } else {
            if (f + 3 < a.N) __builtin_memcpy(yp, &v, 16);
            else
#pragma unroll
              for (int e = 0; e < 3; ++e)
                if (f + e < a.N) reinterpret_cast<float*>(yp)[e] = v[e];
          }
        }
      }
}

// ---- larger layers: a workgroup's rows and weights through LDS ----
//
// The tiles above read each fragment from memory for every 32 x 32 products of a wavefront; with many rows and many outputs the CU's
// address unit (32 rows of 32 bytes an instruction) is what they wait for, at a tenth of the matrix cores' rate, and rows of
// outputs leave eight bytes at a time. Here four wavefronts share a tile of 64 MT x 64 NT outputs: 128 bytes of each row and the weights
// behind them, in fragment order, are brought to LDS once for all of them - rows through registers (they begin anywhere), weights by
// DMA - while the stage before is multiplied. Weights are packed so that a lane ends up with sixteen consecutive features of a row.
// Where the tiles are about as many as the CUs, a stage is a chain - load, store, barrier, fragments, products - that the four wavefronts, one a
// SIMD, wait through (0.6 us): KS such groups of a workgroup take every KS-th stage each, with buffers of their own, and add up at the end.
// Four groups fill the SIMDs' issue (1.0 us for four stages). u8 5008 x 2944 -> 115: 19.0 us on 32 x 32 tiles, 11.5; f16 456 x 1920 -> 1203 18.9,
// 12.8; u8 7621 x 1312 -> 107 11.4 on one group, 9.1. Two groups, and two of 64 x 128 or 128 x 128 tiles, lay between one and four in all but a few.
template <int DT, int MT, int NT, int kStage, int KS>
__global__ void __launch_bounds__(256 * KS) __attribute__((amdgpu_waves_per_eu(KS > 2 ? KS : 2))) FcTileKernel(RowsArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  using mfma = Mfma<DT, 32>;
  using quad = typename Mfma<DT, 16>::acc;
  constexpr int E = DT == kI8 ? 1 : DT == kF16 ? 2 : 4;
  constexpr int kRows = 64 * MT, kPitch = kStage + 16, kSteps = kStage / 32, kPer = kStage / 16;
  constexpr int kX = kRows * kPitch, kBuffer = kX + 2 * NT * kSteps * 1024;  // bytes of one of two buffers: rows, weights
  constexpr int kChunks = kRows * (kStage / 16) / 256;                       // sixteen-byte chunks of rows a thread brings
  const int tid = threadIdx.x & 255, lane = tid & 63, row = lane & 31, part = lane >> 5;
  const int group = KS > 1 ? __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 8)) : 0;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave & 1, wn = wave >> 1;
  const int id = static_cast<int>(blockIdx.x & 7) * a.per_xcd + static_cast<int>(blockIdx.x >> 3);
  if (id >= a.total) return;
  const int tn = DivM(id, a.m_tiles_m), tm = id - tn * a.tiles_m;
  const int stages = a.steps / kSteps;  // (packed to whole stages)

  int64_t at[kChunks];  // of a chunk in the first stage
#pragma unroll
  for (int i = 0; i < kChunks; ++i) {
    const int j = tid + i * 256;
    at[i] = static_cast<int64_t>(min(tm * kRows + (j / kPer), a.M - 1)) * a.row_bytes + (j % kPer) * 16;  // (rows past the end repeat the last and are not stored)
  }
  const int64_t last = a.x_bytes - 16;
  v4i x[kChunks];
  const auto fetch_x = [&](int stage) {
#pragma unroll
    for (int i = 0; i < kChunks; ++i) {
      const int64_t p = at[i] + stage * kStage;
      __builtin_memcpy(&x[i], a.x + (p < last ? p : last), 16);
    }
  };
  const bool ragged = a.row_bytes % kStage != 0;
  const auto store_x = [&](int stage, uint8_t* to) {
#pragma unroll
    for (int i = 0; i < kChunks; ++i) {
      const int j = tid + i * 256;
      v4i v = x[i];
      if (ragged && stage == stages - 1) {  // (uniform) the rows end inside this stage; at the tensor's end a load was moved to the front
        const int64_t over = at[i] + stage * kStage - last;
        const int valid = a.row_bytes - (stage * kStage + (j % kPer) * 16);
        unsigned __int128 b = __builtin_bit_cast(unsigned __int128, v);
        if (over > 0) b = over < 16 ? b >> (8 * static_cast<int>(over)) : 0;
        if (DT == kI8) b ^= __builtin_bit_cast(unsigned __int128, v4i{static_cast<int>(a.xor_mask), static_cast<int>(a.xor_mask), static_cast<int>(a.xor_mask), static_cast<int>(a.xor_mask)});
        if (valid < 16) b = valid > 0 ? b & ((static_cast<unsigned __int128>(1) << (8 * valid)) - 1) : 0;
        v = __builtin_bit_cast(v4i, b);
      } else if (DT == kI8) {
        v ^= static_cast<int>(a.xor_mask);
      }
      *reinterpret_cast<v4i*>(to + (j / kPer) * kPitch + (j % kPer) * 16) = v;
    }
  };
  const v4i* const wt = a.wpk + static_cast<size_t>(tn) * 2 * NT * a.steps * 64 + lane;
  const auto fetch_w = [&](int stage, uint8_t* to) {
    typedef const __attribute__((address_space(1))) void* gptr;
    typedef __attribute__((address_space(3))) void* lptr;
#pragma unroll
    for (int i = 0; i < 2 * NT * kSteps / 4; ++i) {
      const int j = wave + 4 * i, tile = j / kSteps, step = j % kSteps;
      __builtin_amdgcn_global_load_lds((gptr)(wt + static_cast<size_t>(tile * a.steps + stage * kSteps + step) * 64), (lptr)(to + kX + j * 1024), 16, 0, 0);
    }
  };
  typename mfma::acc acc[MT][NT];
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[t][n][i] = 0;
  int rs[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) rs[t] = 0;
  uint8_t* const own = lds + group * 2 * kBuffer;
  if (KS == 1 || group < stages) {
    fetch_x(group);
    fetch_w(group, own);
  }
  // the features' tables, behind the buffers
  uint8_t* const tables = lds + KS * 2 * kBuffer;
  constexpr int kFeatures = 64 * NT;
  for (int i = threadIdx.x; i < kFeatures; i += 256 * KS) {
    if (DT == kI8) reinterpret_cast<tvx_v4i*>(tables)[i] = a.rq[tn * kFeatures + i];
    reinterpret_cast<int*>(tables + kFeatures * 16)[i] = a.bias[tn * kFeatures + i];
  }
  if (KS == 1 || group < stages) store_x(group, own);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (the weights' DMA)
  __syncthreads();
  for (int first = 0, turn = 0; first < stages; first += KS, turn ^= 1) {
    const int stage = first + group;
    const uint8_t* const now = own + turn * kBuffer;
    uint8_t* const then = own + (turn ^ 1) * kBuffer;
    const bool more = stage + KS < stages;
    if (more) {
      fetch_x(stage + KS);
      fetch_w(stage + KS, then);
    }
    if (KS == 1 || stage < stages)  // (uniform)
#pragma unroll
    for (int s = 0; s < kSteps; ++s) {
      v4i fx[MT], fw[NT];
#pragma unroll
      for (int t = 0; t < MT; ++t) fx[t] = *reinterpret_cast<const v4i*>(now + ((wm * MT + t) * 32 + row) * kPitch + s * 32 + part * 16);
#pragma unroll
      for (int n = 0; n < NT; ++n) fw[n] = *reinterpret_cast<const v4i*>(now + kX + ((wn * NT + n) * kSteps + s) * 1024 + lane * 16);
      if (DT == kI8 && a.zws)  // uniform
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
          for (int q = 0; q < 4; ++q) rs[t] = __builtin_amdgcn_sdot4(fx[t][q], 0x01010101, rs[t], false);
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int n = 0; n < NT; ++n) mfma::Step(acc[t][n], fw[n], fx[t]);
    }
    if (more) {
      store_x(stage + KS, then);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    if (first + KS < stages) __syncthreads();
  }
  if constexpr (KS > 1) {  // the groups' sums: the others' into the buffers, the first group adds
    constexpr int kQuads = MT * NT * 4, kSums = kQuads * 4096 + MT * 1024;
    static_assert((KS - 1) * kSums <= KS * 2 * kBuffer);
    __syncthreads();
    if (group) {
      uint8_t* const to = lds + (group - 1) * kSums;
#pragma unroll
      for (int q = 0; q < kQuads; ++q) {
        const auto& c = acc[q / 4 / NT][q / 4 % NT];
        reinterpret_cast<quad*>(to + q * 4096)[tid] = quad{c[4 * (q % 4)], c[4 * (q % 4) + 1], c[4 * (q % 4) + 2], c[4 * (q % 4) + 3]};
      }
      if (DT == kI8)
#pragma unroll
        for (int t = 0; t < MT; ++t) reinterpret_cast<int*>(to + kQuads * 4096 + t * 1024)[tid] = rs[t];
    }
    __syncthreads();
    if (group) return;
#pragma unroll
    for (int g = 0; g < KS - 1; ++g) {
      const uint8_t* const from = lds + g * kSums;
#pragma unroll
      for (int q = 0; q < kQuads; ++q) {
        const quad v = reinterpret_cast<const quad*>(from + q * 4096)[tid];
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[q / 4 / NT][q / 4 % NT][4 * (q % 4) + e] += v[e];
      }
      if (DT == kI8)
#pragma unroll
        for (int t = 0; t < MT; ++t) rs[t] += reinterpret_cast<const int*>(from + kQuads * 4096 + t * 1024)[tid];
    }
  }

  // ---- a lane: sixteen consecutive features of each of its rows ----
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    if (DT == kI8 && a.zws) rs[t] = a.zws * (rs[t] + __shfl_xor(rs[t], 32));
    const int m = tm * kRows + (wm * MT + t) * 32 + row;
    if (m >= a.M) continue;
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      const int f = (wn * NT + n) * 32 + 16 * part, live = a.N - (tn * kFeatures + f);
      if (live <= 0) continue;
      uint8_t* const yp = a.y + (static_cast<int64_t>(m) * a.N + tn * kFeatures + f) * E;
      uint32_t out[4 * E];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const v4i b = reinterpret_cast<const v4i*>(tables + kFeatures * 16)[f / 4 + k];
        if constexpr (DT == kI8) {
          int v[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = acc[t][n][4 * k + e] + (b[e] - rs[t]);
          const tvx_v4i* const rq = reinterpret_cast<const tvx_v4i*>(tables) + f + 4 * k;
          if (a.rq_mode == kRqFastNoTie) {  // uniform
            int c[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) c[e] = Requant8<kRqFastNoTie>(v[e], rq[e], a.out_zp, a.lo, a.hi);
            out[k] = PackBytes(c[0], c[1], c[2], c[3]);
          } else {
            uint32_t r = 0;
#pragma unroll 1
            for (int e = 0; e < 4; ++e) {
              const int c = a.rq_mode == kRqFast ? Requant8<kRqFast>(v[0], rq[e], a.out_zp, a.lo, a.hi) : Requant8<kRqGeneric>(v[0], rq[e], a.out_zp, a.lo, a.hi);
              r = r >> 8 | static_cast<uint32_t>(c) << 24;
              v[0] = v[1]; v[1] = v[2]; v[2] = v[3];
            }
            out[k] = r;
          }
        } else {
          float v[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            v[e] = acc[t][n][4 * k + e] + __builtin_bit_cast(v4f, b)[e];
            if (a.act != TVX_ACT_NONE) v[e] = v[e] < 0.f ? 0.f : v[e];
            if (a.act == TVX_ACT_RELU6) v[e] = v[e] > 6.f ? 6.f : v[e];
          }
          if constexpr (DT == kF16) {
            _Float16 h[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) h[e] = static_cast<_Float16>(v[e]);
            __builtin_memcpy(&out[2 * k], h, 8);
          } else {
            __builtin_memcpy(&out[4 * k], v, 16);
          }
        }
      }
      if (live >= 16) {
        __builtin_memcpy(yp, out, 16 * E);
      } else {
#pragma unroll
        for (int j = 0; j < 15; ++j)
          if (j < live) {
            if constexpr (E == 1) yp[j] = static_cast<uint8_t>(out[j / 4] >> (8 * (j % 4)));
            else if constexpr (E == 2) reinterpret_cast<uint16_t*>(yp)[j] = static_cast<uint16_t>(out[j / 2] >> (16 * (j % 2)));
            else reinterpret_cast<uint32_t*>(yp)[j] = out[j];
          }
      }
    }
  }
}

typedef void (*RowsFn)(RowsArgs);
struct Shape { int ts, rows, features, waves, ks, lds, stage; RowsFn fn[3][2]; };  // stage: steps that are brought to LDS together, or 0
#define TVX_ROWS(TS, WM, WN, KS, MT, NT, R)                                                                                          \
  { TS, WM * MT * TS, WN * NT * TS, WM * WN * KS, KS, KS > 1 ? WM * WN * KS * MT * (NT * TS * TS * 4 + TS * 4) : 0, 0,                 \
    { { FcRowsKernel<kI8, TS, WM, WN, KS, MT, NT, R, false>, FcRowsKernel<kI8, TS, WM, WN, KS, MT, NT, R, true> },                        \
      { FcRowsKernel<kF16, TS, WM, WN, KS, MT, NT, R, false>, FcRowsKernel<kF16, TS, WM, WN, KS, MT, NT, R, true> },                      \
      { FcRowsKernel<kF32, TS, WM, WN, KS, MT, NT, R, false>, nullptr } } }
#define TVX_FC_TILE(MT, NT, STAGE, KS)                                                                                                         \
  { 32, 64 * MT, 64 * NT, 4 * KS, KS, KS * 2 * (64 * MT * (STAGE + 16) + 2 * NT * STAGE * 32) + 64 * NT * 20, STAGE / 32,                                           \
    { { FcTileKernel<kI8, MT, NT, STAGE, KS>, FcTileKernel<kI8, MT, NT, STAGE, KS> }, { FcTileKernel<kF16, MT, NT, STAGE, KS>, FcTileKernel<kF16, MT, NT, STAGE, KS> }, \
      { nullptr, nullptr } } }
const Shape kShapes[] = {
    TVX_ROWS(16, 1, 1, 4, 1, 1, 8),  // 0: 16 x 16, reduction on four wavefronts
    TVX_ROWS(32, 1, 1, 4, 1, 1, 7),  // 1: 32 x 32, on four
    TVX_ROWS(32, 2, 2, 1, 1, 1, 8),  // 2: 64 x 64, not split
    TVX_FC_TILE(1, 1, 128, 1),          // 3: 64 x 64 through LDS, 128 bytes of a row at a time
    TVX_FC_TILE(1, 2, 128, 1),          // 4: 64 rows x 128
    TVX_FC_TILE(2, 2, 128, 1),          // 5: 128 x 128
    TVX_FC_TILE(1, 1, 256, 1),          // 6: 64 x 64, 256 bytes
    TVX_FC_TILE(2, 2, 64, 1),           // 7: 128 x 128, 64 bytes
    TVX_FC_TILE(1, 1, 128, 4),          // 8: 64 x 64, every fourth stage on each of four groups
};
#undef TVX_ROWS
#undef TVX_FC_TILE
constexpr int kShapeCount = sizeof(kShapes) / sizeof(kShapes[0]);

uint32_t Magic(int d) { return d <= 1 ? 0u : static_cast<uint32_t>(((uint64_t{1} << 32) + d - 1) / d); }

// Microseconds of a launch on tiles of a shape: what a launch takes anyway, then per stage of the reduction either its latency, once for
// every round of workgroups a CU holds, or the time its share of the CU's units takes, whichever is longer, and at the end its results. The
// constants are a fit to 310 drawn layers (at least 60000 outputs, int8 and float16) measured back to back in a captured graph, 6 to 15 %
// off each. On 1961 other drawn layers (m 1 to 8192, k 64 to 4096, n 10 to 4096, more 16 x 16 tiles than CUs) the shape chosen takes 0.86
// of the time of 32 x 32 or 64 x 64 tiles by their number (geometric mean) and 1.4 % more than the best of the seven; 18 of them are slower
// than those tiles by more than 3 %, 30 where a cut reduction was charged whole stages (i8 332 x 672 -> 1965: 5.2 us, 6.5 on the tiles that were
// chosen then). u8 4978 x 64 -> 3462: 30.7 -> 15.6 us, i8 3521 x 560 -> 1238: 19.9 -> 13.3, f16 4138 x 3888 -> 603: 82.8 -> 47.9.
struct Fit { int resident; double base, latency, share, end, unaligned; };  // workgroups of a CU; us, and by how much more at any byte
const Fit kFits[2][kShapeCount] = {
    {{}, {4, 1.15, 0.48, 0.80, 0.10, 0.49}, {4, 2.25, 0.11, 0.16, 1.12, 1.33}, {4, 1.53, 0.62, 0.37, 0.55, 0.17}, {2, 2.09, 0.72, 0.56, 1.02, 0.14},
     {2, 3.69, 0.92, 0.97, 2.01, 0.20}, {2, 1.83, 0.95, 0.80, 0.99, 0.19}, {3, 3.21, 0.60, 0.48, 1.61, 0.14},
     {1, 1.21, 1.10, 0.37, 2.51, 0.38}},
    {{}, {4, 1.07, 0.43, 0.76, 0.00, 0.66}, {4, 1.97, 0.11, 0.16, 0.29, 0.79}, {4, 0.96, 0.57, 0.32, 0.89, 0.24}, {2, 1.61, 0.64, 0.55, 1.22, 0.18},
     {2, 3.10, 0.84, 0.94, 3.26, 0.20}, {2, 1.50, 0.80, 0.74, 0.90, 0.22}, {3, 2.40, 0.56, 0.55, 1.93, 0.22},
     {1, 0.98, 1.02, 0.41, 2.30, 0.22}}};
double Cost(const tvx_fc_desc& d, int dt, int shape) {
  const Shape& sp = kShapes[shape];
  const Fit& f = kFits[dt][shape];
  const double row = static_cast<double>(d.k) * (dt == kI8 ? 1 : 2);
  const int stage = sp.stage ? 32 * sp.stage : 32 * sp.ks * (sp.ks > 1 ? 4 : 1), groups = sp.stage ? sp.ks : 1;
  const double per_cu = static_cast<double>((d.m + sp.rows - 1) / sp.rows) * ((d.n + sp.features - 1) / sp.features) / ComputeUnits();
  double stages = std::ceil(row / stage);
  // (a reduction cut over wavefronts may end early in its last stage, which saves half of what is missing; behind one stage alone, nothing)
  if (!sp.stage && sp.ks > 1 && stages > 1) stages = 0.5 * (stages + 0.25 * std::ceil(std::ceil(row / 32) / sp.ks));
  const double each = static_cast<uint64_t>(row) % 4 ? 1 + f.unaligned : 1.0, chain = groups > 1 ? std::ceil(stages / groups) : stages;
  // (tiles on groups leave a CU no room for a second: 259 of them take two rounds - f16 2332 x 2544 -> 401 34.5 us, 24.3 on 32 x 32)
  const double rounds = groups > 1 ? std::ceil(per_cu / f.resident) : std::max(per_cu / f.resident, 1.0);
  const double latency = rounds * chain * each * f.latency, share = per_cu * (f.end + stages * each * f.share);
  return 2.2 + f.base + std::sqrt(std::sqrt(std::pow(latency, 4) + std::pow(share, 4)));
}

// 16 x 16 tiles until there is one for each CU (f16 16 x 4096 -> 4096: 7.5 us against 9.1 on 32 x 32 tiles), 32 x 32 from there on (f32
// 256 x 1024 -> 1024: 8.8 against 11.9), and 64 x 64 - fragments used twice, no exchange at the end - where there are more than one
// of those per CU, or half as many with a reduction too short to split; int8 and float16 otherwise where Cost sees more than it may be
// off by. Stages on four groups are a fit to 260 layers (7 and 10 % off each), which knows nothing of where rows lie: up to two 32 x 32 tiles a CU are ahead of
// them by .96 to 1.28, 1.12 on the average of 29 layers (f16 263 x 1168 -> 1639 7.0 us and 8.7), where all rows fit an XCD's L2 and are no whole cache lines
// apart, and by .90 to 1.33, 1.14 on the average of eight, where more rows than that have up to 2000 bytes (int8 8000 x 1584 -> 41 6.1 us and 7.4). Elsewhere the
// groups, chosen for 380 of 1500 drawn layers, take .81 of the time, 1.04 at most; .88 of it for 144 more of up to two 32 x 32 tiles a CU. float32, whose products take the longest, gains
// nothing by rows through LDS (882 x 3984 -> 1070: 95 us, 101 with).
int ChooseShape(const tvx_fc_desc& d, int dt) {
  const auto tiles = [&](uint32_t side) { return static_cast<uint64_t>((d.m + side - 1) / side) * ((d.n + side - 1) / side); };
  const uint64_t t16 = tiles(16), t64 = tiles(64), row = static_cast<uint64_t>(d.k) * (dt == kI8 ? 1 : 2);
  const uint64_t cus = ComputeUnits();
  if (t16 <= cus) return 0;
  const int direct = 2 * t64 >= 3 * cus || (2 * t64 >= cus && static_cast<uint64_t>(d.k) * (dt == kI8 ? 1 : dt == kF16 ? 2 : 4) <= 384) ? 2 : 1;
  if (dt == kF32) return direct;
  int best = direct;
  double least = 0.94 * Cost(d, dt, direct);  // (what the fit is off by; then the shorter program)
  const bool near_rows = direct == 1 && tiles(32) <= 2 * cus && row % 4 == 0 && row % 128 && (row <= 2000 || d.m * row <= (4u << 20));
  for (int shape = 1; shape < kShapeCount; ++shape) {
    const Shape& sp = kShapes[shape];
    if (sp.stage && sp.ks > 1 && (row <= 64ull * sp.stage * sp.ks || near_rows)) continue;  // (two stages a group at least)
    const double cost = Cost(d, dt, shape);
    if (cost < least) { best = shape; least = cost; }
  }
  return best;
}

// A round of 256 x 256 tiles on all CUs costs its start and end whether full or not (microseconds, from measured layers).
bool LargeTilesWin(const tvx_fc_desc& d, int dt, int shape) {
  if (shape == 0) return false;
  const uint64_t tiles = static_cast<uint64_t>((d.m + 255) / 256) * ((d.n + 255) / 256), cus = ComputeUnits();
  return static_cast<double>((tiles + cus - 1) / cus) * (dt == kI8 ? 17.0 + 0.009 * d.k : 25.0 + 0.0118 * d.k) < Cost(d, dt, shape);
}

struct Plan {
  RowsArgs a;
  RowsFn fn[2];  // rows on whole dwords; at any element
  unsigned grid, threads, lds_bytes;
  int elem;
};

int FcRowsRun(tvx_op* op, const void* in0, const void*, void* out, hipStream_t st) {
  const Plan* plan = reinterpret_cast<const Plan*>(op->host_blob.data());
  if ((reinterpret_cast<uintptr_t>(in0) | reinterpret_cast<uintptr_t>(out)) & (plan->elem - 1))
    return SetError(TVX_E_INVALID, "%s: tensors must be aligned to their elements", op->kernel_name);
  RowsArgs a = plan->a;
  a.x = static_cast<const uint8_t*>(in0);
  a.y = static_cast<uint8_t*>(out);
  hipLaunchKernelGGL(plan->fn[((reinterpret_cast<uintptr_t>(in0) | static_cast<unsigned>(a.row_bytes)) & 3) != 0], dim3(plan->grid), dim3(plan->threads), plan->lds_bytes, st, a);
  TVX_HIP_CHECK(hipGetLastError());
  return TVX_OK;
}

}  // namespace

int FcRowsSetup(tvx_op* op, const tvx_fc_desc* d, const void* w_host, const void* bias_host) {
  if (!w_host) return TVX_E_UNSUPPORTED;
  bool forced = false;
  if (const char* f = getenv("TVX_FC_ROWS")) {  // test lever: 0 declines, 1 claims also where the large tiles are the better choice
    if (atoi(f) == 0) return TVX_E_UNSUPPORTED;
    forced = true;
  } else if (getenv("TVX_FC_TILE_M")) {
    return TVX_E_UNSUPPORTED;  // (a lever of the large tiles)
  }
  int dt;
  if (op->quantized) dt = kI8;
  else if (d->in_dtype == TVX_F16 && d->w_dtype == TVX_F16 && d->out_dtype == TVX_F16) dt = kF16;
  else if (d->in_dtype == TVX_F32 && d->w_dtype == TVX_F32 && d->out_dtype == TVX_F32) dt = kF32;
  else return TVX_E_UNSUPPORTED;
  const int E = dt == kI8 ? 1 : dt == kF16 ? 2 : 4;
  const uint64_t x_bytes = static_cast<uint64_t>(d->m) * d->k * E;
  if (x_bytes < 16 || x_bytes >= (1ull << 40) || static_cast<uint64_t>(d->k) * E >= (1ull << 30) || static_cast<uint64_t>(d->n) * d->k * E >= (1ull << 32) ||
      static_cast<uint64_t>(d->m) >= (1ull << 30) || d->n >= (1u << 30))
    return TVX_E_UNSUPPORTED;
  const bool tiles_take_it = dt == kI8 ? d->k % 16 == 0 : dt == kF16 && d->k % 8 == 0;
  int shape = ChooseShape(*d, dt);
  if (tiles_take_it && !forced && LargeTilesWin(*d, dt, shape)) return TVX_E_UNSUPPORTED;
  // a few hundred quantized outputs: a wavefront per output (fc_generic) is one round trip with nothing to exchange - the same
  // 3.5 us alone, 0.3 us less behind another layer (LeNet's 800 -> 500 at batch 1)
  if (dt == kI8 && !forced && static_cast<uint64_t>(d->m) * d->n <= 1024 && d->k >= 128) return TVX_E_UNSUPPORTED;
  if (const char* f = getenv("TVX_FC_ROWS_SHAPE")) shape = std::max(0, std::min((dt == kF32 ? 3 : kShapeCount) - 1, atoi(f)));  // test lever
  const Shape& sp = kShapes[shape];
  const int kstep = 16 * (64 / sp.ts);
  RowsArgs a{};
  a.M = static_cast<int>(d->m); a.N = static_cast<int>(d->n); a.row_bytes = static_cast<int>(d->k) * E;
  a.x_bytes = static_cast<int64_t>(x_bytes);
  a.steps = (a.row_bytes + kstep - 1) / kstep;
  if (sp.stage) a.steps = (a.steps + sp.stage - 1) / sp.stage * sp.stage;
  a.tiles_m = (a.M + sp.rows - 1) / sp.rows;
  const int tiles_n = (a.N + sp.features - 1) / sp.features;
  const uint64_t total = static_cast<uint64_t>(a.tiles_m) * tiles_n;
  if (total >= (1ull << 30) || total * a.tiles_m >= (1ull << 32)) return TVX_E_UNSUPPORTED;
  a.total = static_cast<int>(total);
  a.per_xcd = (a.total + 7) / 8;
  a.m_tiles_m = Magic(a.tiles_m);
  const bool x_u8 = d->in_dtype == TVX_U8, w_u8 = d->w_dtype == TVX_U8;
  const int zxs = dt == kI8 ? d->in_zp - (x_u8 ? 128 : 0) : 0, zws = dt == kI8 ? op->w_zp - (w_u8 ? 128 : 0) : 0;
  a.xor_mask = dt == kI8 && x_u8 ? 0x80808080u : 0u;
  a.zws = zws;
  a.out_zp = d->out_zp; a.lo = op->act_lo; a.hi = op->act_hi; a.act = d->activation;

  // ---- weights [n][k] -> [feature tile][step][lane = (part, feature)], zero-padded ----
  const size_t n_alloc = static_cast<size_t>(tiles_n) * sp.features;
  std::vector<uint8_t> packed(n_alloc / sp.ts * a.steps * 1024, 0);
  std::vector<int32_t> bias(n_alloc, 0);
  const uint8_t* src = static_cast<const uint8_t*>(w_host);
  const uint8_t flip = w_u8 ? 0x80 : 0;
  for (int n = 0; n < a.N; ++n) {
    // (through LDS: sixteen consecutive features in the accumulators of a lane part)
    const int j = n % sp.ts, at = sp.stage ? j % 16 / 4 * 8 + j / 16 * 4 + j % 4 : j;
    uint8_t* tile = packed.data() + static_cast<size_t>(n / sp.ts) * a.steps * 1024 + static_cast<size_t>(at) * 16;
    const uint8_t* row = src + static_cast<size_t>(n) * a.row_bytes;
    int64_t sw = 0;
    for (int b = 0; b < a.row_bytes; b += 16) {
      uint8_t* to = tile + static_cast<size_t>(b / kstep) * 1024 + static_cast<size_t>(b % kstep / 16) * sp.ts * 16;
      const int len = std::min(16, a.row_bytes - b);
      if (dt != kI8) {
        std::memcpy(to, row + b, len);
      } else {
        int part = 0;
        for (int j = 0; j < len; ++j) {
          const uint8_t v = row[b + j] ^ flip;
          to[j] = v;
          part += static_cast<int8_t>(v);
        }
        sw += part;
      }
    }
    if (dt == kI8) {
      const int64_t v = (bias_host ? static_cast<const int32_t*>(bias_host)[n] : 0) - static_cast<int64_t>(zxs) * sw + static_cast<int64_t>(d->k) * zxs * zws;
      bias[n] = static_cast<int32_t>(static_cast<uint32_t>(v));
    } else if (bias_host) {
      std::memcpy(&bias[n], static_cast<const float*>(bias_host) + n, 4);
    }
  }
  if (dt == kI8) {
    std::vector<int32_t> rqt;
    a.rq_mode = BuildRequantRecords(op->h_mult, op->h_shift, a.N, static_cast<int>(n_alloc), d->out_zp, &rqt, AccumulatorBound(d->k, bias_host, d->n));
    const int s = op->aux2.Upload(rqt.data(), rqt.size() * 4);
    if (s != TVX_OK) return s;
    a.rq = op->aux2.as<tvx_v4i>();
  }
  int s = op->packed.Upload(packed.data(), packed.size());
  if (s == TVX_OK) s = op->aux.Upload(bias.data(), bias.size() * 4);
  if (s != TVX_OK) return s;
  a.wpk = op->packed.as<v4i>();
  a.bias = op->aux.as<int32_t>();
  Plan plan{};
  plan.a = a;
  for (int i = 0; i < 2; ++i) plan.fn[i] = sp.fn[dt][i];
  plan.grid = static_cast<unsigned>(a.per_xcd) * 8;
  plan.threads = 64u * sp.waves;
  plan.lds_bytes = static_cast<unsigned>(sp.lds);
  plan.elem = E;
  if (plan.lds_bytes > 48 * 1024) {
    for (RowsFn fn : plan.fn) {
      const hipError_t e = fn ? hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(plan.lds_bytes)) : hipSuccess;
      if (e != hipSuccess) return SetError(TVX_E_DEVICE, "hipFuncSetAttribute(dynamic LDS %u): %s", plan.lds_bytes, hipGetErrorString(e));
    }
  }
  op->host_blob.assign(reinterpret_cast<const uint8_t*>(&plan), reinterpret_cast<const uint8_t*>(&plan) + sizeof(plan));
  op->run = FcRowsRun;
  op->kernel_name = dt == kF32 ? "fc_rows_f32" : dt == kF16 ? "fc_rows_f16" : "fc_rows_i8";
  if (sp.stage) op->variant = dt == kF16 ? "fc_tile_f16" : "fc_tile_i8";
  return TVX_OK;
}

}  // namespace tvx
