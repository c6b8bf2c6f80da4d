// Rows of a plane in a thread's registers: what the stencils over planes of any width share.
//
// A thread takes R output rows x PX neighbouring outputs of one plane. Each input row behind them is one unaligned run of the
// plane's memory, loaded as whole dwords: a run that leaves its row reads the neighbouring row's elements, which are masked - by
// the column pattern, the same for all of a thread's rows - so that no load depends on the position. Only runs that would leave
// the tensor, at its first and last elements, are read from inside it and shifted. All of a thread's loads are issued before the
// first use. Column and row groups at a plane's end are moved back inside it: they compute some outputs twice, and every store
// but those of planes smaller than a group is a whole vector.
#pragma once

#include <algorithm>

#include "tvx_internal.h"

namespace tvx {

struct PlaneArgs {
  const uint8_t* x;
  uint8_t* y;
  int H, W, OH, OW, pad_t, pad_l;
  int ncg, tpp;           // column groups of a row, threads of a plane
  int planes;
  uint32_t m_tpp, m_ncg;  // reciprocals
  int total;              // elements of the input
  int fill, xor_in;       // what lies outside the image; bits flipped in 8-bit elements (before the fill)
};

// (a sum and not a choice of two: that becomes a branch per division)
__device__ __forceinline__ int DivReciprocal(int u, uint32_t m) {
  const uint32_t one = m ? 0u : ~0u;
  return static_cast<int>(__umulhi(static_cast<uint32_t>(u), m) + (static_cast<uint32_t>(u) & one));
}
inline uint32_t Reciprocal(int d) { return d <= 1 ? 0u : static_cast<uint32_t>(((uint64_t{1} << 32) + d - 1) / d); }

// Planes that share wavefronts: this thread's plane (the last one again past the end, with `live` false), the workgroup's first one,
// and the thread's place in its plane.
__device__ __forceinline__ int SharedPlane(const PlaneArgs& a, int* first_plane, int* t, bool* live) {
  const uint32_t first = blockIdx.x * blockDim.x;
  const int plane0 = __builtin_amdgcn_readfirstlane(static_cast<int>(first / static_cast<uint32_t>(a.tpp)));
  const int local = static_cast<int>(first - static_cast<uint32_t>(plane0) * a.tpp + threadIdx.x);
  const int more = DivReciprocal(local, a.m_tpp);
  *t = local - more * a.tpp;
  *live = plane0 + more < a.planes;
  *first_plane = plane0;
  return min(plane0 + more, a.planes - 1);
}
// ... and its first output
template <int R, int PX>
__device__ __forceinline__ void FirstOutput(const PlaneArgs& a, int t, int* oy, int* ox) {
  const int rg = DivReciprocal(t, a.m_ncg), cg = t - rg * a.ncg;
  *oy = min(rg * R, max(a.OH - R, 0));
  *ox = min(cg * PX, max(a.OW - PX, 0));
}

// NR rows of L elements of E bytes; what lies outside the image is `fill`.
template <int E, int L, int NR>
struct PlaneRows {
  static constexpr int LD = (L * E + 3) / 4;  // dwords of a row
  static constexpr int LE = LD * 4 / E;       // and the elements these load
  uint32_t d[NR][LD];

  // the row's elements by n places up (towards higher columns) or down; where n is a row or more, nothing of it counts
  template <bool UP, int STEP = 1>
  static __device__ __forceinline__ void ShiftDwords(uint32_t (&v)[LD], int dwords) {
    const uint32_t on = dwords & STEP ? ~0u : 0u;
#pragma unroll
    for (int k = 0; k < LD; ++k) {
      const int j = UP ? LD - 1 - k : k;
      const uint32_t from = UP ? (j >= STEP ? v[j >= STEP ? j - STEP : 0] : 0u) : (j + STEP < LD ? v[j + STEP < LD ? j + STEP : 0] : 0u);
      v[j] = (from & on) | (v[j] & ~on);
    }
    if constexpr (2 * STEP <= LD) ShiftDwords<UP, 2 * STEP>(v, dwords);
  }
  template <bool UP>
  static __device__ __forceinline__ void Shift(uint32_t (&v)[LD], int n) {
    const int bytes = min(n, LE) * E;
    ShiftDwords<UP>(v, bytes / 4);
    if constexpr (E < 4) {
      const uint32_t rest = 8 * (bytes & 3);
#pragma unroll
      for (int k = 0; k < LD; ++k) {
        const int j = UP ? LD - 1 - k : k;
        const uint64_t lo = UP ? (j > 0 ? v[j > 0 ? j - 1 : 0] : 0u) : v[j], hi = UP ? v[j] : (j + 1 < LD ? v[j + 1 < LD ? j + 1 : 0] : 0u);
        v[j] = static_cast<uint32_t>((hi << 32 | lo) >> (UP ? 32 - rest : rest));
      }
    }
  }

  // the columns of dword j of a row that begins in column ix: ones where the image has them
  static __device__ __forceinline__ uint32_t Columns(const PlaneArgs& a, int ix, int j) {
    constexpr int N = 4 / E;  // elements
    const int c = ix + j * N;
    uint32_t keep;
    if constexpr (N == 1) {
      keep = ~static_cast<uint32_t>((c | (a.W - 1 - c)) >> 31);
    } else if constexpr (N == 2) {
      keep = (static_cast<unsigned>(c) < static_cast<unsigned>(a.W) ? 0xffffu : 0u) | (static_cast<unsigned>(c + 1) < static_cast<unsigned>(a.W) ? 0xffff0000u : 0u);
    } else {  // (by half as many bits twice: a shift by 32 is one by 0)
      const int in_front = 4 * min(max(-c, 0), 4), behind = 4 * min(max(c + 4 - a.W, 0), 4);
      keep = (~0u << in_front << in_front) & (~0u >> behind >> behind);
    }
    // (a mask and a bit operation per dword, not a condition and a choice: chains of choices by VCC take 16 to 23 cycles each, these 4. float32 3x3
    // maximum on 213 of 28 x 28, batch 17: 7.20 -> 6.91 us; float32 5x5 stencil at stride 2 and pointwise layer on 8 of 22 x 22, batch 10: 9.8 -> 9.3)
    asm("" : "+v"(keep));
    return keep;
  }

  __device__ __forceinline__ void Load(const PlaneArgs& a, int plane, int iy, int ix) {
    const int first = plane * (a.H * a.W);
    int moved[NR];  // elements by which a run was moved to lie inside the tensor
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const int at = first + min(max(iy + i, 0), a.H - 1) * a.W + ix, in = min(max(at, 0), a.total - LE);
      __builtin_memcpy(d[i], a.x + static_cast<size_t>(static_cast<uint32_t>(in)) * E, LD * 4);
      moved[i] = in - at;
    }
    // the tensor's first and last elements: back to their places (what is shifted in lies outside the image)
#pragma unroll
    for (int i = 0; i < NR; ++i)
      if (__ballot(moved[i] != 0)) {
        Shift<true>(d[i], max(moved[i], 0));
        Shift<false>(d[i], max(-moved[i], 0));
      }
    if (E == 1) {
#pragma unroll
      for (int i = 0; i < NR; ++i)
#pragma unroll
        for (int j = 0; j < LD; ++j) d[i][j] ^= static_cast<uint32_t>(a.xor_in);
    }
    const uint32_t fill = static_cast<uint32_t>(a.fill);
    // columns: the same pattern in every row; a wavefront without an edge skips it
    if (__ballot(ix < 0 || ix + L > a.W)) {
#pragma unroll
      for (int j = 0; j < LD; ++j) {
        const uint32_t keep = Columns(a, ix, j);
#pragma unroll
        for (int i = 0; i < NR; ++i) d[i][j] = static_cast<uint32_t>(__builtin_amdgcn_bitop3_b32(static_cast<int>(d[i][j]), static_cast<int>(keep), static_cast<int>(fill), 0xe2));  // keep ? d : fill
      }
    }
    if (__ballot(iy < 0 || iy + NR > a.H)) {
#pragma unroll
      for (int i = 0; i < NR; ++i) {
        const int y = iy + i;
        int outside = (y | (a.H - 1 - y)) >> 31;
        asm("" : "+v"(outside));
#pragma unroll
        for (int j = 0; j < LD; ++j) d[i][j] = static_cast<uint32_t>(__builtin_amdgcn_bitop3_b32(static_cast<int>(fill), outside, static_cast<int>(d[i][j]), 0xe2));  // outside ? fill : d
      }
    }
  }
};

// PX results of a row; where the row has fewer than that, but four: its first four and its last four.
template <int E, int N>
__device__ __forceinline__ void StoreRow(uint8_t* to, const uint32_t (&out)[N], int OW) {
  constexpr int PX = N * 4 / E;
  if (OW >= PX) {  // (uniform)
    __builtin_memcpy(to, out, N * 4);
  } else if (PX == 8 && OW >= 4) {
    const int back = (OW - 4) * E;  // bytes in front of the last four
    uint32_t last[E];
#pragma unroll
    for (int j = 0; j < E; ++j) {
      const uint32_t a = back < 4 ? out[j] : out[j + 1], b = back < 4 ? out[j + 1] : j + 2 < N ? out[j + 2 < N ? j + 2 : 0] : 0u;
      last[j] = __builtin_amdgcn_alignbyte(b, a, static_cast<uint32_t>(back & 3));
    }
    __builtin_memcpy(to, out, 4 * E);
    __builtin_memcpy(to + back, last, 4 * E);
  } else {
#pragma unroll
    for (int q = 0; q < PX; ++q)
      if (q < OW) {
        if constexpr (E == 1) to[q] = static_cast<uint8_t>(out[q / 4] >> (8 * (q & 3)));
        else if constexpr (E == 2) reinterpret_cast<uint16_t*>(to)[q] = static_cast<uint16_t>(out[q / 2] >> (16 * (q & 1)));
        else reinterpret_cast<uint32_t*>(to)[q] = out[q];
      }
  }
}

// The geometry of a launch of `threads(R)` threads; false where a kernel's 32-bit places or reciprocals do not reach.
inline bool PlanPlaneRows(PlaneArgs* a, uint64_t planes, uint32_t H, uint32_t W, uint32_t OH, uint32_t OW, uint32_t pad_t, uint32_t pad_l, int px, int rows) {
  const uint64_t in = planes * H * W, out = planes * OH * OW;
  if (H >= (1u << 30) || W >= (1u << 30) || OH >= (1u << 30) || OW >= (1u << 30) || planes >= (1u << 30)) return false;
  if (in >= (1u << 30) || out >= (1u << 30) || pad_l > 1024 || pad_t > 1024) return false;
  a->H = static_cast<int>(H); a->W = static_cast<int>(W); a->OH = static_cast<int>(OH); a->OW = static_cast<int>(OW);
  a->pad_t = static_cast<int>(pad_t); a->pad_l = static_cast<int>(pad_l);
  a->planes = static_cast<int>(planes);
  a->total = static_cast<int>(in);
  a->ncg = (a->OW + px - 1) / px;
  a->tpp = a->ncg * ((a->OH + rows - 1) / rows);
  a->m_tpp = Reciprocal(a->tpp);
  a->m_ncg = Reciprocal(a->ncg);
  return planes * a->tpp < (1u << 30) && static_cast<uint64_t>(a->tpp + 256) * std::max(a->tpp, a->ncg) < (1ull << 32);
}

}  // namespace tvx
