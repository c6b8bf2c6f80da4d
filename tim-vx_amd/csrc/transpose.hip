// Transpose (reference: src/tim/vx/ops/transpose.cc -> vxTensorPermuteNode): any permutation of up to six dimensions of
// elements of 1, 2 or 4 bytes, moved as they are.
//
// The permutation is reduced first: dimensions of one element go, input dimensions that stay neighbours become one. What is
// left either keeps its fastest dimension (rows move whole: a gather of the widest units the rows, their strides and the
// pointers allow) or is a batch of matrices whose rows become columns, read along one and written along the other through LDS:
//  - the layout change of images: a few interleaved channels to planes. A run of pixels is one contiguous piece of the input. Up to eight
//    channels: a thread reads its pixels as they lie and sorts them in registers. More, up to 64 bytes a pixel: the run goes through LDS, from
//    where a thread takes blocks of channels and pixels that it sorts (multiples of four channels of up to two bytes) or single elements.
//  - anything else: tiles of 64 x 64 elements, 4 bytes per thread on either side.
// 32 x 224 x 224 x 3 bytes (9.6 MB read + written) 19.1 -> 4.1 us, 27 x 91 x 91 x 134 bytes (60 MB) 134 -> 26 us against one thread
// per element with 64-bit divisions; the second is bound by rows that cross cache lines. The first spent its time on a byte a lane out of LDS:
// captured 3.6 us, 2.7 in registers (an empty launch: 2.0), 64 x 61 x 61 x 3 2.9 -> 2.1, 8 x 113 x 113 x 8 3.8 -> 2.3, halves 32 x 224 x 224 x 3 5.5
// -> 4.2. Wide pixels met in a bank of LDS: 4 x 224 x 224 x 32 bytes 16.6 -> 3.9, 8 x 113 x 113 x 12 3.8 -> 3.0, halves x 16 4.2 -> 3.8.
#include <algorithm>
#include <cstring>

#include "variants.h"

namespace tvx {
namespace {

constexpr int kThreads = 256;
constexpr int kMaxDims = 6;
constexpr int kChunkBytes = 8192;   // interleaved form: input bytes of a workgroup
constexpr int kTile = 64;
constexpr int kOwn = 2, kMostOwn = 8;  // interleaved form in registers: dwords of a channel a thread moves, most channels

// Everything a kernel is given stays under 112 bytes: from there on a launch took the host 3.6 us instead of 2.8.
struct MatrixArgs {
  const uint8_t* x;
  uint8_t* y;
  uint32_t A, B;            // extents: the input's fastest dimension, the output's fastest dimension
  uint32_t in_b, out_a;     // strides (elements) of B in the input and of A in the output
  uint32_t tiles_a, tiles_b, m_tiles_a, m_tiles_b;
  uint32_t chunk;           // interleaved form: pixels of a workgroup (a multiple of 4)
  uint32_t m_groups;        // ... reciprocal of chunk / V
  uint32_t m_quads;         // ... of A / 4
};
struct Batch {  // the dimensions beside the matrix's two; the first of up to three has its own extent in the grid only
  uint32_t in_stride[3], out_stride[3];  // elements
  uint32_t dims[2], magic[2];
};
struct NoBatch { uint32_t in_stride, out_stride; };  // one such dimension at most

struct GatherArgs {
  const uint8_t* x;
  uint8_t* y;
  uint32_t total, n;
  uint32_t dims[kMaxDims], magic[kMaxDims], stride[kMaxDims];
};
struct GatherLargeArgs {
  const uint8_t* x;
  uint8_t* y;
  uint64_t total;
  uint64_t stride[kMaxDims];
  uint32_t dims[kMaxDims], n;
};

// u / d = mulhi(u, Magic(d)), exact while u * d < 2^32
__device__ __forceinline__ uint32_t DivM(uint32_t u, uint32_t m) { return m ? __umulhi(u, m) : u; }
uint32_t Magic(uint64_t d) { return d <= 1 ? 0u : static_cast<uint32_t>(((uint64_t{1} << 32) + d - 1) / d); }

__device__ __forceinline__ void BatchOffsets(const NoBatch& b, uint32_t i, uint32_t* in, uint32_t* out) {
  *in = i * b.in_stride;
  *out = i * b.out_stride;
}
__device__ __forceinline__ void BatchOffsets(const Batch& b, uint32_t i, uint32_t* in, uint32_t* out) {
  *in = *out = 0;
#pragma unroll
  for (int d = 0; d < 2; ++d) {
    const uint32_t q = DivM(i, b.magic[d]), r = i - q * b.dims[d];
    *in += r * b.in_stride[d];
    *out += r * b.out_stride[d];
    i = q;
  }
  *in += i * b.in_stride[2];
  *out += i * b.out_stride[2];
}

// A channels interleaved (in_b == A): a chunk of pixels is contiguous in the input.
template <typename T, typename BATCH>
__global__ void __launch_bounds__(kThreads) InterleavedKernel(MatrixArgs a, BATCH batch) {
  __shared__ __attribute__((aligned(16))) uint8_t lds[kChunkBytes + 16];
  constexpr uint32_t V = 4 / sizeof(T);  // elements of a store
  const uint32_t bt = DivM(blockIdx.x, a.m_tiles_b), tb = blockIdx.x - bt * a.tiles_b;
  uint32_t in_off, out_off;
  BatchOffsets(batch, bt, &in_off, &out_off);
  const uint32_t b0 = tb * a.chunk, n = min(a.chunk, a.B - b0);
  const uint32_t bytes = n * a.A * sizeof(T);
  const uint8_t* src = a.x + static_cast<uint64_t>(in_off + b0 * a.A) * sizeof(T);
  for (uint32_t i = threadIdx.x * 16; i < bytes; i += kThreads * 16) {
    if (i + 16 <= bytes) {
      uint4 v;
      __builtin_memcpy(&v, src + i, 16);
      *reinterpret_cast<uint4*>(lds + i) = v;
    } else {
      for (uint32_t j = i; j < bytes; ++j) lds[j] = src[j];
    }
  }
  __syncthreads();
  T* y = reinterpret_cast<T*>(a.y) + out_off + b0;
  const T* s = reinterpret_cast<const T*>(lds);
  const uint32_t groups = a.chunk / V;
  for (uint32_t i = threadIdx.x; i < groups * a.A; i += kThreads) {
    const uint32_t c = DivM(i, a.m_groups), p = (i - c * groups) * V;
    if (p >= n) continue;
    T v[V];
#pragma unroll
    for (uint32_t k = 0; k < V; ++k) v[k] = s[(p + k) * a.A + c];  // (past the run's end: inside the array, not stored)
    T* to = y + c * a.out_a + p;
    if (p + V <= n) __builtin_memcpy(to, v, 4);
    else
#pragma unroll
      for (uint32_t k = 0; k < V; ++k)
        if (p + k < n) to[k] = v[k];
  }
}

// ... of a multiple of four channels of one or two bytes: a thread sorts V channels of V pixels, read as dwords, in registers. The run lies in LDS
// with a dword behind every V pixels, a stride of A + 1 dwords: neighbouring lanes, V pixels apart, would meet in a bank otherwise. (Elements of
// four bytes, with nothing to sort, are 5 % slower for the padding at 12 channels and as much faster at 16: they stay with the kernel above.)
// The last V pixels of a run are those before its end, whichever of them another thread moves too: with a store per element where a run's end cuts
// them, matrices whose pixels are no multiple of V took longer than element by element (1041 of 64 bytes x 15 pixels 5.6 us, 5.0 one by one, now 3.1).
template <typename T, typename BATCH>
__global__ void __launch_bounds__(kThreads) InterleavedBlockKernel(MatrixArgs a, BATCH batch) {
  __shared__ uint32_t lds[kChunkBytes / 4 + kChunkBytes / 32];
  constexpr uint32_t V = 4 / sizeof(T);
  static_assert(V > 1);
  const uint32_t bt = DivM(blockIdx.x, a.m_tiles_b), tb = blockIdx.x - bt * a.tiles_b;
  uint32_t in_off, out_off;
  BatchOffsets(batch, bt, &in_off, &out_off);
  uint32_t b0 = tb * a.chunk, n = min(a.chunk, a.B - b0);
  if (n < V) b0 -= V - n, n = V;  // (a matrix has as many)
  const uint32_t bytes = n * a.A * sizeof(T);
  const uint8_t* src = a.x + static_cast<uint64_t>(in_off + b0 * a.A) * sizeof(T);
  for (uint32_t i = threadIdx.x * 16; i < bytes; i += kThreads * 16) {
    uint32_t v[4] = {0, 0, 0, 0};
    if (i + 16 <= bytes) __builtin_memcpy(v, src + i, 16);
    else  // (whole dwords: four channels)
      for (uint32_t j = 0; j < 3; ++j)
        if (i + 4 * j < bytes) __builtin_memcpy(&v[j], src + i + 4 * j, 4);
    uint32_t* to = lds + i / 4 + DivM(i / 16, a.m_quads);
#pragma unroll
    for (int j = 0; j < 4; ++j) to[j] = v[j];
  }
  __syncthreads();
  T* y = reinterpret_cast<T*>(a.y) + out_off + b0;
  const uint32_t groups = a.chunk / V;
  for (uint32_t i = threadIdx.x; i < groups * (a.A / V); i += kThreads) {
    const uint32_t c = DivM(i, a.m_groups), g = i - c * groups;
    if (g * V >= n) continue;
    const uint32_t p = min(g * V, n - V);
    uint32_t w[V], o[V];
#pragma unroll
    for (uint32_t k = 0; k < V; ++k) w[k] = lds[(p + k) * (a.A / V) + (p + k) / V + c];
    if constexpr (V == 4) {
      Transpose4x4(w, o);
    } else {
      o[0] = __builtin_amdgcn_perm(w[1], w[0], 0x05040100);
      o[1] = __builtin_amdgcn_perm(w[1], w[0], 0x07060302);
    }
    T* to = y + c * V * a.out_a + p;
#pragma unroll
    for (uint32_t k = 0; k < V; ++k) __builtin_memcpy(to + k * a.out_a, &o[k], 4);
  }
}

// Two to eight channels interleaved: a thread takes V * G neighbouring pixels, A * G dwords as they lie, and puts the channels' elements together
// with byte permutes. The last threads of a matrix begin at B - V * G and move some pixels a second time. Two dwords of a channel a thread:
// one and four are level for bytes, one is 5 % behind for halves.
template <typename T, int A, typename BATCH>
__global__ void __launch_bounds__(kThreads) InterleavedRegKernel(MatrixArgs a, BATCH batch) {
  constexpr int V = 4 / sizeof(T), G = kOwn;
  const uint32_t bt = DivM(blockIdx.x, a.m_tiles_b), tb = blockIdx.x - bt * a.tiles_b;
  uint32_t in_off, out_off;
  BatchOffsets(batch, bt, &in_off, &out_off);
  uint32_t p = (tb * kThreads + threadIdx.x) * (V * G);
  if (p >= a.B) return;
  p = min(p, a.B - V * G);
  uint32_t d[A * G];
  __builtin_memcpy(d, a.x + static_cast<uint64_t>(in_off + p * A) * sizeof(T), sizeof(d));
  T* y = reinterpret_cast<T*>(a.y) + out_off + p;
#pragma unroll
  for (int c = 0; c < A; ++c) {
    uint32_t o[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      [[maybe_unused]] const uint32_t* w = d + g * A;
      if constexpr (sizeof(T) == 1) {
        const auto pair = [&](int e) {  // elements e and e + 1 of the channel as the low half of a dword
          const int i = e * A + c, j = i + A;
          return __builtin_amdgcn_perm(w[j / 4], w[i / 4], 0x0c0c0400u + (static_cast<uint32_t>(j % 4) << 8) + i % 4);
        };
        o[g] = __builtin_amdgcn_perm(pair(2), pair(0), 0x05040100);
      } else if constexpr (sizeof(T) == 2) {
        o[g] = __builtin_amdgcn_perm(w[(c + A) / 2], w[c / 2], ((c + A) % 2 ? 0x07060000u : 0x05040000u) + (c % 2 ? 0x0302u : 0x0100u));
      } else {
        o[g] = w[c];
      }
    }
    __builtin_memcpy(y + c * a.out_a, o, sizeof(o));
  }
}

// 64 x 64 tiles of a matrix with rows of A elements in_b apart.
template <typename T, typename BATCH>
__global__ void __launch_bounds__(kThreads) TileKernel(MatrixArgs a, BATCH batch) {
  constexpr int V = 4 / sizeof(T), kPitch = kTile + V;  // elements; one dword more than a tile's row
  __shared__ T tile[kTile * kPitch];
  const uint32_t ra = DivM(blockIdx.x, a.m_tiles_a), ta = blockIdx.x - ra * a.tiles_a;
  const uint32_t bt = DivM(ra, a.m_tiles_b), tb = ra - bt * a.tiles_b;
  uint32_t in_off, out_off;
  BatchOffsets(batch, bt, &in_off, &out_off);
  const uint32_t a0 = ta * kTile, b0 = tb * kTile;
  const T* x = reinterpret_cast<const T*>(a.x) + in_off;
  constexpr int kPerRow = kTile / V;
#pragma unroll
  for (int i = 0; i < kTile * kPerRow / kThreads; ++i) {
    const int it = threadIdx.x + i * kThreads, b = it / kPerRow, p = it % kPerRow * V;
    if (b0 + b >= a.B || a0 + p >= a.A) continue;
    const T* src = x + (b0 + b) * a.in_b + a0 + p;
    T v[V];
    if (a0 + p + V <= a.A) __builtin_memcpy(v, src, 4);
    else
#pragma unroll
      for (int k = 0; k < V; ++k) v[k] = a0 + p + k < a.A ? src[k] : T(0);
    __builtin_memcpy(__builtin_assume_aligned(&tile[b * kPitch + p], 4), v, 4);
  }
  __syncthreads();
  T* y = reinterpret_cast<T*>(a.y) + out_off;
#pragma unroll
  for (int i = 0; i < kTile * kPerRow / kThreads; ++i) {
    const int it = threadIdx.x + i * kThreads, r = it / kPerRow, p = it % kPerRow * V;
    if (a0 + r >= a.A || b0 + p >= a.B) continue;
    T v[V];
#pragma unroll
    for (int k = 0; k < V; ++k) v[k] = tile[(p + k) * kPitch + r];
    T* to = y + (a0 + r) * a.out_a + b0 + p;
    if (b0 + p + V <= a.B) __builtin_memcpy(to, v, 4);
    else
#pragma unroll
      for (int k = 0; k < V; ++k)
        if (b0 + p + k < a.B) to[k] = v[k];
  }
}

// Rows that move whole: one unit of T per thread, the output in order.
template <typename T>
__global__ void __launch_bounds__(kThreads) GatherKernel(GatherArgs a) {
  const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
  if (i >= a.total) return;
  uint32_t rest = i, in = 0;
  for (uint32_t d = 0; d + 1 < a.n; ++d) {
    const uint32_t q = DivM(rest, a.magic[d]);
    in += (rest - q * a.dims[d]) * a.stride[d];
    rest = q;
  }
  reinterpret_cast<T*>(a.y)[i] = reinterpret_cast<const T*>(a.x)[in + rest * a.stride[a.n - 1]];
}

// ... where reciprocals would not be exact: plain 64-bit divisions.
template <typename T>
__global__ void __launch_bounds__(kThreads) GatherLargeKernel(GatherLargeArgs a) {
  const uint64_t i = static_cast<uint64_t>(blockIdx.x) * kThreads + threadIdx.x;
  if (i >= a.total) return;
  uint64_t rest = i, in = 0;
  for (uint32_t d = 0; d < a.n; ++d) {
    in += rest % a.dims[d] * a.stride[d];
    rest /= a.dims[d];
  }
  reinterpret_cast<T*>(a.y)[i] = reinterpret_cast<const T*>(a.x)[in];
}

enum Form { kGather, kGatherLarge, kInterleaved, kInterleavedBlock, kInterleavedReg, kTiles };
struct Plan {
  Form form;
  MatrixArgs m;
  Batch batch;
  bool batched;         // more than one dimension beside the matrix's two
  uint32_t grid;
  GatherLargeArgs g;    // in elements
  uint32_t row_bytes;   // gather: its trailing zero bits up to 16 say in which units rows may move
};

// in units of T, a multiple of the element's bytes
template <typename T>
void LaunchGather(const Plan& p, uint32_t elem, const void* in0, void* out, hipStream_t st) {
  const uint32_t f = sizeof(T) / elem;
  const uint64_t total = p.g.total / f;
  const dim3 grid(static_cast<unsigned>((total + kThreads - 1) / kThreads));
  if (p.form == kGather) {
    GatherArgs a{static_cast<const uint8_t*>(in0), static_cast<uint8_t*>(out), static_cast<uint32_t>(total), p.g.n, {}, {}, {}};
    for (uint32_t d = 0; d < p.g.n; ++d) {
      a.dims[d] = d ? p.g.dims[d] : p.g.dims[d] / f;
      a.magic[d] = Magic(a.dims[d]);
      a.stride[d] = static_cast<uint32_t>(d ? p.g.stride[d] / f : p.g.stride[d]);
    }
    hipLaunchKernelGGL(GatherKernel<T>, grid, dim3(kThreads), 0, st, a);
  } else {
    GatherLargeArgs a = p.g;
    a.x = static_cast<const uint8_t*>(in0);
    a.y = static_cast<uint8_t*>(out);
    a.total = total;
    a.dims[0] /= f;
    for (uint32_t d = 1; d < a.n; ++d) a.stride[d] /= f;
    hipLaunchKernelGGL(GatherLargeKernel<T>, grid, dim3(kThreads), 0, st, a);
  }
}

template <typename T, int A>
void LaunchInterleavedReg(const Plan& p, const MatrixArgs& a, hipStream_t st) {
  const dim3 grid(p.grid), block(kThreads);
  if (p.batched) hipLaunchKernelGGL((InterleavedRegKernel<T, A, Batch>), grid, block, 0, st, a, p.batch);
  else hipLaunchKernelGGL((InterleavedRegKernel<T, A, NoBatch>), grid, block, 0, st, a, NoBatch{p.batch.in_stride[0], p.batch.out_stride[0]});
}

template <typename T>
void LaunchMatrix(const Plan& p, const MatrixArgs& a, hipStream_t st) {
  const dim3 grid(p.grid), block(kThreads);
  const NoBatch one{p.batch.in_stride[0], p.batch.out_stride[0]};
  if (p.form == kInterleavedReg) {
    switch (a.A) {
      case 2: LaunchInterleavedReg<T, 2>(p, a, st); break;
      case 3: LaunchInterleavedReg<T, 3>(p, a, st); break;
      case 4: LaunchInterleavedReg<T, 4>(p, a, st); break;
      case 5: LaunchInterleavedReg<T, 5>(p, a, st); break;
      case 6: LaunchInterleavedReg<T, 6>(p, a, st); break;
      case 7: LaunchInterleavedReg<T, 7>(p, a, st); break;
      default: LaunchInterleavedReg<T, kMostOwn>(p, a, st);
    }
  } else if (p.form == kInterleavedBlock) {
    if constexpr (sizeof(T) <= 2) {
      if (p.batched) hipLaunchKernelGGL((InterleavedBlockKernel<T, Batch>), grid, block, 0, st, a, p.batch);
      else hipLaunchKernelGGL((InterleavedBlockKernel<T, NoBatch>), grid, block, 0, st, a, one);
    }
  } else if (p.form == kInterleaved) {
    if (p.batched) hipLaunchKernelGGL((InterleavedKernel<T, Batch>), grid, block, 0, st, a, p.batch);
    else hipLaunchKernelGGL((InterleavedKernel<T, NoBatch>), grid, block, 0, st, a, one);
  } else {
    if (p.batched) hipLaunchKernelGGL((TileKernel<T, Batch>), grid, block, 0, st, a, p.batch);
    else hipLaunchKernelGGL((TileKernel<T, NoBatch>), grid, block, 0, st, a, one);
  }
}

int TransposeRun(tvx_op* op, const void* in0, const void*, void* out, hipStream_t st) {
  const Plan& p = *reinterpret_cast<const Plan*>(op->host_blob.data());
  const uint32_t elem = op->tr.elem_bytes;
  const uintptr_t where = reinterpret_cast<uintptr_t>(in0) | reinterpret_cast<uintptr_t>(out);
  if (p.form == kGather || p.form == kGatherLarge) {
    uint32_t unit = 16;
    while (unit > elem && ((p.row_bytes | where) & (unit - 1))) unit /= 2;
    switch (unit) {
      case 1: LaunchGather<uint8_t>(p, elem, in0, out, st); break;
      case 2: LaunchGather<uint16_t>(p, elem, in0, out, st); break;
      case 4: LaunchGather<uint32_t>(p, elem, in0, out, st); break;
      case 8: LaunchGather<uint2>(p, elem, in0, out, st); break;
      default: LaunchGather<uint4>(p, elem, in0, out, st);
    }
  } else {
    MatrixArgs a = p.m;
    a.x = static_cast<const uint8_t*>(in0);
    a.y = static_cast<uint8_t*>(out);
    if (elem == 1) LaunchMatrix<uint8_t>(p, a, st);
    else if (elem == 2) LaunchMatrix<uint16_t>(p, a, st);
    else LaunchMatrix<uint32_t>(p, a, st);
  }
  TVX_HIP_CHECK(hipGetLastError());
  return TVX_OK;
}

}  // namespace

int TransposeSetup(tvx_op* op) {
  const tvx_transpose_desc& d = op->tr;
  // ---- the permutation without dimensions of one element, neighbours that stay neighbours as one; in output order:
  // extent, and the input dimension (after the same reduction) it walks ----
  struct Dim { uint64_t extent; uint32_t from; };
  std::vector<Dim> out;
  for (uint32_t i = 0; i < d.rank; ++i) {
    const uint32_t f = d.perm[i];
    if (d.in_dims[f] == 1) continue;
    bool joined = false;
    if (!out.empty()) {  // does this dimension follow the one before in the input too (but for dimensions of one element)?
      uint32_t next = out.back().from + 1;
      while (next < d.rank && d.in_dims[next] == 1) ++next;
      joined = next == f;
    }
    if (joined) {
      out.back().extent *= d.in_dims[f];
      out.back().from = f;
    } else {
      out.push_back({d.in_dims[f], f});
    }
  }
  if (out.empty()) out.push_back({1, 0});
  const int n = static_cast<int>(out.size());
  uint64_t in_stride[kMaxDims], out_stride[kMaxDims], total = 1;
  for (int i = 0; i < n; ++i) {
    out_stride[i] = total;
    total *= out[i].extent;
  }
  // a reduced dimension's stride: everything in front of its first input dimension; `from` is its last
  for (int i = 0; i < n; ++i) {
    uint64_t s = 1;
    for (uint32_t k = 0; k <= out[i].from; ++k) s *= d.in_dims[k];
    in_stride[i] = s / out[i].extent;
  }
  for (int i = 0; i < n; ++i)
    if (out[i].extent >= (1ull << 32)) return SetError(TVX_E_UNSUPPORTED, "tvx_transpose_create: an extent of 2^32 elements");
  if ((total + kThreads - 1) / kThreads > 0x7fffffffull) return SetError(TVX_E_UNSUPPORTED, "tvx_transpose_create: tensor too large");
  Plan plan{};
  // 32-bit offsets, and reciprocals that are exact for every index they divide
  bool exact = total < (1ull << 31);
  uint64_t rest = total;
  for (int i = 0; i + 1 < n; ++i) {
    exact = exact && rest * out[i].extent < (1ull << 32);
    rest /= out[i].extent;
  }
  int fast = 0;  // the output dimension that is the input's fastest
  for (int i = 0; i < n; ++i) if (in_stride[i] == 1 && out[i].extent > 1) fast = i;
  bool matrix = fast != 0 && total < (1ull << 31);
  if (matrix) {
    MatrixArgs& a = plan.m;
    a.A = static_cast<uint32_t>(out[fast].extent);
    a.B = static_cast<uint32_t>(out[0].extent);
    a.in_b = static_cast<uint32_t>(in_stride[0]);
    a.out_a = static_cast<uint32_t>(out_stride[fast]);
    uint64_t batches = 1, largest = 1;
    std::vector<int> others;
    for (int i = 1; i < n; ++i) {
      if (i == fast) continue;
      others.push_back(i);
      batches *= out[i].extent;
      largest = std::max(largest, out[i].extent);
    }
    plan.batched = others.size() > 1;
    // the last one needs no division; one alone stands first
    for (size_t k = 0; k < others.size() && k < 3; ++k) {
      const bool last = plan.batched && k + 1 == others.size();
      const size_t at = last ? 2 : k;
      plan.batch.in_stride[at] = static_cast<uint32_t>(in_stride[others[k]]);
      plan.batch.out_stride[at] = static_cast<uint32_t>(out_stride[others[k]]);
      if (at < 2) {
        plan.batch.dims[at] = static_cast<uint32_t>(out[others[k]].extent);
        plan.batch.magic[at] = Magic(out[others[k]].extent);
      }
    }
    if (others.size() == 2) plan.batch.dims[1] = 1;
    const uint64_t pixel = static_cast<uint64_t>(a.A) * d.elem_bytes;
    uint64_t grid;
    const uint32_t own = 4 / d.elem_bytes * kOwn;  // pixels of a thread, where they stay in registers
    if (a.in_b == a.A && a.A <= kMostOwn && a.B >= own) {
      plan.form = kInterleavedReg;
      a.tiles_b = (a.B + kThreads * own - 1) / (kThreads * own);
      a.m_tiles_b = Magic(a.tiles_b);
      grid = batches * a.tiles_b;
    } else if (a.in_b == a.A && pixel <= 64) {
      plan.form = a.A % 4 || d.elem_bytes > 2 || a.B < 4 / d.elem_bytes ? kInterleaved : kInterleavedBlock;
      a.m_quads = Magic(a.A / 4);
      a.chunk = static_cast<uint32_t>(std::min<uint64_t>(kChunkBytes / pixel, 1024) & ~uint64_t{3});
      a.m_groups = Magic(a.chunk * d.elem_bytes / 4);
      a.tiles_b = (a.B + a.chunk - 1) / a.chunk;
      a.m_tiles_b = Magic(a.tiles_b);
      grid = batches * a.tiles_b;
    } else {
      plan.form = kTiles;
      a.tiles_a = (a.A + kTile - 1) / kTile;
      a.tiles_b = (a.B + kTile - 1) / kTile;
      a.m_tiles_a = Magic(a.tiles_a);
      a.m_tiles_b = Magic(a.tiles_b);
      grid = batches * a.tiles_a * a.tiles_b;
    }
    largest = std::max<uint64_t>({largest, a.tiles_a, a.tiles_b});
    matrix = others.size() <= 3 && grid <= 0x7fffffffull && grid * largest < (1ull << 32);
    plan.grid = static_cast<uint32_t>(grid);
  }
  if (!matrix) {
    plan.form = exact ? kGather : kGatherLarge;
    plan.g.total = total;
    plan.g.n = static_cast<uint32_t>(n);
    for (int i = 0; i < n; ++i) {
      plan.g.dims[i] = static_cast<uint32_t>(out[i].extent);
      plan.g.stride[i] = in_stride[i];
    }
    plan.row_bytes = fast == 0 ? static_cast<uint32_t>(out[0].extent * d.elem_bytes & 15) | 16u : d.elem_bytes;
  }
  op->host_blob.assign(reinterpret_cast<const uint8_t*>(&plan), reinterpret_cast<const uint8_t*>(&plan) + sizeof(plan));
  op->run = TransposeRun;
  op->kernel_name = plan.form == kInterleaved || plan.form == kInterleavedBlock || plan.form == kInterleavedReg ? "transpose_interleaved" : plan.form == kTiles ? "transpose_tiles" : "transpose_gather";
  if (plan.form == kInterleavedBlock) op->variant = "transpose_interleaved_block";
  if (plan.form == kInterleavedReg) op->variant = "transpose_interleaved_reg";
  return TVX_OK;
}

}  // namespace tvx
