// The remaining ops of the whole-graph plan: residualAdd, swiGlu, siluF16
// and multiplyF16 (Reference.metal:119-136, Graph.metal:70-95), copyHalfView
// (Graph.metal:1-14) and linearF16 (Reference.metal:61-103).
//
//  * The elementwise ops are HBM-bound: 8 halves (16 bytes) per lane when
//    the count is a multiple of 8 and the buffers are 16-byte aligned, else
//    one. Each result is the reference's fp32 expression rounded to fp16:
//    the sum and product of two fp16 values are exact or singly rounded in
//    fp32 (24 >= 2 x 11 + 2 bits), so any instruction form gives the same
//    bits; SiLU goes through the same correctly rounded helper as the
//    projections' epilogue.
//  * linearF16 keeps the reference's arithmetic: each output is one fp32
//    fma chain over k = 0 .. K-1 in order, then storeLinear. The chain runs on
//    v_mfma_f32_16x16x4_f32, which adds its four products to the sum in k
//    order, each step rounded as an fma (checked bit for bit against the
//    scalar chain): 3.4 ns a k value for a 16 x 16 tile at any depth of
//    dependence, where a lane's fma chain takes 3.9. That chain bounds a tile
//    (31 us at K = 9216) and 157 TFLOP/s the chip, so every tile of a step
//    must keep its matrix core fed: waves that compute touch LDS and the
//    matrix core only, other waves load the rows (16 bytes a lane, 256 a row),
//    and stage them as MFMA operands: lane group g = lane / 16 of an operand
//    holds the halves k = 4 s + g of its row, so the halves (g, g + 4) of
//    eight consecutive ones go as a dword to group g's lane, and a 16-byte
//    read gives a lane its values of eight steps. Three buffers: the first
//    chunk of the next step is read before the barrier. The three projections
//    of an MLP (2560 -> 9216 -> 2560) for 93 rows 2751 -> 187 us, for one row
//    2740 -> 97 us, against a lane-per-column fma kernel; what is left above
//    the chains is the conversions (a matrix core's fp32 products and the VALU
//    do not overlap) and the staging.
#include "exact_fp.hpp"
#include "hip_common.hpp"
#include "kernels.hpp"
#include "linear_store.hpp"

#include "llminfer_hip.h"

namespace llmi {
namespace {

__device__ __forceinline__ uint16_t elementwise(ElementwiseKind kind, uint16_t a, uint16_t b) {
  switch (kind) {
  case ElementwiseKind::Add:
    return f2h(__fadd_rn(h2f(a), h2f(b)));
  case ElementwiseKind::SwiGlu:
    return f2h(mul32(h2f(silu16(h2f(a))), h2f(b)));
  case ElementwiseKind::Silu:
    return silu16(h2f(a));
  case ElementwiseKind::Multiply:
    return f2h(mul32(h2f(a), h2f(b)));
  }
  return 0;
}

template <ElementwiseKind K>
__global__ __launch_bounds__(256) void elementwise_kernel(const uint16_t *__restrict__ a,
                                                          const uint16_t *__restrict__ b,
                                                          uint16_t *__restrict__ out,
                                                          unsigned count, bool vec) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (vec) {
    if (i * 8 >= count)
      return;
    const uint4_t va = reinterpret_cast<const uint4_t *>(a)[i];
    const uint4_t vb = K == ElementwiseKind::Silu ? va : reinterpret_cast<const uint4_t *>(b)[i];
    uint4_t r;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint16_t lo = elementwise(K, (uint16_t)(va[e] & 0xFFFFu), (uint16_t)(vb[e] & 0xFFFFu));
      const uint16_t hi = elementwise(K, (uint16_t)(va[e] >> 16), (uint16_t)(vb[e] >> 16));
      r[e] = (uint32_t)lo | ((uint32_t)hi << 16);
    }
    reinterpret_cast<uint4_t *>(out)[i] = r;
  } else if (i < count) {
    out[i] = elementwise(K, a[i], K == ElementwiseKind::Silu ? a[i] : b[i]);
  }
}

// Piece i of the view, kPiece halves along its innermost axis. Bound by memory
// and, a half a lane, by the index arithmetic of its three axes, which a piece
// of eight shares (the three views of a DeltaNet layer's 1024 x 8192 halves:
// 22 -> 10 us together).
template <unsigned kPiece>
__global__ __launch_bounds__(256) void copy_view_kernel(const uint16_t *__restrict__ src,
                                                        uint16_t *__restrict__ out,
                                                        HalfViewParams p) {
  const unsigned i = blockIdx.x * 256 + threadIdx.x;
  if (i >= p.count / kPiece)
    return;
  unsigned rest = i * kPiece, offset = p.offset;
#pragma unroll
  for (int d = 2; d >= 0; --d) {
    offset += (rest % p.dims[d]) * p.strides[d];
    rest /= p.dims[d];
  }
  if constexpr (kPiece == 8)
    reinterpret_cast<uint4_t *>(out)[i] = *reinterpret_cast<const uint4_t *>(src + offset);
  else
    out[i] = src[offset];
}

// ------------------------------------------------------------- linearF16

typedef float v4f __attribute__((ext_vector_type(4)));

// Eight consecutive halves of a row from k. kVec: rows start 16-byte aligned
// and hold whole pieces of eight; past the end the last piece again (in
// bounds; zeroed where it is used, so that nothing waits for the load before
// then). Else one half at a time, zeros past the end.
template <bool kVec>
__device__ __forceinline__ uint4_t load_halves8(const uint16_t *__restrict__ row, unsigned k,
                                                unsigned width) {
  if constexpr (kVec)
    return *reinterpret_cast<const uint4_t *>(row + min(k, width - 8));
  uint4_t v;
#pragma unroll
  for (unsigned e = 0; e < 4; ++e) {
    const unsigned k0 = k + 2 * e;
    const uint32_t lo = k0 < width ? row[k0] : 0, hi = k0 + 1 < width ? row[k0 + 1] : 0;
    v[e] = lo | (hi << 16);
  }
  return v;
}

constexpr unsigned kF16Tile = 16, kF16Chunk = 32, kF16Chunks = 4;
constexpr unsigned kF16Step = kF16Chunk * kF16Chunks;      // k values a step
constexpr unsigned kF16ChunkBytes = 1024 + 64;             // 64 lanes x 16 B, and a pad
constexpr unsigned kF16TileBytes = kF16Chunks * kF16ChunkBytes;
constexpr unsigned kF16Buffers = 3, kF16FewTiles = 512;

// kRT x kCT tiles a workgroup, a wave a tile, and kLoaders staging waves whose
// loads run kDepth steps ahead of their staging.
template <int kRT, int kCT, int kLoaders, int kDepth, bool kVec>
__global__ __launch_bounds__(64 * (kRT * kCT + kLoaders)) void linear_f16_kernel(
    const uint16_t *__restrict__ in, const uint16_t *__restrict__ w, void *out, const void *aux,
    const float *bias, LinearParams p, unsigned rowBlocks) {
  constexpr unsigned kThreads = 64 * kLoaders;
  constexpr unsigned kPieces = (kRT + kCT) * kF16Tile * (kF16Step / 8);
  constexpr int kPer = (kPieces + kThreads - 1) / kThreads;
  __shared__ __align__(16) unsigned char lds[kF16Buffers][(kRT + kCT) * kF16TileBytes];
  const unsigned lane = threadIdx.x % 64, wave = threadIdx.x / 64;
  // Row blocks of a column block run side by side on one XCD (blockIdx % 8
  // selects it), so that its L2 serves their common weights.
  const unsigned nwg = gridDim.x, x = blockIdx.x % 8;
  const unsigned v = x * (nwg / 8) + min(x, nwg % 8) + blockIdx.x / 8;
  const unsigned row0 = (v % rowBlocks) * (kF16Tile * kRT);
  const unsigned col0 = (v / rowBlocks) * (kF16Tile * kCT);
  const unsigned steps = (p.inputWidth + kF16Step - 1) / kF16Step;

  if (wave >= kRT * kCT) { // a loader
    const unsigned tid = threadIdx.x - 64 * kRT * kCT;
    const uint16_t *src[kPer];
    unsigned at[kPer];
    const unsigned piece = tid % 16; // of the row's step
#pragma unroll
    for (int e = 0; e < kPer; ++e) {
      // staged row: the rows, then the columns (a piece past the last one
      // repeats it)
      const unsigned r = min((tid + e * kThreads) / 16, (kRT + kCT) * kF16Tile - 1);
      src[e] = r < kRT * kF16Tile
                   ? in + (size_t)min(row0 + r, p.tokens - 1) * p.inputWidth
                   : w + (size_t)min(col0 + r - kRT * kF16Tile, p.rowCount - 1) * p.inputWidth;
      at[e] = (r / kF16Tile) * kF16TileBytes + (piece / 4) * kF16ChunkBytes +
              (r % kF16Tile) * 16 + (piece % 4) * 4;
    }
    uint4_t reg[kDepth][kPer];
    auto load = [&](int slot, unsigned step) {
      const unsigned k = step * kF16Step + 8 * piece;
#pragma unroll
      for (int e = 0; e < kPer; ++e)
        reg[slot][e] = load_halves8<kVec>(src[e], k, p.inputWidth);
    };
    auto stage = [&](int slot, unsigned step) {
      const bool past = step * kF16Step + 8 * piece >= p.inputWidth;
      const unsigned buf = step % kF16Buffers;
#pragma unroll
      for (int e = 0; e < kPer; ++e) {
        uint4_t d = reg[slot][e];
        if (past)
          d = uint4_t{0, 0, 0, 0};
        unsigned char *to = lds[buf] + at[e];
        *reinterpret_cast<uint32_t *>(to) = __builtin_amdgcn_perm(d[2], d[0], 0x05040100u);
        *reinterpret_cast<uint32_t *>(to + 256) = __builtin_amdgcn_perm(d[2], d[0], 0x07060302u);
        *reinterpret_cast<uint32_t *>(to + 512) = __builtin_amdgcn_perm(d[3], d[1], 0x05040100u);
        *reinterpret_cast<uint32_t *>(to + 768) = __builtin_amdgcn_perm(d[3], d[1], 0x07060302u);
      }
    };
    // Steps 0 and 1 staged ahead; inside the loop step s + 2, loads kDepth
    // steps ahead of their staging.
#pragma unroll
    for (int d = 0; d < kDepth; ++d)
      load(d, d); // (zeros past the end)
    stage(0, 0);
    load(0, kDepth);
    stage(1 % kDepth, 1);
    load(1 % kDepth, kDepth + 1);
    lds_sync();
    for (unsigned s0 = 0; s0 < steps; s0 += kDepth) {
#pragma unroll
      for (int d = 0; d < kDepth; ++d) {
        const unsigned step = s0 + d;
        if (step >= steps)
          break;
        if (step + 2 < steps) {
          stage((d + 2) % kDepth, step + 2);
          load((d + 2) % kDepth, step + 2 + kDepth);
        }
        lds_sync();
      }
    }
    return;
  }

  const unsigned wr = wave / kCT, wc = wave % kCT; // the wave's tile
  const bool live = row0 + wr * kF16Tile < p.tokens && col0 + wc * kF16Tile < p.rowCount;
  v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
  uint4_t qa[2], qb[2];
  auto fetch = [&](int to, unsigned buf, unsigned c) {
    const unsigned char *base = lds[buf] + lane * 16 + c * kF16ChunkBytes;
    qa[to] = *reinterpret_cast<const uint4_t *>(base + wr * kF16TileBytes);
    qb[to] = *reinterpret_cast<const uint4_t *>(base + (kRT + wc) * kF16TileBytes);
  };
  lds_sync();
  fetch(0, 0, 0);
  for (unsigned step = 0; step < steps; ++step) {
    if (live) {
#pragma unroll
      for (unsigned c = 0; c < kF16Chunks; ++c) {
        // The next chunk: the next step's first one was staged before the
        // last barrier (after the last step it is read and not used).
        if (c + 1 < kF16Chunks)
          fetch((c + 1) % 2, step % kF16Buffers, c + 1);
        else
          fetch((c + 1) % 2, (step + 1) % kF16Buffers, 0);
        // All conversions, then all products: alternating them costs 25 ns
        // a product against 17.
        float fa[8], fb[8];
#pragma unroll
        for (int s = 0; s < 8; ++s) {
          fa[s] = h2f((uint16_t)(qa[c % 2][s / 2] >> (16 * (s % 2))));
          fb[s] = h2f((uint16_t)(qb[c % 2][s / 2] >> (16 * (s % 2))));
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < 8; ++s)
          acc = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[s], fb[s], acc, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    asm volatile("s_barrier" ::: "memory");
  }
  if (!live)
    return;
  const unsigned g = lane / kF16Tile, col = col0 + kF16Tile * wc + lane % kF16Tile;
  if (col >= p.rowCount)
    return;
  const unsigned column = p.firstRow + col;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const unsigned row = row0 + kF16Tile * wr + 4 * g + r;
    if (row < p.tokens)
      store_linear(out, aux, bias, (size_t)row * p.outputWidth + column, column, p.epilogue,
                   p.epilogueBlock, acc[r]);
  }
}

template <int kRT, int kCT, int kLoaders, int kDepth>
void launch_linear_f16_as(const uint16_t *in, const uint16_t *w, void *out, const void *aux,
                          const float *bias, const LinearParams &p, hipStream_t stream) {
  const unsigned rowBlocks = (p.tokens + kF16Tile * kRT - 1) / (kF16Tile * kRT);
  const unsigned colBlocks = (p.rowCount + kF16Tile * kCT - 1) / (kF16Tile * kCT);
  const dim3 grid(rowBlocks * colBlocks), block(64 * (kRT * kCT + kLoaders));
  if (p.inputWidth % 8 == 0 && aligned16(in) && aligned16(w))
    hipLaunchKernelGGL((linear_f16_kernel<kRT, kCT, kLoaders, kDepth, true>), grid, block, 0,
                       stream, in, w, out, aux, bias, p, rowBlocks);
  else
    hipLaunchKernelGGL((linear_f16_kernel<kRT, kCT, kLoaders, kDepth, false>), grid, block, 0,
                       stream, in, w, out, aux, bias, p, rowBlocks);
}

} // namespace

hipError_t launch_elementwise(ElementwiseKind kind, const uint16_t *a, const uint16_t *b,
                              uint16_t *out, unsigned count, hipStream_t stream) {
  const bool vec = count % 8 == 0 && aligned16(a) && aligned16(out) &&
                   (kind == ElementwiseKind::Silu || aligned16(b));
  const size_t lanes = vec ? count / 8 : count;
  const dim3 grid((unsigned)((lanes + 255) / 256));
  switch (kind) {
  case ElementwiseKind::Add:
    hipLaunchKernelGGL(elementwise_kernel<ElementwiseKind::Add>, grid, dim3(256), 0, stream, a,
                       b, out, count, vec);
    break;
  case ElementwiseKind::SwiGlu:
    hipLaunchKernelGGL(elementwise_kernel<ElementwiseKind::SwiGlu>, grid, dim3(256), 0, stream,
                       a, b, out, count, vec);
    break;
  case ElementwiseKind::Silu:
    hipLaunchKernelGGL(elementwise_kernel<ElementwiseKind::Silu>, grid, dim3(256), 0, stream, a,
                       b, out, count, vec);
    break;
  case ElementwiseKind::Multiply:
    hipLaunchKernelGGL(elementwise_kernel<ElementwiseKind::Multiply>, grid, dim3(256), 0,
                       stream, a, b, out, count, vec);
    break;
  }
  return hipGetLastError();
}

hipError_t launch_copy_half_view(const uint16_t *src, uint16_t *out, const HalfViewParams &p,
                                 hipStream_t stream) {
  // Eight halves a lane where every piece is whole, consecutive and 16-byte
  // aligned on both sides: an innermost extent of whole pieces, the other axes'
  // strides of whole pieces wherever they are stepped along.
  const bool pieces =
      p.strides[2] == 1 && p.dims[2] % 8 == 0 && (p.dims[1] == 1 || p.strides[1] % 8 == 0) &&
      (p.dims[0] == 1 || p.strides[0] % 8 == 0) &&
      (reinterpret_cast<uintptr_t>(src + p.offset) | reinterpret_cast<uintptr_t>(out)) % 16 == 0;
  if (pieces)
    hipLaunchKernelGGL(copy_view_kernel<8>, dim3((p.count / 8 + 255) / 256), dim3(256), 0, stream,
                       src, out, p);
  else
    hipLaunchKernelGGL(copy_view_kernel<1>, dim3((p.count + 255) / 256), dim3(256), 0, stream,
                       src, out, p);
  return hipGetLastError();
}

hipError_t launch_linear_f16(const uint16_t *in, const uint16_t *w, void *out, const void *aux,
                             const float *bias, const LinearParams &p, hipStream_t stream) {
  // Up to kF16FewTiles 16 x 16 tiles, two workgroups a CU, a tile a workgroup
  // spreads the chains; past that a CU's third one waits for its matrix cores,
  // and four waves share what a workgroup stages: four column tiles while there
  // is one row of tiles, else 2 x 2. One tile / 1 x 4 / 2 x 2, us, a width of
  // 2560: one row of 8192 columns (512 tiles) 18.6 / 23.2 / 21.0, of 9216 (576)
  // 24.9 / 23.4 / 32.3, of 16384 30.0 / 27.5 / 33.3, of 248,320 369 / 352 / 404;
  // 33 rows of 2560 columns (480) 17.4 / 22.7 / 20.4, of 4096 (768) 25.4 / 22.8 /
  // 20.5; 93 rows of 9216 95 / 83 / 60.
  const unsigned rowTiles = (p.tokens + kF16Tile - 1) / kF16Tile;
  const uint64_t tiles = (uint64_t)rowTiles * ((p.rowCount + kF16Tile - 1) / kF16Tile);
  if (tiles <= kF16FewTiles)
    launch_linear_f16_as<1, 1, 2, 4>(in, w, out, aux, bias, p, stream);
  else if (rowTiles == 1)
    launch_linear_f16_as<1, 4, 4, 4>(in, w, out, aux, bias, p, stream);
  else
    launch_linear_f16_as<2, 2, 4, 3>(in, w, out, aux, bias, p, stream);
  return hipGetLastError();
}

} // namespace llmi
