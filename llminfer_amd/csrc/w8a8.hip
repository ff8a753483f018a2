// The W8A8 projection path of the whole-graph plan: activation quantization,
// int8 x int8 projections with per-32-group scales and the fused storeLinear
// epilogues, and the embeddings.
//
// Reference kernels: quantizeActivation and embeddingW8 (Graph.metal:16-68),
// linearW8A8Gemv / linearW8A8Gemm (W8A8.metal:28-113), storeLinear and
// embedding (Reference.metal:14-58).
//
//  * quantize: one lane per 32-wide group (64 bytes of fp16 in, 32 int8 and
//    a scale out). x / scale is the IEEE quotient; the reference's
//    floor/fraction tie rule is round half to even (v_rndne_f32).
//  * GEMV (one row, the decode step): bound by the weight stream. A
//    one-wave workgroup serves 4 output columns with 16 lanes each, the
//    reference's linearW8GemvLanes: lane l takes groups l, l + 16, ... of its
//    column, so the 16 lanes of a column read 512 contiguous weight bytes per
//    step. Group dots run on v_dot4_i32_i8 (exact int32); each group adds
//    (float(dot) * a) * w to the lane's fp32 sum in group order and the lanes
//    meet by the xor butterfly, which is the reference's arithmetic order, so
//    outputs are its bits. Eight groups' weight loads go out before their
//    arithmetic.
//  * GEMM (several rows): the group dots come from int8 MFMA over 32 x 32
//    tiles, with the reference's 8 lanes' fp32 sums kept apart and merged in
//    the butterfly's order.
#include "exact_fp.hpp"
#include "gated_norm.hpp"
#include "hip_common.hpp"
#include "kernels.hpp"
#include "linear_store.hpp"

#include "llminfer_hip.h"

namespace llmi {
namespace {

constexpr unsigned kGroup = 32;

__device__ __forceinline__ int dot4x4(uint4_t a, uint4_t b, int acc) {
#pragma unroll
  for (int e = 0; e < 4; ++e)
    acc = __builtin_amdgcn_sdot4((int)a[e], (int)b[e], acc, false);
  return acc;
}

// The group's exact int32 dot: 32 int8 activations by 32 int8 weights.
__device__ __forceinline__ int group_dot(uint4_t a0, uint4_t a1, uint4_t w0, uint4_t w1) {
  return dot4x4(a1, w1, dot4x4(a0, w0, 0));
}

// One group's term added to a lane's sum: acc + (float(dot) * a) * w, each
// operation rounded on its own.
__device__ __forceinline__ float add_term(float acc, int dot, float a, float w) {
  return __fadd_rn(acc, __fmul_rn(__fmul_rn((float)dot, a), w));
}

// --------------------------------------------------------------- quantize

// One 32-wide group (zeros past the row's end): scale = max|x| / 127 (1 for
// an all-zero or non-finite group), q = x / scale clamped to +-127 and
// rounded half to even (zeros for a non-finite group), written as 32 bytes
// at dst (16-byte aligned). Returns the scale.
__device__ __forceinline__ float quantize_group(const float *x, int8_t *dst, bool &finite) {
  float max_abs = 0.0f;
  finite = true;
#pragma unroll
  for (unsigned j = 0; j < kGroup; ++j) {
    finite = finite && __builtin_isfinite(x[j]);
    max_abs = fmaxf(max_abs, fabsf(x[j]));
  }
  const float scale = finite && max_abs > 0.0f ? __fdiv_rn(max_abs, 127.0f) : 1.0f;
  uint4_t packed[2];
#pragma unroll
  for (unsigned j = 0; j < kGroup; j += 4) {
    uint32_t word = 0;
#pragma unroll
    for (unsigned e = 0; e < 4; ++e) {
      int r = 0;
      if (finite) {
        const float v = fminf(fmaxf(__fdiv_rn(x[j + e], scale), -127.0f), 127.0f);
        r = (int)__builtin_rintf(v);
      }
      word |= ((uint32_t)r & 0xFFu) << (8 * e);
    }
    packed[j / 16][(j / 4) % 4] = word;
  }
  uint4_t *d = reinterpret_cast<uint4_t *>(dst);
  d[0] = packed[0];
  d[1] = packed[1];
  return scale;
}


// Rows of whole 32-wide groups from 16-byte-aligned input: a lane per chunk
// of eight values, four lanes a group (quantize_chunk8, the expressions
// above): a group's 32 divides spread over its four lanes instead of one
// lane's sequence.
__global__ __launch_bounds__(256) void quantize_chunks_kernel(const uint16_t *__restrict__ in,
                                                              int8_t *__restrict__ q,
                                                              float *__restrict__ scales,
                                                              unsigned *invalid, unsigned chunks) {
  const unsigned c = blockIdx.x * 256 + threadIdx.x;
  if (c >= chunks) // (chunks is a multiple of 4: a group's lanes leave together)
    return;
  const uint4_t v = reinterpret_cast<const uint4_t *>(in)[c];
  float y[8];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    y[2 * e] = h2f((uint16_t)(v[e] & 0xFFFFu));
    y[2 * e + 1] = h2f((uint16_t)(v[e] >> 16));
  }
  quantize_chunk8(y, q + 8 * (size_t)c, scales + c / 4, invalid, (c & 3u) == 0);
}

__global__ __launch_bounds__(256) void quantize_kernel(const uint16_t *__restrict__ in,
                                                       int8_t *__restrict__ q,
                                                       float *__restrict__ scales,
                                                       unsigned *invalid, unsigned rows,
                                                       unsigned width, unsigned groups,
                                                       bool vec) {
  const unsigned i = blockIdx.x * 256 + threadIdx.x;
  if (i >= rows * groups)
    return;
  const unsigned row = i / groups, begin = (i % groups) * kGroup;
  const unsigned length = min(kGroup, width - begin);
  const uint16_t *group = in + (size_t)row * width + begin;
  float x[kGroup];
  if (vec && length == kGroup) {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const uint4_t v = reinterpret_cast<const uint4_t *>(group)[c];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        x[8 * c + 2 * e] = h2f((uint16_t)(v[e] & 0xFFFFu));
        x[8 * c + 2 * e + 1] = h2f((uint16_t)(v[e] >> 16));
      }
    }
  } else {
#pragma unroll
    for (unsigned j = 0; j < kGroup; ++j)
      x[j] = j < length ? h2f(group[j]) : 0.0f;
  }
  bool finite;
  scales[i] = quantize_group(x, q + (size_t)i * kGroup, finite);
  if (!finite && invalid)
    atomicOr(invalid, 1u);
}

// residualAdd -> rmsNorm -> quantizeActivation of a row, in three phases that
// the fused launches below share (Reference.metal:105-126, Graph.metal:
// 33-68).
//
// Phase 1: the sum fp16(a + b) (the next residual; written when sum_out is
// given) staged in LDS as fp32, the row padded to whole groups by zeros,
// next to 1 + w. Without b the input row is staged as it is.
template <bool kAdd, unsigned kThreads = 256>
__device__ __forceinline__ void stage_norm_row(const uint16_t *__restrict__ a,
                                               const uint16_t *__restrict__ b, uint16_t *sum_out,
                                               const float *__restrict__ w, float *srow,
                                               float *sw, unsigned width, unsigned padded,
                                               unsigned t) {
  // Eight elements a lane in flight at once: one memory round trip per
  // eight, not per element.
  constexpr unsigned kBatch = 8;
  for (unsigned i0 = 0; i0 < padded; i0 += kBatch * kThreads) {
    uint16_t ha[kBatch], hb[kBatch];
    float wi[kBatch];
#pragma unroll
    for (unsigned j = 0; j < kBatch; ++j) {
      const unsigned i = i0 + j * kThreads + t;
      const bool in = i < width;
      ha[j] = in ? a[i] : (uint16_t)0;
      hb[j] = in && kAdd ? b[i] : (uint16_t)0;
      wi[j] = in ? w[i] : 0.0f;
    }
#pragma unroll
    for (unsigned j = 0; j < kBatch; ++j) {
      const unsigned i = i0 + j * kThreads + t;
      if (i >= padded)
        break;
      float x = 0.0f, w1 = 1.0f;
      if (i < width) {
        uint16_t h = ha[j];
        if (kAdd) {
          h = f2h(__fadd_rn(h2f(h), h2f(hb[j])));
          if (sum_out)
            sum_out[i] = h;
        }
        x = h2f(h);
        w1 = 1.0f + wi[j];
      }
      srow[i] = x;
      sw[i] = w1;
    }
  }
}

// Phase 2 (one lane): the norm's sequential fp32 fma sum over the staged row
// (fma(0, 0, sum) == sum for the padding, sum >= +0).
__device__ __forceinline__ float norm_row_sum(const float *srow, unsigned padded) {
  const float4 *v = reinterpret_cast<const float4 *>(srow);
  float sum = 0.0f;
#pragma unroll 8
  for (unsigned c = 0; c < padded / 4; ++c) {
    const float4 x4 = v[c];
    sum = __builtin_fmaf(x4.x, x4.x, sum);
    sum = __builtin_fmaf(x4.y, x4.y, sum);
    sum = __builtin_fmaf(x4.z, x4.z, sum);
    sum = __builtin_fmaf(x4.w, x4.w, sum);
  }
  return sum;
}

// Phase 3: eight lanes a group, four elements a lane: the group's max |y|
// and finiteness by lane swaps (exact in any order), then each lane
// quantizes its four with the standalone kernel's expressions into q (a
// word per lane) and the group's scale into scales.
template <unsigned kThreads = 256>
__device__ __forceinline__ void quantize_norm_row(const float *srow, const float *sw, float scale,
                                                  unsigned width, unsigned groups, unsigned t,
                                                  uint32_t *q, float *scales, unsigned *invalid) {
  const unsigned sub = t % 8;
  for (unsigned g0 = 0; g0 < groups; g0 += kThreads / 8) {
    const unsigned g = g0 + t / 8;
    const bool live = g < groups;
    const unsigned i0 = (live ? g : 0) * kGroup + 4 * sub;
    float y[4];
    float max_abs = 0.0f;
    bool finite = true;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const unsigned i = i0 + e;
      y[e] = i < width ? normed_f(srow[i], scale, sw[i]) : 0.0f;
      finite = finite && __builtin_isfinite(y[e]);
      max_abs = fmaxf(max_abs, fabsf(y[e]));
    }
#pragma unroll
    for (int m = 1; m < 8; m *= 2) {
      max_abs = fmaxf(max_abs, __shfl_xor(max_abs, m, 8));
      finite = __shfl_xor((int)finite, m, 8) && finite;
    }
    if (!live)
      continue;
    const float qs = finite && max_abs > 0.0f ? __fdiv_rn(max_abs, 127.0f) : 1.0f;
    uint32_t word = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      int r = 0;
      if (finite) {
        const float v = fminf(fmaxf(__fdiv_rn(y[e], qs), -127.0f), 127.0f);
        r = (int)__builtin_rintf(v);
      }
      word |= ((uint32_t)r & 0xFFu) << (8 * e);
    }
    q[g * (kGroup / 4) + sub] = word;
    if (sub == 0) {
      scales[g] = qs;
      if (!finite && invalid)
        atomicOr(invalid, 1u);
    }
  }
}

// The three in one launch, a workgroup per row; the bits equal the three
// launches' (residualAdd, rmsNorm, quantizeActivation).
template <bool kAdd>
__global__ __launch_bounds__(256) void add_norm_quantize_kernel(
    const uint16_t *__restrict__ a, const uint16_t *__restrict__ b, uint16_t *sum_out,
    const float *__restrict__ w, int8_t *__restrict__ q, float *__restrict__ scales,
    unsigned *invalid, unsigned width, unsigned groups, float eps) {
  extern __shared__ __align__(16) float srow[]; // the row, then 1 + w, padded
  __shared__ float sscale;
  const unsigned row = blockIdx.x, t = threadIdx.x;
  const size_t base = (size_t)row * width;
  const unsigned padded = groups * kGroup;
  float *sw = srow + padded;
  stage_norm_row<kAdd>(a + base, kAdd ? b + base : nullptr, kAdd ? sum_out + base : nullptr, w,
                       srow, sw, width, padded, t);
  __syncthreads();
  if (t == 0)
    sscale = rms_scale_of(norm_row_sum(srow, padded), width, eps);
  __syncthreads();
  quantize_norm_row(srow, sw, sscale, width, groups, t,
                    reinterpret_cast<uint32_t *>(q + (size_t)row * groups * kGroup),
                    scales + (size_t)row * groups, invalid);
}

// ------------------------------------------------------------------- GEMV

struct W8Args {
  unsigned outputWidth, firstRow, groups, rows, columns, epilogue, block;
};

// One wave per workgroup (4 columns): even the 2560-column down projection
// spreads over 640 workgroups. A lane requests the weights of 8 of its
// groups (256 bytes) before using any; the activations, read by every
// column, come from L1/L2.
constexpr int kGemvLanes = 16, kGemvThreads = 64, kGemvCols = kGemvThreads / kGemvLanes;
constexpr int kGemvUnroll = 8;

__global__ __launch_bounds__(kGemvThreads) void gemv_kernel(
    const int8_t *__restrict__ act, const float *__restrict__ as, const int8_t *__restrict__ w,
    const uint16_t *__restrict__ ws, void *out, const void *aux, const float *bias, W8Args p) {
  const unsigned col = blockIdx.x * kGemvCols + threadIdx.x / kGemvLanes;
  const unsigned l = threadIdx.x % kGemvLanes;
  float acc = 0.0f;
  if (col < p.columns) {
    const uint4_t *wrow = reinterpret_cast<const uint4_t *>(w + (size_t)col * p.groups * kGroup);
    const uint4_t *arow = reinterpret_cast<const uint4_t *>(act);
    const uint16_t *wsrow = ws + (size_t)col * p.groups;
    for (unsigned g0 = l; g0 < p.groups; g0 += kGemvLanes * kGemvUnroll) {
      uint4_t wv[kGemvUnroll][2];
      float wsv[kGemvUnroll];
#pragma unroll
      for (int u = 0; u < kGemvUnroll; ++u) {
        const unsigned g = min(g0 + kGemvLanes * u, p.groups - 1); // clamped: in bounds
        wv[u][0] = __builtin_nontemporal_load(wrow + 2 * g);
        wv[u][1] = __builtin_nontemporal_load(wrow + 2 * g + 1);
        wsv[u] = h2f(wsrow[g]);
      }
#pragma unroll
      for (int u = 0; u < kGemvUnroll; ++u) {
        const unsigned g = g0 + kGemvLanes * u;
        if (g < p.groups)
          acc = add_term(acc, group_dot(arow[2 * g], arow[2 * g + 1], wv[u][0], wv[u][1]),
                         as[g], wsv[u]);
      }
    }
  }
  // The xor butterfly of the column's 16 lanes (every lane ends with the
  // same sum: fp32 addition is commutative).
#pragma unroll
  for (int m = kGemvLanes / 2; m >= 1; m /= 2)
    acc = __fadd_rn(acc, __shfl_xor(acc, m, kGemvLanes));
  if (l == 0 && col < p.columns) {
    const unsigned column = p.firstRow + col;
    store_linear(out, aux, bias, column, column, p.epilogue, p.block, acc);
  }
}

// Long rows (more than 112 groups: 8 steps a lane or more): four waves share the
// same 4 columns. Wave w computes the group terms (float(dot) * a) * w of the
// w-th quarter of every lane's groups (kPer steps of 16 groups), all its
// loads issued at once, into LDS; wave 0 then adds each lane's terms in
// group order -- the same fp32 sums as one lane would form -- and finishes
// as above. The workgroup's threads first request the activation row and
// its scales, then the weights, and stage the row in LDS once its loads
// (the oldest) are back: read from memory in the dot loop, each step's
// activations waited for the whole weight stream before them and for one
// another. kPer is a template parameter so that every load count is fixed
// and the waits count only what they need.
constexpr int kSplitWaves = 4, kSplitMaxSteps = 64; // groups per lane <= 64
constexpr int kSplitPer = kSplitMaxSteps / kSplitWaves;

template <int kPer>
__global__ __launch_bounds__(64 * kSplitWaves) void gemv_split_kernel(
    const int8_t *__restrict__ act, const float *__restrict__ as, const int8_t *__restrict__ w,
    const uint16_t *__restrict__ ws, void *out, const void *aux, const float *bias, W8Args p) {
  constexpr unsigned kThreads = 64 * kSplitWaves, kGroups = kSplitWaves * kPer * kGemvLanes;
  constexpr int kA = (2 * kGroups + kThreads - 1) / kThreads, kS = (kGroups + kThreads - 1) / kThreads;
  __shared__ float sT[kSplitWaves * kPer][64];
  __shared__ uint4_t sAct[2 * kGroups];
  __shared__ float sAs[kGroups];
  const unsigned tid = threadIdx.x, wave = tid / 64, t = tid % 64;
  const unsigned col = blockIdx.x * kGemvCols + t / kGemvLanes;
  const unsigned l = t % kGemvLanes;
  const unsigned i0 = wave * kPer;
  const unsigned nA = 2 * p.groups; // 16-byte pieces of the row
  const uint4_t *arow = reinterpret_cast<const uint4_t *>(act);
  uint4_t aReg[kA];
  float sReg[kS];
#pragma unroll
  for (int k = 0; k < kA; ++k)
    aReg[k] = arow[min(tid + k * kThreads, nA - 1)]; // clamped: in bounds
#pragma unroll
  for (int k = 0; k < kS; ++k)
    sReg[k] = as[min(tid + k * kThreads, p.groups - 1)];
  asm volatile("" ::: "memory"); // (keeps these loads ahead of the weights')
  // The weights (a column past the end reads the last one and stores
  // nothing); the scales stay fp16 bits, one a register, until the
  // products, so that nothing waits for them here.
  const bool live = col < p.columns;
  const unsigned cc = live ? col : p.columns - 1;
  const uint4_t *wrow = reinterpret_cast<const uint4_t *>(w + (size_t)cc * p.groups * kGroup);
  const uint16_t *wsrow = ws + (size_t)cc * p.groups;
  uint4_t wv[kPer][2];
  uint32_t wsv[kPer];
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    const unsigned g = min(l + kGemvLanes * (i0 + u), p.groups - 1); // clamped: in bounds
    wv[u][0] = __builtin_nontemporal_load(wrow + 2 * g);
    wv[u][1] = __builtin_nontemporal_load(wrow + 2 * g + 1);
    wsv[u] = wsrow[g];
  }
#pragma unroll
  for (int k = 0; k < kA; ++k)
    if (tid + k * kThreads < nA)
      sAct[tid + k * kThreads] = aReg[k];
#pragma unroll
  for (int k = 0; k < kS; ++k)
    if (tid + k * kThreads < p.groups)
      sAs[tid + k * kThreads] = sReg[k];
  lds_sync(); // LDS only: the weights stay in flight
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    const unsigned g = l + kGemvLanes * (i0 + u);
    if (live && g < p.groups)
      sT[i0 + u][t] = __fmul_rn(
          __fmul_rn((float)group_dot(sAct[2 * g], sAct[2 * g + 1], wv[u][0], wv[u][1]), sAs[g]),
          h2f((uint16_t)wsv[u]));
  }
  __syncthreads();
  if (wave != 0)
    return;
  float acc = 0.0f;
  if (col < p.columns)
    for (unsigned i = 0; l + kGemvLanes * i < p.groups; ++i)
      acc = __fadd_rn(acc, sT[i][t]);
#pragma unroll
  for (int m = kGemvLanes / 2; m >= 1; m /= 2)
    acc = __fadd_rn(acc, __shfl_xor(acc, m, kGemvLanes));
  if (l == 0 && col < p.columns) {
    const unsigned column = p.firstRow + col;
    store_linear(out, aux, bias, column, column, p.epilogue, p.block, acc);
  }
}

// ------------------------------------------------------------------- GEMM

// Several rows (prefill, a short message): the group dots come from
// v_mfma_i32_32x32x32_i8, one instruction per 32-row x 32-column tile and
// group (K = 32 is exactly one group, so each int32 result is the group's
// exact dot), and the VALU adds (float(dot) * a) * w to fp32 sums. The
// reference's GEMM gives each output 8 lanes, lane l summing groups l, l + 8,
// ... in order before the xor butterfly; here those 8 lane classes are a
// workgroup's eight waves (wave w the groups g = w mod 8), and the sums meet
// through LDS in the butterfly's order ((c0 + c4) + (c2 + c6)) + ((c1 + c5) +
// (c3 + c7)). So the bits are the reference's.
//
// Bounds: from a few hundred rows the fp32 work that this order demands, per
// output and group a conversion (2.3 ns a wave64 operation a SIMD), two
// products (1.2 each) and an addition (1.5): 36 us for 512 rows of a 2560 ->
// 9216 projection, where the kernel takes 60 to 71; below that the latency of a
// step. So waves in flight decide: a tile a workgroup, 64 registers and 37 KB
// of LDS, four workgroups a CU.
//
// A step covers 8 groups: 256 bytes of each of the tile's 32 activation and 32
// weight rows go HBM -> LDS with buffer loads that write LDS directly, double
// buffered; the scales come through registers, requested a step before they
// are staged. One barrier a step, behind a wait for everything but the last
// request of scales.
// Measured (512 rows of 2560 -> 9216, 512 of 9216 -> 2560, 128 of 2560 ->
// 9216, 13 of 9216 -> 2560):
//   through registers and a padded layout      74.4, 73.4, 24.5, 58.1 us
//   this                                       60.5, 61.1, 19.5, 21.2 us
//   traced, uniform random int8 rows           69.8, 69.6, 23.9, 28.0 us
//   the same, the weights in the MALL          70.4, 70.0, 18.4, 14.5 us
// (the first row's fourth ran a kernel of four rows a lane; the two traced rows
// are of another day's card). Not kept: 64 x 32, 32 x 64
// and 64 x 64 tiles (61 - 65 us at 512 rows with half the loads, but four or
// two waves a SIMD; 33 and 49 us at 13 rows); three and four buffers (64 - 90
// us: fewer workgroups a CU); the row scales by DPP broadcast inside the
// product (a DPP product takes 2.0 ns: 71 us); dots accumulated onto 1.5 x
// 2^23 so that a subtraction stands for the conversion (16 registers more: 67).
//
// Operand layout: lane i supplies row (column) i % 32 of the tile and the
// 16 bytes (i / 32) * 16 of the group for both operands; any K order shared
// by the two operands gives the same exact integer dot. Lane i's results are
// column i % 32 and rows 8 * (r / 4) + 4 * (i / 32) + r % 4 of register r.
//
// Workgroups sharing a column tile run on one XCD (blockIdx % 8 selects the
// XCD), so each weight tile is read from HBM once and then from that XCD's L2.
typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

constexpr unsigned kTile = 32, kGemmThreads = 512;
constexpr unsigned kSpan = 8, kStepBytes = kSpan * kGroup; // groups, bytes of a row a step
constexpr unsigned kScalePitch = kTile + 4;                // staged scales a group
constexpr int kBufferWord3 = 0x00020000;                   // gfx9 raw buffer descriptor, dword 3

typedef __attribute__((address_space(3))) void lds_void_t;

// Direct memory -> LDS load of 16 bytes per lane at base + offset (in bounds
// up to `bytes`): lane i's bytes land at dst + 16 i (dst is wave-uniform).
__device__ __forceinline__ void load_lds16(const void *base, unsigned bytes, unsigned char *dst,
                                           unsigned offset) {
  const __amdgpu_buffer_rsrc_t rsrc =
      __builtin_amdgcn_make_buffer_rsrc((void *)base, (short)0, (int)bytes, kBufferWord3);
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_void_t *)dst, 16, offset, 0, 0, 0);
}

__global__ __launch_bounds__(kGemmThreads, 4) void gemm_kernel(
    const int8_t *__restrict__ act, const float *__restrict__ as, const int8_t *__restrict__ w,
    const uint16_t *__restrict__ ws, void *out, const void *aux, const float *bias, W8Args p,
    unsigned rowTiles) {
  // Two buffers (the activation rows, then the weight rows), named one by one
  // so that the compiler can tell the loads in flight from the LDS reads.
  __shared__ __align__(1024) unsigned char s0[2 * kTile * kStepBytes], s1[2 * kTile * kStepBytes];
  __shared__ __align__(16) float sc[2][2 * kSpan * kScalePitch];
  const unsigned nwg = gridDim.x, x = blockIdx.x % 8;
  const unsigned v = x * (nwg / 8) + min(x, nwg % 8) + blockIdx.x / 8;
  const unsigned row0 = (v % rowTiles) * kTile, col0 = (v / rowTiles) * kTile;
  const unsigned tid = threadIdx.x, lane = tid % 64;
  const unsigned wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const unsigned k = p.groups * kGroup;
  const unsigned nsteps = (p.groups + kSpan - 1) / kSpan;

  // A wave moves four rows of each operand, a lane 16 bytes of one: slot s of
  // row r holds chunk s ^ (r % 16), so the operand reads (32 rows, one chunk)
  // meet no bank conflicts. Past a row's end the reads give the next row's
  // bytes or, past the tensor's, nothing: groups that no wave uses.
  const unsigned srow = 4 * wave + lane / 16, schunk = (lane % 16) ^ (srow % 16);
  unsigned oa = min(row0 + srow, p.rows - 1) * k + 16 * schunk;
  unsigned ob = min(col0 + srow, p.columns - 1) * k + 16 * schunk;
  auto load = [&](unsigned char *to) { // the next step
    load_lds16(act, p.rows * k, to + 4 * wave * kStepBytes, oa);
    load_lds16(w, p.columns * k, to + (kTile + 4 * wave) * kStepBytes, ob);
    oa += kStepBytes;
    ob += kStepBytes;
  };
  // The first four waves an activation scale a thread, the others a weight's.
  const bool act_scaler = wave < 4;
  const unsigned sr = (tid % 256) / 8, sg = tid % 8;
  const unsigned os = (act_scaler ? min(row0 + sr, p.rows - 1) : min(col0 + sr, p.columns - 1)) *
                      p.groups;
  uint32_t rs; // fp32 or fp16 bits as loaded
  auto load_scale = [&](unsigned step) {
    const unsigned g = min(step * kSpan + sg, p.groups - 1); // clamped past the end
    if (act_scaler)
      rs = reinterpret_cast<const uint32_t *>(as)[os + g];
    else
      rs = ws[os + g];
  };
  auto stage_scale = [&](float *to) {
    if (act_scaler)
      to[sg * kScalePitch + sr] = __uint_as_float(rs);
    else
      to[(kSpan + sg) * kScalePitch + sr] = h2f((uint16_t)rs);
  };

  const unsigned m = lane % kTile, h = lane / kTile;
  const unsigned from = m * kStepBytes + 16 * ((2 * wave + h) ^ (m % 16));
  const v16i zero = {};
  float acc[16];
#pragma unroll
  for (int r = 0; r < 16; ++r)
    acc[r] = 0.0f;
  // One step of this wave's group.
  auto compute = [&](const unsigned char *st, const float *scl) {
    const v4i a = *reinterpret_cast<const v4i *>(st + from);
    const v4i b = *reinterpret_cast<const v4i *>(st + kTile * kStepBytes + from);
    const float wsv = scl[(kSpan + wave) * kScalePitch + m];
    const v16i dots = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, zero, 0, 0, 0);
    const float4 *sa = reinterpret_cast<const float4 *>(scl + wave * kScalePitch + 4 * h);
    float4 a4[4];
#pragma unroll
    for (int q = 0; q < 4; ++q)
      a4[q] = sa[2 * q];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      acc[4 * q + 0] = add_term(acc[4 * q + 0], dots[4 * q + 0], a4[q].x, wsv);
      acc[4 * q + 1] = add_term(acc[4 * q + 1], dots[4 * q + 1], a4[q].y, wsv);
      acc[4 * q + 2] = add_term(acc[4 * q + 2], dots[4 * q + 2], a4[q].z, wsv);
      acc[4 * q + 3] = add_term(acc[4 * q + 3], dots[4 * q + 3], a4[q].w, wsv);
    }
  };
  // A step: the next one's loads go out, this one's arithmetic runs, and once
  // this wave's loads have landed (the next step's rows and its scale, requested
  // a step ago) that scale is staged and the one after requested, which alone
  // is in flight at the barrier: it ends in a register.
  auto landed = [] { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); };
  auto run = [&](unsigned step, const unsigned char *st, unsigned char *next) {
    if (step + 1 < nsteps)
      load(next);
    if (step * kSpan + wave < p.groups)
      compute(st, sc[step % 2]);
    landed();
    stage_scale(sc[(step + 1) % 2]);
    load_scale(step + 2);
    lds_sync();
  };
  load(s0);
  load_scale(0);
  landed();
  stage_scale(sc[0]);
  load_scale(1);
  lds_sync();
  for (unsigned step = 0; step < nsteps; step += 2) {
    run(step, s0, s1);
    if (step + 1 < nsteps)
      run(step + 1, s1, s0);
  }

  // The classes of half a tile (16 rows) at a time meet in LDS, in the
  // butterfly's order.
  float *sums = reinterpret_cast<float *>(s0);
  constexpr unsigned T = kTile * kTile / 2;
  static_assert(sizeof s0 >= kSpan * T * sizeof(float) && T == kGemmThreads, "half a tile");
#pragma unroll
  for (int half = 0; half < 2; ++half) {
    if (half)
      lds_sync();
#pragma unroll
    for (int r = 0; r < 8; ++r)
      sums[wave * T + (8 * (r / 4) + 4 * h + r % 4) * kTile + m] = acc[8 * half + r];
    lds_sync();
    const unsigned row = row0 + 16 * half + tid / kTile, col = col0 + tid % kTile;
    if (row < p.rows && col < p.columns) {
      const float *c = sums + tid;
      const float total =
          __fadd_rn(__fadd_rn(__fadd_rn(c[0], c[4 * T]), __fadd_rn(c[2 * T], c[6 * T])),
                    __fadd_rn(__fadd_rn(c[T], c[5 * T]), __fadd_rn(c[3 * T], c[7 * T])));
      const unsigned column = p.firstRow + col;
      store_linear(out, aux, bias, (size_t)row * p.outputWidth + column, column, p.epilogue,
                   p.block, total);
    }
  }
}

// ------------------------------------------------- norm + projections, decode

// residualAdd -> rmsNorm -> quantizeActivation of one row and up to four
// W8A8 projections of the quantized row in one launch (the decode step's
// input norms and the projections that read them). The norm's sequential
// sum is one lane's latency-bound chain (~11 us at width 2560) while the
// projections stream their weights: in each 1024-thread workgroup, wave 0
// stages nothing but the norm (every workgroup forms the same bits) and
// runs the chain as soon as the row is in LDS, while waves 1-15 issue their
// weight loads (a wave issues its loads in order, so the chain wave issues
// none: measured, issuing 160 KB of loads a CU takes ~3 us). Waves 1-15
// serve 60 columns of one projection with the GEMV's lanes (16 a column,
// lane l the groups l, l + 16, ...: kLaneGroups of them, 5 up to width 2560,
// 8 up to 4096, one unrolled step) and its arithmetic, so the outputs are
// the separate launches' bits. A paired projection (kPaired, width <= 2560)
// also computes the next one, a SwiGLU projection whose multiplier is this
// one's output, in the same lanes: its weights sit beside the first's and
// the multiplier comes from registers. One workgroup a CU keeps one chain a
// CU (chains sharing a SIMD slow each other down).
constexpr unsigned kNormLinearThreads = 64 + kNormLinearCols * kGemvLanes;
static_assert(kNormLinearThreads == 1024, "the norm wave and 60 columns of 16 lanes");
static_assert(kNormLinearMaxWidth == kGroup * kGemvLanes * 8, "8 groups a lane at most");
static_assert(kNormLinearPairedWidth == kGroup * kGemvLanes * 5, "5 groups a lane paired");

struct NormLinearSeg {
  const int8_t *w;
  const uint16_t *ws;
  void *out;
  const void *aux;
  const float *bias;
  unsigned columns, outputWidth, firstRow, epilogue, block, wgs, paired;
  const uint16_t *cw; // the one-token convolution + SiLU, or null
  uint16_t *ch;
};

// causalConv with applySilu (Reference.metal:137-161) of one token for
// channel c, whose input is the projection's fp32 sum: the input is its
// fp16 rounding, the window the channel's three history values and the
// input, the sum the product of the newest term followed by the fmas of
// the older ones (causal_conv_k4's order), and the history shifts by one.
__device__ __forceinline__ void store_conv_silu(uint16_t *out, const uint16_t *cw, uint16_t *ch,
                                                unsigned c, float acc) {
  const float x = round16(acc);
  const uint16_t h0 = ch[3 * c], h1 = ch[3 * c + 1], h2 = ch[3 * c + 2];
  float y = mul32(x, h2f(cw[4 * c + 3]));
  y = __builtin_fmaf(h2f(h0), h2f(cw[4 * c]), y);
  y = __builtin_fmaf(h2f(h1), h2f(cw[4 * c + 1]), y);
  y = __builtin_fmaf(h2f(h2), h2f(cw[4 * c + 2]), y);
  out[c] = silu16(round16(y));
  ch[3 * c] = h1;
  ch[3 * c + 1] = h2;
  ch[3 * c + 2] = f2h(x);
}

struct NormLinearArgs {
  NormLinearSeg seg[kNormLinearMax];
  unsigned count, width, groups;
  float eps;
  unsigned cols; // columns a workgroup (a multiple of 4, at most 60)
};

// One column's weights for a lane: its kLaneGroups groups (clamped: in
// bounds) and their scales, kept as loaded (fp16 bits): converted where the
// dots use them, so that nothing before then waits for the loads (the norm
// wave issues its own before its chain).
template <int kLaneGroups>
__device__ __forceinline__ void load_lane_weights(const NormLinearSeg &seg, unsigned cc,
                                                  unsigned l, unsigned groups,
                                                  uint4_t (&wv)[kLaneGroups][2],
                                                  uint16_t (&wsv)[kLaneGroups]) {
  const uint4_t *wrow = reinterpret_cast<const uint4_t *>(seg.w + (size_t)cc * groups * kGroup);
  const uint16_t *wsrow = seg.ws + (size_t)cc * groups;
#pragma unroll
  for (int u = 0; u < kLaneGroups; ++u) {
    const unsigned g = min(l + kGemvLanes * u, groups - 1);
    wv[u][0] = __builtin_nontemporal_load(wrow + 2 * g);
    wv[u][1] = __builtin_nontemporal_load(wrow + 2 * g + 1);
    wsv[u] = wsrow[g];
  }
}

// The lane's fp32 sum in group order, then the column's butterfly.
template <int kLaneGroups>
__device__ __forceinline__ float lane_dots(const uint4_t *arow, const float *ss, unsigned l,
                                           unsigned groups, const uint4_t (&wv)[kLaneGroups][2],
                                           const uint16_t (&wsv)[kLaneGroups]) {
  float acc = 0.0f;
#pragma unroll
  for (int u = 0; u < kLaneGroups; ++u) {
    const unsigned g = l + kGemvLanes * u;
    // pinned here (volatile asm keeps its place after the workgroup's
    // barriers): the backend otherwise converts the loaded scale right
    // after its load, which makes the norm wave wait for its weights
    // before its chain
    uint32_t bits = wsv[u];
    asm volatile("" : "+v"(bits));
    if (g < groups)
      acc = add_term(acc, group_dot(arow[2 * g], arow[2 * g + 1], wv[u][0], wv[u][1]), ss[g],
                     h2f((uint16_t)bits));
  }
#pragma unroll
  for (int m = kGemvLanes / 2; m >= 1; m /= 2)
    acc = __fadd_rn(acc, __shfl_xor(acc, m, kGemvLanes));
  return acc;
}

template <bool kAdd, int kLaneGroups, bool kPaired>
__global__ __launch_bounds__(kNormLinearThreads) void norm_linear_kernel(
    const uint16_t *__restrict__ a, const uint16_t *__restrict__ b, uint16_t *sum_out,
    const float *__restrict__ nw, int8_t *q, float *scales, unsigned *invalid,
    NormLinearArgs p) {
  extern __shared__ __align__(16) float srow[]; // row, 1 + w, quantized words, scales
  __shared__ float sscale;
  const unsigned t = threadIdx.x, padded = p.groups * kGroup;
  float *sw = srow + padded;
  uint32_t *sq = reinterpret_cast<uint32_t *>(sw + padded);
  float *ss = reinterpret_cast<float *>(sq + p.groups * (kGroup / 4));
  unsigned blk = blockIdx.x, s = 0;
  bool found = false;
#pragma unroll
  for (unsigned k = 0; k < kNormLinearMax; ++k)
    if (!found && k < p.count) {
      if (blk < p.seg[k].wgs) {
        s = k;
        found = true;
      } else {
        blk -= p.seg[k].wgs;
      }
    }
  // selected with constant indices (no private copy of the table)
  NormLinearSeg seg = p.seg[0], mate = p.seg[0];
#pragma unroll
  for (unsigned k = 1; k < kNormLinearMax; ++k) {
    if (k == s)
      seg = p.seg[k];
    if (kPaired && k == s + 1)
      mate = p.seg[k];
  }
  const bool paired = kPaired && seg.paired;
  const bool norm_wave = t < 64;
  // waves 1-15 serve four columns each, as many as the launch gives a
  // workgroup; the others only help stage and quantize the row
  const unsigned lane_col = (t - 64) / kGemvLanes; // (wraps for the norm wave)
  const unsigned col = blk * p.cols + lane_col;
  const unsigned l = t % kGemvLanes;
  const bool serves = !norm_wave && lane_col < p.cols; // a wave with columns
  const bool live = serves && col < seg.columns;
  const unsigned cc = live ? col : 0; // clamped: in bounds

  // The row, then (waves 1-15) the weights or (wave 0) the chain. The
  // barriers order LDS only: a __syncthreads would wait for the weight
  // stream.
  const bool first = blockIdx.x == 0; // writes the sum, q, scales and the flag
  stage_norm_row<kAdd, kNormLinearThreads>(a, b, first ? sum_out : nullptr, nw, srow, sw,
                                           p.width, padded, t);
  lds_sync();
  uint4_t wv[kLaneGroups][2], mv[kPaired ? kLaneGroups : 1][2];
  uint16_t wsv[kLaneGroups], msv[kPaired ? kLaneGroups : 1];
  if (serves) {
    load_lane_weights<kLaneGroups>(seg, cc, l, p.groups, wv, wsv);
    if constexpr (kPaired)
      if (paired)
        load_lane_weights<kLaneGroups>(mate, cc, l, p.groups, mv, msv);
  }
  if (norm_wave && t == 0)
    sscale = rms_scale_of(norm_row_sum(srow, padded), p.width, p.eps);
  lds_sync();
  quantize_norm_row<kNormLinearThreads>(srow, sw, sscale, p.width, p.groups, t, sq, ss,
                                        first ? invalid : nullptr);
  lds_sync();
  if (first && q)
    for (unsigned i = t; i < p.groups * (kGroup / 4); i += kNormLinearThreads)
      reinterpret_cast<uint32_t *>(q)[i] = sq[i];
  if (first && scales)
    for (unsigned i = t; i < p.groups; i += kNormLinearThreads)
      scales[i] = ss[i];

  if (!serves)
    return;
  const uint4_t *arow = reinterpret_cast<const uint4_t *>(sq);
  const float acc = lane_dots<kLaneGroups>(arow, ss, l, p.groups, wv, wsv);
  if constexpr (kPaired) {
    if (paired) {
      const float macc = lane_dots<kLaneGroups>(arow, ss, l, p.groups, mv, msv);
      if (l == 0 && live) {
        // the first projection has no epilogue: its fp16 output is the
        // SwiGLU multiplier
        const float projected = round16(acc);
        static_cast<uint16_t *>(seg.out)[seg.firstRow + col] = f2h(projected);
        static_cast<uint16_t *>(mate.out)[mate.firstRow + col] =
            silu_mul16(round16(macc), f2h(projected));
      }
      return;
    }
  }
  if (l == 0 && live) {
    const unsigned column = seg.firstRow + col;
    if (seg.cw)
      store_conv_silu(static_cast<uint16_t *>(seg.out), seg.cw, seg.ch, column, acc);
    else
      store_linear(seg.out, seg.aux, seg.bias, column, column, seg.epilogue, seg.block, acc);
  }
}

// ------------------------------------------------------------- embeddings

// embeddingW8 (Graph.metal:16-31): eight outputs per lane (they share a
// 32-wide scale group when hidden is a multiple of 8), or one.
__global__ __launch_bounds__(256) void embedding_w8_kernel(
    const uint32_t *__restrict__ ids, const int8_t *__restrict__ w,
    const uint16_t *__restrict__ sc, uint16_t *__restrict__ out, unsigned tokens,
    unsigned hidden, unsigned first, unsigned count, unsigned groups, unsigned per) {
  const size_t i0 = ((size_t)blockIdx.x * 256 + threadIdx.x) * per;
  if (i0 >= (size_t)tokens * hidden)
    return;
  const uint32_t id = ids[i0 / hidden];
  if (id < first || id - first >= count)
    return;
  const size_t row = id - first;
  const unsigned c0 = (unsigned)(i0 % hidden);
  if (per == 8) {
    const uint2 q = *reinterpret_cast<const uint2 *>(w + row * groups * kGroup + c0);
    const float s = h2f(sc[row * groups + c0 / kGroup]);
    uint4_t o;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t word = e < 2 ? q.x : q.y;
      const int8_t lo = (int8_t)(word >> (16 * (e % 2))), hi = (int8_t)(word >> (16 * (e % 2) + 8));
      o[e] = (uint32_t)f2h(mul32((float)lo, s)) | ((uint32_t)f2h(mul32((float)hi, s)) << 16);
    }
    *reinterpret_cast<uint4_t *>(out + i0) = o;
  } else {
    out[i0] = f2h(mul32((float)w[row * groups * kGroup + c0], h2f(sc[row * groups + c0 / kGroup])));
  }
}

// embedding (Reference.metal:49-58).
__global__ __launch_bounds__(256) void embedding_kernel(const uint32_t *__restrict__ ids,
                                                        const uint16_t *__restrict__ w,
                                                        uint16_t *__restrict__ out,
                                                        unsigned tokens, unsigned hidden,
                                                        unsigned first, unsigned count,
                                                        unsigned per) {
  const size_t i0 = ((size_t)blockIdx.x * 256 + threadIdx.x) * per;
  if (i0 >= (size_t)tokens * hidden)
    return;
  const uint32_t id = ids[i0 / hidden];
  if (id < first || id - first >= count)
    return;
  const size_t src = (size_t)(id - first) * hidden + i0 % hidden;
  if (per == 8)
    *reinterpret_cast<uint4_t *>(out + i0) = *reinterpret_cast<const uint4_t *>(w + src);
  else
    out[i0] = w[src];
}

} // namespace

hipError_t launch_quantize_activation(const uint16_t *in, int8_t *q, float *scales,
                                      unsigned *invalid, unsigned rows, unsigned width,
                                      unsigned groups, hipStream_t stream) {
  const unsigned n = rows * groups;
  const bool vec = width % kGroup == 0 && aligned16(in);
  if (vec) {
    const unsigned chunks = n * (kGroup / 8);
    hipLaunchKernelGGL(quantize_chunks_kernel, dim3((chunks + 255) / 256), dim3(256), 0, stream,
                       in, q, scales, invalid, chunks);
  } else {
    hipLaunchKernelGGL(quantize_kernel, dim3((n + 255) / 256), dim3(256), 0, stream, in, q,
                       scales, invalid, rows, width, groups, vec);
  }
  return hipGetLastError();
}

hipError_t launch_add_norm_quantize(const uint16_t *a, const uint16_t *b, uint16_t *sum_out,
                                   const float *w, int8_t *q, float *scales, unsigned *invalid,
                                   unsigned rows, unsigned width, float eps, hipStream_t stream) {
  const unsigned groups = (width + kGroup - 1) / kGroup;
  const size_t lds = 2 * (size_t)groups * kGroup * sizeof(float);
  if (b)
    hipLaunchKernelGGL(add_norm_quantize_kernel<true>, dim3(rows), dim3(256), lds, stream, a, b,
                       sum_out, w, q, scales, invalid, width, groups, eps);
  else
    hipLaunchKernelGGL(add_norm_quantize_kernel<false>, dim3(rows), dim3(256), lds, stream, a,
                       b, sum_out, w, q, scales, invalid, width, groups, eps);
  return hipGetLastError();
}

// Compute units of the current device (256 on MI355X), read once a device.
static unsigned device_cus() {
  static int cus[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64)
    return 256;
  if (cus[dev] <= 0) {
    int c = 0;
    cus[dev] = hipDeviceGetAttribute(&c, hipDeviceAttributeMultiprocessorCount, dev) ==
                           hipSuccess && c > 0
                   ? c
                   : 256;
  }
  return (unsigned)cus[dev];
}

template <bool kAdd, int kLaneGroups, bool kPaired>
static void launch_norm_linear_as(const uint16_t *a, const uint16_t *b, uint16_t *sum_out,
                                  const float *w, int8_t *q, float *scales, unsigned *invalid,
                                  const NormLinearArgs &p, unsigned wgs, size_t lds,
                                  hipStream_t stream) {
  hipLaunchKernelGGL((norm_linear_kernel<kAdd, kLaneGroups, kPaired>), dim3(wgs),
                     dim3(kNormLinearThreads), lds, stream, a, b, sum_out, w, q, scales, invalid,
                     p);
}

hipError_t launch_add_norm_linear(const uint16_t *a, const uint16_t *b, uint16_t *sum_out,
                                  const float *w, int8_t *q, float *scales, unsigned *invalid,
                                  unsigned width, float eps, const NormLinearProj *proj,
                                  unsigned count, hipStream_t stream) {
  NormLinearArgs p{};
  p.count = count;
  p.width = width;
  p.groups = (width + kGroup - 1) / kGroup;
  p.eps = eps;
  unsigned wgs = 0;
  bool paired = false;
  // The fewest columns a workgroup (a multiple of 4) that still fit the
  // launch in one workgroup a CU: each workgroup's weight stream is then
  // the shortest, with every CU streaming (at 60 columns the MLP's 9216
  // fill 154 CUs, whose streams outlast the norm's chain).
  unsigned perWg = kNormLinearCols;
  const unsigned cus = device_cus();
  for (unsigned c = 4; c < kNormLinearCols; c += 4) {
    unsigned n = 0;
    for (unsigned k = 0; k < count; ++k)
      if (!(k > 0 && proj[k - 1].paired))
        n += (proj[k].shape.columns + c - 1) / c;
    if (n <= cus) {
      perWg = c;
      break;
    }
  }
  p.cols = perWg;
  for (unsigned k = 0; k < count; ++k) {
    const NormLinearProj &x = proj[k];
    const bool mate = k > 0 && proj[k - 1].paired;
    p.seg[k] = {x.w, x.ws, x.out, x.aux, x.bias, x.shape.columns, x.shape.outputWidth,
                x.shape.firstRow, x.shape.epilogue, x.shape.block,
                mate ? 0u : (x.shape.columns + perWg - 1) / perWg, x.paired ? 1u : 0u,
                x.cw, x.ch};
    wgs += p.seg[k].wgs;
    paired = paired || x.paired;
  }
  const size_t lds = 2 * (size_t)p.groups * kGroup * sizeof(float) + (size_t)p.groups * kGroup +
                     (size_t)p.groups * sizeof(float);
  const bool five = width <= kNormLinearPairedWidth;
  if (b) {
    if (paired)
      launch_norm_linear_as<true, 5, true>(a, b, sum_out, w, q, scales, invalid, p, wgs, lds,
                                           stream);
    else if (five)
      launch_norm_linear_as<true, 5, false>(a, b, sum_out, w, q, scales, invalid, p, wgs, lds,
                                            stream);
    else
      launch_norm_linear_as<true, 8, false>(a, b, sum_out, w, q, scales, invalid, p, wgs, lds,
                                            stream);
  } else {
    if (paired)
      launch_norm_linear_as<false, 5, true>(a, b, sum_out, w, q, scales, invalid, p, wgs, lds,
                                            stream);
    else if (five)
      launch_norm_linear_as<false, 5, false>(a, b, sum_out, w, q, scales, invalid, p, wgs, lds,
                                             stream);
    else
      launch_norm_linear_as<false, 8, false>(a, b, sum_out, w, q, scales, invalid, p, wgs, lds,
                                             stream);
  }
  return hipGetLastError();
}

const char *linear_w8a8_kernel(unsigned rows) {
  return rows == 1 ? "linearW8A8Gemv" : "linearW8A8Gemm";
}

// The split GEMV for kPer steps a wave (2 .. kSplitPer).
template <int kPer>
static void launch_gemv_split_as(dim3 grid, hipStream_t stream, const int8_t *act, const float *as,
                                 const int8_t *w, const uint16_t *ws, void *out, const void *aux,
                                 const float *bias, const W8Args &a) {
  hipLaunchKernelGGL(gemv_split_kernel<kPer>, grid, dim3(64 * kSplitWaves), 0, stream, act, as, w,
                     ws, out, aux, bias, a);
}

template <int kPer = kSplitPer>
static void launch_gemv_split(unsigned per, dim3 grid, hipStream_t stream, const int8_t *act,
                              const float *as, const int8_t *w, const uint16_t *ws, void *out,
                              const void *aux, const float *bias, const W8Args &a) {
  if constexpr (kPer > 2)
    if (per < (unsigned)kPer)
      return launch_gemv_split<kPer - 1>(per, grid, stream, act, as, w, ws, out, aux, bias, a);
  launch_gemv_split_as<kPer>(grid, stream, act, as, w, ws, out, aux, bias, a);
}

hipError_t launch_linear_w8a8(const int8_t *act, const float *as, const int8_t *w,
                              const uint16_t *ws, void *out, const void *aux, const float *bias,
                              const W8Shape &s, hipStream_t stream) {
  const W8Args a{s.outputWidth, s.firstRow, s.groups, s.rows, s.columns, s.epilogue, s.block};
  const unsigned steps = (s.groups + kGemvLanes - 1) / kGemvLanes;
  if (s.rows == 1 && steps >= kGemvUnroll && steps <= kSplitMaxSteps)
    launch_gemv_split((steps + kSplitWaves - 1) / kSplitWaves,
                      dim3((s.columns + kGemvCols - 1) / kGemvCols), stream, act, as, w, ws, out,
                      aux, bias, a);
  else if (s.rows == 1)
    hipLaunchKernelGGL(gemv_kernel, dim3((s.columns + kGemvCols - 1) / kGemvCols),
                       dim3(kGemvThreads), 0, stream, act, as, w, ws, out, aux, bias, a);
  else {
    const unsigned rowTiles = (s.rows + kTile - 1) / kTile;
    hipLaunchKernelGGL(gemm_kernel, dim3(rowTiles * ((s.columns + kTile - 1) / kTile)),
                       dim3(kGemmThreads), 0, stream, act, as, w, ws, out, aux, bias, a, rowTiles);
  }
  return hipGetLastError();
}

hipError_t launch_embedding_w8(const uint32_t *ids, const int8_t *w, const uint16_t *sc,
                               uint16_t *out, unsigned tokens, unsigned hidden, unsigned first,
                               unsigned count, unsigned groups, hipStream_t stream) {
  const unsigned per = hidden % 8 == 0 && aligned16(out) && aligned16(w) ? 8u : 1u;
  const size_t n = ((size_t)tokens * hidden + per - 1) / per;
  hipLaunchKernelGGL(embedding_w8_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream,
                     ids, w, sc, out, tokens, hidden, first, count, groups, per);
  return hipGetLastError();
}

hipError_t launch_embedding(const uint32_t *ids, const uint16_t *w, uint16_t *out,
                            unsigned tokens, unsigned hidden, unsigned first, unsigned count,
                            hipStream_t stream) {
  const unsigned per = hidden % 8 == 0 && aligned16(out) && aligned16(w) ? 8u : 1u;
  const size_t n = ((size_t)tokens * hidden + per - 1) / per;
  hipLaunchKernelGGL(embedding_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream,
                     ids, w, out, tokens, hidden, first, count, per);
  return hipGetLastError();
}

} // namespace llmi
