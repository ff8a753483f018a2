// Causal GQA prefill (flash attention) on fp16 MFMA for gfx950.
//
// Replaces gqaFlashAttention (FlashAttention.metal:1-83), which runs one query
// per SIMD group with a scalar per-key reduction. Here:
//
//  * one workgroup = (block of 32 query tokens, KV head, HW query heads of
//    that head's group); wave w computes query head kvh*G + grp*HW + w for the
//    32 tokens, so the waves share every K/V tile staged in LDS.
//  * K/V tiles of 64 keys go HBM -> LDS with buffer loads that write LDS
//    directly (no register staging), double-buffered: tile i+1 is in flight
//    while tile i is consumed. The buffer descriptor's range ends at the
//    block's last visible key, so rows past it read as zero without any
//    per-lane clamping.
//  * LDS rows are XOR-swizzled in 16-byte chunks so the MFMA operand reads
//    are free of bank conflicts: K chunk c of row j sits at c ^ (j % 8), V
//    chunk c of row j at c ^ 2(j % 4).
//  * scores are computed transposed, S^T = K Q^T, with
//    v_mfma_f32_32x32x16_f16: each lane owns one query row (lane % 32) and 32
//    of the tile's keys; the row max needs one exchange with lane ^ 32.
//  * O^T += V^T P^T on the same MFMA; its V^T operand comes straight from
//    the row-major V tile through ds_read_b64_tr_b16 (transposing LDS read),
//    and P^T is the probability tile converted to fp16 in registers.
//  * softmax with a lazily moved reference: probabilities are
//    exp2(s*c - m) with m only raised when a row's maximum would push a
//    probability past 2^15 (then m = max - 7). O and l are rescaled only on
//    such a raise, which after the first tiles is rare; probabilities stay
//    <= 2^15 (fp16-safe) and at least 2^-14 down to 21 binades below the
//    row maximum, so the MFMA sees no fp16 subnormals where they matter.
//  * PV of tile i-1 is issued after the scores of tile i, so its MFMAs
//    overlap the softmax arithmetic of tile i.
//
// At head_dim 256 with four query heads per KV head, grids of 64 workgroups
// or more run gqa_prefill_halves_kernel instead: the single-wave kernel
// needs ~500 registers per lane, one wave per SIMD, and a lone wave cannot
// hide its LDS operand reads behind its MFMAs (measured on gfx950: 55-60
// cycles per 32x32x16 MFMA with a 1 KB operand read each, against 38 with a
// second wave on the SIMD and the reads two MFMAs ahead). The key-split
// kernel gives each head a wave pair that splits the keys, at 248 registers.
//
// A grid that leaves CUs idle on a long history divides the keys over several
// workgroups (SPLIT, split_plan): each leaves its partials in the caller's
// workspace and gqa_prefill_merge_kernel combines and gates them.
//
// The gated call's query rows are normalised by a launch of their own, into
// the output (launch_attention_rows): inside these kernels, one or two waves a
// SIMD, that work took 11 us (333 tokens, traced: 45.3 us with it, 34.8 without,
// 29.0 where the gates are already activated, 20.1 for the attention alone).
#include "hip_common.hpp"
#include "kernels.hpp"
#include "rope_gate.hpp"

#include <algorithm>
#include <math.h>
#include <stdlib.h>
#include <type_traits>

namespace llmi {
namespace {

constexpr int BM = 32;            // query tokens per wave (= MFMA N)
constexpr int BN = 64;            // keys per tile
constexpr int kBufferWord3 = 0x00020000; // gfx9 raw buffer descriptor, dword 3
constexpr float kRaise = 15.0f;   // raise m when a probability would exceed 2^15
constexpr float kHeadroom = 7.0f; // after a raise the largest probability is 2^7

typedef __attribute__((address_space(3))) void lds_void_t;
typedef __fp16 fp16x4_t __attribute__((__vector_size__(4 * sizeof(__fp16))));
typedef __attribute__((address_space(3))) fp16x4_t lds_fp16x4_t;

// Direct HBM -> LDS load of 16 bytes per lane: lane i's bytes land at
// dst + 16 i (dst is wave-uniform).
__device__ __forceinline__ void load_lds16(__amdgpu_buffer_rsrc_t rsrc, char *dst,
                                           unsigned voffset) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_void_t *)dst, 16, voffset, 0, 0, 0);
}

// Hides a value's known bit range from the compiler, so that adding a
// constant to it stays an add (folded into the LDS instruction's offset
// field) instead of becoming an OR of disjoint bits computed on the VALU.
__device__ __forceinline__ void opaque(unsigned &x) { asm volatile("" : "+v"(x)); }

__device__ __forceinline__ void wait_loads() {
  __builtin_amdgcn_s_waitcnt(0x0F70); // vmcnt(0)
}

// ds_read_b64_tr_b16: in each 16-lane group, lane j receives element j % 4 of
// the 8-byte chunks addressed by lanes j/4, 4 + j/4, 8 + j/4, 12 + j/4.
__device__ __forceinline__ half4_t read_tr(const char *base, unsigned off) {
  typedef __attribute__((address_space(3))) char lds_char_t;
  return __builtin_bit_cast(half4_t, __builtin_amdgcn_ds_read_tr16_b64_v4f16(
                                         (lds_fp16x4_t *)((lds_char_t *)base + off)));
}

// The sigmoid gate of one lane's 16 outputs of a 32-channel tile (the
// four half4 groups at g + 8 i): the fast logistic first, then the exact one
// for the few that miss the margin test, one per pass of the wave (as the
// standalone gate kernel does). activated: the gate values are already
// fp16(logistic(.)), and the output is their plain product (multiplyF16).
template <int N = 4>
__device__ __forceinline__ void gate_tile(half4_t (&v)[N], const half_t *g4p, bool activated) {
  float g[4 * N], sg[4 * N];
  unsigned need = 0;
#pragma unroll
  for (int g4 = 0; g4 < N; ++g4) {
    const half4_t gv = *reinterpret_cast<const half4_t *>(g4p + 8 * g4);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      g[4 * g4 + e] = (float)gv[e];
      sg[4 * g4 + e] = activated ? g[4 * g4 + e] : logistic_estimate(g[4 * g4 + e]);
      need |= activated || f16_settled(sg[4 * g4 + e]) ? 0u : 1u << (4 * g4 + e);
    }
  }
  while (need) {
    const unsigned k = __builtin_ctz(need);
    need &= need - 1;
    float gk = g[0];
#pragma unroll
    for (int e = 1; e < 4 * N; ++e)
      gk = k == (unsigned)e ? g[e] : gk;
    const float sk = logistic_exact(gk);
#pragma unroll
    for (int e = 0; e < 4 * N; ++e)
      sg[e] = k == (unsigned)e ? sk : sg[e];
  }
#pragma unroll
  for (int g4 = 0; g4 < N; ++g4)
#pragma unroll
    for (int e = 0; e < 4; ++e)
      v[g4][e] = __builtin_bit_cast(half_t, f2h(mul32(round16(sg[4 * g4 + e]), (float)v[g4][e])));
}

struct NoArgs {}; // an argument the kernel's form does not take

// GATED: the projected rows (per head D query values, then D gate values)
// whose gates the output goes through.
struct GateArgs {
  const half_t *qproj;
  unsigned activated;
};

// A split launch's partials: for each (split, token block, query head) the
// block's 32 row references m and denominators l, and the unnormalised
// O^T / (2^m) tile as the kernels hold it ([output tile][register][lane]).
struct SplitArgs {
  float *ml, *o;
  unsigned splits;
};
// A split launch's workgroups in order of their keys: those that read the
// same ones (a KV head's split: its head groups and row blocks) run side by
// side on one XCD (blockIdx % 8 selects it), whose L2 then serves all but the
// first (61 tokens on 16411 past rows, cold: 34.7 -> 30.2 us against a KV
// head's head pairs on XCDs of their own).
struct SplitPlace {
  unsigned split, kvh, heads, rows;
};
__device__ __forceinline__ SplitPlace split_place(unsigned Hkv, unsigned groups, unsigned blocks) {
  const unsigned nwg = gridDim.x, x = blockIdx.x % 8, members = groups * blocks;
  const unsigned v = x * (nwg / 8) + min(x, nwg % 8) + blockIdx.x / 8;
  const unsigned m = v % members, g = v / members;
  return {g / Hkv, g % Hkv, m % groups, m / groups};
}

__device__ __forceinline__ size_t split_unit(unsigned split, unsigned nb, unsigned block,
                                             unsigned Hq, unsigned h) {
  return ((size_t)split * nb + block) * Hq + h;
}

// GATED: the output goes through the sigmoid gate, with the bits of the
// standalone sigmoidMul. The query rows may be the output's own (the gated
// call normalises them there): a wave reads the rows it writes, at its start.
// SPLIT: the block's tiles are divided over sa.splits workgroups, each of
// which leaves its (m, l, O^T) for gqa_prefill_merge_kernel. The host gives a
// split at least three tiles, so that its first one is visible to every row
// of the block (the mask reaches into the last two tiles at most).
template <int D, int HW, bool GATED, bool SPLIT>
__global__ __attribute__((amdgpu_flat_work_group_size(64 * HW, 64 * HW),
                          amdgpu_waves_per_eu(HW > 4 ? 2 : 1, HW > 4 ? 2 : 1)))
void gqa_prefill_kernel(const half_t *q, const half_t *__restrict__ kc,
                        const half_t *__restrict__ vc, half_t *out,
                        unsigned T, unsigned Hq, unsigned Hkv, unsigned P,
                        unsigned groups, unsigned nb, float c,
                        typename std::conditional<GATED, GateArgs, NoArgs>::type ga,
                        typename std::conditional<SPLIT, SplitArgs, NoArgs>::type sa) {
  static_assert(!(GATED && SPLIT), "the merge gates a split launch's rows");
  constexpr int KS = D / 16;         // k-steps of S^T over channels
  constexpr int DT = D / 32;         // 32-channel output tiles
  constexpr int ROWB = 2 * D;        // bytes per K/V row
  constexpr int TILEB = BN * ROWB;   // bytes per K or V tile
  constexpr int NIW = TILEB / 1024 / HW; // 1-KB LDS loads per wave per tile
  constexpr int CPR = D / 8;         // 16-byte chunks per row
  constexpr int RPI = 64 / CPR;      // rows per 1-KB load
  static_assert(NIW >= 1 && TILEB % (1024 * HW) == 0, "tile/waves");
  // V is staged transposed (V^T rows of BN keys, padded) when one pass of
  // the workgroup's threads covers the tile in (8-key run, 8-channel) units;
  // smaller workgroups read V with the transposing LDS read instead.
  constexpr int VUNITS = (BN / 8) * (D / 8);
  constexpr bool kStagedV = VUNITS <= 64 * HW;
  constexpr int VTROW = 2 * BN;       // bytes per V^T row (8 chunks of 16 B)
  constexpr int VBUF = kStagedV ? D * VTROW : TILEB;

  __shared__ __attribute__((aligned(1024))) char sK0[TILEB], sK1[TILEB];
  __shared__ __attribute__((aligned(1024))) char sV0[VBUF], sV1[VBUF];

  // Workgroup -> (head group, token block). Each XCD (workgroups are dealt
  // round-robin over 8) serves as few head groups as possible, so its L2
  // holds their K/V; token blocks go longest (most keys) first.
  const unsigned NH = Hkv * groups;
  const unsigned id = blockIdx.x, xcd = id % 8, j8 = id / 8;
  unsigned hg, tbr, split = 0;
  if constexpr (SPLIT) {
    const SplitPlace at = split_place(Hkv, groups, nb);
    hg = at.kvh * groups + at.heads, tbr = at.rows, split = at.split;
  } else if (8 % NH == 0 && nb % (8 / NH) == 0) {
    const unsigned X = 8 / NH;
    hg = xcd / X;
    tbr = j8 * X + xcd % X;
  } else if (NH % 8 == 0) {
    const unsigned per = NH / 8;
    hg = xcd * per + j8 % per;
    tbr = j8 / per;
  } else {
    hg = id % NH;
    tbr = id / NH;
  }
  const unsigned tb = nb - 1 - tbr;
  const unsigned kvh = hg / groups, grp = hg % groups;
  const unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const unsigned lane = threadIdx.x % 64, r = lane % 32, hi = lane / 32;
  const unsigned h = (kvh * groups + grp) * HW + wave;
  const unsigned t0 = tb * BM, tq = t0 + r;
  const bool rowValid = tq < T;
  const unsigned tLast = min(t0 + BM, T) - 1;
  unsigned kend = P + tLast + 1; // keys [0, kend) can be visible
  unsigned tbeg = 0, tiles = (kend + BN - 1) / BN; // this workgroup's [tbeg, tiles)
  if constexpr (SPLIT) {
    tbeg = (unsigned)((uint64_t)tiles * split / sa.splits);
    tiles = (unsigned)((uint64_t)tiles * (split + 1) / sa.splits);
    kend = min(kend, tiles * BN);
  }
  const size_t rowBytes = (size_t)Hkv * D * 2;
  const char *kbase = reinterpret_cast<const char *>(kc) + (size_t)kvh * D * 2;
  const char *vbase = reinterpret_cast<const char *>(vc) + (size_t)kvh * D * 2;

  // Load i of this wave writes tile rows (wave + HW i) RPI + [0, RPI). The
  // swizzle repeats every 8 rows (K) or 4 rows (V), so the lane offsets
  // repeat every PK / PV loads up to a uniform row shift, added per load.
  constexpr int STEP = HW * RPI;
  constexpr int PK = STEP >= 8 ? 1 : 8 / STEP, PV = STEP >= 4 ? 1 : 4 / STEP;
  unsigned koff[PK], voff[PV];
#pragma unroll
  for (int p = 0; p < PK; ++p) {
    const unsigned row = wave * RPI + lane / CPR + STEP * p, slot = lane % CPR;
    koff[p] = row * (unsigned)rowBytes + 16 * (slot ^ (row & 7));
  }
#pragma unroll
  for (int p = 0; p < PV; ++p) {
    const unsigned row = wave * RPI + lane / CPR + STEP * p, slot = lane % CPR;
    voff[p] = row * (unsigned)rowBytes + 16 * (slot ^ ((row & 3) << 1));
  }
  // One descriptor per tile over its rows below kend (none for a tile past
  // the end, whose loads then do nothing).
  auto tile_rsrc = [&](const char *base, unsigned tile) {
    const unsigned first = tile * BN;
    const unsigned rows = kend > first ? min((unsigned)BN, kend - first) : 0u;
    return __builtin_amdgcn_make_buffer_rsrc((void *)(base + (size_t)first * rowBytes),
                                             (short)0, (int)(rows * rowBytes), kBufferWord3);
  };
  // A tile's loads go out in NPART parts spread over the score MFMAs, so the
  // vector memory pipeline takes them while the matrix cores work.
  constexpr int NPART = 4;
  auto issue = [&](__amdgpu_buffer_rsrc_t rs, const unsigned *off, int period, char *dst,
                   int part) {
#pragma unroll
    for (int i = 0; i < NIW; ++i)
      if (i * NPART / NIW == part)
        load_lds16(rs, dst + 1024 * (wave + HW * i),
                   off[i % period] + (unsigned)(STEP * (i - i % period)) * (unsigned)rowBytes);
  };
  auto issue_k = [&](unsigned tile, char *dst) {
    const __amdgpu_buffer_rsrc_t rs = tile_rsrc(kbase, tile);
#pragma unroll
    for (int part = 0; part < NPART; ++part)
      issue(rs, koff, PK, dst, part);
  };
  auto issue_v = [&](unsigned tile, char *dst) {
    const __amdgpu_buffer_rsrc_t rs = tile_rsrc(vbase, tile);
#pragma unroll
    for (int part = 0; part < NPART; ++part)
      issue(rs, voff, PV, dst, part);
  };

  // Staged V: thread t owns unit t = (run, 8-channel block cb). A run is the
  // 8 keys 16G + 4hh + {0..3} and 16G + 8 + 4hh + {0..3} of a 16-key group
  // G; V^T stores them at key positions 16G + 8hh + [0, 8), i.e. bits 2 and
  // 3 of the key index swapped within each group, which is exactly the key
  // order the probability operand holds (lane half hi, slots e: key
  // 16G + 8(e/4) + 4hi + e%4). So one 16-byte read gives an MFMA operand.
  // The 16-byte chunk c of V^T row j sits at c ^ ((j / 8) % 8): the eight
  // threads writing rows 8 cb + ch for consecutive cb hit distinct banks.
  const unsigned vunit = threadIdx.x, vcb = vunit % (D / 8), vrun = vunit / (D / 8);
  const unsigned vG = vrun / 2, vhh = vrun % 2;
  const bool vowner = VUNITS == 64 * HW || vunit < (unsigned)VUNITS;
  const unsigned vsrc = (16 * vG + 4 * vhh) * (unsigned)rowBytes + 16 * vcb;
  const unsigned vdst = (8 * vcb) * VTROW + 16 * ((2 * vG + vhh) ^ (vcb % 8));
  half8_t vst[8];
  auto load_v_part = [&](__amdgpu_buffer_rsrc_t rs, int part) {
    if (vowner) {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (e * NPART / 8 == part)
          vst[e] = __builtin_bit_cast(
              half8_t,
              __builtin_amdgcn_raw_buffer_load_b128(
                  rs, vsrc, (unsigned)((e % 4) + 8 * (e / 4)) * (unsigned)rowBytes, 0));
    }
  };
  auto load_v = [&](unsigned tile) {
    const __amdgpu_buffer_rsrc_t rs = tile_rsrc(vbase, tile);
#pragma unroll
    for (int part = 0; part < NPART; ++part)
      load_v_part(rs, part);
  };
  auto store_vt = [&](char *dst) {
    if (vowner) {
#pragma unroll
      for (int ch = 0; ch < 8; ++ch)
        *reinterpret_cast<half8_t *>(dst + vdst + ch * VTROW) =
            half8_t{vst[0][ch], vst[1][ch], vst[2][ch], vst[3][ch],
                    vst[4][ch], vst[5][ch], vst[6][ch], vst[7][ch]};
    }
  };

  // Operand read offsets. K (A of S^T, row 32kt + r, chunk 2s + hi): the
  // swizzle only touches the low 3 chunk bits, so s = 4a + b reads
  // kread[b] + 128a. V^T via the transposing read: lane j of a 16-lane group
  // addresses row k0 + j/4, channels 16g + 4(j%4) .. +3 of an output tile.
  unsigned kread[4];
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    kread[b] = r * ROWB + 16 * ((2 * b + hi) ^ (r & 7));
    opaque(kread[b]);
  }
  const unsigned j16 = lane % 16, g = (lane / 16) % 2;
  const unsigned vx = 2 * (j16 / 4), vb = (j16 % 4) / 2;
  const unsigned vrow = (4 * hi + j16 / 4) * ROWB + 8 * (j16 % 2);
  const unsigned vread[2] = {vrow + 16 * ((2 * g + vb) ^ vx),
                             vrow + 16 * ((4 + 2 * g + vb) ^ vx)};
  // Staged V^T: lane reads row 32 dt + r, key positions 16 G + 8 hi + [0, 8),
  // i.e. chunk (2G + hi) ^ ((4 dt + r / 8) % 8): one offset per (dt % 2, G).
  unsigned vtread[2][4];
#pragma unroll
  for (int dp = 0; dp < 2; ++dp)
#pragma unroll
    for (int G = 0; G < 4; ++G) {
      vtread[dp][G] = r * VTROW + 16 * ((2 * G + hi) ^ ((4 * dp + r / 8) % 8));
      opaque(vtread[dp][G]);
    }
  // PV operand of a tile: output tile dt, 16-key group G = 2 kt + m.
  auto vop = [&](const char *sv, int dt, int kt, int m) {
    if constexpr (kStagedV) {
      return load8(reinterpret_cast<const half_t *>(sv + vtread[dt % 2][2 * kt + m] +
                                                    32 * dt * VTROW));
    } else {
      const unsigned o = vread[dt % 2] + 128 * (dt / 2) + ROWB * (32 * kt + 16 * m);
      const half4_t lo = read_tr(sv, o), up = read_tr(sv, o + 8 * ROWB);
      return half8_t{lo[0], lo[1], lo[2], lo[3], up[0], up[1], up[2], up[3]};
    }
  };

  // Q^T as the MFMA B operand: lane holds query row r, channels
  // 16 s + 8 hi + [0, 8). Rows past T use zeros (their output is dropped).
  half8_t qb[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s)
    qb[s] = rowValid ? load8(q + ((size_t)tq * Hq + h) * D + 16 * s + 8 * hi)
                     : half8_t{0, 0, 0, 0, 0, 0, 0, 0};

  float16_t oacc[DT];
#pragma unroll
  for (int i = 0; i < DT; ++i)
    oacc[i] = float16_t{0};
  // l (the softmax denominator) is accumulated by the MFMA as ones x P^T,
  // from the same fp16 probabilities that multiply V: every register of
  // lacc holds the row sum of the lane's query.
  float mRef = -INFINITY;
  float16_t lacc = float16_t{0};
  const half8_t ones{1, 1, 1, 1, 1, 1, 1, 1};
  half8_t pb[2][2]; // P^T B operands, [32-key half][16-key step]

  auto pv = [&](const char *svl) {
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int m = 0; m < 2; ++m) {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
          oacc[dt] = mfma32x32x16(vop(svl, dt, kt, m), pb[kt][m], oacc[dt]);
        lacc = mfma32x32x16(ones, pb[kt][m], lacc);
      }
  };
  // Causal mask as the scores' initial accumulator: -inf where key > P + tq
  // (a finite K row plus -inf stays -inf), 0 elsewhere.
  auto mask_init = [&](unsigned base, float16_t (&init)[2]) {
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int v = 0; v < 16; ++v)
        init[kt][v] = base + 32 * kt + mfma_c_row(v, hi) > P + tq ? -INFINITY : 0.0f;
  };
  // Softmax, first half: the tile's row maximum decides whether the
  // reference moves (then O must be rescaled by the returned factor, which
  // the caller does when any row of the wave moved); l follows at once.
  auto reference = [&](float mx, bool &raised) {
    const LanePair pr = pair32(mx);
    const float tm = fmaxf(pr.a, pr.b) * c;
    const bool need = tm - mRef > kRaise;
    const float mNew = need ? tm - kHeadroom : mRef;
    const float alpha = SPLIT && !need ? 1.0f : fast_exp2(mRef - mNew);
    mRef = mNew;
    raised = __builtin_amdgcn_ballot_w64(need) != 0;
    return alpha;
  };
  // Softmax, second half: the fp16 probabilities of scores sp against the
  // current reference, as PV operand pb, and their sum into l.
  auto prob = [&](const float (&sp)[32], int j, float negm) {
    const int kt = j / 16, m = (j / 8) % 2, e = j % 8;
    pb[kt][m][e] = (half_t)fast_exp2(fmaf(sp[16 * kt + 8 * m + e], c, negm));
  };

  // Phase A of step i: the score MFMAs of tile i, each K operand read three
  // k-steps ahead, with the probabilities of tile i-1 (scores sp) computed
  // on the VALU in between.
  auto phase_a = [&](const char *sk, const float16_t *init, const float (&sp)[32],
                     float16_t (&sacc)[2], auto &&feed) {
    constexpr int PER = 32 / KS; // probabilities per k-step
    auto kld = [&](int st, int kt) {
      return load8(reinterpret_cast<const half_t *>(sk + kread[st % 4] + 128 * (st / 4) +
                                                    32 * ROWB * kt));
    };
    const float negm = SPLIT && mRef == -INFINITY ? 0.0f : -mRef;
    constexpr int AHEAD = 3;
    half8_t ka[AHEAD + 1][2];
#pragma unroll
    for (int st = 0; st < AHEAD; ++st) {
      ka[st][0] = kld(st, 0);
      ka[st][1] = kld(st, 1);
    }
    sacc[0] = init ? init[0] : float16_t{0};
    sacc[1] = init ? init[1] : float16_t{0};
#pragma unroll
    for (int st = 0; st < KS; ++st) {
      if (st + AHEAD < KS) {
        ka[(st + AHEAD) % (AHEAD + 1)][0] = kld(st + AHEAD, 0);
        ka[(st + AHEAD) % (AHEAD + 1)][1] = kld(st + AHEAD, 1);
      }
      sacc[0] = mfma32x32x16(ka[st % (AHEAD + 1)][0], qb[st], sacc[0]);
      sacc[1] = mfma32x32x16(ka[st % (AHEAD + 1)][1], qb[st], sacc[1]);
#pragma unroll
      for (int u = 0; u < PER; ++u)
        prob(sp, st * PER + u, negm);
      if (st % (KS / NPART) == 0)
        feed(st / (KS / NPART));
    }
  };
  // Phase B of step i: the PV MFMAs of tile i-1, each V^T operand read two
  // MFMAs ahead, with the row maximum of tile i taken in between.
  auto phase_b = [&](const char *svl, const float16_t (&sacc)[2], float (&sv)[32],
                     bool &raised) {
    constexpr int NPV = 4 * DT, PER = 32 / NPV;
    // Consecutive MFMAs go to different output tiles (independent chains).
    auto vld = [&](int n) { return vop(svl, n % DT, n / (2 * DT), (n / DT) % 2); };
    half8_t va[3];
    va[0] = vld(0);
    va[1] = vld(1);
    float mx = -INFINITY;
#pragma unroll
    for (int n = 0; n < NPV; ++n) {
      if (n + 2 < NPV)
        va[(n + 2) % 3] = vld(n + 2);
      const int dt = n % DT, kt = n / (2 * DT), m = (n / DT) % 2;
      oacc[dt] = mfma32x32x16(va[n % 3], pb[kt][m], oacc[dt]);
      if (dt == DT - 1)
        lacc = mfma32x32x16(ones, pb[kt][m], lacc);
#pragma unroll
      for (int u = 0; u < PER; ++u) {
        const int j = n * PER + u;
        sv[j] = sacc[j / 16][j % 16];
        mx = fmaxf(mx, sv[j]);
      }
    }
    return reference(mx, raised);
  };

  // Buffers start zeroed: rows past the block's last key may keep what was
  // there before, which must be finite (a probability of 0 times V, and the
  // -inf mask plus a K dot product, must stay exact).
  {
    const uint4_t z{0, 0, 0, 0};
    for (unsigned i = threadIdx.x * 16; i < (unsigned)TILEB; i += 64 * HW * 16) {
      *reinterpret_cast<uint4_t *>(sK0 + i) = z;
      *reinterpret_cast<uint4_t *>(sK1 + i) = z;
    }
    for (unsigned i = threadIdx.x * 16; i < (unsigned)VBUF; i += 64 * HW * 16) {
      *reinterpret_cast<uint4_t *>(sV0 + i) = z;
      *reinterpret_cast<uint4_t *>(sV1 + i) = z;
    }
  }
  __syncthreads();
  issue_k(tbeg, sK0);
  if constexpr (kStagedV)
    load_v(tbeg);
  else
    issue_v(tbeg, sV0);
  wait_loads();
  __syncthreads();
  if (tiles > tbeg + 1)
    issue_k(tbeg + 1, sK1);

  // The first tile: scores and reference only (O is still zero).
  float sv[32]; // scores of the last tile, raw (masked keys -inf)
  {
    float16_t init[2], sacc[2];
    const bool masked = (tbeg + 1) * BN > P + t0 + 1;
    if (masked)
      mask_init(tbeg * BN, init);
    const float zero[32] = {};
    phase_a(sK0, masked ? init : nullptr, zero, sacc, [](int) {});
    float mx = -INFINITY;
#pragma unroll
    for (int j = 0; j < 32; ++j) {
      sv[j] = sacc[j / 16][j % 16];
      mx = fmaxf(mx, sv[j]);
    }
    bool raised;
    reference(mx, raised);
  }

  // Step i: phase A (scores of tile i, probabilities of tile i-1), phase B
  // (PV of tile i-1, row maximum of tile i), with the loads of K(i+1) and
  // V(i) in flight. Buffers are named statically so the compiler can tell
  // the loads in flight from the LDS reads and need not wait for them;
  // tiles below the block's first query (the steady state, run in pairs)
  // skip the mask.
  auto step = [&](unsigned i, bool masked, const char *kcur, char *vprev, char *knext,
                  char *vdst) {
    wait_loads();
    if constexpr (kStagedV)
      store_vt(vprev); // V(i-1), loaded during the previous step
    __syncthreads();
    // K(i+1) (none past the last tile) and V(i), spread over phase A.
    const __amdgpu_buffer_rsrc_t krs = tile_rsrc(kbase, i + 1), vrs = tile_rsrc(vbase, i);
    auto feed = [&](int part) {
      issue(krs, koff, PK, knext, part);
      if constexpr (kStagedV)
        load_v_part(vrs, part);
      else
        issue(vrs, voff, PV, vdst, part);
    };
    float16_t init[2], sacc[2];
    if (masked)
      mask_init(i * BN, init);
    bool raised;
    phase_a(kcur, masked ? init : nullptr, sv, sacc, feed);
    const float alpha = phase_b(vprev, sacc, sv, raised);
    if (raised) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
        oacc[dt] *= alpha;
      lacc *= alpha;
    }
  };
  // Tiles [1, iu) lie wholly below the block's first query.
  const unsigned iu = max(tbeg + 1, min(tiles, (P + t0 + 1) / BN));
  unsigned i = tbeg + 1;
  for (; i + 1 < iu; i += 2) {
    step(i, false, sK1, sV0, sK0, sV1);
    step(i + 1, false, sK0, sV1, sK1, sV0);
  }
  // The rest (at most three tiles) with the mask, which is all-pass on an
  // unmasked tile.
  for (; i < tiles; i += 2) {
    step(i, true, sK1, sV0, sK0, sV1);
    if (i + 1 < tiles)
      step(i + 1, true, sK0, sV1, sK1, sV0);
  }
  {
    const float negm = SPLIT && mRef == -INFINITY ? 0.0f : -mRef;
#pragma unroll
    for (int j = 0; j < 32; ++j)
      prob(sv, j, negm);
  }
  wait_loads();
  if constexpr (kStagedV)
    store_vt((tiles - 1 - tbeg) % 2 == 0 ? sV0 : sV1);
  __syncthreads();
  if ((tiles - 1 - tbeg) % 2 == 0)
    pv(sV0);
  else
    pv(sV1);

  if (!rowValid)
    return;
  if constexpr (SPLIT) {
    const size_t u = split_unit(split, nb, tb, Hq, h);
    if (hi == 0) {
      sa.ml[u * 2 * BM + r] = mRef;
      sa.ml[u * 2 * BM + BM + r] = lacc[0];
    }
    float *o = sa.o + u * BM * D + lane;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int v = 0; v < 16; ++v)
        o[(dt * 16 + v) * 64] = oacc[dt][v];
    return;
  }
  const float inv = 1.0f / lacc[0];
  half_t *orow = out + ((size_t)tq * Hq + h) * D;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) {
    half4_t v[4];
#pragma unroll
    for (int g4 = 0; g4 < 4; ++g4)
      v[g4] = half4_t{f16_of(oacc[dt][4 * g4 + 0] * inv), f16_of(oacc[dt][4 * g4 + 1] * inv),
                      f16_of(oacc[dt][4 * g4 + 2] * inv), f16_of(oacc[dt][4 * g4 + 3] * inv)};
    if constexpr (GATED)
      gate_tile(v, ga.qproj + ((size_t)tq * Hq + h) * 2 * D +
                       D + 32 * dt + 4 * hi, ga.activated);
#pragma unroll
    for (int g4 = 0; g4 < 4; ++g4)
      *reinterpret_cast<half4_t *>(orow + 32 * dt + 8 * g4 + 4 * hi) = v[g4];
  }
}

// d = 256 with an even number of query heads per KV head: eight waves, two
// per SIMD, over a pair of token blocks (nb - 1 - p and p: their key counts
// add up to the same total for every pair, which balances the causal
// triangle across workgroups) and two query heads. Wave w serves block
// w / 4 (the long one first), head (w / 2) % 2 and key half w % 2: each
// (block, head) has a wave pair that splits the keys by 32-key tiles, the
// even tiles to one wave, the odd ones to the other, each with its own
// (m, l, O). SIMD j (a workgroup's waves are dealt to the SIMDs in turn)
// runs wave j of the long block and wave j of the short one: while one
// waits on LDS operands or runs its softmax the other keeps the matrix core
// busy, and once the short block is done the long block's wave has the
// SIMD to itself. A lane holds O^T (128 registers), Q^T (64) and one 32x32
// score block; the row sums are fp32 sums of the fp16 probabilities that
// multiply V (v_dot2). At the end each odd-tile wave hands its (m, l, O) to
// its partner through LDS. One step = one barrier: the four tiles of the
// next step (K and V of tiles 2s + 2 and 2s + 3, shared by both blocks) go
// HBM -> LDS as the step begins. GATED as in gqa_prefill_kernel.
// SPLIT as in gqa_prefill_kernel, over the pair's steps: a workgroup leaves
// the (m, l, O^T) that its wave pairs merged (m = -inf, l = 0, O = 0 for rows
// that see none of its keys).
template <bool GATED, bool SPLIT>
__global__ __attribute__((amdgpu_flat_work_group_size(512, 512), amdgpu_waves_per_eu(2, 2)))
void gqa_prefill_halves_kernel(const half_t *q, const half_t *__restrict__ kc,
                               const half_t *__restrict__ vc, half_t *out,
                               unsigned T, unsigned Hq, unsigned Hkv, unsigned P,
                               unsigned hpairs, unsigned nb, float c,
                               typename std::conditional<GATED, GateArgs, NoArgs>::type ga,
                               typename std::conditional<SPLIT, SplitArgs, NoArgs>::type sa) {
  static_assert(!(GATED && SPLIT), "the merge gates a split launch's rows");
  constexpr int D = 256, KS = D / 16, DT = D / 32;
  constexpr int BK = 32;           // keys per tile
  constexpr int ROWB = 2 * D;      // bytes per K/V row
  constexpr int TILEB = BK * ROWB; // 16 KB per K or V tile
  // [set][half]: set s % 2 holds what step s reads. Named one by one so the
  // compiler can tell the loads in flight from the LDS reads.
  __shared__ __attribute__((aligned(1024))) char sK00[TILEB], sK01[TILEB], sK10[TILEB],
      sK11[TILEB];
  __shared__ __attribute__((aligned(1024))) char sV00[TILEB], sV01[TILEB], sV10[TILEB],
      sV11[TILEB];
  __shared__ float sML[4][2][64];

  // Workgroup -> (block pair, KV head, head pair): each XCD (workgroups are
  // dealt round-robin over 8) serves as few KV heads as possible, so its L2
  // holds their K/V.
  const unsigned NH = Hkv * hpairs, npairs = (nb + 1) / 2;
  const unsigned id = blockIdx.x, xcd = id % 8, j8 = id / 8;
  unsigned hg, pr, split = 0;
  if constexpr (SPLIT) {
    const SplitPlace at = split_place(Hkv, hpairs, npairs);
    hg = at.kvh * hpairs + at.heads, pr = at.rows, split = at.split;
  } else if (8 % NH == 0 && npairs % (8 / NH) == 0) {
    const unsigned X = 8 / NH;
    hg = xcd / X;
    pr = j8 * X + xcd % X;
  } else if (NH % 8 == 0) {
    const unsigned per = NH / 8;
    hg = xcd * per + j8 % per;
    pr = j8 / per;
  } else {
    hg = id % NH;
    pr = id / NH;
  }
  const unsigned kvh = hg / hpairs, hp = hg % hpairs;
  const unsigned bL = nb - 1 - pr, bS = pr;
  const unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const unsigned blk = wave / 4, hs = (wave / 2) % 2, half = wave % 2;
  const unsigned pi = 2 * blk + hs; // (block, head) of this wave
  const bool idle = blk == 1 && bS == bL; // nb odd: the middle block pairs with itself
  const unsigned lane = threadIdx.x % 64, r = lane % 32, hi = lane / 32;
  const unsigned h = (kvh * hpairs + hp) * 2 + hs;
  const unsigned t0 = (blk ? bS : bL) * BM, tq = t0 + r;
  const bool rowValid = tq < T && !idle;
  // Keys [0, kend) can be visible to the long block; this wave's block needs
  // its first `mine` tiles.
  unsigned kend = P + min(bL * BM + BM, T);
  const unsigned ntiles = (kend + BK - 1) / BK;
  unsigned sbeg = 0, steps = (ntiles + 1) / 2; // this workgroup's [sbeg, steps)
  if constexpr (SPLIT) {
    sbeg = (unsigned)((uint64_t)steps * split / sa.splits);
    steps = (unsigned)((uint64_t)steps * (split + 1) / sa.splits);
    kend = min(kend, steps * 2 * BK);
  }
  const unsigned mine = idle ? 0u : (P + min(t0 + BM, T) + BK - 1) / BK;
  const unsigned ju = (P + t0 + 1) / BK; // tiles [0, ju) need no mask
  const size_t rowBytes = (size_t)Hkv * D * 2;
  const char *kbase = reinterpret_cast<const char *>(kc) + (size_t)kvh * D * 2;
  const char *vbase = reinterpret_cast<const char *>(vc) + (size_t)kvh * D * 2;

  // Wave w moves the 1-KB pieces w and w + 8 (tile rows 2p, 2p + 1) of each
  // tile; the XOR swizzles (K chunk c of row j at c ^ (j % 8), V chunk c at
  // c ^ 2(j % 4)) repeat every 16 rows, so piece w + 8 is piece w 16 rows on.
  const unsigned prow = 2 * wave + lane / 32, slot = lane % 32;
  const unsigned koff = prow * (unsigned)rowBytes + 16 * (slot ^ (prow & 7));
  const unsigned voff = prow * (unsigned)rowBytes + 16 * (slot ^ ((prow & 3) << 1));
  const unsigned pstep = 16 * (unsigned)rowBytes;
  auto tile_rsrc = [&](const char *base, unsigned tile) {
    const unsigned first = tile * BK;
    const unsigned rows = kend > first ? min((unsigned)BK, kend - first) : 0u;
    return __builtin_amdgcn_make_buffer_rsrc((void *)(base + (size_t)first * rowBytes),
                                             (short)0, (int)(rows * rowBytes), kBufferWord3);
  };
  auto load_tile = [&](const char *base, unsigned tile, unsigned off, char *dst) {
    const __amdgpu_buffer_rsrc_t rs = tile_rsrc(base, tile);
    load_lds16(rs, dst + 1024 * wave, off);
    load_lds16(rs, dst + 1024 * (wave + 8), off + pstep);
  };

  // Operand reads. K (A of S^T, row r, chunk 2s + hi): kread[s % 4] +
  // 128 (s / 4). V^T through the transposing read: lane j of a 16-lane
  // group addresses row k0 + j / 4, channels 16 g + 4 (j % 4) .. +3.
  unsigned kread[4];
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    kread[b] = r * ROWB + 16 * ((2 * b + hi) ^ (r & 7));
    opaque(kread[b]);
  }
  const unsigned j16 = lane % 16, g = (lane / 16) % 2;
  const unsigned vx = 2 * (j16 / 4), vb = (j16 % 4) / 2;
  const unsigned vrow = (4 * hi + j16 / 4) * ROWB + 8 * (j16 % 2);
  unsigned vread[2] = {vrow + 16 * ((2 * g + vb) ^ vx), vrow + 16 * ((4 + 2 * g + vb) ^ vx)};
  opaque(vread[0]);
  opaque(vread[1]);

  half8_t qb[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s)
    qb[s] = rowValid ? load8(q + ((size_t)tq * Hq + h) * D + 16 * s + 8 * hi)
                     : half8_t{0, 0, 0, 0, 0, 0, 0, 0};

  float16_t oacc[DT];
#pragma unroll
  for (int i = 0; i < DT; ++i)
    oacc[i] = float16_t{0};
  float mRef = -INFINITY, lsum = 0.0f;
  float16_t sacc = float16_t{0};
  half8_t pb[2]; // P^T B operands, [16-key step]

  // Scores of one tile into sacc (the causal mask as the initial
  // accumulator where the tile reaches past the block's first query).
  auto scores = [&](const char *kb, unsigned tile) {
    auto kld = [&](int st) {
      return load8(reinterpret_cast<const half_t *>(kb + kread[st % 4] + 128 * (st / 4)));
    };
    constexpr int KA = 2; // operand reads run KA MFMAs ahead
    half8_t ka[KA + 1];
#pragma unroll
    for (int st = 0; st < KA; ++st)
      ka[st] = kld(st);
    if (tile >= ju) {
#pragma unroll
      for (int v = 0; v < 16; ++v)
        sacc[v] = tile * BK + mfma_c_row(v, hi) > P + tq ? -INFINITY : 0.0f;
    } else {
      sacc = float16_t{0};
    }
#pragma unroll
    for (int st = 0; st < KS; ++st) {
      if (st + KA < KS)
        ka[(st + KA) % (KA + 1)] = kld(st + KA);
      sacc = mfma32x32x16(ka[st % (KA + 1)], qb[st], sacc);
      __builtin_amdgcn_sched_barrier(0); // operand reads stay KA ahead, no further
    }
  };
  // Softmax of sacc against the lazily moved reference (raised only when a
  // probability would pass 2^15; O and l rescaled then), the fp16
  // probabilities into pb, their sum into l.
  auto softmax = [&]() {
    float mx = sacc[0];
#pragma unroll
    for (int v = 1; v < 16; ++v)
      mx = fmaxf(mx, sacc[v]);
    const LanePair pr = pair32(mx);
    const float tm = fmaxf(pr.a, pr.b) * c;
    const bool need = tm - mRef > kRaise; // false while every key so far is masked
    const float mNew = need ? tm - kHeadroom : mRef;
    const float alpha = need ? fast_exp2(mRef - mNew) : 1.0f;
    mRef = mNew;
    if (__builtin_amdgcn_ballot_w64(need) != 0) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
        oacc[dt] *= alpha;
      lsum *= alpha;
    }
    const float negm = mRef == -INFINITY ? 0.0f : -mRef;
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int e = 0; e < 8; ++e)
        pb[m][e] = (half_t)fast_exp2(fmaf(sacc[8 * m + e], c, negm));
    const half2_t one2{1, 1};
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int e = 0; e < 8; e += 2)
        lsum = __builtin_amdgcn_fdot2(half2_t{pb[m][e], pb[m][e + 1]}, one2, lsum, false);
  };
  // O^T += V^T P^T for one tile: output tile dt, 16-key step m.
  auto pv = [&](const char *vbuf) {
    auto vld = [&](int n) {
      const int dt = n % DT, m = n / DT;
      const unsigned o = vread[dt % 2] + 128 * (dt / 2) + ROWB * 16 * m;
      const half4_t lo = read_tr(vbuf, o), up = read_tr(vbuf, o + 8 * ROWB);
      return half8_t{lo[0], lo[1], lo[2], lo[3], up[0], up[1], up[2], up[3]};
    };
    constexpr int VA = 2;
    half8_t va[VA + 1];
#pragma unroll
    for (int n = 0; n < VA; ++n)
      va[n] = vld(n);
#pragma unroll
    for (int n = 0; n < 2 * DT; ++n) {
      if (n + VA < 2 * DT)
        va[(n + VA) % (VA + 1)] = vld(n + VA);
      oacc[n % DT] = mfma32x32x16(va[n % (VA + 1)], pb[n / DT], oacc[n % DT]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // LDS starts zeroed: rows past the block's last key keep whatever an
  // earlier tile left there, which must be finite.
  {
    const uint4_t z{0, 0, 0, 0};
    for (unsigned i = threadIdx.x * 16; i < (unsigned)TILEB; i += 512 * 16) {
      *reinterpret_cast<uint4_t *>(sK00 + i) = z;
      *reinterpret_cast<uint4_t *>(sK01 + i) = z;
      *reinterpret_cast<uint4_t *>(sK10 + i) = z;
      *reinterpret_cast<uint4_t *>(sK11 + i) = z;
      *reinterpret_cast<uint4_t *>(sV00 + i) = z;
      *reinterpret_cast<uint4_t *>(sV01 + i) = z;
      *reinterpret_cast<uint4_t *>(sV10 + i) = z;
      *reinterpret_cast<uint4_t *>(sV11 + i) = z;
    }
  }
  __syncthreads();
  load_tile(kbase, 2 * sbeg, koff, sK00);
  load_tile(kbase, 2 * sbeg + 1, koff, sK01);
  load_tile(vbase, 2 * sbeg, voff, sV00);
  load_tile(vbase, 2 * sbeg + 1, voff, sV01);

  // Step s: set s % 2 holds K and V of tiles 2s and 2s + 1; the other set
  // receives those of 2s + 2 and 2s + 3, requested as the step begins. Each
  // half runs its own loop (one barrier per step in both) over its
  // statically named buffers.
  auto loads = [&](unsigned s, char *nkA, char *nkB, char *nvA, char *nvB) {
    load_tile(kbase, 2 * s + 2, koff, nkA);
    load_tile(kbase, 2 * s + 3, koff, nkB);
    load_tile(vbase, 2 * s + 2, voff, nvA);
    load_tile(vbase, 2 * s + 3, voff, nvB);
  };
  auto run = [&](unsigned first, const char *k0, const char *v0, const char *k1,
                 const char *v1) {
    auto step = [&](unsigned s, const char *kc_, const char *vc_, char *nkA, char *nkB,
                    char *nvA, char *nvB) {
      wait_loads();
      __syncthreads();
      loads(s, nkA, nkB, nvA, nvB);
      if (2 * s + first < mine) {
        scores(kc_, 2 * s + first);
        softmax();
        pv(vc_);
      }
    };
    unsigned s = sbeg;
    for (; s + 1 < steps; s += 2) {
      step(s, k0, v0, sK10, sK11, sV10, sV11);
      step(s + 1, k1, v1, sK00, sK01, sV00, sV01);
    }
    if (s < steps)
      step(s, k0, v0, sK10, sK11, sV10, sV11);
  };
  if (half == 0)
    run(0, sK00, sV00, sK10, sV10);
  else
    run(1, sK01, sV01, sK11, sV11);
  wait_loads();
  __syncthreads(); // every wave is done with the K/V buffers

  // The odd half's (m, l, O^T) to LDS, lane-major (conflict-free): pair pi
  // uses two 16 KB buffers, output tiles 0-3 in the first.
  char *ma = pi == 0 ? sK00 : pi == 1 ? sK10 : pi == 2 ? sV00 : sV10;
  char *mb = pi == 0 ? sK01 : pi == 1 ? sK11 : pi == 2 ? sV01 : sV11;
  if (half == 1) {
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int v = 0; v < 16; ++v)
        reinterpret_cast<float *>(dt < 4 ? ma : mb)[((dt % 4) * 16 + v) * 64 + lane] =
            oacc[dt][v];
    sML[pi][0][lane] = mRef;
    sML[pi][1][lane] = lsum;
  }
  __syncthreads();
  if (half == 1 || !rowValid)
    return;
  const float m1 = sML[pi][0][lane], l1 = sML[pi][1][lane];
  // (unsplit, mRef is finite: key 0 is visible to every row)
  const float M = fmaxf(mRef, m1);
  const bool none = SPLIT && M == -INFINITY;
  const float a0 = none ? 0.0f : fast_exp2(mRef - M), a1 = none ? 0.0f : fast_exp2(m1 - M);
  const LanePair lp = pair32(lsum * a0 + l1 * a1);
  if constexpr (SPLIT) {
    const size_t u = split_unit(split, nb, blk ? bS : bL, Hq, h);
    if (hi == 0) {
      sa.ml[u * 2 * BM + r] = M;
      sa.ml[u * 2 * BM + BM + r] = lp.a + lp.b;
    }
    float *o = sa.o + u * BM * D + lane;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      const float *o1 = reinterpret_cast<const float *>(dt < 4 ? ma : mb) + (dt % 4) * 16 * 64;
#pragma unroll
      for (int v = 0; v < 16; ++v)
        o[(dt * 16 + v) * 64] = oacc[dt][v] * a0 + o1[v * 64 + lane] * a1;
    }
    return;
  }
  const float inv = 1.0f / (lp.a + lp.b);
  half_t *orow = out + ((size_t)tq * Hq + h) * D;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) {
    const float *o1 = reinterpret_cast<const float *>(dt < 4 ? ma : mb) + (dt % 4) * 16 * 64;
    half4_t v[4];
#pragma unroll
    for (int g4 = 0; g4 < 4; ++g4)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int i = 4 * g4 + e;
        v[g4][e] = f16_of((oacc[dt][i] * a0 + o1[i * 64 + lane] * a1) * inv);
      }
    if constexpr (GATED)
      gate_tile(v, ga.qproj + ((size_t)tq * Hq + h) * 2 * D +
                       D + 32 * dt + 4 * hi, ga.activated);
#pragma unroll
    for (int g4 = 0; g4 < 4; ++g4)
      *reinterpret_cast<half4_t *>(orow + 32 * dt + 8 * g4 + 4 * hi) = v[g4];
  }
}

// The merge of a split launch: a wave per (token block, query head, 32-channel
// output tile, 8-channel half pair g4): lane (r, hi) owns row r and channels
// 32 dt + 8 g4 + 4 hi + [0, 4). Every split's partials are rescaled to the
// largest reference, as the kernels rescale their own; the gate follows.
template <int D, bool GATED>
__global__ __launch_bounds__(256) void gqa_prefill_merge_kernel(
    const float *__restrict__ ml, const float *__restrict__ po, half_t *__restrict__ out,
    unsigned T, unsigned Hq, unsigned nb, unsigned splits, const half_t *qproj,
    unsigned activated) {
  constexpr unsigned DT = D / 32;
  const unsigned w = blockIdx.x * 4 + threadIdx.x / 64, lane = threadIdx.x % 64;
  const unsigned g4 = w % 4, dt = (w / 4) % DT, bh = w / (4 * DT);
  const unsigned h = bh % Hq, blk = bh / Hq, r = lane % 32, hi = lane / 32;
  const unsigned tq = blk * BM + r;
  if (blk >= nb || tq >= T)
    return;
  const size_t stride = (size_t)nb * Hq; // units a split
  const float *m = ml + split_unit(0, nb, blk, Hq, h) * 2 * BM + r;
  const float *o = po + split_unit(0, nb, blk, Hq, h) * BM * D + (dt * 16 + 4 * g4) * 64 + lane;
  float M = -INFINITY;
#pragma unroll 8
  for (unsigned s = 0; s < splits; ++s)
    M = fmaxf(M, m[s * stride * 2 * BM]);
  float l = 0.0f, acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 8
  for (unsigned s = 0; s < splits; ++s) {
    const float a = fast_exp2(m[s * stride * 2 * BM] - M);
    l = fmaf(m[s * stride * 2 * BM + BM], a, l);
#pragma unroll
    for (int e = 0; e < 4; ++e)
      acc[e] = fmaf(o[s * stride * BM * D + e * 64], a, acc[e]);
  }
  const float inv = 1.0f / l;
  half4_t v[1] = {half4_t{f16_of(acc[0] * inv), f16_of(acc[1] * inv), f16_of(acc[2] * inv),
                          f16_of(acc[3] * inv)}};
  const size_t ch = 32 * dt + 8 * g4 + 4 * hi;
  if constexpr (GATED)
    gate_tile<1>(v, qproj + ((size_t)tq * Hq + h) * 2 * D + D + ch, activated);
  *reinterpret_cast<half4_t *>(out + ((size_t)tq * Hq + h) * D + ch) = v[0];
}

template <int D> constexpr unsigned heads_per_wg(unsigned G) {
  return G < (D == 256 ? 4u : 8u) ? G : (D == 256 ? 4u : 8u);
}

template <int D, int HW, bool GATED = false, bool SPLIT = false, typename Rows = NoArgs>
hipError_t launch_dw(const GqaShape &s, const uint16_t *q, const uint16_t *k,
                     const uint16_t *v, uint16_t *out, hipStream_t stream,
                     const Rows &rows = Rows{}, const SplitArgs &split = SplitArgs{}) {
  const float c = kLog2e / sqrtf((float)D);
  const unsigned G = s.Hq / s.Hkv, groups = G / HW, nb = (s.T + BM - 1) / BM;
  typename std::conditional<SPLIT, SplitArgs, NoArgs>::type sa;
  if constexpr (SPLIT)
    sa = split;
  hipLaunchKernelGGL((gqa_prefill_kernel<D, HW, GATED, SPLIT>),
                     dim3(nb * s.Hkv * groups * (SPLIT ? split.splits : 1)), dim3(64 * HW), 0,
                     stream, reinterpret_cast<const half_t *>(q),
                     reinterpret_cast<const half_t *>(k), reinterpret_cast<const half_t *>(v),
                     reinterpret_cast<half_t *>(out), s.T, s.Hq, s.Hkv, s.P, groups, nb, c,
                     rows, sa);
  return hipGetLastError();
}

template <bool GATED, bool SPLIT = false, typename Rows = NoArgs>
hipError_t launch_halves(const GqaShape &s, const uint16_t *q, const uint16_t *k,
                         const uint16_t *v, uint16_t *out, hipStream_t stream,
                         const Rows &rows = Rows{}, const SplitArgs &split = SplitArgs{}) {
  const float c = kLog2e / sqrtf(256.0f);
  const unsigned G = s.Hq / s.Hkv, hpairs = G / 2, nb = (s.T + BM - 1) / BM;
  typename std::conditional<SPLIT, SplitArgs, NoArgs>::type sa;
  if constexpr (SPLIT)
    sa = split;
  hipLaunchKernelGGL((gqa_prefill_halves_kernel<GATED, SPLIT>),
                     dim3((nb + 1) / 2 * s.Hkv * hpairs * (SPLIT ? split.splits : 1)), dim3(512),
                     0, stream, reinterpret_cast<const half_t *>(q),
                     reinterpret_cast<const half_t *>(k), reinterpret_cast<const half_t *>(v),
                     reinterpret_cast<half_t *>(out), s.T, s.Hq, s.Hkv, s.P, hpairs, nb, c,
                     rows, sa);
  return hipGetLastError();
}

// LLMI_PREFILL_HALVES=0 selects the single-wave kernel always, =1 the
// key-split one wherever it runs (for A/B timing): 0, 1, or -1 unset.
int forced_halves() {
  static const int forced = [] {
    const char *e = getenv("LLMI_PREFILL_HALVES");
    return e && *e ? (*e == '0' ? 0 : 1) : -1;
  }();
  return forced;
}

// The key-split kernel once the grid has at least 64 workgroups (below
// that, as at 128 tokens, the single-wave kernel's shorter prologue wins by
// ~1 us). The plain and gated launches take the same choice, so the two stay
// bit-identical.
bool use_halves(const GqaShape &s) {
  if (forced_halves() >= 0)
    return forced_halves() == 1;
  const unsigned nb = (s.T + BM - 1) / BM, hpairs = s.Hq / s.Hkv / 2;
  return (nb + 1) / 2 * s.Hkv * hpairs >= 64;
}

// Query heads a single-wave-kernel workgroup serves: four share each K/V
// tile, but a grid of fewer than 32 such workgroups (a short prefill, e.g.
// 128 tokens at 16 / 4 heads: 16 workgroups) leaves most CUs idle, and two
// heads a workgroup twice as many workgroups ran faster (measured at 128
// tokens: 13.2 us with four, 10.9 with two, 12.3 with one). Every head's
// arithmetic is its own, so the choice changes no bits.
template <int D> unsigned prefill_heads(const GqaShape &s) {
  const unsigned G = s.Hq / s.Hkv, hw = heads_per_wg<D>(G);
  const unsigned nb = (s.T + BM - 1) / BM;
  return hw == 4 && nb * s.Hkv * (G / hw) < 32 ? 2u : hw;
}

template <int D>
hipError_t launch_gated_d(const GqaShape &s, const uint16_t *q, const uint16_t *k,
                          const uint16_t *v, uint16_t *out, const GateArgs &ga,
                          hipStream_t stream) {
  switch (prefill_heads<D>(s)) {
  case 1:
    return launch_dw<D, 1, true>(s, q, k, v, out, stream, ga);
  case 2:
    return launch_dw<D, 2, true>(s, q, k, v, out, stream, ga);
  case 4:
    if (D == 256 && use_halves(s))
      return launch_halves<true>(s, q, k, v, out, stream, ga);
    return launch_dw<D, 4, true>(s, q, k, v, out, stream, ga);
  }
  return hipErrorInvalidValue;
}

template <int D>
hipError_t launch_d(const GqaShape &s, const uint16_t *q, const uint16_t *k,
                    const uint16_t *v, uint16_t *out, hipStream_t stream) {
  switch (prefill_heads<D>(s)) {
  case 1:
    return launch_dw<D, 1>(s, q, k, v, out, stream);
  case 2:
    return launch_dw<D, 2>(s, q, k, v, out, stream);
  case 4:
    if (D == 256 && use_halves(s))
      return launch_halves<false>(s, q, k, v, out, stream);
    return launch_dw<D, 4>(s, q, k, v, out, stream);
  case 8:
    if constexpr (D == 128)
      return launch_dw<D, 8>(s, q, k, v, out, stream);
  }
  return hipErrorInvalidValue;
}

// The split of a prefill's keys. Without one a short chunk on a long history
// keeps a few CUs busy (61 tokens, 16 / 4 heads: 8 workgroups, 391 us at
// 16411 past rows at head_dim 256 and 290 at 128; split 37 and 26), so the
// keys are divided until every CU has a workgroup. A split takes at least
// kSplitSteps tiles of 64 keys, counted over the past rows, which every row
// sees: its O^T is written out and merged for what it saves (2 tokens on 1024
// rows: 32.8 us unsplit, 19.7 / 21.6 / 27.0 at 3 / 4 / 6 tiles a split; 512
// tokens on 500: 31.7 unsplit, 33.8 at 3), so at 511 past rows and fewer
// nothing is split. At head_dim 256 two blocks of rows and more run as the
// key-split kernel's pairs. A block's keys are divided by a whole number, so a
// grid of more than half the CUs stays as it is: 1024 tokens on 4096 rows take
// 99 us in two splits, 1025 tokens 123 in none (head_dim 128: 64 and 89). In two
// splits from 64 workgroups on and at few past rows the plain call pays more for
// the partials than it saves, and the gated one, whose gates then leave the
// attention kernel, gains (undivided / divided): 500 tokens of 16 / 4 heads of 256
// on 512 rows 31.6 / 32.9 us plain, 68.6 / 42.6 gated; 128 of 64 / 16 heads 26.2 /
// 31.1 and 62.6 / 38.0; 500 of 32 / 8 heads of 128 23.7 / 25.1. Both take one rule,
// so that their bits agree.
constexpr unsigned kSplitSteps = 4, kSplitWorkgroups = 256;
static_assert(kSplitSteps >= 3, "a split's first tile is visible to every row of its block");

struct SplitPlan {
  unsigned splits = 1;
  bool halves = false;
};
SplitPlan split_plan(const GqaShape &s) {
  SplitPlan p;
  if (s.T < 2 || !prefill_supported(s))
    return p;
  const unsigned G = s.Hq / s.Hkv, nb = (s.T + BM - 1) / BM;
  const unsigned hw = s.D == 256 ? heads_per_wg<256>(G) : heads_per_wg<128>(G);
  p.halves = s.D == 256 && hw == 4 && (forced_halves() >= 0 ? forced_halves() == 1 : nb >= 2);
  const uint64_t base = p.halves ? (uint64_t)(nb + 1) / 2 * s.Hkv * (G / 2)
                                 : (uint64_t)nb * s.Hkv * (G / hw);
  const unsigned most = s.P / BN / kSplitSteps;
  if (2 * base <= kSplitWorkgroups && most >= 2)
    p.splits = std::min((unsigned)(kSplitWorkgroups / base), most);
  return p;
}

template <int D>
hipError_t launch_split_d(const GqaShape &s, const uint16_t *q, const uint16_t *k,
                          const uint16_t *v, uint16_t *out, void *workspace,
                          const GateArgs *ga, hipStream_t stream) {
  const SplitPlan p = split_plan(s);
  const unsigned nb = (s.T + BM - 1) / BM;
  const size_t units = (size_t)p.splits * nb * s.Hq;
  SplitArgs sa;
  sa.ml = static_cast<float *>(workspace);
  sa.o = sa.ml + units * 2 * BM;
  sa.splits = p.splits;
  hipError_t rc = hipErrorInvalidValue;
  if (p.halves) {
    rc = launch_halves<false, true>(s, q, k, v, out, stream, NoArgs{}, sa);
  } else {
    switch (heads_per_wg<D>(s.Hq / s.Hkv)) {
    case 1:
      rc = launch_dw<D, 1, false, true>(s, q, k, v, out, stream, NoArgs{}, sa);
      break;
    case 2:
      rc = launch_dw<D, 2, false, true>(s, q, k, v, out, stream, NoArgs{}, sa);
      break;
    case 4:
      rc = launch_dw<D, 4, false, true>(s, q, k, v, out, stream, NoArgs{}, sa);
      break;
    case 8:
      if constexpr (D == 128)
        rc = launch_dw<D, 8, false, true>(s, q, k, v, out, stream, NoArgs{}, sa);
      break;
    }
  }
  if (rc != hipSuccess)
    return rc;
  const dim3 grid(nb * s.Hq * (D / 32)); // four waves a workgroup
  half_t *o = reinterpret_cast<half_t *>(out);
  if (ga)
    hipLaunchKernelGGL((gqa_prefill_merge_kernel<D, true>), grid, dim3(256), 0, stream, sa.ml,
                       sa.o, o, s.T, s.Hq, nb, p.splits, ga->qproj, ga->activated);
  else
    hipLaunchKernelGGL((gqa_prefill_merge_kernel<D, false>), grid, dim3(256), 0, stream, sa.ml,
                       sa.o, o, s.T, s.Hq, nb, p.splits, (const half_t *)nullptr, 0u);
  return hipGetLastError();
}

} // namespace

bool prefill_supported(const GqaShape &s) {
  const unsigned G = s.Hkv ? s.Hq / s.Hkv : 0;
  // A 64-key slice of one cache must stay within a buffer descriptor's
  // 32-bit range.
  const uint64_t sliceBytes = (uint64_t)BN * s.Hkv * s.D * 2;
  return (s.D == 128 || s.D == 256) && (G == 1 || G == 2 || G == 4 || G == 8) &&
         s.T >= 1 && sliceBytes < (1ull << 31);
}

bool prefill_gated_supported(const GqaShape &s, unsigned rot) {
  // The shapes that the call has always taken: those whose normalised query
  // tile and its tables fit a key tile's LDS, where they once lay. At head_dim
  // 128 rotary widths to 96 and up to four heads, at 256 to 224.
  const unsigned HW = s.D == 256 ? heads_per_wg<256>(s.Hkv ? s.Hq / s.Hkv : 0)
                                 : heads_per_wg<128>(s.Hkv ? s.Hq / s.Hkv : 0);
  const size_t need = (size_t)BM * (s.D + 8) * 2 + BM * 4 + (size_t)s.D * 4 +
                      (size_t)BM * (rot / 2) * 4;
  return prefill_supported(s) && HW <= 4 && need <= (size_t)BN * 2 * s.D &&
         rot % 16 == 0 && rot <= s.D;
}

hipError_t launch_gqa_prefill_gated(const uint16_t *q, const uint16_t *k, const uint16_t *v,
                                    uint16_t *out, const GqaShape &s, const uint16_t *qproj,
                                    unsigned activated, hipStream_t stream) {
  const GateArgs ga{reinterpret_cast<const half_t *>(qproj), activated};
  if (s.D == 128)
    return launch_gated_d<128>(s, q, k, v, out, ga, stream);
  return launch_gated_d<256>(s, q, k, v, out, ga, stream);
}

hipError_t launch_gqa_prefill(const uint16_t *q, const uint16_t *k,
                              const uint16_t *v, uint16_t *out,
                              const GqaShape &s, hipStream_t stream) {
  if (s.D == 128)
    return launch_d<128>(s, q, k, v, out, stream);
  return launch_d<256>(s, q, k, v, out, stream);
}

bool prefill_split(const GqaShape &s) { return split_plan(s).splits > 1; }

size_t prefill_workspace_bytes(const GqaShape &s) {
  const SplitPlan p = split_plan(s);
  const size_t units = (size_t)p.splits * ((s.T + BM - 1) / BM) * s.Hq;
  return p.splits > 1 ? units * BM * (2 + s.D) * sizeof(float) : 0;
}

hipError_t launch_gqa_prefill_split(const uint16_t *q, const uint16_t *k, const uint16_t *v,
                                    uint16_t *out, void *workspace, const GqaShape &s,
                                    const uint16_t *qproj, unsigned activated,
                                    hipStream_t stream) {
  const GateArgs gate{reinterpret_cast<const half_t *>(qproj), activated};
  const GateArgs *ga = qproj ? &gate : nullptr;
  if (s.D == 128)
    return launch_split_d<128>(s, q, k, v, out, workspace, ga, stream);
  return launch_split_d<256>(s, q, k, v, out, workspace, ga, stream);
}

} // namespace llmi
