// pa_prefill.hpp -- causal paged prefill on CDNA4 matrix cores (gfx950).
//
// Replaces the reference's WMMA tile kernel (kernels/paged_attn_wmma.cu:36-210)
// with a design built around v_mfma_f32_32x32x16_{f16,bf16}:
//
//  * A work-group (4 waves) owns one (sequence b, KV head, block of 128
//    packed query rows); wave w owns 32 of those rows, one MFMA n-tile.  The
//    rows of a GQA group's heads are packed: row R of the block numbering is
//    head R % G of chunk row R / G, so rows stay ordered by position, a block
//    spans QB / G positions (fewer half-masked diagonal tiles) and a chunk
//    shorter than a block still fills its rows with its heads (groups of 4 and
//    8: the 8-wave kernel 5-17 % faster than
//    with a block per query head, this one up to 12 %, none slower).  The kernel
//    is sized for two work-groups per CU (<= 256 registers per lane, 68 KB of
//    LDS), so every SIMD holds two waves and one wave's softmax arithmetic
//    overlaps the other's matrix work.
//  * Key tiles (64 keys for D <= 128, 32 for D = 256) are gathered from the
//    paged pool (block table -> page -> row, 64-bit offsets) straight into
//    LDS with global_load_lds_dwordx4: no registers or VALU stores on the way,
//    and the next tile's loads are in flight while the current one is used.
//    Rows are XOR-swizzled in 16-byte chunks (the swizzle is applied on the
//    global side, since a wave's direct load fills 1 KB of LDS in lane order).
//  * Scores are computed transposed, S^T = K . Q^T: K rows are the MFMA A
//    operand read from LDS (16 bytes per lane), the wave's 32 query rows are
//    the B operand held in registers for the whole loop.  In the 32x32 S^T
//    accumulator layout a lane holds 16 keys of one query column, eight of
//    which are exactly the B operand slots of one 16-key step of
//    O^T += V^T . P^T -- probabilities never leave registers.  The V^T A
//    operand is two ds_read_b64_tr_b16 per step.
//  * The softmax is done in log2 units with the scale folded into one FMA per
//    score; the running max is only raised when a tile's max exceeds it by
//    more than 2^8 (probabilities stay <= 256, exact in fp16/bf16 range), so
//    the O^T rescale is a rare wave-uniform branch instead of a per-tile
//    multiply.  Masking runs only on tiles that cross a wave's diagonal.
//  * Work-groups are ordered by query block, longest first, across all
//    (sequence, head) pairs.  (Grouping one (sequence, head)'s blocks on one
//    XCD, for L2 reuse, put three blocks of the same length on each CU when
//    all work-groups are resident: config 4a ran 22 % slower.)
//
// Semantics follow kernels/paged_attn_wmma.cu:80-205: query row r of the
// chunk sits at ctx - S + r and sees keys [0, ctx - S + r]; accumulation and
// the softmax are fp32; a row that sees no key is written as zeros (:200).
// Precision: P is carried in fp16 (11-bit significand) as the reference does.
// A bf16 V tile is converted to fp16 while it is staged, so P.V runs in fp16
// too; if any staged |v| reaches 65520 (fp16 overflow, or inf) the
// work-group restarts in a mode that keeps V in bf16 and carries P as a bf16
// hi + lo pair (two P.V products, ~16-bit significand).  q that does not
// arrive in the KV type is likewise split into hi + lo for Q.K^T.
#pragma once

#include "pa_device.hpp"

#include <algorithm>
#include <atomic>

namespace pa {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef short short4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) short4_t lds_short4_t;
typedef __attribute__((address_space(3))) void lds_void_t;
typedef uint64_t u64x2_t __attribute__((ext_vector_type(2)));

// 16 bytes per lane from global memory straight into LDS (global_load_lds_dwordx4):
// lane i writes lds + 16*i; lds must be wave-uniform.  (A function of its own:
// used directly in the kernel template, the builtin stops the host pass from
// emitting the launch stubs.)
__device__ inline void lds_dma16(const void* g, lds_void_t* lds) {
  __builtin_amdgcn_global_load_lds(g, lds, 16, 0, 0);
}

// The same load as inline asm (M0 set by the compiler from the operand).  The
// compiler does not see it write LDS, so it places no wait for it before later
// LDS reads; the caller waits (vmcnt) before the barrier that publishes the data.
__device__ inline void lds_dma16_async(const void* g, lds_void_t* lds) {
  const uint32_t m = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)lds);
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(g), "{m0}"(m));
}

template <bool kBf16>
__device__ inline f32x16_t mfma32(const u32x4_t& a, const u32x4_t& b, const f32x16_t& c) {
  if constexpr (kBf16) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                   __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
  } else {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8_t, a),
                                                  __builtin_bit_cast(half8_t, b), c, 0, 0, 0);
  }
}

// Two fp32 values -> one packed 16-bit pair, round to nearest even.
template <bool kBf16>
__device__ inline uint32_t pack2(float x, float y) {
  if constexpr (kBf16) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(float2_t{x, y}, bf16x2_t));
  } else {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(float2_t{x, y}, half2_t));
  }
}

// The two fp32 values of a packed 16-bit pair.
template <bool kBf16>
__device__ inline float2_t unpack2(uint32_t w) {
  if constexpr (kBf16) {
    return float2_t{__builtin_bit_cast(float, w << 16), __builtin_bit_cast(float, w & 0xffff0000u)};
  } else {
    const half2_t h = __builtin_bit_cast(half2_t, w);
    return float2_t{(float)h[0], (float)h[1]};
  }
}

// Eight consecutive q elements (16-byte aligned) as fp32.
__device__ inline void load8f(const void* q, int dtype, int64_t idx, float (&x)[8]) {
  if (dtype == kF32) {
    const float4_t a = *reinterpret_cast<const float4_t*>(static_cast<const float*>(q) + idx);
    const float4_t b = *reinterpret_cast<const float4_t*>(static_cast<const float*>(q) + idx + 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      x[e] = a[e];
      x[4 + e] = b[e];
    }
  } else {
    const u32x4_t r = *reinterpret_cast<const u32x4_t*>(static_cast<const uint16_t*>(q) + idx);
    if (dtype == kF16) {
      KvF16::widen(r, x);
    } else {
      KvBF16::widen(r, x);
    }
  }
}

constexpr int kPfThreads = 256;   // 4 waves
constexpr int kPfBtStage = 1024;  // block-table entries staged in LDS
constexpr float kLazyRescale = 8.0f;  // raise the running max only past 2^8
constexpr float kWeightCap = 32768.0f;  // 8-wave kernel: raise it when a lane's weights sum past 2^15
                                        // (weights up to 2^15 are exact in fp16 and bf16 range)


// How a tile's P.V product is formed.
enum PvMode : int {
  kPvDirect = 0,   // V tile loaded straight into LDS; P and V in fp16
  kPvConvert = 1,  // bf16 V converted to fp16 while staged; P and V in fp16
  kPvSplit = 2,    // bf16 V in LDS; P as bf16 hi + lo, two products
  kPvF8 = 3,       // FP8 K and V codes staged in registers, written to LDS as fp16 (exact)
  kPvScalar = 4,   // fp32-precision kernel, non-finite data: both products on the vector ALU
};
template <int M>
struct PvTag {
  static constexpr int value = M;
};

// FP8 (E4M3) caches: the codes convert exactly to fp16 and to bf16, so K tiles
// take q's 16-bit type (no hi + lo split of a bf16 q) and V tiles fp16 (P
// stays fp16).  KvFP8 serves fp16 and fp32 q, KvFP8QkBf16 bf16 q.
struct KvFP8QkBf16 : KvFP8 {
  static constexpr const char* kName = "pa::KvFP8QkBf16";
};
template <typename KV>
struct QkBf16 {  // Q.K^T on bf16 MFMA
  static constexpr bool value = KV::kCode == kBF16;
};
template <>
struct QkBf16<KvFP8QkBf16> {
  static constexpr bool value = true;
};

template <int D>
struct PfShape {
  static constexpr int QW = 32;                  // query rows per wave (one MFMA n-tile)
  static constexpr int QB = 4 * QW;              // query rows per work-group
  static constexpr int KB = D <= 128 ? 64 : 32;  // keys per tile
  static constexpr int MT = KB / 32;             // 32-key m-tiles of S^T
  static constexpr int KS = D / 16;              // 16-dim k-steps of Q.K^T
  static constexpr int DT = D / 32;              // 32-dim m-tiles of O^T
  static constexpr int NCH = D / 8;              // 16-byte chunks per row
  // LDS chunk swizzles (chunk cc of row r sits at position cc ^ f(r)), one per
  // read pattern, so that every 256-byte LDS pass hits 64 distinct banks:
  //  K, read as the S^T A operand (16 consecutive rows, one chunk):
  //    f(r) = (r >> KSH) & KSW;
  //  V, read transposed (4 consecutive rows x 4 consecutive chunks per 32
  //  lanes): f(r) = ((r >> VSH) & VSW) << 2.
  static constexpr int KSW = (NCH < 16 ? NCH : 16) - 1;
  static constexpr int KSH = NCH >= 16 ? 0 : NCH == 8 ? 1 : 2;
  static constexpr int VSW = NCH >= 16 ? 3 : NCH == 8 ? 1 : 0;
  static constexpr int VSH = NCH >= 16 ? 0 : 1;
  static constexpr int CPT = KB * NCH / kPfThreads;    // chunks per thread per tile
  static constexpr int WAVES_PER_EU = D <= 128 ? 2 : 1;
  static_assert(KB * NCH % kPfThreads == 0, "tile chunks must divide the work-group");
};

// LDS element offsets of (row, chunk cc) in the swizzled [KB][D] K and V tiles.
template <int D>
__device__ inline int kpos(int row, int cc) {
  return cc ^ ((row >> PfShape<D>::KSH) & PfShape<D>::KSW);
}
template <int D>
__device__ inline int vpos(int row, int cc) {
  return cc ^ (((row >> PfShape<D>::VSH) & PfShape<D>::VSW) << 2);
}
template <int D>
__device__ inline int swk(int row, int cc) {
  return row * D + (kpos<D>(row, cc) << 3);
}
template <int D>
__device__ inline int swv(int row, int cc) {
  return row * D + (vpos<D>(row, cc) << 3);
}

// The i-th head group that sequence b's work-groups take.  Pairs reach the 8 XCDs
// round robin, so with eight packed KV heads each XCD kept to one of them: its K and
// V rows lie a whole token row apart and share few of the L2's channels.  The heads'
// order therefore moves on with the sequence.  8-wave kernel, fp16, 64/8 heads of
// 128, one block per query head before packing -> packed in a fixed order -> this:
// 8 prompts of 256 rows 42 -> 58 -> 36 us, 16 prompts 80 -> 104 -> 69 us; 32/8 heads,
// 16 prompts of 512 rows 94 -> 96 -> 83 us.
__device__ __forceinline__ int pf_turn(const PrefillParams& p, int b, int i) {
  if (p.gp == 1) return i;
  i += (b & 7) * p.HG >> 3;
  return i >= p.HG ? i - p.HG : i;
}

// Sum over the wave, in scalar registers: rotations within rows of 16 lanes, then one
// lane of each row.
__device__ __forceinline__ int pf_wave_sum(int s) {
  s += __builtin_amdgcn_update_dpp(0, s, 0x128, 0xf, 0xf, false);  // row_ror:8
  s += __builtin_amdgcn_update_dpp(0, s, 0x124, 0xf, 0xf, false);
  s += __builtin_amdgcn_update_dpp(0, s, 0x122, 0xf, 0xf, false);
  s += __builtin_amdgcn_update_dpp(0, s, 0x121, 0xf, 0xf, false);
  return __builtin_amdgcn_readlane(s, 0) + __builtin_amdgcn_readlane(s, 16) + __builtin_amdgcn_readlane(s, 32) +
         __builtin_amdgcn_readlane(s, 48);
}

// Work-group x -> partition (context split, the slow index) and unit (b, head
// group, block of QB packed rows); false past the last unit of a compacted
// grid (work-group uniform).
template <int QB, bool kPart>
__device__ __forceinline__ bool pf_unit(const PrefillParams& p, int64_t x, int lane, int& part, int64_t& unit, int& qt,
                                        int& hg, int& b) {
  part = 0;
  // Work-group -> unit (b, h, query block).  Units are numbered with the
  // query block as the slow index, longest first across all (sequence, head)
  // pairs.  When the grid is more than one resident wave, work-group x takes
  // unit x: the dispatcher hands the longest remaining unit to each CU slot
  // that frees.  When every work-group is resident at once (p.wg_cus = C
  // CUs), the dispatcher places work-groups x, x + C, x + 2C, ... on one CU;
  // odd generations then take their units mirrored, so each CU's units add
  // up to about the same number of key tiles (config 4a: 27-28 per CU instead
  // of 20-34).  The mirror keeps x mod 8 (work-groups go to the 8 XCDs round
  // robin), so a (sequence, head) pair's blocks, which read the same keys,
  // stay on one XCD's L2.
  const int nq = p.q_tiles;
  const int64_t nbh = (int64_t)p.B * p.HG;
  if (p.vl_compact) {
    // Variable-length batch, compacted grid: the work-groups take only the
    // (query block, sequence, head) units that have rows -- query blocks
    // from the last (longest) down, then sequences, then heads -- and those
    // past the last unit exit.  A grid sized by the longest sequence would
    // dispatch a work-group for every block of every sequence, most of them
    // (decode rows of a mixed batch, blocks past a short sequence's rows)
    // exiting only after a memory round trip, and spread the working ones
    // across the launch.  Per-sequence block counts sit in the lanes
    // (kVlMaxSeqs / 64 per lane).
    int nbk[kVlMaxSeqs / 64];
#pragma unroll
    for (int c = 0; c < kVlMaxSeqs / 64; ++c) {
      const int i = c * 64 + lane;
      nbk[c] = 0;
      if (i < p.B) {
        const int qa = p.cu_q[i], qb = p.cu_q[i + 1];
        int len = qa >= 0 && qb >= qa && (int64_t)qb <= p.q_total ? qb - qa : 0;
        if (p.skip_single && len == 1) len = 0;
        nbk[c] = (min(len, p.S) * p.gp + QB - 1) / QB;
      }
    }
    if constexpr (kPart) {  // the partitions of the units there are, so that the idle work-groups come last
      int mine = 0;
#pragma unroll
      for (int c = 0; c < kVlMaxSeqs / 64; ++c) mine += nbk[c];
      mine = pf_wave_sum(mine);
      // No more than the grid and the workspace hold: a cu_q whose ranges overlap
      // ([0, 512, 0, 512] of 512 rows) has more rows than T.  The units past them
      // stay unserved, as past the end of the unsplit kernel's grid.
      const int64_t rows = (int64_t)mine * p.HG;
      const int64_t total = rows < p.units ? rows : p.units;
      if (x >= total * p.parts) return false;
      part = (int)(x / total);
      x -= part * total;
    }
    unit = x;
    // The largest block t with more units from it on than x, by bisection (a walk
    // down from the last block costs up to 0.6 us a step, and packed heads have many:
    // fp16, 8/1 heads of 128, one prompt of 512 rows at 1024, split, 60.3 -> 22.3 us;
    // of 1024 at 2048 121.9 -> 35.0; of 2048, unsplit, 68.5 -> 44.6).
    int ft = 0, hi = nq;
    int64_t past = 0;  // units of the blocks past it
    while (hi - ft > 1) {  // wave-uniform
      const int mid = (ft + hi) >> 1;
      int s = 0;
#pragma unroll
      for (int c = 0; c < kVlMaxSeqs / 64; ++c) s += max(nbk[c] - mid, 0);
      const int64_t from = (int64_t)pf_wave_sum(s) * p.HG;
      if (x < from) {
        ft = mid;
      } else {
        hi = mid;
        past = from;
      }
    }
    int64_t rem = x - past;
    int fb = -1, fh = 0;
#pragma unroll
    for (int c = 0; c < kVlMaxSeqs / 64; ++c) {
      const uint64_t m = __builtin_amdgcn_ballot_w64(nbk[c] > ft);
      const int64_t cnt = (int64_t)__builtin_popcountll(m) * p.HG;
      if (fb < 0) {
        if (rem < cnt) {
          const int k = (int)(rem / p.HG);
          const int rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
          const uint64_t sel = __builtin_amdgcn_ballot_w64(((m >> lane) & 1u) != 0 && rank == k);
          fb = c * 64 + __builtin_ctzll(sel);
          fh = (int)(rem - (int64_t)k * p.HG);
        } else {
          rem -= cnt;
        }
      }
    }
    if (fb < 0) return false;
    qt = ft;
    b = fb;
    hg = pf_turn(p, b, fh);
  } else {
    if constexpr (kPart) {
      part = (int)(x / p.units);
      x -= (int64_t)part * p.units;
    }
    unit = x;
    if (p.wg_cus > 0) {
      const int64_t C = p.wg_cus, g = x / C, j = x - g * C;
      if ((g & 1) && (g + 1) * C <= nbh * nq) x = g * C + (C % 8 == 0 ? C - 8 - (j & ~(int64_t)7) + (j & 7) : C - 1 - j);
    }
    qt = nq - 1 - (int)(x / nbh);
    const int64_t bh = x % nbh;
    b = (int)(bh / p.HG);
    hg = pf_turn(p, b, (int)(bh % p.HG));
  }
  return true;
}

// A sequence's query rows: `S` of them (row r at position ctx - S + r)
// starting at token tok0 of q/out, of which `served` are; false when the
// decode kernel serves the sequence.
__device__ __forceinline__ bool pf_rows(const PrefillParams& p, int b, int& S, int64_t& tok0, int& served) {
  // Uniform batches: p.S rows each.  Variable-length batches: rows cu_q[b] ..
  // cu_q[b+1] of the packed [T, H, D] q/out, at most p.S (the caller's
  // max_q_len) of them served; a malformed range (negative, decreasing or
  // past T) is treated as empty.
  S = p.S;
  tok0 = (int64_t)b * p.S;
  if (p.cu_q) {
    const int qa = p.cu_q[b], qb = p.cu_q[b + 1];
    const bool ok = qa >= 0 && qb >= qa && (int64_t)qb <= p.q_total;
    S = ok ? qb - qa : 0;
    tok0 = ok ? qa : 0;
    if (p.skip_single && S == 1) return false;
  }
  served = min(S, p.S);
  return true;
}

// kSplit (key-split mode, tiles of two 32-key m-tiles): a work-group serves
// 64 query rows; waves 0-1 own rows 0-31 / 32-63 over the first 32 keys of
// every tile, waves 2-3 the same rows over the second 32, and the two halves
// are merged through LDS at the end (log-sum-exp rule).  The loads and the
// LDS layout are those of the plain mode; each wave does half of a tile's
// work, so a query block's chain of tiles takes half as long and twice as
// many work-groups share the work.  Chosen when the plain grid is too short
// for the dispatcher to balance causal blocks (config 4a: 768 work-groups,
// chains of 2 to 16 tiles, on 768 slots).
//
// kQP: q is carried as kQP 16-bit pieces (1: it arrives in the Q.K^T type).
//
// kX (fp32-precision mode, prefill32_kernel): q and the weights are carried as
// two fp16 pieces (three bf16 pieces over a bf16 cache) whose sum is the fp32
// value to 2^-24 of it or the pieces' smallest step (bf16: exactly), and every
// product of a piece with a K or V element is exact in the matrix cores' fp32
// accumulation, so both products keep fp32 precision at two (three) 16-bit
// products each.  fp16 pieces need the range: each q row is scaled by a power of
// two that puts its largest element in [2^14, 2^15), and the weights by 2^7 (they
// are at most 2^8 by the lazy maximum, which is kept an integer so that these
// shifts are exact).  The smallest step, half of fp16's 2^-24, is then 2^-32 of a
// weight of 1 and 2^-39 of a row's largest q: below those the rounding is
// absolute, under the 2^-24 that fp32 sums of the largest terms carry.
// Bound by the matrix and vector work of the pieces (the 16-bit-weight kernel's
// chain of tiles with four products for its three and ~180 more vector
// instructions per 64 keys).  B = 4, S = 512, context 2048, 12 heads of 64,
// fp16 cache, fp32 q: 1105 us as a decode problem per query row on the vector
// ALU -> 42 us (10 -> 266 TFLOP/s; the fp32 matrix rate is 154), error against
// 64 bits 3.2e-7 -> 2.5e-7.
//
// kPart (context split, split_prefill*_kernel): the work-group computes one
// partition of its block's key tiles and writes partial sums.  An instance of
// its own: as a run-time choice it cost the others 1-6 %.
template <typename KV, int D, int kQP, bool kSplit, bool kX, bool kPart>
__device__ __forceinline__ void prefill_body(const PrefillParams& p) {
  using Sh = PfShape<D>;
  constexpr int QW = Sh::QW, KB = Sh::KB, MT = Sh::MT, KS = Sh::KS, DT = Sh::DT;
  static_assert(!kSplit || MT == 2, "the key-split mode halves tiles of two m-tiles");
  constexpr int MTW = kSplit ? 1 : MT;           // 32-key m-tiles of each tile this wave computes
  constexpr int QB = kSplit ? 2 * QW : Sh::QB;   // query rows per work-group
  constexpr int NCH = Sh::NCH, CPT = Sh::CPT;
  constexpr bool kBf16 = QkBf16<KV>::value;  // Q.K^T operand type (and the type of a split q)
  constexpr bool kF8 = KV::kCode == kFP8;    // tiles converted from FP8 codes; P.V in fp16
  constexpr int EB = KV::kBytes;
  constexpr bool kXBf16 = kX && KV::kCode == kBF16;     // weights and V as bf16 (three pieces)
  constexpr bool kXScale = kX && !kBf16 && kQP > 1;     // fp16 q pieces of a scaled row
  constexpr float kXBias = kX && !kXBf16 ? 7.0f : 0.0f;  // log2 of the weights' scale

  __shared__ __attribute__((aligned(16))) uint16_t sK0[KB * D];
  __shared__ __attribute__((aligned(16))) uint16_t sK1[KB * D];
  __shared__ __attribute__((aligned(16))) uint16_t sV0[KB * D];
  __shared__ __attribute__((aligned(16))) uint16_t sV1[KB * D];
  __shared__ int32_t s_bt[kPfBtStage];  // window of the work-group's block ids
  __shared__ int s_badkey;              // first key whose page has an invalid block id
  __shared__ u64x2_t s_off0[KB];        // per-row K/V byte offsets of a tile (even / odd tiles)
  __shared__ u64x2_t s_off1[KB];
  __shared__ int s_ovf;                 // the fp16 pass produced a non-finite O

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int rw = kSplit ? (wave & 1) : wave;   // this wave's 32 query rows of the block
  const int par = kSplit ? (wave >> 1) : 0;    // key half of every tile (key-split mode)
  const int n = lane & 31;   // query column of this lane (S^T, O^T) / key row (K operand)
  const int hh = lane >> 5;  // lane half: k-slot block of the operands

  int part, qt, hg, b;
  int64_t unit;
  if (!pf_unit<QB, kPart>(p, blockIdx.x, lane, part, unit, qt, hg, b)) return;  // past the last unit (work-group uniform)
  const int h0 = hg * p.gp;  // first query head of the unit
  const int kvh = h0 / p.G;

  int S, served;
  int64_t tok0;
  if (!pf_rows(p, b, S, tok0, served)) return;
  const int Sr = served * p.gp;  // packed rows served
  const int ctx = p.context_lens[b];
  const int maxctx = p.MB * p.BS;
  const int qs0 = qt * QB;
  if (qs0 >= Sr) return;            // no served rows of this sequence here (work-group uniform)
  const int qw0 = qs0 + rw * QW;    // this wave's first query row
  const int qrow = qw0 + n;
  const bool live = qrow < Sr;
  // Packed row -> chunk row and head; the row's offset in q and out.
  auto chunk_row = [&](int r) { return (int)fastdiv((uint32_t)r, p.gp_div); };
  const int srow = chunk_row(qrow);
  auto row_offset = [&](int r) {
    const int sr = chunk_row(r);
    return ((tok0 + sr) * p.H + h0 + (r - sr * p.gp)) * D;
  };

  if (ctx > maxctx) {  // context longer than the block table: poison rows that attend keys
    if (live && hh == 0 && (!kPart || part == 0)) {
      const float fillv = ctx - S + srow < 0 ? 0.0f : __builtin_nanf("");
      const int64_t row_at = row_offset(qrow);
      for (int d = 0; d < D; ++d) store_elem(p.out, p.out_dtype, row_at + d, fillv);
    }
    return;
  }
  if (threadIdx.x == 0) {
    s_badkey = 0x7fffffff;
    s_ovf = 0;
  }

  // Keys the work-group's rows can see: [0, kend); this wave's rows: [0, wave_kend).
  int kend = min(ctx, ctx - S + chunk_row(min(qs0 + QB, Sr) - 1) + 1);
  int ntiles = kend > 0 ? (kend + KB - 1) / KB : 0;
  const int wave_last = min(qw0 + QW - 1, Sr - 1);
  int wave_kend = qw0 < Sr ? min(ctx, ctx - S + chunk_row(wave_last) + 1) : 0;
  int wave_kfull = ctx - S + chunk_row(qw0) + 1;  // keys below this are visible to every row of the wave
  const int qpos = ctx - S + srow;
  int qlim = min(qpos, kend - 1);        // last key this column may see
  const int npages = kend > 0 ? (int)fastdiv((uint32_t)(kend - 1), p.bs_div) + 1 : 0;
  // Context split: partition `part` of the unit's tiles, whose keys are
  // numbered from its first one, key0, from here on.  A unit of one partition
  // writes its output rows, the others their partial sums.
  int key0 = 0;
  bool whole = true;
  if constexpr (kPart) {
    const int n = (ntiles + p.part_tiles - 1) / p.part_tiles;
    if (part >= max(n, 1)) return;  // work-group uniform
    whole = n <= 1;
    key0 = part * p.part_tiles * KB;
    ntiles = min(p.part_tiles, ntiles - part * p.part_tiles);
    kend -= key0;
    wave_kend -= key0;
    wave_kfull -= key0;
    qlim -= key0;
  }

  // Q^T operand (row qrow, dims ks*16 + hh*8 .. +8) in the KV type.  The sign of
  // the scale is applied here (exactly), so the softmax scale below is positive.
  u32x4_t qf[kQP][KS];
  float qs_row = p.qscale;  // softmax scale of this lane's row (kXScale: less the row's power of two)
  const int64_t qoff = row_offset(live ? qrow : 0) + hh * 8;
  if constexpr (kQP == 1) {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      u32x4_t r = u32x4_t{0u, 0u, 0u, 0u};
      if (live) r = *reinterpret_cast<const u32x4_t*>(static_cast<const uint16_t*>(p.q) + qoff + ks * 16);
      qf[0][ks] = (r & p.q_and) ^ p.q_xor;
    }
  } else {
    float sgn = p.q_sign;
    auto load_row = [&](int ks, float (&xv)[8]) {
      if (live) {
        load8f(p.q, p.q_dtype, qoff + ks * 16, xv);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) xv[e] = 0.0f;
      }
    };
    if constexpr (kXScale) {
      float mxq = 0.0f;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        float xv[8];
        load_row(ks, xv);
#pragma unroll
        for (int e = 0; e < 8; ++e) mxq = fmaxf(mxq, __builtin_fabsf(xv[e]));
      }
      mxq = fmaxf(mxq, __shfl_xor(mxq, 32, 64));
      // 2^k with mxq 2^k in [2^14, 2^15); k within [-100, 100] (a smaller row's
      // scores are below 2^-60 whatever its keys hold), none for Inf.
      const int ex = (int)(__builtin_bit_cast(uint32_t, mxq) >> 23) - 127;
      const int k = ex > 127 ? 0 : max(-100, min(100, 14 - ex));
      sgn *= __builtin_bit_cast(float, (uint32_t)(127 + k) << 23);
      qs_row *= __builtin_bit_cast(float, (uint32_t)(127 - k) << 23);
    }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      float xv[8];
      load_row(ks, xv);
#pragma unroll
      for (int e = 0; e < 8; ++e) xv[e] *= sgn;
#pragma unroll
      for (int pc = 0; pc < kQP; ++pc) {
        uint32_t w[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          w[j] = pack2<kBf16>(xv[2 * j], xv[2 * j + 1]);
          const float2_t r = unpack2<kBf16>(w[j]);
          xv[2 * j] -= r[0];
          xv[2 * j + 1] -= r[1];
        }
        qf[pc][ks] = u32x4_t{w[0], w[1], w[2], w[3]};
      }
    }
  }
  const float qscale = kXScale ? qs_row : p.qscale;

  const int32_t* bt_row = p.block_tables + (int64_t)b * p.bt_stride;
  // Block ids of the pages this work-group reads live in an LDS window of
  // kPfBtStage pages starting at page win0, so a tile's loads never wait
  // behind a dependent block-table load.  The window moves (at a tile
  // boundary, between barriers) when the next tile to load leaves it.
  int win0 = 0;
  auto stage = [&](int first) {
    win0 = first;
    const int cnt = min(kPfBtStage, npages - first);
    for (int i = threadIdx.x; i < cnt; i += kPfThreads) s_bt[i] = bt_row[first + i];
  };
  auto ensure_window = [&](int t) {  // work-group uniform
    const int last = key0 + min(t * KB + KB, kend) - 1;
    const int plast = (int)fastdiv((uint32_t)last, p.bs_div);
    if (plast >= win0 + kPfBtStage) {
      __syncthreads();
      stage((int)fastdiv((uint32_t)(key0 + t * KB), p.bs_div));
      __syncthreads();
    }
  };

  const char* kbase = static_cast<const char*>(p.k) + (int64_t)kvh * p.k_sh * EB;
  const char* vbase = static_cast<const char*>(p.v) + (int64_t)kvh * p.v_sh * EB;
  const uint32_t k_sbb = (uint32_t)(p.k_sb * EB), k_stb = (uint32_t)(p.k_st * EB);
  const uint32_t v_sbb = (uint32_t)(p.v_sb * EB), v_stb = (uint32_t)(p.v_st * EB);
  const uint64_t nb = (uint64_t)p.num_blocks;

  // This thread's chunks of a tile: chunk c fills LDS chunk position
  // pos = (c*4 + wave)*64 + lane (wave-contiguous 1 KB per direct load), i.e.
  // row pos / NCH at swizzled position pos % NCH; it loads the source chunk
  // whose swizzled position that is (an involution: the same XOR).
  int prow[CPT], ksrc[CPT], vsrc[CPT];
#pragma unroll
  for (int c = 0; c < CPT; ++c) {
    const int pos = (c * 4 + wave) * 64 + lane;
    prow[c] = pos / NCH;
    ksrc[c] = kpos<D>(prow[c], pos % NCH) * 8 * EB;  // byte offset of the 8-element source chunk
    vsrc[c] = vpos<D>(prow[c], pos % NCH) * 8 * EB;
  }
  int badkey = 0x7fffffff;

  // Row offsets of a tile, built once per tile by the first KB / 64 waves (one
  // row per lane) two tiles ahead, so the other waves' loads cost one LDS read and an add
  // per chunk.  Entry r = {K byte offset, V byte offset | use}; a row past
  // kend, or on a page with an invalid block id, points at row 0 of block 0
  // (in bounds, NB >= 1) with use = 0.  Offsets are multiples of 16 bytes, so
  // bit 0 of the V offset is free for the flag.
  auto build = [&](int t, u64x2_t* tb) {
    if (wave * 64 + lane < KB) {
      const int row = wave * 64 + lane;
      const int kabs = t * KB + row;
      const bool valid = kabs < kend;
      const int kk = key0 + (valid ? kabs : 0);
      const int pg = (int)fastdiv((uint32_t)kk, p.bs_div);
      const int off = kk - pg * p.BS;
      const int blk = s_bt[valid ? pg - win0 : 0];
      const bool okb = (uint64_t)(int64_t)blk < nb;
      if (valid && !okb) badkey = min(badkey, key0 + kabs);
      const bool use = valid && okb;
      const uint32_t ub = use ? (uint32_t)blk : 0u, uo = use ? (uint32_t)off : 0u;
      tb[row] = u64x2_t{(uint64_t)ub * k_sbb + uo * k_stb,
                        ((uint64_t)ub * v_sbb + uo * v_stb) | (use ? 1u : 0u)};
    }
  };

  f32x16_t o[DT];
  float m = -__builtin_inff(), l = 0.0f;  // running max (log2 units); this lane half's row sum

  // Both products of one tile on the vector ALU (kX, non-finite data): each
  // row attends its own keys only (a masked key's V never meets its weight:
  // 0 * Inf is NaN), and Inf or NaN reach the row as a chain of fp32 products
  // would carry them.  Same lane layout as the matrix products; a loop step
  // serves one accumulator slot (a key of each lane half), rotated to slot 0.
  auto scalar_tile = [&](int t, const uint16_t* cK, const uint16_t* cV) {
    cK += par * 32 * D;
    cV += par * 32 * D;
    const int tk0 = t * KB + par * 32;
    auto elem = [&](const uint16_t* x, bool bf) {
      return bf ? __builtin_bit_cast(float, (uint32_t)*x << 16) : (float)*reinterpret_cast<const _Float16*>(x);
    };
#pragma unroll 1
    for (int mt = 0; mt < MTW; ++mt) {
      float s[16];
      float mx = -__builtin_inff();
#pragma unroll 1
      for (int r = 0; r < 16; ++r) {
        const int key = mt * 32 + 8 * (r >> 2) + 4 * hh + (r & 3);
        float d = 0.0f;
#pragma unroll 1
        for (int c = 0; c < NCH; ++c) {
          float xv[8];
          load8f(p.q, p.q_dtype, qoff - hh * 8 + c * 8, xv);
          const uint16_t* kr = cK + swk<D>(key, c);
#pragma unroll
          for (int e = 0; e < 8; ++e) d = fmaf(xv[e] * p.q_sign, elem(kr + e, kBf16), d);
        }
        const float sv = tk0 + key > qlim ? -__builtin_inff() : d * p.qscale;
        mx = fmaxf(mx, sv);
#pragma unroll
        for (int i = 0; i < 15; ++i) s[i] = s[i + 1];
        s[15] = sv;
      }
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
      const float mn = fmaxf(m, mx);
      const float corr = mn == -__builtin_inff() ? 1.0f : fast_exp2(m - mn);
      m = mn;
      l *= corr;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) o[dt] *= corr;
      // (The weights carry the matrix pass's scale: partitions of a context split
      // that took either pass are merged.)
      const float negm = (m == -__builtin_inff() ? 0.0f : -m) + kXBias;
#pragma unroll 1
      for (int r = 0; r < 16; ++r) {
        const int key0 = mt * 32 + 8 * (r >> 2) + (r & 3);  // lane half 0's key; half 1's is 4 further
        const float pv = fast_exp2(s[0] + negm);
        l += tk0 + key0 + 4 * hh > qlim ? 0.0f : pv;
#pragma unroll
        for (int i = 0; i < 15; ++i) s[i] = s[i + 1];
        const float other = __shfl_xor(pv, 32, 64);
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          const int key = key0 + 4 * k;
          const float w = k == hh ? pv : other;
          if (tk0 + key > qlim) continue;
#pragma unroll
          for (int dt = 0; dt < DT; ++dt) {
#pragma unroll
            for (int i = 0; i < 16; ++i) {
              const int d = dt * 32 + 8 * (i >> 2) + 4 * hh + (i & 3);
              o[dt][i] = fmaf(w, elem(cV + swv<D>(key, d >> 3) + (d & 7), kXBf16), o[dt][i]);
            }
          }
        }
      }
    }
  };

  // One pass over the key tiles in PV mode kMode.  Returns false (work-group
  // uniform) when kPvConvert produced a non-finite O (a V value that fp16
  // cannot hold, or non-finite data): the caller reruns in kPvSplit.
  auto run = [&](auto mode_tag) -> bool {
    constexpr int kMode = decltype(mode_tag)::value;
    constexpr bool kStage8 = kF8 && (kMode == kPvF8 || kMode == kPvScalar);  // FP8 codes through registers
    constexpr bool kDirectV = kMode != kPvConvert && !kStage8;
    constexpr bool kPvBf16 = kMode == kPvSplit || kXBf16;
    constexpr int kPP = kX ? (kXBf16 ? 3 : 2) : kMode == kPvSplit ? 2 : 1;  // pieces of the weights

#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
#pragma unroll
      for (int r = 0; r < 16; ++r) o[dt][r] = 0.0f;
    }
    m = -__builtin_inff();
    l = 0.0f;

    u32x4_t vreg[kDirectV || kStage8 ? 1 : CPT];
    u32x2_t kreg8[kStage8 ? CPT : 1], vreg8[kStage8 ? CPT : 1];  // FP8 codes of this thread's chunks
    uint32_t umask = 0;

    // Loads of a tile into (dK, dV) from its offset table: entries() reads
    // this thread's table entries, chunk(c) issues chunk c's K (and V unless
    // converted) loads straight to LDS.
    u64x2_t ent[CPT];
    auto entries = [&](const u64x2_t* tb) {
#pragma unroll
      for (int c = 0; c < CPT; ++c) ent[c] = tb[prow[c]];
      umask = 0;
    };
    auto chunk = [&](int c, uint16_t* dK, uint16_t* dV) {
      const uint32_t use = (uint32_t)ent[c][1] & 1u;
      umask |= use << c;
      const char* va = vbase + (ent[c][1] - use) + vsrc[c];
      if constexpr (kStage8) {
        kreg8[c] = *reinterpret_cast<const u32x2_t*>(kbase + ent[c][0] + ksrc[c]);
        vreg8[c] = *reinterpret_cast<const u32x2_t*>(va);
        return;
      }
      lds_dma16(kbase + ent[c][0] + ksrc[c], (lds_void_t*)(dK + (c * 4 + wave) * 512));
      if constexpr (kDirectV) {
        lds_dma16(va, (lds_void_t*)(dV + (c * 4 + wave) * 512));
      } else {
        vreg[c] = *reinterpret_cast<const u32x4_t*>(va);
      }
    };
    auto issue = [&](const u64x2_t* tb, uint16_t* dK, uint16_t* dV) {
      entries(tb);
#pragma unroll
      for (int c = 0; c < CPT; ++c) chunk(c, dK, dV);
      __builtin_amdgcn_sched_barrier(0);
    };
    // After a tile's loads are complete: zero V rows that were substituted
    // (their probabilities are 0, but substituted data may not be finite),
    // or convert the register-staged bf16 V to fp16 (exact for
    // 2^-17 <= |v| < 65504; smaller values round to fp16 subnormals).
    auto finish = [&](uint16_t* dK, uint16_t* dV) {
      if constexpr (kStage8) {
        // Codes -> 16-bit pairs (v_cvt_scalef32_pk_{f16,bf16}_fp8 at scale 1:
        // exact for every code), K in the Q.K^T type, V in fp16; V rows that were
        // substituted are zeroed (their codes may be NaN), K rows need not be
        // (their scores are masked).
#pragma unroll
        for (int c = 0; c < CPT; ++c) {
          uint32_t wk[4], wv[4];
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            if constexpr (kBf16) {
              wk[2 * j] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(kreg8[c][j], 1.0f, false));
              wk[2 * j + 1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(kreg8[c][j], 1.0f, true));
            } else {
              wk[2 * j] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(kreg8[c][j], 1.0f, false));
              wk[2 * j + 1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(kreg8[c][j], 1.0f, true));
            }
            wv[2 * j] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(vreg8[c][j], 1.0f, false));
            wv[2 * j + 1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(vreg8[c][j], 1.0f, true));
          }
          const bool used = (umask >> c) & 1u;
#pragma unroll
          for (int j = 0; j < 4; ++j) wv[j] = used ? wv[j] : 0u;
          const int at = ((c * 4 + wave) * 64 + lane) * 8;
          *reinterpret_cast<u32x4_t*>(dK + at) = u32x4_t{wk[0], wk[1], wk[2], wk[3]};
          *reinterpret_cast<u32x4_t*>(dV + at) = u32x4_t{wv[0], wv[1], wv[2], wv[3]};
        }
      } else if constexpr (kDirectV) {
        if (umask != (1u << CPT) - 1u) {
#pragma unroll
          for (int c = 0; c < CPT; ++c) {
            if (!((umask >> c) & 1u))
              *reinterpret_cast<u32x4_t*>(dV + ((c * 4 + wave) * 64 + lane) * 8) = u32x4_t{0u, 0u, 0u, 0u};
          }
        }
      } else {
        // Rows are substituted only at the end of the keys or on a bad block
        // id: the zeroing selects run only when some lane of the wave has one.
        const bool all_used = __builtin_amdgcn_ballot_w64(umask != (1u << CPT) - 1u) == 0;
#pragma unroll
        for (int c = 0; c < CPT; ++c) {
          u32x4_t w;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const uint32_t x = vreg[c][j];
            w[j] = pack2<false>(__builtin_bit_cast(float, x << 16), __builtin_bit_cast(float, x & 0xffff0000u));
          }
          if (!all_used) {
            asm volatile("");
            if (!((umask >> c) & 1u)) w = u32x4_t{0u, 0u, 0u, 0u};
          }
          *reinterpret_cast<u32x4_t*>(dV + ((c * 4 + wave) * 64 + lane) * 8) = w;
        }
      }
    };

    // S^T, softmax and O^T update for tile t from LDS (cK, cV).
    auto compute = [&](int t, const uint16_t* cK, const uint16_t* cV) {
      if constexpr (kMode == kPvScalar) {
        scalar_tile(t, cK, cV);
        return;
      }
      // Key-split mode: this wave's 32 keys are rows par*32 .. of the tile;
      // the swizzles depend on row bits below 32 only, so its m-tile is the
      // tile's shifted by par*32 rows.
      cK += par * 32 * D;
      cV += par * 32 * D;
      f32x16_t st[MTW];
#pragma unroll
      for (int mt = 0; mt < MTW; ++mt) {
#pragma unroll
        for (int r = 0; r < 16; ++r) st[mt][r] = 0.0f;
      }
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
        for (int mt = 0; mt < MTW; ++mt) {
          const u32x4_t a = *reinterpret_cast<const u32x4_t*>(cK + swk<D>(mt * 32 + n, 2 * ks + hh));
#pragma unroll
          for (int pc = kX ? kQP - 1 : 0; kX ? pc >= 0 : pc < kQP; pc += kX ? -1 : 1)  // (kX: small pieces first)
            st[mt] = mfma32<kBf16>(a, qf[pc][ks], st[mt]);
        }
      }
      // Keys of this lane: t*KB + mt*32 + 8*(r/4) + 4*hh + r%4.  Only tiles
      // that cross the wave's diagonal (or the end of the keys) are masked;
      // the empty asm keeps this a branch rather than selects on every tile.
      const int tk0 = t * KB + par * 32;
      if (tk0 + MTW * 32 > wave_kfull) {
        asm volatile("");
        const int thr = qlim - tk0 - 4 * hh;
#pragma unroll
        for (int mt = 0; mt < MTW; ++mt) {
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            if (mt * 32 + 8 * (r >> 2) + (r & 3) > thr) st[mt][r] = -__builtin_inff();
          }
        }
      }
      // Max over this lane half's keys of the column; the other half holds the
      // column's other keys.  The two halves share m, and m only has to move
      // when some half exceeds m + 2^8, so the cross-half max is formed only
      // on that (rare) branch.
      float mx = -__builtin_inff();
#pragma unroll
      for (int mt = 0; mt < MTW; ++mt) {
#pragma unroll
        for (int r = 0; r < 16; ++r) mx = fmaxf(mx, st[mt][r]);
      }
      const float mxh = mx * qscale;
      if (__builtin_amdgcn_ballot_w64(mxh > m + kLazyRescale) != 0) {
        asm volatile("");  // rare: keep the O^T rescale behind the branch
        const float mxs = fmaxf(mxh, __shfl_xor(mxh, 32, 64));
        const float mn = kX ? __builtin_ceilf(fmaxf(m, mxs)) : fmaxf(m, mxs);
        const float corr = mn == -__builtin_inff() ? 1.0f : fast_exp2(m - mn);
        m = mn;
        l *= corr;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) o[dt] *= corr;
      }
      float negm = m == -__builtin_inff() ? 0.0f : -m;
      if constexpr (kXBias != 0.0f) negm += kXBias;

      // Per 32-key m-tile: P^T operands of its two 16-key steps (accumulator
      // slots 8s .. 8s+7 of step s), then O^T += V^T . P^T.  V^T operand of
      // step (mt, s): lane l of 16-lane group g supplies row
      // mt*32 + 16s + 4*hh + (l%16)/4 (and +8), dims dt*32 + 16*(g%2) +
      // (l%4)*4 .. +4, and receives dim dt*32 + lane%32.
      const int li = lane & 15;
      const int trow = 4 * hh + (li >> 2);
      const int tcol = 16 * ((lane >> 4) & 1) + (li & 3) * 4;
#pragma unroll
      for (int mt = 0; mt < MTW; ++mt) {
        u32x4_t pb[kPP][2];
        float lt = 0.0f;  // kX: this m-tile's sum of weights
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          uint32_t w[kPP][4];
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            float p0 = fast_exp2(fmaf(st[mt][8 * s + 2 * j], qscale, negm));
            float p1 = fast_exp2(fmaf(st[mt][8 * s + 2 * j + 1], qscale, negm));
            if constexpr (kX) lt += p0 + p1;
            if constexpr (kPP == 2 && !kX) l += p0 + p1;
            w[0][j] = pack2<kPvBf16>(p0, p1);
#pragma unroll
            for (int pc = 1; pc < kPP; ++pc) {
              const float2_t r = unpack2<kPvBf16>(w[pc - 1][j]);
              p0 -= r[0];
              p1 -= r[1];
              w[pc][j] = pack2<kPvBf16>(p0, p1);
            }
            if constexpr (kPP == 1)
              l = __builtin_amdgcn_fdot2(__builtin_bit_cast(half2_t, w[0][j]), half2_t{1.0f16, 1.0f16}, l, false);
          }
#pragma unroll
          for (int pc = 0; pc < kPP; ++pc) pb[pc][s] = u32x4_t{w[pc][0], w[pc][1], w[pc][2], w[pc][3]};
        }
        if constexpr (kX) l += lt;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
          // kX: the m-tile's products are summed on their own and added to O
          // once, so O is rounded once per 32 keys (the output's error against
          // 64 bits at a 2048-token context: 3.4e-7 -> 2.5e-7, +5 % time).
          f32x16_t ot;
          if constexpr (kX) {
#pragma unroll
            for (int r = 0; r < 16; ++r) ot[r] = 0.0f;
          }
          f32x16_t& oa = kX ? ot : o[dt];
#pragma unroll
          for (int s = 0; s < 2; ++s) {
            const int r0 = mt * 32 + 16 * s + trow;
            const int col = dt * 32 + tcol;
            const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (lds_short4_t*)(cV + swv<D>(r0, col >> 3) + (col & 7)));
            const short4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (lds_short4_t*)(cV + swv<D>(r0 + 8, col >> 3) + (col & 7)));
            const uint64_t lo64 = __builtin_bit_cast(uint64_t, lo), hi64 = __builtin_bit_cast(uint64_t, hi);
            const u32x4_t a = u32x4_t{(uint32_t)lo64, (uint32_t)(lo64 >> 32), (uint32_t)hi64,
                                      (uint32_t)(hi64 >> 32)};
#pragma unroll
            for (int pc = kX ? kPP - 1 : 0; kX ? pc >= 0 : pc < kPP; pc += kX ? -1 : 1)
              oa = mfma32<kPvBf16>(a, pb[pc][s], oa);
          }
          if constexpr (kX) o[dt] += ot;
        }
      }
    };

    // Double-buffered tiles, unrolled by two so each LDS buffer (and offset
    // table) is a distinct object: tile t+1's loads and tile t+2's offset
    // table are produced while tile t is computed; one barrier per tile.
    stage((int)fastdiv((uint32_t)key0, p.bs_div));
    __syncthreads();
    build(0, s_off0);
    if (ntiles > 1) {
      ensure_window(1);
      build(1, s_off1);
    }
    __syncthreads();
    if (ntiles > 0) {
      issue(s_off0, sK0, sV0);
      __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this thread's loads are in LDS
      finish(sK0, sV0);
    }
    __syncthreads();
    for (int t = 0; t < ntiles; t += 2) {
      if (t + 2 < ntiles) ensure_window(t + 2);
      if (t + 2 < ntiles) build(t + 2, s_off0);
      const bool more1 = t + 1 < ntiles;
      if (more1) issue(s_off1, sK1, sV1);
      if (t * KB + par * 32 < wave_kend) compute(t, sK0, sV0);
      if (more1) {
        __builtin_amdgcn_s_waitcnt(0x0F70);
        finish(sK1, sV1);
      }
      __syncthreads();
      if (!more1) break;
      if (t + 3 < ntiles) ensure_window(t + 3);
      if (t + 3 < ntiles) build(t + 3, s_off1);
      const bool more2 = t + 2 < ntiles;
      if (more2) issue(s_off0, sK0, sV0);
      if ((t + 1) * KB + par * 32 < wave_kend) compute(t + 1, sK1, sV1);
      if (t + 2 < ntiles) {
        __builtin_amdgcn_s_waitcnt(0x0F70);
        finish(sK0, sV0);
      }
      __syncthreads();
    }
    if constexpr (kMode == kPvConvert || (kX && kMode != kPvScalar)) {
      bool bad = kX && !__builtin_isfinite(l);
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
#pragma unroll
        for (int r = 0; r < 16; ++r) bad |= !__builtin_isfinite(o[dt][r]);
      }
      if (bad) s_ovf = 1;
      __syncthreads();
      if (s_ovf) return false;
    }
    return true;
  };

  if constexpr (kX) {
    if (!run(PvTag<kF8 ? kPvF8 : kPvDirect>{})) {
      badkey = 0x7fffffff;
      run(PvTag<kPvScalar>{});
    }
  } else if constexpr (kF8) {
    run(PvTag<kPvF8>{});
  } else if constexpr (kBf16) {
    if (!run(PvTag<kPvConvert>{})) {
      badkey = 0x7fffffff;
      run(PvTag<kPvSplit>{});
    }
  } else {
    run(PvTag<kPvDirect>{});
  }

  if (badkey != 0x7fffffff) atomicMin(&s_badkey, badkey);
  __syncthreads();
  const int bad_from = s_badkey;

  // Key-split mode: waves 2-3 hand their (m, l, O^T) to waves 0-1 through
  // the (now idle) tile buffers; the lanes of the two waves hold the same
  // rows and dims, so the merge is lane by lane (log-sum-exp rule on the
  // reference points m, which are -inf where a wave saw no key).
  if constexpr (kSplit) {
    float* xo = reinterpret_cast<float*>(rw == 0 ? sK0 : sK1);  // [DT * 16][64]: KB * D halves hold it
    float* xm = reinterpret_cast<float*>(sV0) + rw * 128;       // m [64], l [64]
    if (par == 1) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
#pragma unroll
        for (int r = 0; r < 16; ++r) xo[(dt * 16 + r) * 64 + lane] = o[dt][r];
      }
      xm[lane] = m;
      xm[64 + lane] = l;
    }
    __syncthreads();
    if (par == 1) return;
    const float m2 = xm[lane], l2 = xm[64 + lane];
    const float mn = fmaxf(m, m2);
    const float a = m == -__builtin_inff() ? 0.0f : fast_exp2(m - mn);
    const float c = m2 == -__builtin_inff() ? 0.0f : fast_exp2(m2 - mn);
    l = l * a + l2 * c;
    m = mn;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
#pragma unroll
      for (int r = 0; r < 16; ++r) o[dt][r] = o[dt][r] * a + xo[(dt * 16 + r) * 64 + lane] * c;
    }
  }

  // Row sum over the two lane halves, normalise, write.  O^T slot r of lane
  // (n, hh) in m-tile dt is dim dt*32 + 8*(r/4) + 4*hh + r%4 of row qrow.
  const float lt = l + __shfl_xor(l, 32, 64);
  if (!live) return;
  // The row's position and offset again from its number, behind an empty asm:
  // kept across the tile loop they cost it registers.
  int qrow_e = qrow;
  asm volatile("" : "+v"(qrow_e));
  const int qpos_e = ctx - S + chunk_row(qrow_e);
  const int64_t row_at = row_offset(qrow_e);
  const bool bad = bad_from <= qpos_e;
  if (kPart && !whole) {  // this partition's sums (a row with an unreadable key: NaN)
    const int64_t e = (unit * p.parts + part) * QB + rw * QW + n;
    if (hh == 0) {
      p.ws_m[e] = m;
      p.ws_l[e] = bad ? __builtin_nanf("") : lt;
    }
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        *reinterpret_cast<float4_t*>(p.ws_acc + e * D + dt * 32 + 8 * j + 4 * hh) =
            float4_t{o[dt][4 * j], o[dt][4 * j + 1], o[dt][4 * j + 2], o[dt][4 * j + 3]};
    }
    return;
  }
  // (kX: a row whose weights are all 0, every score -Inf, is 0 / 0.)
  const float inv = lt > 0.0f || (kX && qpos_e >= 0) ? p.vscale / lt : 0.0f;
  // Slots 4j .. 4j+3 of m-tile dt are 4 consecutive dims: one 8-byte (16-bit
  // out) or 16-byte (fp32 out) store when the output base allows it.
  const uintptr_t oa = reinterpret_cast<uintptr_t>(p.out);
  const bool vec = (p.out_dtype == kF32 ? (oa & 15) == 0 : (oa & 7) == 0);
  if (!vec) {
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int d = dt * 32 + 8 * (r >> 2) + 4 * hh + (r & 3);
        store_elem(p.out, p.out_dtype, row_at + d, bad ? __builtin_nanf("") : o[dt][r] * inv);
      }
    }
    return;
  }
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = bad ? __builtin_nanf("") : o[dt][4 * j + i] * inv;
      const int64_t e = row_at + dt * 32 + 8 * j + 4 * hh;
      if (p.out_dtype == kF32) {
        u64x2_t w = u64x2_t{(uint64_t)__builtin_bit_cast(uint32_t, v[0]) | ((uint64_t)__builtin_bit_cast(uint32_t, v[1]) << 32),
                            (uint64_t)__builtin_bit_cast(uint32_t, v[2]) | ((uint64_t)__builtin_bit_cast(uint32_t, v[3]) << 32)};
        *reinterpret_cast<u64x2_t*>(static_cast<float*>(p.out) + e) = w;
      } else {
        const uint32_t w0 = p.out_dtype == kF16 ? pack2<false>(v[0], v[1]) : pack2<true>(v[0], v[1]);
        const uint32_t w1 = p.out_dtype == kF16 ? pack2<false>(v[2], v[3]) : pack2<true>(v[2], v[3]);
        const uint64_t w = (uint64_t)w0 | ((uint64_t)w1 << 32);
        *reinterpret_cast<uint64_t*>(static_cast<uint16_t*>(p.out) + e) = w;
      }
    }
  }
}

template <typename KV, int D, bool kSplitQ, bool kSplit>
__global__ __launch_bounds__(kPfThreads) __attribute__((amdgpu_waves_per_eu(PfShape<D>::WAVES_PER_EU)))
void prefill_mfma_kernel(const PrefillParams p) {
  prefill_body<KV, D, kSplitQ ? 2 : 1, kSplit, false, false>(p);
}

// The fp32-precision kernel (kX above).
template <typename KV, int D, int kQP, bool kSplit>
__global__ __launch_bounds__(kPfThreads) __attribute__((amdgpu_waves_per_eu(PfShape<D>::WAVES_PER_EU)))
void prefill32_kernel(const PrefillParams p) {
  prefill_body<KV, D, kQP, kSplit, true, false>(p);
}

// One partition of a context split.
template <typename KV, int D, bool kSplitQ, bool kSplit>
__global__ __launch_bounds__(kPfThreads) __attribute__((amdgpu_waves_per_eu(PfShape<D>::WAVES_PER_EU)))
void split_prefill_mfma_kernel(const PrefillParams p) {
  prefill_body<KV, D, kSplitQ ? 2 : 1, kSplit, false, true>(p);
}

template <typename KV, int D, int kQP, bool kSplit>
__global__ __launch_bounds__(kPfThreads) __attribute__((amdgpu_waves_per_eu(PfShape<D>::WAVES_PER_EU)))
void split_prefill32_kernel(const PrefillParams p) {
  prefill_body<KV, D, kQP, kSplit, true, true>(p);
}

// Merge of a context split's partitions (log-sum-exp rule, as the decode
// split's): one thread per 4 dims of a row, the unit's rows in blocks along
// grid y.  Partition states and sums are a few MB: eight partitions' rows are
// in flight per thread, since the loads' latency is what it takes.
template <int D>
struct PfReduce {
  static constexpr int QB = D <= 128 ? 64 : 128;  // rows per unit of a split grid
  static constexpr int ROWS = kPfThreads / (D / 4);
};

template <int D, bool kX>
__global__ __launch_bounds__(kPfThreads) void prefill_reduce_kernel(const PrefillParams p) {
  constexpr int QB = PfReduce<D>::QB, KB = PfShape<D>::KB;
  int part, qt, hg, b, S, served;
  int64_t unit, tok0;
  if (!pf_unit<QB, true>(p, blockIdx.x, threadIdx.x & 63, part, unit, qt, hg, b) || part > 0) return;
  if (!pf_rows(p, b, S, tok0, served)) return;
  const int Sr = served * p.gp, qs0 = qt * QB;
  const int r = blockIdx.y * PfReduce<D>::ROWS + threadIdx.x / (D / 4), d = threadIdx.x % (D / 4) * 4;
  const int ctx = p.context_lens[b];
  if (qs0 + r >= Sr || ctx > p.MB * p.BS) return;
  auto chunk_row = [&](int x) { return (int)fastdiv((uint32_t)x, p.gp_div); };
  const int kend = min(ctx, ctx - S + chunk_row(min(qs0 + QB, Sr) - 1) + 1);
  const int n = kend > 0 ? ((kend + KB - 1) / KB + p.part_tiles - 1) / p.part_tiles : 0;
  if (n <= 1) return;  // the unit's one partition wrote its rows
  const int64_t e0 = unit * p.parts * QB + r;
  float M = -__builtin_inff(), L = 0.0f;
  float4_t acc = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
  constexpr int NL = 8;
  for (int j0 = 0; j0 < n; j0 += NL) {
    float mj[NL], lj[NL];
    float4_t x[NL];
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int64_t e = e0 + (int64_t)min(j0 + i, n - 1) * QB;
      mj[i] = p.ws_m[e];
      lj[i] = p.ws_l[e];
      x[i] = *reinterpret_cast<const float4_t*>(p.ws_acc + e * D + d);
    }
    float mn = M;
#pragma unroll
    for (int i = 0; i < NL; ++i) mn = fmaxf(mn, mj[i]);
    const float ref = mn == -__builtin_inff() ? 0.0f : mn;  // (no key so far: every weight is 0)
    const float corr = fast_exp2(M - ref);
    M = mn;
    L *= corr;
    acc *= corr;
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const float w = fast_exp2(mj[i] - ref);
      if (j0 + i < n) {
        L += w * lj[i];
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[c] = fmaf(w, x[i][c], acc[c]);
      }
    }
  }
  const int row = qs0 + r, sr = chunk_row(row), qpos = ctx - S + sr;
  const float inv = L > 0.0f || L != L || (kX && qpos >= 0) ? p.vscale / L : 0.0f;
  const int64_t at = ((tok0 + sr) * p.H + hg * p.gp + row - sr * p.gp) * D + d;
#pragma unroll
  for (int c = 0; c < 4; ++c) store_elem(p.out, p.out_dtype, at + c, acc[c] * inv);
}

// Ping-pong prefill (64-key tiles; 16-bit caches with q in the KV type, or
// FP8 caches with fp16 or bf16 q, the codes staged in registers).  A
// work-group of 8 waves serves 256 query rows (wave w owns rows 32w ..) and
// is the only one on its CU, so each SIMD holds wave s of group 0 (waves 0-3)
// and wave s + 4 of group 1.  Every phase ends at a work-group barrier, and
// group 1 runs one phase behind group 0: in each phase one group does its
// matrix step (O^T += V^T . P^T of tile j - 1, then S^T = K . Q^T of tile j)
// while the other does its vector step (the softmax of its S^T of tile j),
// so each SIMD issues one wave's MFMAs against the other wave's vector work.
// In the four-wave kernel the two waves of a SIMD belong to different
// work-groups, drift into the same step and queue behind each other.
//
// Phase ph, group g: step e = ph - g; even e = matrix step e / 2, odd e =
// vector step e / 2.  Tile j's K is read in phases 2j (group 0) and 2j + 1
// (group 1), its V (by the P.V of step j + 1) in 2j + 2 and 2j + 3.  Loads
// (at D >= 64 every thread of both groups loads its share of every K and V
// tile, so the two groups' vector steps carry the same work; at D = 32, one
// 16-byte chunk per thread of a group, group 1 loads K and group 0 V):
//  * in its vector step j (phase 2j + 1 + g) a thread issues its chunks of K
//    of tile j + 2 and of V of tile j + 1: direct to LDS, except a bf16 V
//    tile and FP8 codes, which go to registers -- both buffers were last
//    read in phase 2j - 1;
//  * at the end of its matrix step j + 1 (phase 2j + 2 + g) it waits for
//    them and finishes them (bf16 V converted to fp16, FP8 K and V codes to
//    16-bit pairs, and stored; substituted V rows zeroed), before the
//    barrier ahead of their first read (phase 2j + 4).
// Per-row offset tables (three, tile t in t % 3) are built by wave 0 in its
// vector step j for tile j + 3.
template <int N>
struct Slot {  // a compile-time buffer index
  static constexpr int value = N;
};

constexpr int kPpThreads = 512;  // 8 waves
constexpr int kPpRows = 256;     // query rows per work-group

template <typename KV, int D>
__global__ __launch_bounds__(kPpThreads) __attribute__((amdgpu_waves_per_eu(2)))
void prefill_pp_kernel(const PrefillParams p) {
  using Sh = PfShape<D>;
  static_assert(Sh::KB == 64 && Sh::MT == 2, "64-key tiles");
  constexpr int QW = 32, QB = kPpRows, KB = 64, MT = 2, KS = Sh::KS, DT = Sh::DT, NCH = Sh::NCH;
  constexpr int CPT = Sh::CPT;  // chunks per thread of one group (256 threads) per tile
  constexpr bool kBf16 = QkBf16<KV>::value;  // Q.K^T operand type
  constexpr bool kF8 = KV::kCode == kFP8;    // tiles converted from FP8 codes; P.V in fp16
  constexpr int EB = KV::kBytes;
  static_assert(EB == 2 || kF8, "16-bit or FP8 caches");

  __shared__ __attribute__((aligned(16))) uint16_t sK[3][KB * D];
  __shared__ __attribute__((aligned(16))) uint16_t sV[3][KB * D];
  __shared__ int32_t s_bt[kPfBtStage];
  __shared__ u64x2_t s_off[3][KB];
  __shared__ int s_badkey;
  __shared__ int s_ovf;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int grp = wave >> 2;
  const int n = lane & 31;
  const int hh = lane >> 5;

  // Work-group -> unit (b, h, query block), as the four-wave kernel; also compacted:
  // a work-group without rows held a CU to exit, and with packed heads the few with
  // rows came singly between them (fp16, 64/8 heads of 128, 16 decode rows and one
  // prompt of 2048 at 4096: unpacked 248 us, packed 297, compacted 235).
  int part, qt, hg, b;
  int64_t unit;
  if (!pf_unit<QB, false>(p, blockIdx.x, lane, part, unit, qt, hg, b)) return;
  const int h0 = hg * p.gp;  // first query head of the unit
  const int kvh = h0 / p.G;

  int S, served;
  int64_t tok0;
  if (!pf_rows(p, b, S, tok0, served)) return;
  const int Sr = served * p.gp;  // packed rows served
  const int qs0 = qt * QB;
  if (qs0 >= Sr) return;
  const int qw0 = qs0 + wave * QW;
  const int qrow = qw0 + n;
  const bool live = qrow < Sr;
  // Packed row -> chunk row and head; the row's offset in q and out.
  auto chunk_row = [&](int r) { return (int)fastdiv((uint32_t)r, p.gp_div); };
  const int srow = chunk_row(qrow);
  auto row_offset = [&](int r) {
    const int sr = chunk_row(r);
    return ((tok0 + sr) * p.H + h0 + (r - sr * p.gp)) * D;
  };

  // Issued before the context length arrives: the block table's first
  // min(MB, kPfBtStage) entries (the window; the host serves only tables that
  // fit it) and this lane's q.
  const int32_t* bt_row = p.block_tables + (int64_t)b * p.bt_stride;
  const int nbt = min(p.MB, kPfBtStage);
  static_assert(kPfBtStage == 2 * kPpThreads, "two entries per thread");
  int32_t btp0 = 0, btp1 = 0;
  if ((int)threadIdx.x < nbt) btp0 = bt_row[threadIdx.x];
  if ((int)threadIdx.x + kPpThreads < nbt) btp1 = bt_row[threadIdx.x + kPpThreads];
  u32x4_t qf[KS];
  {
    const int64_t qoff = row_offset(live ? qrow : 0) + hh * 8;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      u32x4_t r = u32x4_t{0u, 0u, 0u, 0u};
      if (live) r = *reinterpret_cast<const u32x4_t*>(static_cast<const uint16_t*>(p.q) + qoff + ks * 16);
      qf[ks] = (r & p.q_and) ^ p.q_xor;
    }
  }
  const int ctx = p.context_lens[b];
  const int maxctx = p.MB * p.BS;

  if (ctx > maxctx) {
    if (live && hh == 0) {
      const float fillv = ctx - S + srow < 0 ? 0.0f : __builtin_nanf("");
      const int64_t row_at = row_offset(qrow);
      for (int d = 0; d < D; ++d) store_elem(p.out, p.out_dtype, row_at + d, fillv);
    }
    return;
  }
  if (threadIdx.x == 0) {
    s_badkey = 0x7fffffff;
    s_ovf = 0;
  }

  const int kend = min(ctx, ctx - S + chunk_row(min(qs0 + QB, Sr) - 1) + 1);
  const int ntiles = kend > 0 ? (kend + KB - 1) / KB : 0;
  const int wave_last = min(qw0 + QW - 1, Sr - 1);
  const int wave_kend = qw0 < Sr ? min(ctx, ctx - S + chunk_row(wave_last) + 1) : 0;
  const int wave_kfull = ctx - S + chunk_row(qw0) + 1;
  const int qpos = ctx - S + srow;
  const int qlim = min(qpos, kend - 1);

  const float qscale = p.qscale;

  // The block ids of every page the work-group reads.
  const int npages = kend > 0 ? min((int)fastdiv((uint32_t)(kend - 1), p.bs_div) + 1, nbt) : 0;
  if ((int)threadIdx.x < npages) s_bt[threadIdx.x] = btp0;
  if ((int)threadIdx.x + kPpThreads < npages) s_bt[threadIdx.x + kPpThreads] = btp1;

  const char* kbase = static_cast<const char*>(p.k) + (int64_t)kvh * p.k_sh * EB;
  const char* vbase = static_cast<const char*>(p.v) + (int64_t)kvh * p.v_sh * EB;
  const uint32_t k_sbb = (uint32_t)(p.k_sb * EB), k_stb = (uint32_t)(p.k_st * EB);
  const uint32_t v_sbb = (uint32_t)(p.v_sb * EB), v_stb = (uint32_t)(p.v_st * EB);
  const uint64_t nb = (uint64_t)p.num_blocks;

  // This thread's chunks of a tile.  With two or more chunks per thread of a
  // group (D >= 64), both groups load half of every K tile and half of every
  // V tile (CH chunks of each per thread), so the two groups' vector steps
  // carry the same work; at D = 32 (one chunk) group 1 loads K, group 0 V.
  constexpr bool kHalves = CPT % 2 == 0;
  constexpr int CH = kHalves ? CPT / 2 : CPT;
  auto cpos = [&](int c) { return kHalves ? c * 8 + wave : c * 4 + (wave & 3); };  // 64-chunk group of chunk c
  const bool do_k = kHalves || grp == 1, do_v = kHalves || grp == 0;  // wave-uniform
  int prow[CH], ksrc[CH], vsrc[CH];
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    const int pos = cpos(c) * 64 + lane;
    prow[c] = pos / NCH;
    ksrc[c] = kpos<D>(prow[c], pos % NCH) * 8 * EB;
    vsrc[c] = vpos<D>(prow[c], pos % NCH) * 8 * EB;
  }
  int badkey = 0x7fffffff;

  // Wave 0: the offset table of tile t (entry r = {K byte offset, V byte
  // offset | use}; a row past kend or on an invalid block id reads row 0 of
  // block 0 with use = 0).
  auto build = [&](auto slot, int t) {
    const int row = lane;
    const int kabs = t * KB + row;
    const bool valid = kabs < kend;
    const int kk = valid ? kabs : 0;
    const int pg = (int)fastdiv((uint32_t)kk, p.bs_div);
    const int off = kk - pg * p.BS;
    const int blk = s_bt[valid ? pg : 0];
    const bool okb = (uint64_t)(int64_t)blk < nb;
    if (valid && !okb) badkey = min(badkey, kabs);
    const bool use = valid && okb;
    const uint32_t ub = use ? (uint32_t)blk : 0u, uo = use ? (uint32_t)off : 0u;
    s_off[decltype(slot)::value][row] = u64x2_t{(uint64_t)ub * k_sbb + uo * k_stb,
                                ((uint64_t)ub * v_sbb + uo * v_stb) | (use ? 1u : 0u)};
  };

  f32x16_t o[DT];
  float m = -__builtin_inff(), l = 0.0f;

  auto run = [&](auto mode_tag) -> bool {
    constexpr int kMode = decltype(mode_tag)::value;
    constexpr bool kDirectV = kMode != kPvConvert && kMode != kPvF8;
    constexpr bool kPvBf16 = kMode == kPvSplit;

#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
#pragma unroll
      for (int r = 0; r < 16; ++r) o[dt][r] = 0.0f;
    }
    m = -__builtin_inff();
    l = 0.0f;

    u32x4_t vreg[kDirectV || kF8 ? 1 : CH];
    u32x2_t kreg8[kF8 ? CH : 1], vreg8[kF8 ? CH : 1];  // FP8 codes of this thread's chunks
    uint32_t umask = 0;

    // This thread's K chunks of tile t: straight to LDS, or (FP8) codes into
    // registers `kr`.
    auto issue_k = [&](auto slot, u32x2_t (&kr)[kF8 ? CH : 1]) {
      if (!do_k) return;
      const u64x2_t* tb = s_off[decltype(slot)::value];
      uint16_t* dK = sK[decltype(slot)::value];
      uint64_t e[CH];  // the K halves of the table entries first: one LDS round trip
#pragma unroll
      for (int c = 0; c < CH; ++c) e[c] = reinterpret_cast<const uint64_t*>(tb + prow[c])[0];
#pragma unroll
      for (int c = 0; c < CH; ++c) {
        if constexpr (kF8) {
          kr[c] = *reinterpret_cast<const u32x2_t*>(kbase + e[c] + ksrc[c]);
        } else {
          lds_dma16_async(kbase + e[c] + ksrc[c], (lds_void_t*)(dK + cpos(c) * 512));
        }
      }
    };
    // FP8, after this thread's K loads of tile t are complete: codes -> Q.K^T
    // type pairs (exact for every code; rows past the keys need no zeroing:
    // their scores are masked).
    auto finish_k = [&](auto slot, const u32x2_t (&kr)[kF8 ? CH : 1]) {
      if constexpr (kF8) {
        if (!do_k) return;
        uint16_t* dK = sK[decltype(slot)::value];
#pragma unroll
        for (int c = 0; c < CH; ++c) {
          uint32_t w[4];
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            if constexpr (kBf16) {
              w[2 * j] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(kr[c][j], 1.0f, false));
              w[2 * j + 1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(kr[c][j], 1.0f, true));
            } else {
              w[2 * j] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(kr[c][j], 1.0f, false));
              w[2 * j + 1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(kr[c][j], 1.0f, true));
            }
          }
          *reinterpret_cast<u32x4_t*>(dK + (cpos(c) * 64 + lane) * 8) = u32x4_t{w[0], w[1], w[2], w[3]};
        }
      }
    };
    // This thread's V chunks of tile t (to LDS, or to registers for conversion).
    auto issue_v = [&](auto slot) {
      if (!do_v) return;
      const u64x2_t* tb = s_off[decltype(slot)::value];
      uint16_t* dV = sV[decltype(slot)::value];
      umask = 0;
      uint64_t e[CH];  // the V halves of the table entries first: one LDS round trip
#pragma unroll
      for (int c = 0; c < CH; ++c) e[c] = reinterpret_cast<const uint64_t*>(tb + prow[c])[1];
#pragma unroll
      for (int c = 0; c < CH; ++c) {
        const uint32_t use = (uint32_t)e[c] & 1u;
        umask |= use << c;
        const char* va = vbase + (e[c] - use) + vsrc[c];
        if constexpr (kF8) {
          vreg8[c] = *reinterpret_cast<const u32x2_t*>(va);
        } else if constexpr (kDirectV) {
          lds_dma16_async(va, (lds_void_t*)(dV + cpos(c) * 512));
        } else {
          vreg[c] = *reinterpret_cast<const u32x4_t*>(va);
        }
      }
    };
    // After this thread's V loads are complete: zero substituted rows, or
    // convert the staged bf16 V to fp16 (exact for 2^-17 <= |v| < 65504), or
    // the FP8 codes to fp16 (exact; substituted rows zeroed: their codes may
    // be NaN).
    auto finish_v = [&](auto slot) {
      if (!do_v) return;
      uint16_t* dV = sV[decltype(slot)::value];
      if constexpr (kF8) {
#pragma unroll
        for (int c = 0; c < CH; ++c) {
          uint32_t w[4];
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            w[2 * j] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(vreg8[c][j], 1.0f, false));
            w[2 * j + 1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(vreg8[c][j], 1.0f, true));
          }
          const bool used = (umask >> c) & 1u;
#pragma unroll
          for (int j = 0; j < 4; ++j) w[j] = used ? w[j] : 0u;
          *reinterpret_cast<u32x4_t*>(dV + (cpos(c) * 64 + lane) * 8) = u32x4_t{w[0], w[1], w[2], w[3]};
        }
      } else if constexpr (kDirectV) {
        __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the direct loads are not tracked by the compiler
        if (umask != (1u << CH) - 1u) {
#pragma unroll
          for (int c = 0; c < CH; ++c) {
            if (!((umask >> c) & 1u))
              *reinterpret_cast<u32x4_t*>(dV + (cpos(c) * 64 + lane) * 8) = u32x4_t{0u, 0u, 0u, 0u};
          }
        }
      } else {
        const bool all_used = __builtin_amdgcn_ballot_w64(umask != (1u << CH) - 1u) == 0;
#pragma unroll
        for (int c = 0; c < CH; ++c) {
          u32x4_t w;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const uint32_t xv = vreg[c][j];
            w[j] = pack2<false>(__builtin_bit_cast(float, xv << 16), __builtin_bit_cast(float, xv & 0xffff0000u));
          }
          if (!all_used) {
            asm volatile("");
            if (!((umask >> c) & 1u)) w = u32x4_t{0u, 0u, 0u, 0u};
          }
          *reinterpret_cast<u32x4_t*>(dV + (cpos(c) * 64 + lane) * 8) = w;
        }
      }
    };

    f32x16_t st[MT];
    u32x4_t pb[MT][2], pb_lo[kPvBf16 ? MT : 1][2];
    // Softmax of tile t: mask, lazy maximum, P^T operands (see the four-wave kernel).
    auto softmax = [&](int t) {
      const int tk0 = t * KB;
      if (tk0 + KB > wave_kfull) {
        asm volatile("");
        const int thr = qlim - tk0 - 4 * hh;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            if (mt * 32 + 8 * (r >> 2) + (r & 3) > thr) st[mt][r] = -__builtin_inff();
          }
        }
      }
      // Weights against the running maximum m, packed as the P^T operands,
      // and their row sum over the rounded weights (four chains, added at the
      // end): each lane's sum over its 16 keys of the row.
      auto weights = [&](float negm) __attribute__((always_inline)) {
        float ls[MT][2];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
          for (int s2 = 0; s2 < 2; ++s2) {
            uint32_t w[4], wl[4];
            float lc = 0.0f;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              const float p0 = fast_exp2(fmaf(st[mt][8 * s2 + 2 * j], qscale, negm));
              const float p1 = fast_exp2(fmaf(st[mt][8 * s2 + 2 * j + 1], qscale, negm));
              w[j] = pack2<kPvBf16>(p0, p1);
              if constexpr (kPvBf16) {
                const float2_t r = unpack2<true>(w[j]);
                wl[j] = pack2<true>(p0 - r[0], p1 - r[1]);
                lc += p0 + p1;
              } else {
                lc = __builtin_amdgcn_fdot2(__builtin_bit_cast(half2_t, w[j]), half2_t{1.0f16, 1.0f16}, lc, false);
              }
            }
            ls[mt][s2] = lc;
            pb[mt][s2] = u32x4_t{w[0], w[1], w[2], w[3]};
            if constexpr (kPvBf16) pb_lo[mt][s2] = u32x4_t{wl[0], wl[1], wl[2], wl[3]};
          }
        }
        return (ls[0][0] + ls[0][1]) + (ls[1][0] + ls[1][1]);
      };
      // The maximum is raised only when needed: on the first tile (every
      // live row sees key 0), or when a lane's weights could leave the range
      // they are exact in (a sum above 2^15, or not finite: a weight past
      // 2^15).  The tile maximum is computed only then.
      float lsum = weights(m == -__builtin_inff() ? 0.0f : -m);
      if (__builtin_amdgcn_ballot_w64(t == 0 || !(lsum <= kWeightCap)) != 0) {
        asm volatile("");
        // Maximum over four independent chains (short dependency chains).
        float mc[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          mc[c] = st[c >> 1][(c & 1) * 8];
#pragma unroll
          for (int r = 1; r < 8; ++r) mc[c] = fmaxf(mc[c], st[c >> 1][(c & 1) * 8 + r]);
        }
        const float mxh = fmaxf(fmaxf(mc[0], mc[1]), fmaxf(mc[2], mc[3])) * qscale;
        const float mxs = fmaxf(mxh, __shfl_xor(mxh, 32, 64));
        const float mn = fmaxf(m, mxs);
        const float corr = mn == -__builtin_inff() ? 1.0f : fast_exp2(m - mn);
        m = mn;
        l *= corr;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) o[dt] *= corr;
        lsum = weights(m == -__builtin_inff() ? 0.0f : -m);
      }
      l += lsum;
    };
    // Matrix step: O^T += V^T . P^T of tile j - 1 (V in slot SV), then
    // S^T = K . Q^T of tile j (K in slot SK).  Each LDS operand is read two
    // MFMAs ahead into a ring of three, in this order (fences keep the
    // scheduler from regrouping the reads next to their uses), and the first
    // two K operands are read before the P.V products.
    const int li = lane & 15;
    const int trow = 4 * hh + (li >> 2);
    const int tcol = 16 * ((lane >> 4) & 1) + (li & 3) * 4;
    auto mstep = [&](auto sk, auto sv, bool do_pv, bool do_qk) {
      const uint16_t* cK = sK[decltype(sk)::value];
      const uint16_t* cV = sV[decltype(sv)::value];
      u32x4_t ka[3][MT];
      auto rdk = [&](int ks, u32x4_t (&dst)[MT]) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          dst[mt] = *reinterpret_cast<const u32x4_t*>(cK + swk<D>(mt * 32 + n, 2 * ks + hh));
      };
      if (do_qk) {
        rdk(0, ka[0]);
        rdk(1, ka[1]);
      }
      if (do_pv) {
        // Product i: m-tile mt = i / (2 DT), step s2 = (i / DT) % 2, dims dt = i % DT.
        constexpr int NP = MT * 2 * DT;
        u32x4_t va[3];
        auto rdv = [&](int i, u32x4_t& dst) {
          const int mt = i / (2 * DT), s2 = (i / DT) % 2, dt = i % DT;
          const int r0 = mt * 32 + 16 * s2 + trow;
          const int col = dt * 32 + tcol;
          const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (lds_short4_t*)(cV + swv<D>(r0, col >> 3) + (col & 7)));
          const short4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (lds_short4_t*)(cV + swv<D>(r0 + 8, col >> 3) + (col & 7)));
          const uint64_t lo64 = __builtin_bit_cast(uint64_t, lo), hi64 = __builtin_bit_cast(uint64_t, hi);
          dst = u32x4_t{(uint32_t)lo64, (uint32_t)(lo64 >> 32), (uint32_t)hi64, (uint32_t)(hi64 >> 32)};
        };
        rdv(0, va[0]);
        rdv(1, va[1]);
#pragma unroll
        for (int i = 0; i < NP; ++i) {
          if (i + 2 < NP) rdv(i + 2, va[(i + 2) % 3]);
          __builtin_amdgcn_sched_barrier(0);
          const int mt = i / (2 * DT), s2 = (i / DT) % 2, dt = i % DT;
          o[dt] = mfma32<kPvBf16>(va[i % 3], pb[mt][s2], o[dt]);
          if constexpr (kPvBf16) o[dt] = mfma32<true>(va[i % 3], pb_lo[mt][s2], o[dt]);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      if (do_qk) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
          for (int r = 0; r < 16; ++r) st[mt][r] = 0.0f;
        }
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          if (ks + 2 < KS) rdk(ks + 2, ka[(ks + 2) % 3]);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) st[mt] = mfma32<kBf16>(ka[ks % 3][mt], qf[ks], st[mt]);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    };

    // Prologue: tables 0-2, K of tiles 0 and 1, V of tile 0.
    __syncthreads();
    if (wave == 0) {
      if (ntiles > 0) build(Slot<0>{}, 0);
      if (ntiles > 1) build(Slot<1>{}, 1);
      if (ntiles > 2) build(Slot<2>{}, 2);
    }
    __syncthreads();
    if (ntiles > 0) {
      u32x2_t kreg8b[kF8 ? CH : 1];
      issue_k(Slot<0>{}, kreg8);
      if (ntiles > 1) issue_k(Slot<1>{}, kreg8b);
      issue_v(Slot<0>{});
      finish_k(Slot<0>{}, kreg8);
      if (ntiles > 1) finish_k(Slot<1>{}, kreg8b);
      finish_v(Slot<0>{});
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
    __syncthreads();

    // Step j (buffer slot j % 3, a compile-time index: every LDS address is a
    // loop-invariant lane offset plus an immediate).  Every wave runs the
    // same steps; group 1 passes one barrier first, so its k-th barrier of
    // the loop meets group 0's (k + 1)-th: one phase behind.  Loads for a
    // later tile start at the top of a vector step and are finished at the
    // end of the next matrix step, two phases later.
    auto step = [&](auto slot, int j) {
      constexpr int B0 = decltype(slot)::value;  // tile j
      constexpr int B1 = (B0 + 1) % 3;           // tile j + 1
      constexpr int B2 = (B0 + 2) % 3;           // tiles j + 2 and j - 1
      // Matrix step j.
      // The matrix step issues at a raised wave priority: a SIMD otherwise
      // issues the older wave (group 0) first, so group 1's MFMAs queued
      // behind group 0's vector work (config 4b +0.7 %, FP8 +0.4 %).
      __builtin_amdgcn_s_setprio(1);
      mstep(Slot<B0>{}, Slot<B2>{}, j >= 1 && (j - 1) * KB < wave_kend, j < ntiles && j * KB < wave_kend);
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_setprio(0);
      // This thread's loads of vector step j - 1: V of tile j and K of tile j + 1.
      __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the direct loads are not tracked by the compiler
      if (j >= 1 && j + 1 < ntiles) finish_k(Slot<B1>{}, kreg8);
      if (j >= 1 && j < ntiles) finish_v(Slot<B0>{});
      __syncthreads();
      // Vector step j.
      if (j + 1 < ntiles) issue_v(Slot<B1>{});
      if (j + 2 < ntiles) issue_k(Slot<B2>{}, kreg8);
      if (j < ntiles && j * KB < wave_kend) softmax(j);
      if (wave == 0 && j + 3 < ntiles) build(Slot<B0>{}, j + 3);
      __syncthreads();
    };
    if (grp == 1) __syncthreads();
    for (int j = 0; j <= ntiles; j += 3) {  // work-group uniform exits
      step(Slot<0>{}, j);
      if (j + 1 > ntiles) break;
      step(Slot<1>{}, j + 1);
      if (j + 2 > ntiles) break;
      step(Slot<2>{}, j + 2);
    }
    if (grp == 0) __syncthreads();
    if constexpr (kMode == kPvConvert) {
      bool bad = false;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
#pragma unroll
        for (int r = 0; r < 16; ++r) bad |= !__builtin_isfinite(o[dt][r]);
      }
      if (bad) s_ovf = 1;
      __syncthreads();
      if (s_ovf) return false;
    }
    return true;
  };

  if constexpr (kF8) {
    run(PvTag<kPvF8>{});
  } else if constexpr (KV::kCode == kBF16) {
    if (!run(PvTag<kPvConvert>{})) {
      badkey = 0x7fffffff;
      run(PvTag<kPvSplit>{});
    }
  } else {
    run(PvTag<kPvDirect>{});
  }

  if (badkey != 0x7fffffff) atomicMin(&s_badkey, badkey);
  __syncthreads();
  const int bad_from = s_badkey;

  const float lt = l + __shfl_xor(l, 32, 64);
  if (!live) return;
  // The row's position and offset again from its number, behind an empty asm:
  // kept across the tile loop they cost it registers.
  int qrow_e = qrow;
  asm volatile("" : "+v"(qrow_e));
  const int qpos_e = ctx - S + chunk_row(qrow_e);
  const int64_t row_at = row_offset(qrow_e);
  const bool bad = bad_from <= qpos_e;
  const float inv = lt > 0.0f ? p.vscale / lt : 0.0f;
  const uintptr_t oa = reinterpret_cast<uintptr_t>(p.out);
  const bool vec = (p.out_dtype == kF32 ? (oa & 15) == 0 : (oa & 7) == 0);
  if (!vec) {
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int d = dt * 32 + 8 * (r >> 2) + 4 * hh + (r & 3);
        store_elem(p.out, p.out_dtype, row_at + d, bad ? __builtin_nanf("") : o[dt][r] * inv);
      }
    }
    return;
  }
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = bad ? __builtin_nanf("") : o[dt][4 * j + i] * inv;
      const int64_t e = row_at + dt * 32 + 8 * j + 4 * hh;
      if (p.out_dtype == kF32) {
        u64x2_t w = u64x2_t{(uint64_t)__builtin_bit_cast(uint32_t, v[0]) | ((uint64_t)__builtin_bit_cast(uint32_t, v[1]) << 32),
                            (uint64_t)__builtin_bit_cast(uint32_t, v[2]) | ((uint64_t)__builtin_bit_cast(uint32_t, v[3]) << 32)};
        *reinterpret_cast<u64x2_t*>(static_cast<float*>(p.out) + e) = w;
      } else {
        const uint32_t w0 = p.out_dtype == kF16 ? pack2<false>(v[0], v[1]) : pack2<true>(v[0], v[1]);
        const uint32_t w1 = p.out_dtype == kF16 ? pack2<false>(v[2], v[3]) : pack2<true>(v[2], v[3]);
        const uint64_t w = (uint64_t)w0 | ((uint64_t)w1 << 32);
        *reinterpret_cast<uint64_t*>(static_cast<uint16_t*>(p.out) + e) = w;
      }
    }
  }
}

// CU count of the current device and resident work-groups per CU of one
// kernel instance, cached per device; {0, 0} if unknown.
template <typename F>
static void residency(F kernel, std::atomic<int64_t> (&cache)[64], int64_t* cus, int64_t* per_cu,
                      int threads = kPfThreads) {
  *cus = *per_cu = 0;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0) return;
  if (dev < 64) {
    const int64_t c = cache[dev].load(std::memory_order_relaxed);
    if (c > 0) {
      *cus = c >> 8;
      *per_cu = c & 0xff;
      return;
    }
  }
  int n = 0, k = 0;
  if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) return;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&k, kernel, threads, 0) != hipSuccess || k <= 0 ||
      k > 0xff)
    return;
  if (dev < 64) cache[dev].store(((int64_t)n << 8) | k, std::memory_order_relaxed);
  *cus = n;
  *per_cu = k;
}

// Grid of a prefill kernel of QB-row blocks: its work-groups, and the fields of
// q that number them.
template <typename F>
static int64_t pf_grid(F kernel, std::atomic<int64_t> (&cache)[64], int QB, PrefillParams& q, int threads = kPfThreads) {
  q.q_tiles = (int32_t)(((int64_t)q.S * q.gp + QB - 1) / QB);
  int64_t units = (int64_t)q.B * q.HG * q.q_tiles;
  int64_t cus = 0, per_cu = 0;
  residency(kernel, cache, &cus, &per_cu, threads);
  q.wg_cus = units > cus && units <= cus * per_cu ? (int32_t)cus : 0;  // one resident wave
  // Variable-length batches of up to kVlMaxSeqs sequences: a compacted grid
  // of at most the units with rows (sum over sequences of ceil(rows / QB) <
  // T / QB + sequences).
  q.vl_compact = 0;
  if (q.cu_q && q.B <= kVlMaxSeqs) {
    units = pf_compact_units(q, QB);
    q.vl_compact = 1;
    q.wg_cus = 0;
  }
  return units;
}

// Whether `plain` blocks of 128 packed rows of the fp32-precision prefill run
// faster as twice as many key-split ones of 64 (per_cu of them resident per CU):
// where all of those are resident at once, up to three per CU.  384 plain blocks
// on 256 CUs take two blocks' time, 768 halves at three per CU one and a half.
// fp16, D = 64: 12 heads, S = 4096 91.2 -> 74.1 us; 24 heads, four 512-row
// chunks at 4096 121 -> 106.  Two per CU (D = 128, bf16 q): 256 blocks, one prompt
// of 1024 rows of 32/8 heads, 55 -> 35; but 384, 24 heads, fp16, four chunks at
// 4096, 209 -> 234.  Past that the halves only pay their second reading of K and V
// (D = 64, 448 blocks: 34.5 -> 40.6).
inline bool key_split_pays(int64_t plain, int64_t cus, int64_t per_cu) {
  return 2 * plain <= cus * std::clamp<int64_t>(per_cu, 2, 3);
}

}  // namespace pa
