// pa_common.hpp -- types shared by the host launchers and the gfx950 kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace pa {

enum Dtype : int32_t { kF32 = 0, kF16 = 1, kBF16 = 2, kF64 = 3, kI32 = 4, kI64 = 5, kFP8 = 6 };

constexpr float kNegBig = -3.0e38f;          // empty-softmax sentinel (kernels/paged_attn_v3.cu:21)
constexpr float kLog2e = 1.4426950408889634f;

// Unsigned division by a runtime constant d (1 <= d < 2^31) for n < 2^31:
// q = (umulhi(n, m) + n) >> s with s = ceil(log2 d), m = floor(2^32 (2^s - d) / d) + 1
// (Granlund & Montgomery, "Division by invariant integers using multiplication", 1994).
struct FastDiv {
  uint32_t d, m, s;
};

inline FastDiv make_fastdiv(uint32_t d) {
  FastDiv f;
  f.d = d;
  f.s = 0;
  while ((1ull << f.s) < d) ++f.s;
  f.m = (uint32_t)(((1ull << 32) * ((1ull << f.s) - d)) / d + 1);
  return f;
}

__host__ __device__ inline uint32_t fastdiv(uint32_t n, const FastDiv& f) {
#if defined(__HIP_DEVICE_COMPILE__)
  const uint32_t hi = __umulhi(n, f.m);
#else
  const uint32_t hi = (uint32_t)(((uint64_t)n * f.m) >> 32);
#endif
  return (hi + n) >> f.s;
}

// Everything one decode launch needs.  q/out are [Bq, Sq, H, D] contiguous;
// decode has Sq = 1.  For the fp32 prefill path every query row is its own
// decode problem with context ctx_b - Sq + s + 1 (kernels/paged_attn_prefill.cu:62-65).
struct DecodeParams {
  const void* q;
  void* out;
  const void* k;
  const void* v;
  const int32_t* block_tables;
  const int32_t* context_lens;
  float* ws_acc;  // [B][H][parts][D]
  float* ws_m;    // [B][H][parts]
  float* ws_l;    // [B][H][parts]
  int64_t k_sb, k_st, k_sh;  // element strides of k_cache: block, token, head
  int64_t v_sb, v_st, v_sh;
  int64_t bt_stride;   // elements between block-table rows
  int64_t num_blocks;  // NB: valid block ids are [0, NB)
  int32_t B, Sq, H, HKV, G, D, BS, MB;
  int32_t head_chunks;  // ceil(G / GC): WGs per KV head
  int32_t q_dtype, out_dtype;
  int32_t parts;        // partitions per (sequence, KV head) in the grid
  int32_t part_tokens;  // > 0: fixed partition length; 0: chunk = ceil(ctx / parts)
  int32_t direct;       // 1: one partition, every WG writes the normalised output
  int32_t hp;           // KV heads per work-group (head packing: MHA, or GQA groups of four); <= 1: one
  int32_t pprio;        // 1: the whole grid is resident at once; waves lower their priority as they progress
  int32_t wave_parts;   // explicit splits into short chunks: 1 from the host (the launcher picks the
                        // mode: a partition per wave or per token slot); 0 otherwise
  int32_t uniform_whole;  // part_len(): nearly equal contexts are not cut (B <= 64)
  int32_t fp32_weights;   // matrix-core decode over a bf16 cache: weights (and fp32 q) in 24 bits, not 16
  int32_t seq_order;    // explicit split into long partitions, B <= 64, Sq = 1: sequences dispatched
                        // longest first
  FastDiv bs_div;
  float qscale;         // scale * k_scale * log2(e): scores come out in log2 units
  float vscale;         // v_scale (FP8 caches): applied to the weighted V sum
  // Variable-length batches (Sq = 1): [B + 1] row offsets into packed [T, H, D]
  // q/out; only sequences of exactly one row are served (else null).
  const int32_t* cu_q;
  int64_t q_total;
};

struct ReduceParams {
  void* out;
  const float* ws_acc;
  const float* ws_m;
  const float* ws_l;
  const int32_t* context_lens;
  int32_t B, H, D, MB, BS;
  int32_t out_dtype;
  int32_t parts;
  int32_t part_tokens;
  int32_t uniform_whole;
  const int32_t* cu_q;  // variable-length batches: as DecodeParams
  int64_t q_total;
};

struct PrefillParams {
  const void* q;   // [B, S, H, D]
  void* out;       // [B, S, H, D]
  const void* k;
  const void* v;
  const int32_t* block_tables;
  const int32_t* context_lens;
  int64_t k_sb, k_st, k_sh;
  int64_t v_sb, v_st, v_sh;
  int64_t bt_stride;
  int64_t num_blocks;
  int32_t B, S, H, HKV, G, D, BS, MB;
  int32_t q_dtype, out_dtype;
  int32_t gp;        // heads packed into the rows: the GQA group, or 1
  int32_t HG;        // H / gp
  FastDiv gp_div;
  int32_t q_tiles;   // ceil(S * gp / QBLOCK)
  int32_t wg_cus;    // > 0: the whole grid is resident on this many CUs (work-group order)
  const int32_t* cu_q;  // variable-length batches: [B + 1] row offsets into [T, H, D] q/out (else null)
  int64_t q_total;      // T (variable-length batches)
  int32_t skip_single;  // variable-length batches: sequences of one row are served by the decode kernel
  int32_t vl_compact;   // variable-length batches (B <= kVlMaxSeqs): the grid holds only units with rows
  int32_t q_split;   // q is not exactly the KV type: add a low-part product
  FastDiv bs_div;
  float qscale;      // |scale| * log2(e), or 1 when scale == 0 (always positive)
  float q_sign;      // sign of scale applied to q (+1, -1, or 0 when scale == 0)
  float vscale;      // v_scale of a scaled (FP8) cache: multiplies the output rows
  uint32_t q_and;    // the same on packed 16-bit q: bits & q_and ^ q_xor
  uint32_t q_xor;
  // Context split (parts > 1).
  int32_t units;       // units of the grid, per partition
  int32_t parts;       // most partitions per unit
  int32_t part_tiles;  // key tiles per partition
  float* ws_acc;       // [units][parts][rows][D] un-normalised sums
  float* ws_m;         // [units][parts][rows] reference points (log2 units; -inf: no key)
  float* ws_l;         // [units][parts][rows] row sums (NaN: an unreadable key)
};

constexpr int kPfMinPartTiles = 4;  // fewest key tiles per partition of a prefill split
constexpr int kVlMaxSeqs = 256;  // variable-length batches numbered compactly (four sequences per lane)

// Rows per unit of a context-split prefill grid and keys per tile.
inline int pf_split_rows(int D) { return D <= 128 ? 64 : 128; }
inline int pf_tile_keys(int D) { return D <= 128 ? 64 : 32; }

// Most units of a compacted variable-length grid of QB-row blocks.
inline int64_t pf_compact_units(const PrefillParams& p, int QB) {
  const int64_t tiles = ((int64_t)p.S * p.gp + QB - 1) / QB;
  const int64_t by_rows = (p.q_total * p.gp + QB - 1) / QB + (p.B < p.q_total ? p.B : p.q_total);
  return p.HG * (p.B * tiles < by_rows ? p.B * tiles : by_rows);
}

// Context split of a prefill grid on `cus` compute units: sets parts and
// part_tiles, returns the bytes of workspace the partitions' sums take (0: no
// split).
// A work-group alone on its CU takes tile_us per 64-key tile (measured: D = 64
// 0.86, D = 128 1.3), two take 1.25-1.35 times that between them, and a third
// or fourth adds nothing: so a grid is brought to at most two work-groups per
// CU, and only where the shorter chains save more than the second launch and
// the partial sums cost (5-7 us; a variable-length batch, whose grid holds idle
// work-groups and whose prompts may be shorter than its longest context, 12, and 20
// where the partitions outnumber the CUs: 90 decode rows and six chunks of 128 at
// context 1024, fp16, unsplit / split: 8/1 heads of 128 71 / 78 us, 8/2 heads
// 51 / 56; at 4096 217 / 143 and 156 / 118).  The times are those of 16-bit weights;
// fp32 weights and the 32-key tiles of D = 256 take longer.  B = 1, S = 16, context 12288: 12 heads of
// 64 150 -> 20 us, 32/8 heads of 128 242 -> 27 us; B = 1, S = 64, context
// 1024: 17.5 -> 12.5 and 27.8 -> 15.7; B = 1, S = 512, context 8192, 32/8
// heads (256 blocks, two partitions): 161 -> 111.  Without the two bounds
// B = 4, S = 512, context 2048, 12 heads (384 blocks) took 37.1 instead of
// 33.5 us, S = 1024 of 16/4 heads of 64 (256 blocks, 16 tiles) 19.9 instead
// of 17.9.
inline size_t plan_prefill_split(PrefillParams& p, bool varlen, int cus) {
  p.parts = 1;
  p.part_tiles = 0;
  if (varlen && p.B > kVlMaxSeqs) return 0;
  const int QB = pf_split_rows(p.D), KB = pf_tile_keys(p.D);
  const int64_t tiles = ((int64_t)p.S * p.gp + QB - 1) / QB;
  const int64_t units = varlen ? pf_compact_units(p, QB) : (int64_t)p.B * p.HG * tiles;
  // Blocks with rows (a variable-length batch's: about its rows over QB).
  const int64_t by_rows = p.HG * ((p.q_total * p.gp + QB - 1) / QB);
  const int64_t busy = varlen && by_rows < units ? by_rows : units;
  const int64_t key_tiles = ((int64_t)p.MB * p.BS + KB - 1) / KB;
  if (busy <= 0) return 0;
  int64_t n = 2 * (int64_t)cus / busy;
  if (n > key_tiles / kPfMinPartTiles) n = key_tiles / kPfMinPartTiles;
  const double tile_us = p.D <= 64 ? 0.86 : 1.3;
  if (n < 2 || (double)key_tiles * tile_us * (1.0 - 1.35 / (double)n) < (varlen ? (n * busy > cus ? 20.0 : 12.0) : 7.0)) return 0;
  p.part_tiles = (int32_t)((key_tiles + n - 1) / n);
  p.parts = (int32_t)((key_tiles + p.part_tiles - 1) / p.part_tiles);
  return (size_t)units * p.parts * QB * (p.D + 2) * 4;
}
// The workspace's sections for that plan.
inline void bind_prefill_split(PrefillParams& p, void* ws, size_t bytes) {
  const size_t rows = bytes / ((size_t)(p.D + 2) * 4);
  p.ws_acc = static_cast<float*>(ws);
  p.ws_m = p.ws_acc + rows * p.D;
  p.ws_l = p.ws_m + rows;
}

// KV-cache write: new [T, HKV, D] rows -> paged pool slots (element strides).
struct WriteParams {
  void* kc;            // k_cache / v_cache [NB, BS, HKV, D]
  void* vc;
  const void* key;     // [T, HKV, D]
  const void* value;
  const void* slots;   // [T] int32 or int64
  int64_t kc_sb, kc_st, kc_sh;
  int64_t vc_sb, vc_st, vc_sh;
  int64_t key_st, key_sh;
  int64_t val_st, val_sh;
  int64_t nslots;      // NB * BS (< 2^31)
  int32_t T, HKV, D, BS;
  int32_t src_dtype, cache_dtype, slot_i64;
  int32_t unit_scale;  // 1: k_scale == v_scale == 1 (no division)
  float k_scale, v_scale;  // the cache holds key / k_scale and value / v_scale
  float k_rcp, v_rcp;      // 1 / k_scale, 1 / v_scale rounded to nearest (fp32)
  int32_t k_fast, v_fast;  // |k_rcp|, |v_rcp| in [2^-60, 2^60]: the reciprocal-based division applies
  FastDiv bs_div;
  FastDiv chunk_div, hkv_div;  // D / 8 and HKV (work item -> token, head, chunk)
  int32_t t_base;              // first token of this launch (large writes take several)
};

constexpr int kDecodeWaves = 4;
constexpr int kDecodeThreads = 64 * kDecodeWaves;
constexpr int kBtChunk = 256;  // block-table entries a decode work-group stages in LDS at a time

// Explicit short partitions (DecodeParams::wave_parts): one per wave, or one
// per token slot of a wave (TPI per wave).
constexpr int kWavePart = 1;
constexpr int kSlotPart = 2;

// Records the kernel instance a launcher is about to dispatch, as profilers
// print its demangled name, for pa_last_launch() (host side, per thread).
void note_launch(const char* fmt, ...) __attribute__((format(printf, 1, 2)));

// Host launchers (defined in the kernel translation units).
hipError_t launch_decode(const DecodeParams& p, int kv_dtype, int gc, hipStream_t stream);
hipError_t launch_reduce(const ReduceParams& p, hipStream_t stream);
hipError_t launch_prefill_mfma(const PrefillParams& p, int kv_dtype, hipStream_t stream);
hipError_t launch_prefill_part(const PrefillParams& p, int kv_dtype, hipStream_t stream);
hipError_t launch_prefill32_part(const PrefillParams& p, int kv_dtype, hipStream_t stream);
hipError_t launch_prefill32(const PrefillParams& p, int kv_dtype, hipStream_t stream);
hipError_t launch_write_kv(const WriteParams& p, hipStream_t stream);

// Head packing (heads contiguous in the pool; MHA, or GQA groups of four over
// 16-bit caches): one decode work-group
// serves HP adjacent KV heads, whose rows of a token are contiguous, as one
// row of HP * D elements.  Wider contiguous reads keep more of each DRAM row
// access useful: at B = 256, ctx 2048, fp16 D = 64 one head per work-group
// streams 6.42 TB/s, two 6.66, four 6.80.  Rows shorter than a 128-byte line
// are always packed (two heads at least), since a half-line request costs
// a whole line.  The planner chooses HP per call (DecodeParams::hp); it sees
// only K (the workspace-size query has no V), and the kernel also needs V's
// heads contiguous, else it serves one head per work-group under the same
// plan.
constexpr int kPackRowBytes = 512;  // widest packed row
constexpr int kPackMax = 4;         // most KV heads per work-group
constexpr int kPackGqaMax = 2;      // most KV heads per work-group for GQA groups of four

// Widest packing the layout allows (1 = none).  GQA groups of four query
// heads over 8/16-bit caches pack too: each lane still serves one KV head's
// group, so the vector work per lane is unchanged and only the rows read
// together get wider (two KV heads: config 3 5819 -> 5968 GB/s, FP8 config 3
// 4550 -> 4753).
inline int decode_pack_max(int D, int kv_bytes, int G, int HKV, int64_t k_sh) {
  if (k_sh != D || !(G == 1 || (G == 4 && kv_bytes <= 2))) return 1;
  const int most = G == 1 ? kPackMax : kPackGqaMax;
  const int64_t row = kPackRowBytes;
  int hp = 1;
  for (int c = 2; c <= most; c *= 2)
    if ((int64_t)D * kv_bytes * c <= row && HKV % c == 0) hp = c;
  return hp;
}

// Narrowest packing worth running: two heads when a row is under a line.
inline int decode_pack_min(int D, int kv_bytes, int G, int HKV, int64_t k_sh) {
  return (D * kv_bytes < 128 && decode_pack_max(D, kv_bytes, G, HKV, k_sh) >= 2) ? 2 : 1;
}

// Heads per decode work-group for a GQA group of G query heads.
inline int decode_heads_per_wg(int G) {
  if (G <= 1) return 1;
  if (G <= 2) return 2;
  if (G <= 4) return 4;
  if (G <= 8) return 8;
  if (G % 8 == 0) return 8;
  if (G % 4 == 0) return 4;
  if (G % 2 == 0) return 2;
  return 1;
}

}  // namespace pa
