// pa_prefill.hip -- launches of the matrix-core prefill kernels of pa_prefill.hpp
// (16-bit weights): which kernel serves a call, and its grid.
#include "pa_prefill.hpp"

namespace pa {

template <typename KV, int D, bool kSplitQ, bool kSplit>
static hipError_t launch_pf_q(const PrefillParams& p, hipStream_t stream) {
  static std::atomic<int64_t> cache[64];
  const auto kernel = prefill_mfma_kernel<KV, D, kSplitQ, kSplit>;
  PrefillParams q = p;
  const int64_t blocks = pf_grid(kernel, cache, kSplit ? 2 * PfShape<D>::QW : PfShape<D>::QB, q);
  note_launch("pa::prefill_mfma_kernel<%s, %d, %s, %s>", KV::kName, D, kSplitQ ? "true" : "false",
              kSplit ? "true" : "false");
  hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(kPfThreads), 0, stream, q);
  return hipGetLastError();
}

template <typename KV, int D>
static hipError_t launch_pp(const PrefillParams& p, hipStream_t stream) {
  static std::atomic<int64_t> cache[64];
  const auto kernel = prefill_pp_kernel<KV, D>;
  PrefillParams q = p;
  const int64_t units = pf_grid(kernel, cache, kPpRows, q, kPpThreads);
  note_launch("pa::prefill_pp_kernel<%s, %d>", KV::kName, D);
  hipLaunchKernelGGL(kernel, dim3((unsigned)units), dim3(kPpThreads), 0, stream, q);
  return hipGetLastError();
}

// Key-split mode when the plain grid (blocks of 128 query rows) has fewer
// work-groups than CUs: chunks of a long context
// (the reference's 512-token chunk at context 2048: 192 work-groups, +19 %).
// Above that, twice the tiles cost more than the shorter chains save
// (config 4a, 768 work-groups: -17 %).
// The choice counts the blocks that have rows to serve as if each query head had
// its own: a uniform batch's B * ceil(S / rows) per head; a variable-length batch
// brings T rows in all (its grid is sized by the longest sequence, and the
// work-groups past a sequence's rows exit at once), so about ceil(T / rows) of its
// blocks carry work.  (A mixed batch of 64 decode rows and four 256-row chunks had
// taken the 8-wave kernel for its 816-block grid: 48 blocks with rows, on 256 CUs.)
// A group's heads are packed into shared blocks, so where the rows of a head do not
// fill a block the launch has fewer of them, down to count / gp.  fp16, 64/8 heads
// of 128, one block per query head -> packed, 8-wave / 4-wave: 16 prompts of 32 rows
// 32 -> 14.4 / 11.4 us (64 blocks), of 64 rows at 564 tokens 78 -> 33.3 / 33.7 us,
// of 128 rows 46 -> 33.8 / 29.4 us; 4 prompts of 512 rows 49 -> 40 / 42 us.
template <typename KV, int D>
static hipError_t launch_pf(const PrefillParams& p, hipStream_t stream) {
  if constexpr (PfShape<D>::MT == 2) {
    static std::atomic<int64_t> cache[64];
    int64_t cus = 0, per_cu = 0;
    residency(prefill_mfma_kernel<KV, D, false, false>, cache, &cus, &per_cu);
    auto busy = [&](int rows) {
      const int64_t grid = (int64_t)p.B * ((p.S + rows - 1) / rows);
      return (int64_t)p.H * (p.cu_q ? std::min<int64_t>(grid, (p.q_total + rows - 1) / rows) : grid);
    };
    const int64_t plain = busy(PfShape<D>::QB);
    if ((cus > 0 && plain < cus) || (!p.cu_q && (int64_t)p.S * p.gp <= 64))
      return p.q_split ? launch_pf_q<KV, D, true, true>(p, stream) : launch_pf_q<KV, D, false, true>(p, stream);
    // The 8-wave kernel (one work-group per CU) from two of its blocks per CU on;
    // with fewer and one head to a block its 256-row blocks leave CUs idle at the
    // end of the launch (config 4a: 384 work-groups, -20 %).
    if constexpr (KV::kCode == kF16 || KV::kCode == kBF16 || KV::kCode == kFP8) {
      const int64_t pp_units = busy(kPpRows);
      if (!p.q_split && p.MB <= kPfBtStage && cus > 0 && pp_units >= 2 * cus) return launch_pp<KV, D>(p, stream);
    }
  }
  return p.q_split ? launch_pf_q<KV, D, true, false>(p, stream) : launch_pf_q<KV, D, false, false>(p, stream);
}

template <typename KV>
static hipError_t launch_pf_kv(const PrefillParams& p, hipStream_t stream) {
  switch (p.D) {
    case 32: return launch_pf<KV, 32>(p, stream);
    case 64: return launch_pf<KV, 64>(p, stream);
    case 128: return launch_pf<KV, 128>(p, stream);
    case 256: return launch_pf<KV, 256>(p, stream);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_prefill_mfma(const PrefillParams& p, int kv_dtype, hipStream_t stream) {
  if (p.parts > 1) return launch_prefill_part(p, kv_dtype, stream);
  if (kv_dtype == kF16) return launch_pf_kv<KvF16>(p, stream);
  if (kv_dtype == kBF16) return launch_pf_kv<KvBF16>(p, stream);
  if (kv_dtype == kFP8) return p.q_dtype == kBF16 ? launch_pf_kv<KvFP8QkBf16>(p, stream) : launch_pf_kv<KvFP8>(p, stream);
  return hipErrorInvalidValue;
}

}  // namespace pa
