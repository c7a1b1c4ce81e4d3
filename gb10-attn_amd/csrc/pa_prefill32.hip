// pa_prefill32.hip -- launches of the fp32-precision matrix-core prefill
// (prefill32_kernel of pa_prefill.hpp): paged_attention_prefill over 16-bit
// and FP8 caches.
#include "pa_prefill.hpp"

namespace pa {

template <typename KV, int D, int kQP, bool kSplit>
static hipError_t launch_p32_q(const PrefillParams& p, hipStream_t stream) {
  static std::atomic<int64_t> cache[64];
  const auto kernel = prefill32_kernel<KV, D, kQP, kSplit>;
  PrefillParams q = p;
  const int64_t blocks = pf_grid(kernel, cache, kSplit ? 2 * PfShape<D>::QW : PfShape<D>::QB, q);
  note_launch("pa::prefill32_kernel<%s, %d, %d, %s>", KV::kName, D, kQP, kSplit ? "true" : "false");
  hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(kPfThreads), 0, stream, q);
  return hipGetLastError();
}

// Key-split mode (64 packed query rows per work-group) or the plain one (128):
// see key_split_pays(); up to 64 rows take it too (half of the plain mode's
// waves would have none).  At D = 128 q in several pieces takes it always: the
// plain mode's two row tiles per wave overflow the registers there (60 to 100
// spilled, none to 45 in the key-split mode): fp32 q, fp16 cache, 12 heads,
// S = 4096 321 -> 128 us, eight of 1024 rows 151 -> 100, 32/8 heads, eight
// 256-row chunks at 4096 457 -> 296; bf16 355 -> 165, 173 -> 127, 574 -> 397.
template <typename KV, int D, int kQP>
static hipError_t launch_p32(const PrefillParams& p, hipStream_t stream) {
  if constexpr (PfShape<D>::MT == 2) {
    if constexpr (D == 128 && kQP > 1) {
      return launch_p32_q<KV, D, kQP, true>(p, stream);
    } else {
      static std::atomic<int64_t> cache[64];
      int64_t cus = 0, per_cu = 0;
      residency(prefill32_kernel<KV, D, kQP, true>, cache, &cus, &per_cu);
      const int64_t rows = (int64_t)p.S * p.gp, QB = PfShape<D>::QB;
      if (rows <= 64 || key_split_pays((int64_t)p.B * p.HG * ((rows + QB - 1) / QB), cus, per_cu))
        return launch_p32_q<KV, D, kQP, true>(p, stream);
    }
  }
  if constexpr (!(D == 128 && kQP > 1)) return launch_p32_q<KV, D, kQP, false>(p, stream);
}

template <typename KV, int kQP>
static hipError_t launch_p32_kv(const PrefillParams& p, hipStream_t stream) {
  switch (p.D) {
    case 32: return launch_p32<KV, 32, kQP>(p, stream);
    case 64: return launch_p32<KV, 64, kQP>(p, stream);
    case 128: return launch_p32<KV, 128, kQP>(p, stream);
    case 256: return launch_p32<KV, 256, kQP>(p, stream);
    default: return hipErrorInvalidValue;
  }
}

// q in the cache's 16-bit type is one exact piece; else two fp16 pieces (fp16
// and FP8 caches) or three bf16 ones.
hipError_t launch_prefill32(const PrefillParams& p, int kv_dtype, hipStream_t stream) {
  if (p.parts > 1) return launch_prefill32_part(p, kv_dtype, stream);
  if (kv_dtype == kF16)
    return p.q_dtype == kF16 ? launch_p32_kv<KvF16, 1>(p, stream) : launch_p32_kv<KvF16, 2>(p, stream);
  if (kv_dtype == kBF16)
    return p.q_dtype == kBF16 ? launch_p32_kv<KvBF16, 1>(p, stream) : launch_p32_kv<KvBF16, 3>(p, stream);
  if (kv_dtype == kFP8) return launch_p32_kv<KvFP8, 2>(p, stream);
  return hipErrorInvalidValue;
}

}  // namespace pa
