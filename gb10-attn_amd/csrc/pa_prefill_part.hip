// pa_prefill_part.hip -- context split of the 16-bit-weight prefill.
#include "pa_prefill_part.hpp"

namespace pa {

template <typename KV>
static hipError_t launch_part_q(const PrefillParams& p, hipStream_t stream) {
  return p.q_split ? launch_part_kv<KV, 2, false>(p, stream) : launch_part_kv<KV, 1, false>(p, stream);
}

hipError_t launch_prefill_part(const PrefillParams& p, int kv_dtype, hipStream_t stream) {
  if (kv_dtype == kF16) return launch_part_q<KvF16>(p, stream);
  if (kv_dtype == kBF16) return launch_part_q<KvBF16>(p, stream);
  if (kv_dtype == kFP8)
    return p.q_dtype == kBF16 ? launch_part_kv<KvFP8QkBf16, 1, false>(p, stream) : launch_part_q<KvFP8>(p, stream);
  return hipErrorInvalidValue;
}

}  // namespace pa
