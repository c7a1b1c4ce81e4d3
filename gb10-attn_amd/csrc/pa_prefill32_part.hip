// pa_prefill32_part.hip -- context split of the fp32-precision prefill (the
// pieces of launch_prefill32).
#include "pa_prefill_part.hpp"

namespace pa {

hipError_t launch_prefill32_part(const PrefillParams& p, int kv_dtype, hipStream_t stream) {
  if (kv_dtype == kF16)
    return p.q_dtype == kF16 ? launch_part_kv<KvF16, 1, true>(p, stream) : launch_part_kv<KvF16, 2, true>(p, stream);
  if (kv_dtype == kBF16)
    return p.q_dtype == kBF16 ? launch_part_kv<KvBF16, 1, true>(p, stream) : launch_part_kv<KvBF16, 3, true>(p, stream);
  if (kv_dtype == kFP8) return launch_part_kv<KvFP8, 2, true>(p, stream);
  return hipErrorInvalidValue;
}

}  // namespace pa
