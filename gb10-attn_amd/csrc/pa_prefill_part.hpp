// pa_prefill_part.hpp -- launches of a prefill's context split: the partitions
// (split_prefill*_kernel), then their merge (prefill_reduce_kernel).
#pragma once

#include "pa_prefill.hpp"

namespace pa {

template <typename KV, int D, int kQP, bool kX>
static hipError_t launch_part(const PrefillParams& p, hipStream_t stream) {
  static_assert((PfShape<D>::MT == 2 ? 2 * PfShape<D>::QW : PfShape<D>::QB) == PfReduce<D>::QB, "rows per unit");
  static std::atomic<int64_t> cache[64];
  constexpr bool kSplit = PfShape<D>::MT == 2;  // key-split mode where there is one
  auto kernel = [] {
    if constexpr (kX) {
      return split_prefill32_kernel<KV, D, kQP, kSplit>;
    } else {
      return split_prefill_mfma_kernel<KV, D, (kQP > 1), kSplit>;
    }
  }();
  PrefillParams q = p;
  q.units = (int32_t)pf_grid(kernel, cache, PfReduce<D>::QB, q);
  q.wg_cus = 0;
  const char* split = kSplit ? "true" : "false";
  if (kX)
    note_launch("pa::split_prefill32_kernel<%s, %d, %d, %s>", KV::kName, D, kQP, split);
  else
    note_launch("pa::split_prefill_mfma_kernel<%s, %d, %s, %s>", KV::kName, D, kQP > 1 ? "true" : "false", split);
  hipLaunchKernelGGL(kernel, dim3((unsigned)q.units * (unsigned)q.parts), dim3(kPfThreads), 0, stream, q);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  note_launch("pa::prefill_reduce_kernel<%d, %s>", D, kX ? "true" : "false");
  hipLaunchKernelGGL((prefill_reduce_kernel<D, kX>),
                     dim3((unsigned)q.units, (unsigned)(PfReduce<D>::QB / PfReduce<D>::ROWS)), dim3(kPfThreads), 0,
                     stream, q);
  return hipGetLastError();
}

template <typename KV, int kQP, bool kX>
static hipError_t launch_part_kv(const PrefillParams& p, hipStream_t stream) {
  switch (p.D) {
    case 32: return launch_part<KV, 32, kQP, kX>(p, stream);
    case 64: return launch_part<KV, 64, kQP, kX>(p, stream);
    case 128: return launch_part<KV, 128, kQP, kX>(p, stream);
    case 256: return launch_part<KV, 256, kQP, kX>(p, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace pa
