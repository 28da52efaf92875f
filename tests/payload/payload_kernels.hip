// The churn kernels' wave_fill and wave_verify on buffers the test made: lane l
// of one wave owns the buffer at ptrs[l] of words[l] 64-bit words (0: none)
// and fills it with pats[l], or counts the words that differ from pats[l].
// Built into tests/payload/libpayload_kernels.so by tests/payload/build.py;
// driven from tests/test_gpu_payload.py.
#include <hip/hip_runtime.h>

#include "gallatin/allocators/alloc_utils.hpp"

using namespace gallatin;

namespace {

#include "payload.hpp"

__global__ __launch_bounds__(64) void k_payload(uint64_t* const* ptrs, const uint32_t* words,
                                                const uint64_t* pats, uint32_t* bad, int verify) {
  __shared__ chunk_map m;
  const uint32_t l = threadIdx.x;
  const bool on = words[l] != 0;
  if (verify)
    bad[l] = wave_verify(m, on, ptrs[l], words[l], pats[l]);
  else
    wave_fill(m, on, ptrs[l], words[l], pats[l]);
}

}  // namespace

// Arrays of 64 entries on the device; words at most 512, buffers 16-byte
// aligned with room for an even word count.  Synchronous; 0 or a negative error.
extern "C" int payload_run(uint64_t* const* ptrs, const uint32_t* words, const uint64_t* pats,
                           uint32_t* bad, int verify) {
  if (!ptrs || !words || !pats || !bad) return -1;
  k_payload<<<1, 64>>>(ptrs, words, pats, bad, verify);
  return hipDeviceSynchronize() == hipSuccess ? 0 : -2;
}
