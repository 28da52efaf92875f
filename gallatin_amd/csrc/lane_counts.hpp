// Per-lane counts of the workload kernels and their per-workgroup sums.
// Included inside an anonymous namespace of each workload source.
#ifndef GALLATIN_AMD_LANE_COUNTS_HPP
#define GALLATIN_AMD_LANE_COUNTS_HPP

// Sum of a per-lane value over the wave (every lane of the wave active).
__device__ inline uint64_t wave_sum(uint64_t v) {
  for (int off = 32; off >= 1; off >>= 1)
    v += gallatin::wave::fetch(v, (int)(gallatin::wave::lane() ^ (uint32_t)off));
  return v;
}

// Adds each wave's totals (v[i], the same on every lane) to ctr[i], summed
// over the workgroup in LDS first: one global atomic per nonzero counter per
// workgroup.  The counters share one cache line, where device atomics
// serialise (88 M/s), and the loads of waves still at work queue behind
// them: one atomic per counter per wave took 0.28 ms of a 0.63 ms launch of
// 2^20 threads, and in the cleanup of a batched stream the loads of the last
// chunks took 30 us instead of 2 beside the atomics of the waves that had
// ended.  Every thread of the workgroup calls it once, at the end.
template <int kN>
__device__ inline void add_wave_totals(uint64_t* ctr, const uint64_t (&v)[kN]) {
  // One large workgroup alone: nobody queues behind its waves' atomics, and
  // its barriers cost more (66 batches of at most 287 requests through the
  // slice cache, a launch each: 1,024 threads 1,091 us with the barriers, 1,054
  // without; 256 threads 945 and 954).
  if (gridDim.x == 1 && blockDim.x > 256) {
    if (gallatin::wave::lane() == 0) {
#pragma unroll
      for (int i = 0; i < kN; ++i)
        if (v[i]) gallatin::utils::atomic_add(&ctr[i], v[i]);
    }
    return;
  }
  __shared__ unsigned long long wg[kN];
  if (threadIdx.x < kN) wg[threadIdx.x] = 0;
  __syncthreads();
  if (gallatin::wave::lane() == 0) {
#pragma unroll
    for (int i = 0; i < kN; ++i)
      if (v[i]) atomicAdd(&wg[i], (unsigned long long)v[i]);
  }
  __syncthreads();
  if (threadIdx.x < kN && wg[threadIdx.x])
    gallatin::utils::atomic_add(&ctr[threadIdx.x], (uint64_t)wg[threadIdx.x]);
}

// Per-lane counts of one thread.
struct lane_counts {
  uint32_t pairs = 0, misses = 0, bad = 0, mallocs = 0;
  uint64_t bytes = 0;
};

__device__ inline void add_counters(uint64_t* ctr, const lane_counts& c) {
  const uint64_t v[5] = {wave_sum(c.pairs), wave_sum(c.misses), wave_sum(c.bad),
                         wave_sum(c.bytes), wave_sum(c.mallocs)};
  add_wave_totals(ctr, v);
}

#endif
