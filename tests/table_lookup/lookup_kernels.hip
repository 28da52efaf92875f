// Hash table operations on an XCD whose caches hold directory entries from
// before the buckets were published: one workgroup reads the empty entries,
// one on another XCD publishes them, and the first looks up and inserts.
// Built into tests/table_lookup/liblookup_kernels.so by
// tests/table_lookup/build.py; driven from tests/test_gpu_table_lookup.py.
#include <hip/hip_runtime.h>

#include "gallatin/data_structs/extendible_ht.hpp"

using namespace gallatin::allocators;
using namespace gallatin::data_structs;
using table = extendible_hash_table<uint64_t, 0ULL, ~0ULL, uint64_t, 15, 4, 10>;

namespace {

constexpr uint64_t kEntries = table::min_items;
constexpr uint32_t kPolls = 1u << 18;  // bound of each wait

struct meeting {
  uint64_t saved[kEntries];
  uint32_t xcd;        // 1 + the reader's XCD
  uint32_t seen;       // the reader has the empty entries in its caches
  uint32_t taken;      // one workgroup of another XCD publishes
  uint32_t published;
  uint64_t result[6];  // 1 when the run took place, empty entries seen, found, value, stored, found
};

__global__ void k_fill(table* t, uint64_t key, uint64_t val) { t->insert(key, val); }

__global__ void k_empty(table* t, meeting* m) {
  for (uint64_t i = 0; i < kEntries; ++i) {
    uint64_t* e = reinterpret_cast<uint64_t*>(&t->directory[i]);
    m->saved[i] = table::ld(e);
    table::st(e, 0);
  }
}

__device__ bool wait_for(uint32_t* word) {
  for (uint32_t n = 0; n < kPolls; ++n) {
    if (gallatin::utils::atomic_load(word)) return true;
    __builtin_amdgcn_s_sleep(8);
  }
  return false;
}

__global__ __launch_bounds__(64) void k_meet(table* t, meeting* m, uint64_t key, uint64_t other) {
  if (threadIdx.x != 0) return;
  const uint32_t here = 1 + (uint32_t)(__smid() >> 6);
  if (blockIdx.x == 0) {
    gallatin::utils::atomic_store(&m->xcd, here);
    uint64_t empty = 0;
    for (uint64_t i = 0; i < kEntries; ++i)
      empty += table::ld_cached(reinterpret_cast<uint64_t*>(&t->directory[i])) == 0;
    __builtin_amdgcn_s_waitcnt(0);
    gallatin::utils::atomic_store(&m->seen, 1u);
    if (!wait_for(&m->published)) return;
    uint64_t v = 0;
    m->result[1] = empty;
    m->result[2] = t->query(key, v);
    m->result[3] = v;
    m->result[4] = t->insert(other, other + 1);
    m->result[5] = t->query(other, v) && v == other + 1;
    m->result[0] = 1;
    return;
  }
  if (!wait_for(&m->seen) || gallatin::utils::atomic_load(&m->xcd) == here) return;
  if (gallatin::utils::atomic_exch(&m->taken, 1u)) return;
  for (uint64_t i = 0; i < kEntries; ++i)
    table::st(reinterpret_cast<uint64_t*>(&t->directory[i]), m->saved[i]);
  __builtin_amdgcn_s_waitcnt(0);
  gallatin::utils::atomic_store(&m->published, 1u);
}

}  // namespace

// result: meeting::result.  0 or a negative error.
extern "C" int table_lookup(unsigned long long* result) {
  init_global_allocator(1ULL << 30, 42, false);
  table* t = table::generate_on_device(9);
  meeting* m = nullptr;
  int rc = -1;
  if (t && hipMalloc(&m, sizeof(*m)) == hipSuccess &&
      hipMemset(m, 0, sizeof(*m)) == hipSuccess) {
    k_fill<<<1, 1>>>(t, 77, 78);
    k_empty<<<1, 1>>>(t, m);
    k_meet<<<32, 64>>>(t, m, 77, 99);
    if (hipMemcpy(result, m->result, sizeof(m->result), hipMemcpyDeviceToHost) == hipSuccess)
      rc = 0;
    (void)hipFree(m);
  }
  table::free_on_device(t);
  free_global_allocator();
  return rc;
}
