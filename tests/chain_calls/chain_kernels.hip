// The chaining table's device functions called by a program of its own:
// chaining_block::init(defaultKey) and chaining_table::attach_block(link).
// Built into tests/chain_calls/libchain_kernels.so by tests/chain_calls/build.py;
// driven from tests/test_gpu_chain_calls.py.
#include <hip/hip_runtime.h>

#include "gallatin/data_structs/chaining_table.hpp"

using namespace gallatin::allocators;
using namespace gallatin::data_structs;

namespace {

template <typename Key, typename Val, int size>
__global__ void k_calls(chaining_table<Key, Val, size>* t, Key key, unsigned long long* errors) {
  using block = chaining_block<Key, Val, size>;
  // an own block, used before: init empties it
  block* b = static_cast<block*>(global_malloc(sizeof(block)));
  if (!b) {
    errors[0] = 1;
    return;
  }
  b->next = 5;
  b->ready = 7;
  for (int i = 0; i < size; ++i) b->keys[i] = (Key)(key + 1 + i);
  __threadfence();
  b->init(key);
  __builtin_amdgcn_s_waitcnt(0);
  __threadfence();
  if (gallatin::utils::atomic_load(&b->next) != 0 || gallatin::utils::atomic_load(&b->ready) != 0)
    atomicAdd(&errors[1], 1ULL);
  for (int i = 0; i < size; ++i)
    if (gallatin::utils::atomic_load(&b->keys[i]) != key) atomicAdd(&errors[1], 1ULL);
  // an empty link gets an empty block, a filled one stays as it is
  uint64_t* link = reinterpret_cast<uint64_t*>(&t->pointer_list[0]);
  const bool first = t->attach_block(link);
  const uint64_t at = gallatin::utils::atomic_load(link);
  const bool again = t->attach_block(link);
  if (first != true || again != true || at == 0 || gallatin::utils::atomic_load(link) != at) {
    atomicAdd(&errors[2], 1ULL);
    return;
  }
  block* n = reinterpret_cast<block*>(at);
  if (gallatin::utils::atomic_load(&n->next) != 0 || gallatin::utils::atomic_load(&n->ready) != 0)
    atomicAdd(&errors[3], 1ULL);
  for (int i = 0; i < size; ++i)
    if (gallatin::utils::atomic_load(&n->keys[i]) != key) atomicAdd(&errors[3], 1ULL);
  global_free(b);
}

template <typename Key, typename Val, int size>
int run(Key key, unsigned long long* errors) {
  auto* t = chaining_table<Key, Val, size>::generate_on_device(size, key, 7);
  unsigned long long* d = nullptr;
  if (!t || hipMalloc(&d, 4 * sizeof(*d)) != hipSuccess) return -2;
  if (hipMemset(d, 0, 4 * sizeof(*d)) != hipSuccess) return -2;
  k_calls<Key, Val, size><<<1, 1>>>(t, key, d);
  const hipError_t e = hipMemcpy(errors, d, 4 * sizeof(*d), hipMemcpyDeviceToHost);
  (void)hipFree(d);
  chaining_table<Key, Val, size>::free_on_device(t);
  return e == hipSuccess ? 0 : -2;
}

}  // namespace

// errors: [0] no memory, [1] init, [2] attach_block's results, [3] the block
// it attached.  Layouts: 64-bit keys, 4 a block; 32-bit keys, 3 a block.
extern "C" int chain_calls(unsigned long long* errors8) {
  init_global_allocator(1ULL << 30, 42, false);
  int rc = run<uint64_t, uint64_t, 4>(11, errors8);
  if (rc == 0) rc = run<uint32_t, uint64_t, 3>(11u, errors8 + 4);
  free_global_allocator();
  return rc;
}
