// Allocator-backed extendible hash table of 64-bit keys and values
// (extendible_ht.cuh:132-1437).
//
// Layout.  Buckets of items_per_bucket pairs come from the global allocator.
// Bucket b has a home index h(b) and a depth d(b) >= min_bits and owns the
// keys whose hash agrees with h(b) in the low d(b) bits.  The directory has
// 2^max_bits entries (taken from the global allocator and zeroed once);
// entry i holds the bucket whose home is i, or nothing if no bucket with
// that home exists yet.  The owner of a hash is found by looking at the
// entry of its low `level` bits, then of its low level - 1 bits, ... and
// taking the first bucket present (the reference's refinement from the
// global level down, extendible_ht.cuh:842-1115); the entries of four
// depths are loaded together.  Entries [0, 2^min_bits) are filled at
// creation.
//
// Writes (insert, remove) lock the owner bucket, check that it still owns
// the key and work under the lock.  The lock bit, the depth and the home
// share one word, so the atomic that takes the lock also returns both.  A full
// bucket is split: a new bucket with home h(b) + 2^d(b) and depth d(b) + 1
// receives the keys whose bit d(b) is set, is published in the directory,
// then the old bucket's depth is raised and the moved keys are cleared from
// it (the reference's promotion, extendible_ht.cuh:1118-1289).  Queries
// take no lock: they read the owner's depth, scan its keys, and when the key
// is missing look again if the depth changed meanwhile, so a key is never
// missed while it moves; a found key's value counts only if the key is still
// in its slot after the value was read (the slot may have been emptied and
// reused).  Every bucket word is read and written with device-coherent
// atomics; a value is written before its key and a moved key before the new
// bucket is published.  Lock attempts per operation are bounded.
//
// What bounds it: coherent requests.  A lane that reads its own bucket's 17
// words one by one issues 17 of them per key, and the device serves 250 G/s of
// such scattered requests.  So a bucket of 15 pairs starts with one 128-byte
// line, the control word and the keys, and the lanes of a whole wave read the
// lines together: eight lanes per bucket, 16 bytes each, so that a line is
// one request.  The first look at the directory goes through the XCD's
// caches (see owner).  2^20 operations on a table of 2^21 keys: query
// 114 -> 76 us, insert 215 -> 157 us, remove 183 -> 99 us (the last two are then
// bound by their lock atomics and stores, 4 and 3 an operation at 26 G/s).
//
// Differences from the reference: insert of a present key replaces its
// value; remove() exists (the reference has none, so its behaviour is not
// pinned by it); a table that cannot split further, or cannot get memory,
// makes insert return false instead of trapping.
#ifndef GALLATIN_EXTENDIBLE_HT_HPP
#define GALLATIN_EXTENDIBLE_HT_HPP

#include <hip/hip_runtime.h>

#include "gallatin/allocators/global_allocator.hpp"
#include "gallatin/allocators/murmurhash.hpp"

namespace gallatin {
namespace data_structs {

template <typename table>
__global__ void ext_ht_alloc_directory(table* t) {
  if (blockIdx.x == 0 && threadIdx.x == 0) t->alloc_directory();
}

template <typename table>
__global__ void ext_ht_first_buckets(table* t, uint64_t n) {
  const uint64_t i = gallatin::utils::get_tid();
  if (i < n) t->make_first_bucket(i);
}

template <typename table>
__global__ void ext_ht_free_buckets(table* t, uint64_t n) {
  const uint64_t i = gallatin::utils::get_tid();
  if (i < n) t->free_bucket_at(i);
}

template <typename table>
__global__ void ext_ht_free_directory(table* t) {
  if (blockIdx.x == 0 && threadIdx.x == 0) t->free_directory();
}

// Keys present (out[0]) and buckets (out[1]): a bucket is the one directory
// entry at its home.  One atomic per wave and counter.
template <typename table>
__global__ void ext_ht_count(table* t, uint64_t n, unsigned long long* out) {
  const uint64_t i = gallatin::utils::get_tid();
  uint64_t keys = 0, buckets = 0;
  if (i < n) {
    keys = t->bucket_fill(i);
    buckets = t->directory && t->directory[i] ? 1 : 0;
  }
  for (int off = 32; off >= 1; off >>= 1) {
    const int src = (int)(gallatin::wave::lane() ^ (uint32_t)off);
    keys += gallatin::wave::fetch(keys, src);
    buckets += gallatin::wave::fetch(buckets, src);
  }
  if (gallatin::wave::lane() == 0) {
    if (keys) atomicAdd(out, (unsigned long long)keys);
    if (buckets) atomicAdd(out + 1, (unsigned long long)buckets);
  }
}

template <typename Key, Key defaultKey, Key tombstoneKey, typename Val, int items_per_bucket,
          uint64_t min_bits, uint64_t max_bits>
struct extendible_hash_table {
  using my_type = extendible_hash_table<Key, defaultKey, tombstoneKey, Val, items_per_bucket,
                                        min_bits, max_bits>;
  static_assert(sizeof(Key) == 8 && sizeof(Val) == 8, "64-bit keys and values");
  static_assert(min_bits >= 1 && min_bits <= max_bits && max_bits <= 40, "table bits");
  static_assert(items_per_bucket >= 2 && items_per_bucket <= 64, "bucket size");

  static constexpr uint64_t min_items = 1ULL << min_bits;
  static constexpr uint64_t max_items = 1ULL << max_bits;
  static constexpr uint32_t kTries = 1u << 22;  // lock attempts per operation
  static constexpr uint32_t kSameBucket = 6;    // lost lock attempts before looking up again
  static constexpr uint32_t kTogether = 8;      // lanes from which a wave reads lines together

  struct bucket {
    uint64_t ctl;  // (home << 8) | (depth << 1) | lock bit
    uint64_t keys[items_per_bucket];
    uint64_t vals[items_per_bucket];
  };
  // the control word and the keys fill one 128-byte line of an aligned bucket
  static constexpr bool kLine = items_per_bucket == 15;

  bucket** directory;  // max_items entries
  uint64_t level;      // deepest bucket depth
  uint64_t seed;
  uint64_t reserved;   // (buckets are counted by count_keys)
  uint64_t failed;     // inserts refused (table full or no memory)

  // ---- host ----
  // extendible_ht.cuh:441-476.  Needs the global allocator.
  static __host__ my_type* generate_on_device(uint64_t seed = 42) {
    my_type host{};
    host.level = min_bits;
    host.seed = seed;
    my_type* dev = nullptr;
    if (hipMalloc(&dev, sizeof(my_type)) != hipSuccess) return nullptr;
    if (hipMemcpy(dev, &host, sizeof(my_type), hipMemcpyHostToDevice) != hipSuccess) {
      (void)hipFree(dev);
      return nullptr;
    }
    ext_ht_alloc_directory<my_type><<<1, 1>>>(dev);
    bucket** dir = nullptr;
    if (hipDeviceSynchronize() != hipSuccess ||
        hipMemcpy(&dir, &dev->directory, sizeof(dir), hipMemcpyDeviceToHost) != hipSuccess ||
        dir == nullptr || hipMemset(dir, 0, sizeof(bucket*) * max_items) != hipSuccess) {
      (void)hipFree(dev);
      return nullptr;
    }
    ext_ht_first_buckets<my_type><<<(unsigned)((min_items + 255) / 256), 256>>>(dev, min_items);
    if (hipDeviceSynchronize() != hipSuccess) return nullptr;
    return dev;
  }

  // extendible_ht.cuh:479-494.
  static __host__ void free_on_device(my_type* dev) {
    if (!dev) return;
    ext_ht_free_buckets<my_type><<<(unsigned)((max_items + 255) / 256), 256>>>(dev, max_items);
    ext_ht_free_directory<my_type><<<1, 1>>>(dev);
    (void)hipDeviceSynchronize();
    (void)hipFree(dev);
  }

  // Keys present (calculate_fill's count, extendible_ht.cuh:1379-1411) and,
  // into *buckets, the buckets in use.
  static __host__ uint64_t count_keys(my_type* dev, uint64_t* buckets = nullptr) {
    unsigned long long* c = nullptr;
    if (hipMalloc(&c, 2 * sizeof(*c)) != hipSuccess) return 0;
    (void)hipMemset(c, 0, 2 * sizeof(*c));
    ext_ht_count<my_type><<<(unsigned)((max_items + 255) / 256), 256>>>(dev, max_items, c);
    unsigned long long n[2] = {0, 0};
    (void)hipMemcpy(n, c, sizeof(n), hipMemcpyDeviceToHost);
    (void)hipFree(c);
    if (buckets) *buckets = n[1];
    return n[0];
  }

  // ---- device: set-up and teardown ----
  __device__ void alloc_directory() {
    directory = static_cast<bucket**>(
        gallatin::allocators::global_malloc(sizeof(bucket*) * max_items));
  }

  __device__ bucket* new_bucket(uint64_t home, uint32_t depth) {
    bucket* b = static_cast<bucket*>(gallatin::allocators::global_malloc(sizeof(bucket)));
    if (!b) return nullptr;
    // device-coherent stores: another XCD may read the bucket as soon as
    // it is published
    gallatin::utils::atomic_store(&b->ctl, ctl_of(home, depth));
    for (int i = 0; i < items_per_bucket; ++i)
      gallatin::utils::atomic_store(&b->keys[i], (uint64_t)defaultKey);
    return b;
  }

  __device__ void make_first_bucket(uint64_t i) {
    bucket* b = new_bucket(i, (uint32_t)min_bits);
    if (!b) {
      gallatin::utils::atomic_add(&failed, (uint64_t)1);
      return;
    }
    __builtin_amdgcn_s_waitcnt(0);
    gallatin::utils::atomic_store(reinterpret_cast<uint64_t*>(&directory[i]),
                                  reinterpret_cast<uint64_t>(b));
  }

  __device__ void free_bucket_at(uint64_t i) {
    if (directory && directory[i]) gallatin::allocators::global_free(directory[i]);
  }

  __device__ void free_directory() {
    if (directory) gallatin::allocators::global_free(directory);
    directory = nullptr;
  }

  __device__ uint64_t bucket_fill(uint64_t i) {
    bucket* b = directory ? directory[i] : nullptr;
    if (!b) return 0;
    uint64_t c = 0;
    for (int s = 0; s < items_per_bucket; ++s)
      c += b->keys[s] != defaultKey && b->keys[s] != tombstoneKey;
    return c;
  }

  // ---- device: operations ----
  static __device__ __forceinline__ uint64_t mask(uint64_t d) { return (1ULL << d) - 1; }
  static __device__ __forceinline__ uint64_t ld(const uint64_t* p) {
    return gallatin::utils::atomic_load(p);
  }
  static __device__ __forceinline__ void st(uint64_t* p, uint64_t v) {
    gallatin::utils::atomic_store(p, v);
  }
  // A read that may return an old value: a workgroup-scope load, served by
  // this XCD's caches.  (A volatile read compiles to a system-scope load,
  // which goes to memory like a device-coherent one.)
  static __device__ __forceinline__ uint64_t ld_cached(const uint64_t* p) {
    return __hip_atomic_load(const_cast<uint64_t*>(p), __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_WORKGROUP);
  }

  __device__ uint64_t hash(Key k) const { return hashers::MurmurHash64A_u64((uint64_t)k, seed); }

  typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

  // Eight device-coherent 16-byte loads in flight together (each 8-byte half
  // is read whole).  The wait is part of the block, so no output register is
  // reused while its load is still on the way.
  static __device__ __forceinline__ void load8(const uint64_t (&a)[8], u32x4 (&w)[8]) {
    asm volatile(
        "global_load_dwordx4 %0, %8, off sc1\n\t"
        "global_load_dwordx4 %1, %9, off sc1\n\t"
        "global_load_dwordx4 %2, %10, off sc1\n\t"
        "global_load_dwordx4 %3, %11, off sc1\n\t"
        "global_load_dwordx4 %4, %12, off sc1\n\t"
        "global_load_dwordx4 %5, %13, off sc1\n\t"
        "global_load_dwordx4 %6, %14, off sc1\n\t"
        "global_load_dwordx4 %7, %15, off sc1\n\t"
        "s_waitcnt vmcnt(0)"
        : "=&v"(w[0]), "=&v"(w[1]), "=&v"(w[2]), "=&v"(w[3]), "=&v"(w[4]), "=&v"(w[5]),
          "=&v"(w[6]), "=&v"(w[7])
        : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]), "v"(a[4]), "v"(a[5]), "v"(a[6]), "v"(a[7])
        : "memory");
  }
  static __device__ __forceinline__ uint64_t lo(u32x4 v) {
    return (uint64_t)v.x | (uint64_t)v.y << 32;
  }
  static __device__ __forceinline__ uint64_t hi(u32x4 v) {
    return (uint64_t)v.z | (uint64_t)v.w << 32;
  }
  static __device__ __forceinline__ bool is_free(uint64_t k) {
    return k == (uint64_t)defaultKey || k == (uint64_t)tombstoneKey;
  }

  // Bucket b's control word, the slot holding `key` or -1, and the first free
  // slot or -1, for every lane with `on` (the others get nothing of use).  All
  // words are loaded first, so the loads are in flight together, then
  // compared.
  __device__ void scan(bool on, bucket* b, uint64_t key, uint64_t& ctl, int& match, int& empty) {
    const uint64_t todo = __ballot(on);
    match = -1;
    empty = -1;
    ctl = 0;
    if (!todo) return;
    if constexpr (kLine) {
      uint64_t a[8];
      u32x4 w[8];
      if (__ballot(1) == ~0ULL && gallatin::wave::count(todo) >= kTogether) {
        // round r serves lanes 8r .. 8r + 7: lane l reads the l % 8-th 16
        // bytes of the bucket of lane 8r + l / 8
        const uint32_t lane = gallatin::wave::lane();
        const int any = gallatin::wave::first(todo);  // stands in for lanes that ask nothing
        const uint64_t mine = reinterpret_cast<uint64_t>(b);
        const uint64_t at = on ? mine : gallatin::wave::readlane(mine, any);
#pragma unroll
        for (int r = 0; r < 8; ++r)
          a[r] = gallatin::wave::fetch(at, 8 * r + (int)(lane >> 3)) + 16 * (lane & 7);
        load8(a, w);
        uint64_t m0 = 0, m1 = 0, e0 = 0, e1 = 0;  // this lane's round's answers
#pragma unroll
        for (int r = 0; r < 8; ++r) {
          const uint64_t k = gallatin::wave::fetch(key, 8 * r + (int)(lane >> 3));
          const uint64_t x0 = lo(w[r]), x1 = hi(w[r]);
          const bool first = (lane & 7) == 0;  // x0 is the control word
          const uint64_t q0 = __ballot(!first && x0 == k), q1 = __ballot(x1 == k);
          const uint64_t f0 = __ballot(!first && is_free(x0)), f1 = __ballot(is_free(x1));
          const uint64_t c = gallatin::wave::fetch(x0, (int)(8 * (lane & 7)));
          const bool me = (int)(lane >> 3) == r;
          m0 = me ? q0 : m0;
          m1 = me ? q1 : m1;
          e0 = me ? f0 : e0;
          e1 = me ? f1 : e1;
          ctl = me ? c : ctl;
        }
        // byte l % 8: bit j of m0 is slot 2j - 1, of m1 slot 2j
        const uint32_t sh = 8 * (lane & 7);
        const uint32_t q0 = (uint32_t)(m0 >> sh) & 255u, q1 = (uint32_t)(m1 >> sh) & 255u;
        const uint32_t f0 = (uint32_t)(e0 >> sh) & 255u, f1 = (uint32_t)(e1 >> sh) & 255u;
        if (q0 | q1) match = q0 ? 2 * __builtin_ctz(q0) - 1 : 2 * __builtin_ctz(q1);
        const int s0 = f0 ? 2 * __builtin_ctz(f0) - 1 : 15, s1 = f1 ? 2 * __builtin_ctz(f1) : 15;
        const int s = s0 < s1 ? s0 : s1;
        if (s < 15) empty = s;
      } else if (on) {  // few, or some lanes are elsewhere: each its own bucket's line
#pragma unroll
        for (int r = 0; r < 8; ++r) a[r] = reinterpret_cast<uint64_t>(b) + 16 * r;
        load8(a, w);
        ctl = lo(w[0]);
#pragma unroll
        for (int r = 7; r >= 0; --r) {
          if (hi(w[r]) == key) match = 2 * r;
          if (is_free(hi(w[r]))) empty = 2 * r;
          if (r > 0 && lo(w[r]) == key) match = 2 * r - 1;
          if (r > 0 && is_free(lo(w[r]))) empty = 2 * r - 1;
        }
      }
    } else if (on) {
      uint64_t k[items_per_bucket];
      ctl = ld(&b->ctl);
#pragma unroll
      for (int s = 0; s < items_per_bucket; ++s) k[s] = ld(&b->keys[s]);
#pragma unroll
      for (int s = items_per_bucket - 1; s >= 0; --s) {
        if (k[s] == key) match = s;
        if (is_free(k[s])) empty = s;
      }
    }
  }

  // The bucket owning hash h: the entry of its low `level` bits, or of
  // fewer bits when that home has no bucket yet.  Entries are only ever
  // set, so the deepest one present among the loaded depths is the owner
  // (or a bucket being split, which the callers' home check rejects).
  //
  // `fresh` = false reads `level` and the entries through the caches: they
  // may be behind, and since the level only grows and entries are only ever
  // set that only leads to an ancestor of the owner, or to none; every caller
  // checks the bucket's home against its depth and looks again (with fresh =
  // true), and where the caches show no entry at all this does.  nullptr: no
  // bucket.
  // Device-coherent reads of one word from the whole device queue at one
  // memory channel, and scattered ones run at half the rate of cached ones.
  static constexpr int kOwnerFan = 4;
  __device__ bucket* owner(uint64_t h, bool fresh) {
    uint64_t top = fresh ? ld(&level) : ld_cached(&level);
    for (;;) {
      uint64_t e[kOwnerFan];
#pragma unroll
      for (int j = 0; j < kOwnerFan; ++j) {
        const uint64_t d = top >= min_bits + j ? top - j : min_bits;
        const uint64_t* at = reinterpret_cast<const uint64_t*>(&directory[h & mask(d)]);
        e[j] = fresh ? ld(at) : ld_cached(at);
      }
#pragma unroll
      for (int j = 0; j < kOwnerFan; ++j)
        if (e[j]) return reinterpret_cast<bucket*>(e[j]);
      if (top >= min_bits + kOwnerFan) {
        top -= kOwnerFan;
      } else {
        if (fresh) return nullptr;
        fresh = true;
        top = ld(&level);
      }
    }
  }

  static __device__ __forceinline__ uint32_t depth_of(uint64_t ctl) {
    return (uint32_t)(ctl >> 1) & 127u;
  }
  static __device__ __forceinline__ uint64_t home_of(uint64_t ctl) { return ctl >> 8; }
  static __device__ __forceinline__ uint64_t ctl_of(uint64_t home, uint32_t d) {
    return (home << 8) | ((uint64_t)d << 1);
  }
  // Whether the bucket of this control word owns hash h.
  static __device__ __forceinline__ bool owns(uint64_t ctl, uint64_t h) {
    return (h & mask(depth_of(ctl))) == home_of(ctl);
  }

  // One attempt; on success `ctl` is the bucket's control word.  Lock users
  // retry in a loop whose every iteration holds the whole critical section: a
  // lane that gets the lock releases it in the same iteration, so lanes of one
  // wave waiting for the same bucket never keep its holder from running (a
  // spin-then-work loop would).
  __device__ bool try_lock(bucket* b, uint64_t& ctl) {
    ctl = gallatin::utils::atomic_or(&b->ctl, (uint64_t)1);
    return (ctl & 1) == 0;
  }

  __device__ void unlock(bucket* b, uint64_t ctl) {
    __builtin_amdgcn_s_waitcnt(0);  // the critical section's stores land first
    gallatin::utils::atomic_store(&b->ctl, ctl);
  }

  // Split full bucket b (locked, depth d): keys with bit d set move to a new
  // bucket with home h(b) + 2^d.  False when no bucket could be had.
  __device__ bool split(bucket* b, uint32_t d, uint64_t old_home) {
    uint64_t k[items_per_bucket], v[items_per_bucket];
#pragma unroll
    for (int s = 0; s < items_per_bucket; ++s) {
      k[s] = ld(&b->keys[s]);
      v[s] = ld(&b->vals[s]);
    }
    const uint64_t home = old_home | (1ULL << d);
    bucket* nb = static_cast<bucket*>(gallatin::allocators::global_malloc(sizeof(bucket)));
    if (!nb) return false;
    uint64_t moved = 0;
#pragma unroll
    for (int s = 0; s < items_per_bucket; ++s) {
      const bool live = k[s] != (uint64_t)defaultKey && k[s] != (uint64_t)tombstoneKey;
      const bool go = live && ((hash((Key)k[s]) >> d) & 1);
      moved |= (uint64_t)go << s;
      if (go) st(&nb->vals[s], v[s]);
      st(&nb->keys[s], go ? k[s] : (uint64_t)defaultKey);
    }
    st(&nb->ctl, ctl_of(home, d + 1));
    __builtin_amdgcn_s_waitcnt(0);  // the new bucket is whole before it is published
    st(reinterpret_cast<uint64_t*>(&directory[home]), reinterpret_cast<uint64_t>(nb));
    // level only grows: a cached value at or above d + 1 needs no update
    if (ld_cached(&level) < d + 1)
      gallatin::utils::atomic_max(&level, (uint64_t)(d + 1));
    __builtin_amdgcn_s_waitcnt(0);
    st(&b->ctl, ctl_of(old_home, d + 1) | 1);  // still locked
    __builtin_amdgcn_s_waitcnt(0);  // new depth visible before keys leave
#pragma unroll
    for (int s = 0; s < items_per_bucket; ++s)
      if ((moved >> s) & 1) st(&b->keys[s], (uint64_t)defaultKey);
    return true;
  }

  // Insert (or replace) the pair of every lane with `put`, remove the key of
  // every other; true when stored or found.  The operations of a wave run
  // together, whichever they are, so that the lanes can read buckets together
  // (scan); a lane that is done stays in the loop for the others.
  __device__ bool update(bool put, Key key, Val val) {
    const bool valid = !put || ((uint64_t)key != (uint64_t)defaultKey &&
                                (uint64_t)key != (uint64_t)tombstoneKey);
    const uint64_t h = hash(key);
    int state = valid ? 0 : 3;  // 0 pending, 1 done, 2 refused or absent, 3 not a key
    bucket* b = nullptr;
    bool fresh = false;
    uint32_t losses = 0;
    for (uint32_t tries = 0; __ballot(state == 0) && tries < kTries; ++tries) {
      uint64_t ctl = 0;
      bool held = false;
      if (state == 0) {
        if (!b) {
          b = owner(h, fresh);
          fresh = true;
        }
        if (!b)
          state = 2;
        else
          held = try_lock(b, ctl);
      }
      const bool none = __ballot(held) == 0;  // the wave got no lock this time
      int match, free_slot;
      uint64_t seen;
      scan(held, b, (uint64_t)key, seen, match, free_slot);
      if (held) {
        if (!owns(ctl, h)) {
          unlock(b, ctl);
          b = nullptr;  // split since the look-up: look again
          continue;
        }
        if (match >= 0) {
          if (put)
            st(&b->vals[match], (uint64_t)val);
          else
            st(&b->keys[match], (uint64_t)defaultKey);
          state = 1;
        } else if (!put) {
          state = 2;
        } else if (free_slot >= 0) {
          st(&b->vals[free_slot], (uint64_t)val);
          __builtin_amdgcn_s_waitcnt(0);  // value before key
          st(&b->keys[free_slot], (uint64_t)key);
          state = 1;
        } else if (depth_of(ctl) < max_bits && split(b, depth_of(ctl), home_of(ctl))) {
          ctl = ctl_of(home_of(ctl), depth_of(ctl) + 1);  // full: split, try again
        } else {
          state = 2;
        }
        unlock(b, ctl);
        if (state == 0) b = nullptr;
      } else if (state == 0) {
        // Locked: the same bucket again, and after a few passes in which
        // another wave kept this one from every lock, look up again: that
        // keeps the waiting lanes off the word that the holder has to unlock
        // (trying the same bucket until its word shows a split, 512 inserts of
        // one key take 3.5 ms, not 1.6).  A lane that only waits for lanes of
        // its own wave has nobody to make room for, and its look-up would hold
        // them up: 64 inserts of one key 165 us with look-ups there, now 132;
        // 256 keys in about 18 buckets 71, now 62; 1,000 keys 54, now 50.
        if ((none && ++losses > kSameBucket) || !owns(ctl, h)) b = nullptr;
        __builtin_amdgcn_s_sleep(2);
      }
    }
    if (put && (state == 0 || state == 2)) gallatin::utils::atomic_add(&failed, (uint64_t)1);
    return state == 1;
  }

  // extendible_ht.cuh:842-1115.  Insert or replace; false when the table
  // cannot hold the key.
  __device__ bool insert(Key key, Val val) { return update(true, key, val); }

  // Remove key; true if it was present.  (No counterpart in the reference.)
  __device__ bool remove(Key key) { return update(false, key, Val{}); }

  // extendible_ht.cuh:1291-1375.  The control word and the keys are loaded
  // together; a missing key is reported only if the depth is unchanged
  // when looked at again after the keys (a split raises the depth before
  // it clears moved keys), and a found key's value is taken only if the
  // key is still in its slot after the value was read.
  __device__ bool query(Key key, Val& val) {
    const uint64_t h = hash(key);
    bool pending = true, found = false;
    for (uint32_t tries = 0; __ballot(pending) && tries < kTries; ++tries) {
      bucket* b = nullptr;
      if (pending) {
        b = owner(h, tries > 0);
        pending = b != nullptr;
      }
      uint64_t ctl;
      int match, empty;
      scan(pending, b, (uint64_t)key, ctl, match, empty);
      if (!pending || !owns(ctl, h)) continue;  // being split: look again
      if (match >= 0) {
        const uint64_t v = ld(&b->vals[match]);
        __builtin_amdgcn_s_waitcnt(0);  // the value is read before the key is read again
        // Between the two reads the key may have left the slot (moved by a
        // split or removed) and another insert may have reused it, value
        // first: the value belongs to the key only if the key is still there.
        if (ld(&b->keys[match]) == (uint64_t)key) {
          val = (Val)v;
          found = true;
          pending = false;
        }
      } else if (depth_of(ld(&b->ctl)) == depth_of(ctl)) {
        pending = false;
      }
    }
    return found;
  }
};

}  // namespace data_structs
}  // namespace gallatin

#endif
