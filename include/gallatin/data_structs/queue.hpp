// Allocator-backed multi-producer multi-consumer FIFO queue (queue.cuh:59-192)
// and the ring of queues built on it (queue.cuh:196-253).
//
// Nodes come from the backing allocator (`allocator->malloc` / `->free`, as
// in the reference).  The list always starts with a dummy node: enqueue
// appends after the last node; dequeue reads the item of the node after the
// dummy, swings `head` to it (which becomes the dummy) and frees the old
// dummy at once.
//
// The reference links nodes with plain pointers and frees dequeued nodes at
// once, so a dequeuer that read `head` before another dequeuer freed and
// re-linked the same node can swing `head` to a node that is gone (ABA),
// and a queue emptied to one node can have `tail` left on a freed node.
// Here `head` is a tagged word, (count << 48) | address, and each update
// bumps the count, so a stale compare-and-swap fails.  A node another
// dequeuer freed may still be read before such a compare-and-swap fails; its
// memory stays in the allocator's pool (it is never unmapped), and an
// address read from it is used only if it could be a node of the pool.  Node
// words are read and written with device-coherent atomics, since producers
// and consumers may run on different XCDs.  Every retry loop is bounded.
//
// Lanes of one wave that work on the same queue act as one, where the
// reference makes every lane compete for the same word:
//  - Enqueues append one chain of nodes: one exchange of `tail` takes the
//    place at the end, then the node that was last gets its link.  No wave
//    ever retries.  A node is freed only after its link is written and
//    `head` has moved past it, so the link always goes to a live node and
//    `tail` never names a freed one.  A dequeuer that finds no link after the
//    last node it reached, while `tail` names another node, waits for it.
//  - Dequeues take as many nodes as the group has lanes with one
//    compare-and-swap of `head`.  The nodes of a chain usually are evenly
//    spaced slices (one claim of its wave's malloc, every lane or every n-th
//    of it), and a link says how many nodes follow the one it leads to at
//    which spacing, so 64 nodes are found with one load.  Items are read after the compare-and-swap, when
//    the nodes belong to the group; only the last one, the new dummy, may be
//    left by another dequeue meanwhile, so it is freed by whichever of the
//    two comes second (a bit of its link word tells).
//  - A group that lost a compare-and-swap takes a ticket and waits, without
//    touching `head`, until few tickets before it are open.  The ticket only
//    spares the words: the compare-and-swap alone decides, and the wait is
//    bounded.
//
// What bounds it: one word takes 88 M device atomics/s, and a dequeue by a
// wave is the chain head -> link -> compare-and-swap, about 1.6 us, after
// the one before it.  65,003 items of 8 bytes, enqueued and then dequeued by
// 1,016 waves: 0.04 and 1.6 ms.  With a compare-and-swap of the last node's
// link for enqueues and a walk node by node for dequeues it was 88 and
// 17.9 ms; without the tickets the dequeues take 6.8 ms, and with 1, 3 or 16
// tickets open instead of 8, 2.6, 1.75 and 1.55 ms.
#ifndef GALLATIN_QUEUE_HPP
#define GALLATIN_QUEUE_HPP

#include <hip/hip_runtime.h>

#include "gallatin/allocators/alloc_utils.hpp"

namespace gallatin {
namespace data_structs {

// head: (update count << 48) | address.  A node's link: the address of the
// next node (0: none yet), how many evenly spaced nodes follow that one (bits
// 48..53) and their spacing in slices (bits 54..62), and kLeft, set in the
// link of a node taken as the last of a group by the first of its two
// leavers.
namespace tagged {
constexpr uint64_t kAddrMask = (1ULL << 48) - 1;
constexpr uint64_t kLeft = 1ULL << 63;
__device__ __forceinline__ uint64_t addr(uint64_t w) { return w & kAddrMask; }
__device__ __forceinline__ uint64_t count(uint64_t w) { return w >> 48; }
constexpr uint32_t kMaxStep = 511;
__device__ __forceinline__ uint32_t run(uint64_t w) { return (uint32_t)(w >> 48) & 63u; }
__device__ __forceinline__ uint32_t step(uint64_t w) { return (uint32_t)(w >> 54) & kMaxStep; }
__device__ __forceinline__ uint64_t make(uint64_t a, uint64_t c) {
  return (a & kAddrMask) | (c << 48);
}
}  // namespace tagged

// queue.cuh:19-43.  `item` is kept in 8-byte words.
template <typename T>
struct queue_node {
  static constexpr int kWords = (int)((sizeof(T) + 7) / 8);
  uint64_t next;
  uint64_t words[kWords];

  __device__ void store_item(const T& v) {
    uint64_t tmp[kWords] = {};
    __builtin_memcpy(tmp, &v, sizeof(T));
    for (int i = 0; i < kWords; ++i) gallatin::utils::atomic_store(&words[i], tmp[i]);
  }
  __device__ T load_item() {
    uint64_t tmp[kWords];
    for (int i = 0; i < kWords; ++i) tmp[i] = gallatin::utils::atomic_load(&words[i]);
    T v;
    __builtin_memcpy(&v, tmp, sizeof(T));
    return v;
  }
};

template <typename queue_type, typename allocator>
__global__ void queue_init_kernel(queue_type* q, allocator* a, uint32_t* ok) {
  if (blockIdx.x == 0 && threadIdx.x == 0) *ok = q->init(a) ? 1u : 0u;
}

template <typename queue_type>
__global__ void queue_teardown_kernel(queue_type* q) {
  if (blockIdx.x == 0 && threadIdx.x == 0) q->teardown();
}

template <typename T, typename allocator>
struct queue {
  using my_type = queue<T, allocator>;
  using node = queue_node<T>;
  static constexpr uint32_t kTries = 1u << 20;

  // dequeues and enqueues work on words of different cache lines
  alignas(128) uint64_t head;  // tagged; the dummy
  uint32_t gate_next;          // tickets given to groups that lost a compare-and-swap
  uint32_t gate_done;          // tickets whose group is through
  alignas(128) uint64_t tail;  // address of the last node
  alignas(128) allocator* my_backing_allocator;
  uint64_t pool_lo, pool_hi;  // the allocator's pool, for address checks
  uint64_t stride;            // bytes of a slice of a node's size class (a power of two)

  // queue.cuh:72-81.  Returns nullptr on failure.
  static __host__ my_type* generate_on_device(allocator* backing_allocator) {
    my_type* dev = nullptr;
    uint32_t* ok = nullptr;
    if (hipMalloc(&dev, sizeof(my_type)) != hipSuccess) return nullptr;
    if (hipMalloc(&ok, sizeof(uint32_t)) != hipSuccess) {
      (void)hipFree(dev);
      return nullptr;
    }
    queue_init_kernel<my_type, allocator><<<1, 1>>>(dev, backing_allocator, ok);
    uint32_t h = 0;
    const bool good = hipMemcpy(&h, ok, sizeof(h), hipMemcpyDeviceToHost) == hipSuccess && h;
    (void)hipFree(ok);
    if (!good) {
      (void)hipFree(dev);
      return nullptr;
    }
    return dev;
  }

  // Frees every node left in the queue and the queue object.
  static __host__ void free_on_device(my_type* dev) {
    if (!dev) return;
    queue_teardown_kernel<my_type><<<1, 1>>>(dev);
    (void)hipDeviceSynchronize();
    (void)hipFree(dev);
  }

  // queue.cuh:83-88, with the dummy node.
  __device__ bool init(allocator* a) {
    my_backing_allocator = a;
    pool_lo = (uint64_t)a->memory;
    pool_hi = pool_lo + (a->num_segments << a->seg_shift);
    stride = a->smallest;
    while (stride < sizeof(node)) stride *= 2;
    node* d = static_cast<node*>(a->malloc(sizeof(node)));
    if (!d) return false;
    // no group took the first dummy: its only leaver is the first dequeue
    gallatin::utils::atomic_store(&d->next, tagged::kLeft);
    __builtin_amdgcn_s_waitcnt(0);
    gate_next = gate_done = 0;
    head = tagged::make((uint64_t)d, 0);
    tail = (uint64_t)d;
    return true;
  }

  __device__ void teardown() {
    uint64_t h = tagged::addr(head);
    while (h) {
      node* n = reinterpret_cast<node*>(h);
      h = tagged::addr(n->next);
      my_backing_allocator->free(n);
    }
    head = tail = 0;
  }

  // An address that may be a node: inside the pool, with room for a whole
  // node, and aligned as every slice is (16 bytes).
  __device__ __forceinline__ bool in_pool(uint64_t a) const {
    return a >= pool_lo && a <= pool_hi - sizeof(node) && (a & 15) == 0;
  }

  // queue.cuh:90-135.  False when no node could be allocated.  The lanes of
  // a wave that enqueue into this queue together link their nodes into one
  // chain in lane order; one lane takes the end of the queue for the chain
  // with an exchange of `tail` and links the node that was there to it.
  __device__ bool try_enqueue(T item) {
    node* nd = static_cast<node*>(my_backing_allocator->malloc(sizeof(node)));
    const bool have = nd != nullptr;
    const uint64_t group = gallatin::wave::match(__ballot(have), have, (uint64_t)this);
    if (!have) return false;
    nd->store_item(item);
    const uint64_t below = gallatin::wave::lanes_below();
    const uint64_t above = group & ~below & ~(1ULL << gallatin::wave::lane());
    const int me = (int)gallatin::wave::lane();
    const int leader = gallatin::wave::first(group);
    const int last = 63 - __builtin_clzll(group);
    const int next_lane = above ? gallatin::wave::first(above) : me;
    const uint64_t succ = gallatin::wave::fetch((uint64_t)nd, next_lane);
    // the spacing of the first two nodes, and the nodes that follow this one
    // at it: up to the first lane whose successor lies elsewhere (the last
    // lane has none)
    const uint64_t gap = gallatin::wave::fetch(succ - (uint64_t)nd, leader);
    const uint64_t step = gap >> __builtin_ctzll(stride);
    const bool even = step >= 1 && step <= tagged::kMaxStep && step * stride == gap;
    const uint64_t ends =
        group & ~__ballot(above && even && succ - (uint64_t)nd == gap) & ~below;
    const uint32_t run =
        gallatin::wave::count(group & ~below & ((1ULL << gallatin::wave::first(ends)) - 1));
    const uint64_t tag = run ? run | (step << 6) : 0;
    const uint64_t succ_tag = gallatin::wave::fetch(tag, next_lane);
    gallatin::utils::atomic_store(&nd->next, above ? tagged::make(succ, succ_tag) : (uint64_t)0);
    __builtin_amdgcn_s_waitcnt(0);  // every node of the chain is complete before it is linked
    const uint64_t last_node = gallatin::wave::fetch((uint64_t)nd, last);
    if (me == leader) {
      const uint64_t before = gallatin::utils::atomic_exch(&tail, last_node);
      gallatin::utils::atomic_or(&reinterpret_cast<node*>(before)->next,
                                 tagged::make((uint64_t)nd, tag));
    }
    return true;
  }

  __device__ void enqueue(T item) { (void)try_enqueue(item); }

  // Waits about n / 10 microseconds.
  static __device__ __forceinline__ void pause(uint32_t n) {
    for (uint32_t i = 0; i < n; ++i) __builtin_amdgcn_s_sleep(4);
  }

  static constexpr int32_t kGateOpen = 8;       // groups with a ticket that may compete
  static constexpr uint32_t kGatePolls = 4096;  // polls after which a group competes anyway

  // The second of the two leavers of node `a` frees it.
  static __device__ __forceinline__ bool leave(uint64_t a) {
    return (gallatin::utils::atomic_or(&reinterpret_cast<node*>(a)->next, tagged::kLeft) &
            tagged::kLeft) != 0;
  }

  // queue.cuh:139-187.  False when the queue is empty.  Lanes of a group
  // that got no node look again until the group sees the queue empty.
  __device__ bool dequeue(T& return_val) {
    // A wave may hold groups of several queues: values are broadcast from a
    // group's leader, so every branch is uniform within the group.
    bool pending = true, took = false, is_last = false, ticketed = false, open = true;
    uint64_t mine = 0, dummy = 0;  // the node taken; for the last one, the dummy left
    uint32_t ticket = 0, polls = 0;
    uint64_t h = gallatin::utils::atomic_load(&head);
    for (uint32_t tries = 0; tries < kTries && __ballot(pending); ++tries) {
      const uint64_t group = gallatin::wave::match(__ballot(pending), pending, (uint64_t)this);
      if (!pending) continue;
      const int leader = gallatin::wave::first(group);
      const bool leads = (int)gallatin::wave::lane() == leader;
      if (!open) {
        const uint32_t done =
            gallatin::wave::fetch(gallatin::utils::atomic_load(&gate_done), leader);
        const int32_t ahead = (int32_t)(ticket - done);
        if (ahead >= kGateOpen && ++polls < kGatePolls) {
          // groups of other queues in this wave stand still meanwhile
          const bool alone = __ballot(1) == group;
          pause(!alone ? 1u : ahead < 32 ? 8u * (uint32_t)ahead : 256u);
          continue;
        }
        open = true;
        h = gallatin::utils::atomic_load(&head);
      }
      const uint32_t k = gallatin::wave::count(group);
      const uint32_t rank = gallatin::wave::count(group & gallatin::wave::lanes_below());
      h = gallatin::wave::fetch(h, leader);
      // Find up to k nodes: `base` is the last one reached, m are found.  What
      // is read of nodes that another dequeue freed meanwhile makes the
      // compare-and-swap fail, whatever it says.
      uint64_t base = tagged::addr(h);
      uint32_t m = 0;
      bool end = false, stale = false;
      while (m < k && !end && !stale) {
        const uint64_t link = gallatin::wave::fetch(
            gallatin::utils::atomic_load(&reinterpret_cast<node*>(base)->next), leader);
        const uint64_t a = tagged::addr(link);
        if (a == 0) {
          end = true;
          continue;
        }
        const uint32_t more = tagged::run(link) < k - m - 1 ? tagged::run(link) : k - m - 1;
        const uint64_t by = stride * tagged::step(link), e = a + by * more;
        stale = !in_pool(a) || !in_pool(e);
        if (stale) continue;
        if (rank >= m && rank <= m + more) mine = a + by * (rank - m);
        m += more + 1;
        base = e;
      }
      bool through = false;  // this look settled something
      if (stale || m == 0) {
        const uint64_t t = gallatin::wave::fetch(gallatin::utils::atomic_load(&tail), leader);
        __builtin_amdgcn_s_waitcnt(0);  // tail first: an unchanged head then dates both
        const uint64_t h2 = gallatin::wave::fetch(gallatin::utils::atomic_load(&head), leader);
        if (!stale && h2 == h && t == tagged::addr(h)) {  // empty
          pending = false;
          through = true;
        } else if (h2 == h) {  // the next chain's link is on its way
          __builtin_amdgcn_s_sleep(1);
        }
        h = h2;
      } else {
        const uint64_t moved = tagged::make(base, tagged::count(h) + 1);
        uint64_t seen = 0;
        if (leads) seen = gallatin::utils::atomic_cas(&head, h, moved);
        seen = gallatin::wave::fetch(seen, leader);
        if (seen == h) {
          if (rank < m) {
            took = true;
            pending = false;
            is_last = rank + 1 == m;
            dummy = tagged::addr(h);
          }
          h = moved;
          through = true;
        } else {
          h = seen;
          if (!ticketed) {
            if (leads) ticket = gallatin::utils::atomic_add(&gate_next, 1u);
            ticket = gallatin::wave::fetch(ticket, leader);
            ticketed = true;
            open = false;
            polls = 0;
          }
        }
      }
      if (through && ticketed) {
        if (leads) gallatin::utils::atomic_add(&gate_done, 1u);
        ticketed = false;
        open = true;
      }
    }
    if (ticketed) {  // out of tries: the ticket is given back all the same
      const uint64_t group = gallatin::wave::match(__ballot(1), true, (uint64_t)this);
      if ((int)gallatin::wave::lane() == gallatin::wave::first(group))
        gallatin::utils::atomic_add(&gate_done, 1u);
    }
    if (took) return_val = reinterpret_cast<node*>(mine)->load_item();
    __builtin_amdgcn_s_waitcnt(0);  // the items are read before their nodes are freed
    // the group's nodes but the last are its own; its last node and the
    // dummy before its first one are left, each by the second leaver
    uint64_t out[2] = {0, 0};
    if (took && !is_last) out[0] = mine;
    if (took && is_last) {
      if (leave(dummy)) out[0] = dummy;
      if (leave(mine)) out[1] = mine;
    }
    for (int i = 0; i < 2; ++i)
      if (out[i]) my_backing_allocator->free(reinterpret_cast<node*>(out[i]));
    return took;
  }
};

template <typename queue_type>
__global__ void ring_init_kernel(queue_type* q, typename queue_type::alloc_type* a,
                                 uint32_t* ok) {
  if (blockIdx.x == 0 && threadIdx.x == 0) *ok = q->init(a) ? 1u : 0u;
}

// queue.cuh:196-253: `width` queues used round robin, one counter for
// enqueues and one for dequeues, to spread the contention of one queue.
template <typename T, int width, typename allocator>
struct circular_CAS_queue {
  using my_type = circular_CAS_queue<T, width, allocator>;
  using alloc_type = allocator;

  uint64_t malloc_counter;
  uint64_t free_counter;
  queue<T, allocator> queue_list[width];

  __device__ bool init(allocator* a) {
    malloc_counter = 0;
    free_counter = 0;
    for (int i = 0; i < width; ++i)
      if (!queue_list[i].init(a)) return false;
    return true;
  }

  static __host__ my_type* generate_on_device(allocator* a) {
    my_type* dev = nullptr;
    uint32_t* ok = nullptr;
    if (hipMalloc(&dev, sizeof(my_type)) != hipSuccess) return nullptr;
    if (hipMalloc(&ok, sizeof(uint32_t)) != hipSuccess) {
      (void)hipFree(dev);
      return nullptr;
    }
    ring_init_kernel<my_type><<<1, 1>>>(dev, a, ok);
    uint32_t h = 0;
    const bool good = hipMemcpy(&h, ok, sizeof(h), hipMemcpyDeviceToHost) == hipSuccess && h;
    (void)hipFree(ok);
    if (!good) {
      (void)hipFree(dev);
      return nullptr;
    }
    return dev;
  }

  __device__ void teardown() {
    for (int i = 0; i < width; ++i) queue_list[i].teardown();
  }

  static __host__ void free_on_device(my_type* dev) {
    if (!dev) return;
    queue_teardown_kernel<my_type><<<1, 1>>>(dev);
    (void)hipDeviceSynchronize();
    (void)hipFree(dev);
  }

  __device__ bool try_enqueue(T item) {
    const uint64_t i = gallatin::utils::atomic_add(&malloc_counter, (uint64_t)1) % width;
    return queue_list[i].try_enqueue(item);
  }
  __device__ void enqueue(T item) { (void)try_enqueue(item); }

  // As in the reference, a dequeue looks at one queue only, so it can find
  // that queue empty while others hold items.
  __device__ bool dequeue(T& return_val) {
    const uint64_t i = gallatin::utils::atomic_add(&free_counter, (uint64_t)1) % width;
    return queue_list[i].dequeue(return_val);
  }
};

}  // namespace data_structs
}  // namespace gallatin

#endif
