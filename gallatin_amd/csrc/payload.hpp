// Payload fill and verify of the churn kernels.  Included inside an anonymous
// namespace of each source that uses it.
#ifndef GALLATIN_AMD_PAYLOAD_HPP
#define GALLATIN_AMD_PAYLOAD_HPP

// Payload fill and verify, spread over the whole wave: the buffers of the
// participating lanes are cut into 16-byte chunks numbered buffer after
// buffer (lane order), and lane r handles chunks r, r + 64, r + 128, ...
// Needs all 64 lanes of the wave active.
//
// The owner of a chunk comes from a map in LDS, made once per fill or verify:
// a bit per chunk that is set on each buffer's last one, and the buffers'
// addresses and patterns in order.  For 64 consecutive chunks the owners are
// the set bits below each lane's (v_mbcnt on one uniform word), and one
// 16-byte LDS read then gives address and pattern: two LDS reads per chunk.
// A binary search over the lanes' chunk prefixes took eleven ds_bpermute per
// chunk, six of them one after another, and kept the LDS pipes busy for about
// half of a round of the batched churn: with it a launch of 2^24 threads of
// ten rounds took 22.9 ms, now 21.1 (4.6 TB/s of HBM
// traffic, where a copy of scattered 2 KiB pieces reaches 4.9).
//
// A buffer of w words (w = ceil(size / 8)) lives in a slice whose size is a
// multiple of 16 bytes and at least 8 * w, so for odd w the slice extends at
// least 8 bytes past the last word: every chunk is accessed as one aligned
// 16-byte vector, and the verify ignores the upper half of a buffer's last
// chunk when w is odd.  Accesses go through global-address-space pointers
// (global_load / global_store), so stores never hold up the LDS waits, and
// the verify keeps kVerifyDepth loads per lane in flight.
typedef unsigned long long u64x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(1))) u64x2 global_u64x2;

constexpr int kVerifyDepth = 8;
constexpr uint32_t kMaxChunks = 256;  // of one buffer: 4096 bytes

// One wave's map of a fill or verify.
struct chunk_map {
  u64x2 own[64];            // r-th buffer: address - 16 * its first chunk's number, with bit 0
                            // set when its word count is odd; pattern
  uint64_t last[kMaxChunks];  // bit c % 64 of word c / 64: chunk c ends its buffer
};

// LDS operations of a wave run in order; this keeps the compiler to it.
__device__ __forceinline__ void wave_lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Inclusive sum over the lanes up to this one, all 64 active.
__device__ __forceinline__ uint32_t wave_prefix(uint32_t v) {
  int x = (int)v;
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, true);   // row_shr:1
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, true);   // row_shr:2
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, true);   // row_shr:4
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, true);   // row_shr:8
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);  // row_bcast:15
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);  // row_bcast:31
  return (uint32_t)x;
}

// Fills the map; returns the wave's chunks.
__device__ inline uint32_t map_chunks(chunk_map& m, bool on, const void* p, uint64_t words,
                                      uint64_t pat) {
  const uint32_t n = on ? (uint32_t)((words + 1) / 2) : 0u;
  const uint32_t upto = wave_prefix(n);
  const uint32_t total = wave::readlane(upto, 63);
  const uint32_t lane = wave::lane();
  for (uint32_t i = lane; 64 * i < total; i += 64) m.last[i] = 0;
  wave_lds_order();
  const uint64_t owners = __ballot(n != 0);
  if (n) {
    const uint64_t end = upto - 1;
    atomicOr((unsigned long long*)&m.last[end >> 6], 1ULL << (end & 63));
    m.own[wave::count(owners & wave::lanes_below())] =
        u64x2{((uint64_t)p - 16ULL * (upto - n)) | (words & 1), pat};
  }
  wave_lds_order();
  return total;
}

// Buffers ended before this lane's chunk among the 64 of `ends`.
__device__ __forceinline__ uint32_t ended_below(uint64_t ends) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(ends >> 32),
                                   __builtin_amdgcn_mbcnt_lo((uint32_t)ends, 0u));
}

__device__ inline void wave_fill(chunk_map& m, bool on, uint64_t* p, uint64_t words,
                                 uint64_t pat) {
  const uint32_t total = map_chunks(m, on, p, words, pat);
  const uint32_t lane = wave::lane();
  uint32_t before = 0;  // buffers ended before `base`
  for (uint32_t base = 0; base < total; base += 64) {
    const uint64_t ends = wave::readfirst(m.last[base >> 6]);
    const uint32_t c = base + lane;
    if (c < total) {
      const u64x2 o = m.own[before + ended_below(ends)];
      const uint64_t a = (o.x & ~1ULL) + 16ULL * c;
      *reinterpret_cast<global_u64x2*>(a) = u64x2{o.y, o.y};
    }
    before += wave::count(ends);
  }
  wave_lds_order();
}

// Returns this lane's share of the mismatching words.
__device__ inline uint32_t wave_verify(chunk_map& m, bool on, const uint64_t* p, uint64_t words,
                                       uint64_t pat) {
  const uint32_t total = map_chunks(m, on, p, words, pat);
  const uint32_t lane = wave::lane();
  uint32_t bad = 0, before = 0;
  for (uint32_t base = 0; base < total; base += 64 * kVerifyDepth) {
    uint64_t v[kVerifyDepth];
    uint32_t half = 0;  // bit k: only the lower word of chunk k counts
    u64x2 x[kVerifyDepth];
#pragma unroll
    for (int k = 0; k < kVerifyDepth; ++k) {
      const uint32_t c = base + 64u * k + lane;
      // past the last chunk: the last word again, which no lane uses
      const uint32_t at = base + 64u * k < total ? base + 64u * k : total - 1;
      const uint64_t ends = wave::readfirst(m.last[at >> 6]);
      if (c < total) {
        const u64x2 o = m.own[before + ended_below(ends)];
        v[k] = o.y;
        half |= ((uint32_t)o.x & (uint32_t)(ends >> lane) & 1u) << k;
        x[k] = *reinterpret_cast<const global_u64x2*>((o.x & ~1ULL) + 16ULL * c);
      }
      before += wave::count(ends);
    }
#pragma unroll
    for (int k = 0; k < kVerifyDepth; ++k)
      if (base + 64u * k + lane < total)
        bad += (x[k].x != v[k]) + (!((half >> k) & 1) && x[k].y != v[k]);
  }
  wave_lds_order();
  return bad;
}

#endif
