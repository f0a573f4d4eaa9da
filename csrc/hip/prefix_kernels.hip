// prefix_kernels.hip — gfx950 kernels for the router's prefix-cache hot path.
//
// These are the MI355X-native replacement for the reference's CPU hot loops
// `approximateprefix/hashing.go:80-95` (chained xxhash over prompt blocks)
// and `approximateprefix/indexer.go:86-102` (hash -> pod-set longest-prefix
// match under RWMutex). Re-design for CDNA4:
//   * batched across the whole admission queue — one launch hashes and
//     matches EVERY queued request (the Go version is per-request serial);
//   * one 64-lane wave per request: contents are hashed and the table probed
//     lane-parallel, 64 blocks at a time; what follows block by block is
//     uniform over the wave and runs on the scalar unit, whose multiplies take
//     a quarter of the vector unit's time for one lane;
//   * the hash->endpoint-mask table is a device-resident open-addressing
//     table (sized for 288 GB HBM budgets) probed directly by the match
//     kernel.
// The chain of 64-bit multiplies bounds the hash. 48 prompts of 1000 tokens
// (62 blocks): hash 10.2 us, match 4.6; with chain and match on one vector lane
// and results cleared beforehand 16.8 and 20.3; 96 of 256 blocks: 35 and 5.3
// (52.8 and 72.4).
// The chain definition is shared bit-exactly with the CPU core via
// csrc/common/xxhash64.h.
#include "hip_common.h"
#include "../common/xxhash64.h"

using ldsr::block_content_hash;

namespace {

__device__ __forceinline__ uint64_t lane_value(uint64_t x, int lane) {
  const uint32_t lo = __builtin_amdgcn_readlane((int)(uint32_t)x, lane);
  const uint32_t hi = __builtin_amdgcn_readlane((int)(x >> 32), lane);
  return (uint64_t)hi << 32 | lo;
}

// chain_hash(content, prev) in two halves: what the content adds to the state,
// and what follows once the hash before it is known
__device__ __forceinline__ uint64_t chain_head(uint64_t content) {
  using namespace ldsr;
  const uint64_t h = (PRIME64_5 + 16) ^ xxh_round(0, content);
  return xxh_rotl64(h, 27) * PRIME64_1 + PRIME64_4;
}
__device__ __forceinline__ uint64_t chain_tail(uint64_t head, uint64_t prev) {
  using namespace ldsr;
  uint64_t h = head ^ xxh_round(0, prev);
  h = xxh_rotl64(h, 27) * PRIME64_1 + PRIME64_4;
  h = (h ^ (h >> 33)) * PRIME64_2;
  h = (h ^ (h >> 29)) * PRIME64_3;
  return h ^ (h >> 32);
}

// ---------------------------------------------------------------------------
// hash_prompts: one wave per request.
//  tokens:   flat int32 token buffer
//  offsets:  int64 [R+1] request start offsets into tokens
//  out:      uint64 [R, max_blocks] chained hashes, 0 behind the last
//  counts:   int32 [R] number of complete blocks hashed
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(WAVE) void hash_prompts_kernel(
    const int32_t* __restrict__ tokens, const int64_t* __restrict__ offsets,
    int block_tokens, int max_blocks, uint64_t seed0,
    uint64_t* __restrict__ out, int32_t* __restrict__ counts) {
  const int req = blockIdx.x, lane = threadIdx.x;
  const int64_t beg = offsets[req], end = offsets[req + 1];
  const int n_blocks =
      (int)min((end - beg) / block_tokens, (int64_t)max_blocks);
  if (lane == 0) counts[req] = n_blocks;
  uint64_t* dst = out + (int64_t)req * max_blocks;
  uint64_t prev = seed0;                       // uniform
  for (int b0 = 0; b0 < max_blocks; b0 += WAVE) {
    const int b = b0 + lane, n = min(n_blocks - b0, WAVE);
    uint64_t head = 0, mine = 0;
    if (lane < n)
      head = chain_head(block_content_hash(
          tokens + beg + (int64_t)b * block_tokens, block_tokens, seed0));
    for (int i = 0; i < n; ++i) {
      prev = chain_tail(lane_value(head, i), prev);
      if (lane == i) mine = prev;
    }
    if (b < max_blocks) dst[b] = mine;
  }
}

// ---------------------------------------------------------------------------
// Device hash table: open addressing, linear probing.
// keys[cap] (0 = empty; real hash 0 is remapped to 1), masks[cap].
// The host-side C++ PrefixIndex owns LRU policy; inserts/removals are
// mirrored here in batches.
// ---------------------------------------------------------------------------

__device__ __forceinline__ uint64_t norm_key(uint64_t h) { return h ? h : 1; }

__global__ void table_insert_kernel(uint64_t* __restrict__ keys,
                                    unsigned long long* __restrict__ masks,
                                    uint32_t cap_mask,  // cap-1, cap = 2^k
                                    const uint64_t* __restrict__ hashes,
                                    int64_t n, unsigned long long bit) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  uint64_t key = norm_key(hashes[i]);
  uint32_t slot = (uint32_t)key & cap_mask;
  for (uint32_t probe = 0; probe <= cap_mask; ++probe) {
    uint64_t prev = atomicCAS((unsigned long long*)&keys[slot], 0ULL,
                              (unsigned long long)key);
    if (prev == 0 || prev == key) {
      atomicOr(&masks[slot], bit);
      return;
    }
    slot = (slot + 1) & cap_mask;
  }
  // table full: drop (host monitors load factor and rebuilds)
}

__global__ void table_remove_kernel(const uint64_t* __restrict__ keys,
                                    unsigned long long* __restrict__ masks,
                                    uint32_t cap_mask,
                                    const uint64_t* __restrict__ hashes,
                                    int64_t n, unsigned long long bit) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  uint64_t key = norm_key(hashes[i]);
  uint32_t slot = (uint32_t)key & cap_mask;
  for (uint32_t probe = 0; probe <= cap_mask; ++probe) {
    uint64_t k = keys[slot];
    if (k == 0) return;  // not present
    if (k == key) {
      atomicAnd(&masks[slot], ~bit);
      return;
    }
    slot = (slot + 1) & cap_mask;
  }
}

__device__ __forceinline__ unsigned long long table_lookup(
    const uint64_t* __restrict__ keys,
    const unsigned long long* __restrict__ masks, uint32_t cap_mask,
    uint64_t key) {
  uint32_t slot = (uint32_t)key & cap_mask;
  for (uint32_t probe = 0; probe <= cap_mask; ++probe) {
    const uint64_t k = keys[slot];
    const unsigned long long mask = masks[slot];    // one wait for both
    if (k == 0) return 0;
    if (k == key) return mask;
    slot = (slot + 1) & cap_mask;
  }
  return 0;
}

// ---------------------------------------------------------------------------
// match_longest: one wave per request. Probes the table for 64 chain hashes at
// a time; the blocks that an endpoint holds are then the bits of a ballot.
//  hashes:  uint64 [R, max_blocks]
//  counts:  int32 [R]
//  out:     int32 [R, n_endpoints] consecutive matched blocks per endpoint
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(WAVE) void match_longest_kernel(
    const uint64_t* __restrict__ keys,
    const unsigned long long* __restrict__ masks, uint32_t cap_mask,
    const uint64_t* __restrict__ hashes, const int32_t* __restrict__ counts,
    int max_blocks, int n_endpoints, int32_t* __restrict__ out) {
  const int req = blockIdx.x, lane = threadIdx.x;
  const int n_blocks = min(counts[req], max_blocks);
  const uint64_t* h = hashes + (int64_t)req * max_blocks;
  // endpoints that hold every block so far (the table knows 64)
  unsigned long long active =
      n_endpoints >= 64 ? ~0ULL : (1ULL << n_endpoints) - 1;
  int mine = 0;                                // of endpoint `lane`
  for (int b0 = 0; b0 < n_blocks && active; b0 += WAVE) {
    unsigned long long holds = 0;
    if (b0 + lane < n_blocks)
      holds = table_lookup(keys, masks, cap_mask, norm_key(h[b0 + lane]));
    for (unsigned long long left = active; left; left &= left - 1) {
      const int e = __builtin_ctzll(left);
      const unsigned long long missing = ~__ballot((holds >> e) & 1);
      if (lane == e) mine = b0 + (missing ? __builtin_ctzll(missing) : WAVE);
      if (missing) active &= ~(1ULL << e);
    }
  }
  for (int e = lane; e < n_endpoints; e += WAVE)
    out[(int64_t)req * n_endpoints + e] = e < WAVE ? mine : 0;
}

}  // namespace

// ---- host-side launchers (called from the torch binding) ----

extern "C" {

hipError_t lds_hash_prompts(const int32_t* tokens, const int64_t* offsets,
                            int n_requests, int block_tokens, int max_blocks,
                            uint64_t seed0, uint64_t* out, int32_t* counts,
                            hipStream_t stream) {
  if (n_requests == 0) return hipSuccess;
  hipLaunchKernelGGL(hash_prompts_kernel, dim3(n_requests), dim3(WAVE), 0,
                     stream, tokens, offsets, block_tokens, max_blocks, seed0,
                     out, counts);
  HIP_CHECK_LAST();
  return hipSuccess;
}

hipError_t lds_table_update(uint64_t* keys, unsigned long long* masks,
                            uint32_t cap_mask, const uint64_t* hashes,
                            int64_t n, int endpoint, int is_remove,
                            hipStream_t stream) {
  if (n == 0) return hipSuccess;
  unsigned long long bit = 1ULL << endpoint;
  int threads = 256;
  int blocks = (int)((n + threads - 1) / threads);
  if (is_remove) {
    hipLaunchKernelGGL(table_remove_kernel, dim3(blocks), dim3(threads), 0,
                       stream, keys, masks, cap_mask, hashes, n, bit);
  } else {
    hipLaunchKernelGGL(table_insert_kernel, dim3(blocks), dim3(threads), 0,
                       stream, keys, masks, cap_mask, hashes, n, bit);
  }
  HIP_CHECK_LAST();
  return hipSuccess;
}

hipError_t lds_match_longest(const uint64_t* keys,
                             const unsigned long long* masks,
                             uint32_t cap_mask, const uint64_t* hashes,
                             const int32_t* counts, int n_requests,
                             int max_blocks, int n_endpoints, int32_t* out,
                             hipStream_t stream) {
  if (n_requests == 0) return hipSuccess;
  hipLaunchKernelGGL(match_longest_kernel, dim3(n_requests), dim3(WAVE), 0,
                     stream, keys, masks, cap_mask, hashes, counts, max_blocks,
                     n_endpoints, out);
  HIP_CHECK_LAST();
  return hipSuccess;
}

}  // extern "C"
