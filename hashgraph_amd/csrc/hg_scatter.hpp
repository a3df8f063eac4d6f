// hg_scatter.hpp -- one tile of a partition pass with at most BLOCK buckets.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>
#include "hg_common.hpp"
#include "hg_device.hpp"

namespace hg {

template <typename K>
__host__ __device__ constexpr uint32_t scatter_tile_keys(int block) {
  return (uint32_t)block * (sizeof(K) == 4 ? 16 : 8);
}

// 44 KB (64-bit keys) or 53 KB at 512 threads: three workgroups share a CU, and
// one's loads and stores run under another's LDS phases.
template <typename K, int BLOCK>
struct ScatterLds {
  K key[scatter_tile_keys<K>(BLOCK)];
  uint16_t bkt[scatter_tile_keys<K>(BLOCK)];
  uint32_t cnt[BLOCK], adj[BLOCK];
  uint32_t tmp[BLOCK / 64 + 1];
};

// The cnt keys from keys[k0] on: ranked with LDS atomics, staged bucket by
// bucket in LDS and written run by run.  bucket(key) < ncols <= BLOCK;
// take(c) gives thread b the place of bucket b's run of c keys (called by
// threads b < ncols, its result used only after the staging, so that a
// global reservation's latency is hidden).
// dst(b) is the array that bucket b's places count in.
// PACK: the keys are 32-bit and the output 8-byte records (position << 32 | key).
template <typename K, int BLOCK, bool PACK, typename DST, typename BUCKET, typename TAKE>
__device__ __forceinline__ void scatter_tile(const void *__restrict__ keys, uint64_t k0, uint32_t cnt, uint32_t ncols,
                                             ScatterLds<K, BLOCK> &s, DST dst, BUCKET bucket, TAKE take) {
  constexpr int KPT = scatter_tile_keys<K>(BLOCK) / BLOCK;
  using IN = typename std::conditional<PACK, uint32_t, K>::type;
  const uint32_t b = threadIdx.x;
  const bool col = b < ncols;
  const __amdgpu_buffer_rsrc_t rs = make_rsrc((const IN *)keys + k0, cnt * (uint32_t)sizeof(IN));
  IN kr[KPT];
#pragma unroll
  for (int j = 0; j < KPT; j++)
    kr[j] = buf_load<IN>(rs, threadIdx.x * (uint32_t)sizeof(IN), j * BLOCK * (uint32_t)sizeof(IN));
  if (col) s.cnt[b] = 0;
  __syncthreads();
  uint32_t pk[KPT];
#pragma unroll
  for (int j = 0; j < KPT; j++) pk[j] = bucket(kr[j]);
#pragma unroll
  for (int j = 0; j < KPT; j++) {
    const bool valid = j * BLOCK + threadIdx.x < cnt;
    if (valid) pk[j] = (pk[j] << 16) | atomicAdd(&s.cnt[pk[j]], 1u);
  }
  __syncthreads();
  const uint32_t c = col ? s.cnt[b] : 0u;
  uint32_t place = 0;
  if (col) place = take(c);
  uint32_t tt;
  const uint32_t ex = block_exclusive_sum<BLOCK, uint32_t>(c, s.tmp, tt);
  if (col) s.cnt[b] = ex;
  __syncthreads();
#pragma unroll
  for (int j = 0; j < KPT; j++)
    if (j * BLOCK + threadIdx.x < cnt) {
      const uint32_t q = s.cnt[pk[j] >> 16] + (pk[j] & 0xFFFFu);
      if constexpr (PACK)
        s.key[q] = ((k0 + j * BLOCK + threadIdx.x) << 32) | kr[j];
      else
        s.key[q] = kr[j];
      s.bkt[q] = (uint16_t)(pk[j] >> 16);
    }
  if (col) s.adj[b] = place - ex;
  __syncthreads();
#pragma unroll
  for (int j = 0; j < KPT; j++) {
    const uint32_t q = j * BLOCK + threadIdx.x;
    if (q < cnt) {
      const uint32_t c = s.bkt[q];
      dst(c)[s.adj[c] + q] = s.key[q];
    }
  }
  __syncthreads();
}

}  // namespace hg
