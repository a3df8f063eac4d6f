// hg_final.hpp -- final stage of one bucket, shared by the per-bucket kernel
// and the one-workgroup build.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "hg_common.hpp"
#include "hg_device.hpp"

namespace hg {

// Leaves of a learned model a bucket-local kernel stages in LDS (the range
// between its smallest and largest key's leaves; wider ranges are read from
// global memory).
constexpr uint32_t RANGE_LEAVES = 512;

// Final-stage store of an index-carrying build of 32-bit keys (SPLIT): the
// 8-byte record (input position << 32 | key) goes to the CSR key array as its
// low half and to the position array as its high half.
__device__ __forceinline__ void split_store(uint32_t *keys, uint64_t *pos, uint64_t i, uint64_t rec) {
  keys[i] = (uint32_t)rec;
  pos[i] = rec >> 32;
}

// One workgroup's bucket (count <= BLOCK*KPT, count <= 65535, nbins <= 65535).
// Keys stay in VGPRs; the bucket-local bin (16 bit) is computed once and kept
// packed.  LDS (smem32, lds_bytes) holds nbins u16 counters (two per word);
// their exclusive scan gives the offsets, a second atomic pass gives every
// key's slot, then LDS is reused to stage the bin-ordered keys.  Every key is
// read before the first store, so csr may be part itself.
template <typename K, typename OFF, int BLOCK, int KPT, int HK, bool SPLIT = false>
__device__ __forceinline__ void final_bucket(const K *part, K *csr, OFF *__restrict__ off,
                                             const FinItem &it, const BinMap &mp, uint32_t *smem32, uint32_t lds_bytes,
                                             uint64_t *__restrict__ csr_index) {
  __shared__ uint32_t s_tmp[BLOCK / 64 + 1];
  const uint32_t W = it.nbins, cnt = it.count;
  const uint32_t nw = (W + 1) >> 1;
  for (uint32_t i = threadIdx.x; i < nw; i += BLOCK) smem32[i] = 0;
  __syncthreads();
  const K *kp = part + it.key_start;
  const uint32_t nv = cnt > threadIdx.x ? (cnt - threadIdx.x + BLOCK - 1) / BLOCK : 0;
  // slots below nfull are valid in every lane: a uniform (scalar) branch, so
  // no per-slot exec mask has to stay live across the unrolled loops
  const uint32_t nfull = cnt / BLOCK;
  const __amdgpu_buffer_rsrc_t rs = make_rsrc(kp, cnt * (uint32_t)sizeof(K));
  K kr[KPT];
  uint32_t lb[(KPT + 1) / 2];
#pragma unroll
  for (int j = 0; j < KPT; j++) kr[j] = buf_load<K>(rs, threadIdx.x * (uint32_t)sizeof(K), j * BLOCK * (uint32_t)sizeof(K));
#pragma unroll
  for (int j = 0; j < (KPT + 1) / 2; j++) lb[j] = 0;
  // a learned model: bins from the leaves this bucket's keys reach, copied
  // to LDS (one or a few leaves on most buckets)
  __shared__ RmiLeaf s_leaf[HK == HK_RMI ? RANGE_LEAVES : 1];
  if (HK == HK_RMI)
    rmi_local_bins<K, BLOCK, KPT>(kr, nv, lb, mp.rmi, s_leaf, RANGE_LEAVES, (uint32_t)it.bin_lo, mp.M);
  auto count_slot = [&](int j) {
    uint32_t l;
    if (HK == HK_RMI) {
      l = (lb[j >> 1] >> ((j & 1) * 16)) & 0xFFFFu;
    } else {
      l = bin_of<K, HK>(kr[j], mp) - (uint32_t)it.bin_lo;
      lb[j >> 1] |= l << ((j & 1) * 16);
    }
    atomicAdd(&smem32[l >> 1], 1u << ((l & 1) * 16));
  };
#pragma unroll
  for (int j = 0; j < KPT; j++) {
    if (__builtin_amdgcn_readfirstlane(j < (int)nfull)) count_slot(j);
    else if (j < nv) count_slot(j);
  }
  __syncthreads();
  // exclusive scan of the u16 counts (bucket total <= 65535, so every
  // prefix fits 16 bits and the packed halves never carry into each other)
  {
    const uint32_t per = (nw + BLOCK - 1) / BLOCK;
    const uint32_t w0 = min(threadIdx.x * per, nw), w1 = min(w0 + per, nw);
    uint32_t s = 0;
    for (uint32_t w = w0; w < w1; w++) {
      const uint32_t v = smem32[w];
      s += (v & 0xFFFFu) + (v >> 16);
    }
    uint32_t tot;
    uint32_t ex = block_exclusive_sum<BLOCK, uint32_t>(s, s_tmp, tot);
    for (uint32_t w = w0; w < w1; w++) {
      const uint32_t v = smem32[w];
      const uint32_t lo = v & 0xFFFFu;
      smem32[w] = ex | ((ex + lo) << 16);
      ex += lo + (v >> 16);
    }
  }
  __syncthreads();
  const uint64_t obase = it.key_start - it.key_rel;
  for (uint32_t l = threadIdx.x; l < W; l += BLOCK) {
    const uint32_t pre = (smem32[l >> 1] >> ((l & 1) * 16)) & 0xFFFFu;
    off[it.off_pos + l] = (OFF)(obase + pre);
  }
  if (it.end_pos != ~0ull && threadIdx.x == 0) off[it.end_pos] = (OFF)(obase + cnt);
  __syncthreads();
  auto place_slot = [&](int j) {
    const uint32_t sh = (j & 1) * 16;
    const uint32_t l = (lb[j >> 1] >> sh) & 0xFFFFu;
    const uint32_t old = atomicAdd(&smem32[l >> 1], 1u << ((l & 1) * 16));
    const uint32_t pos = (old >> ((l & 1) * 16)) & 0xFFFFu;
    lb[j >> 1] = (lb[j >> 1] & ~(0xFFFFu << sh)) | (pos << sh);
  };
#pragma unroll
  for (int j = 0; j < KPT; j++) {
    if (__builtin_amdgcn_readfirstlane(j < (int)nfull)) place_slot(j);
    else if (j < nv) place_slot(j);
  }
  __syncthreads();
  K *st = (K *)smem32;
  const uint32_t cap = lds_bytes / sizeof(K);
  K *dst = csr + it.key_start;
  for (uint32_t r0 = 0; r0 < cnt; r0 += cap) {
    auto stage_slot = [&](int j) {
      const uint32_t q = ((lb[j >> 1] >> ((j & 1) * 16)) & 0xFFFFu) - r0;
      if (q < cap) st[q] = kr[j];
    };
#pragma unroll
    for (int j = 0; j < KPT; j++) {
      if (__builtin_amdgcn_readfirstlane(j < (int)nfull)) stage_slot(j);
      else if (j < nv) stage_slot(j);
    }
    __syncthreads();
    const uint32_t n = min(cap, cnt - r0);
    if constexpr (SPLIT) {
      uint32_t *dk = (uint32_t *)csr + it.key_start;
      uint64_t *di = csr_index + it.key_start;
      for (uint32_t q = threadIdx.x; q < n; q += BLOCK) split_store(dk, di, r0 + q, st[q]);
    } else {
      for (uint32_t q = threadIdx.x; q < n; q += BLOCK) dst[r0 + q] = st[q];
    }
    __syncthreads();
  }
}

}  // namespace hg
