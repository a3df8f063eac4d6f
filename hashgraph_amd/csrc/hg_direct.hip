// hg_direct.hip -- gfx950 kernels for tables that need no partition pass.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "hg_common.hpp"
#include "hg_device.hpp"
#include "hg_final.hpp"
#include "hg_kernels.hpp"

namespace hg {

// ---------------------------------------------------------------------------
// One-workgroup build: the table is one bucket of the final stage, so the
// input keys are its bucket as they stand (no hash pass, no count matrix, no
// partitioned copy, no descriptors).  Bound by the launch and by the latency
// of one workgroup's phases: 1000 uint32 keys take 8 us (52 us through the
// partition pass and its 16 launches), 16384 keys 14 us (87 us).
// ---------------------------------------------------------------------------
template <typename K, typename OFF, int BLOCK, int KPT, int HK>
__global__ __launch_bounds__(BLOCK) void k_build_one(const K *keys, K *csr, OFF *__restrict__ off, uint32_t n,
                                                     uint32_t bin_lo, uint32_t nbins, BinMap mp, uint32_t lds_bytes) {
  extern __shared__ __align__(16) uint32_t smem32[];
  FinItem it;
  it.key_start = 0;
  it.key_rel = 0;
  it.off_pos = 0;
  it.end_pos = nbins;
  it.count = n;
  it.nbins = nbins;
  it.bin_lo = bin_lo;
  it.table = 0;
  final_bucket<K, OFF, BLOCK, KPT, HK>(keys, csr, off, it, mp, smem32, lds_bytes, nullptr);
}

// ---------------------------------------------------------------------------
// Direct probe: every thread hashes U probe keys, reads their bins' offsets
// and walks the bins in global memory; the probe keys are not partitioned.
// Bound by the latency of three dependent reads per key (probe key, offsets,
// bin), so the U reads of a step are all issued before the first is used, and
// from about 10^5 keys on by the lines those reads bring in: 2^20 uint32 keys
// against 2^20 take 49 us (105 us through the wide partition pass), about 22
// keys/ns beyond.
// Matches, and the keys of bins longer than PROBE_BIN_LIMIT (listed in `heavy`
// for the caller): one block scan and one reservation of each per workgroup.
//
// `st` (a DirectState, zero between calls) collects the counts; the last
// workgroup to finish stores them to `res` in pinned host memory and zeroes
// the state again, so a call needs no fill and no copy back.
// ---------------------------------------------------------------------------
struct DirectState {
  unsigned long long cursor;  // matches
  unsigned int heavy;         // keys listed
  unsigned int ticket;        // workgroups done
};
static_assert(sizeof(DirectState) <= DIRECT_STATE_BYTES, "DirectState");

template <typename OFF>
__device__ __forceinline__ void load_pair(const OFF *p, OFF &a, OFF &b) {
  OFF v[2];
  __builtin_memcpy(v, p, sizeof(v));  // one load (element alignment is enough on gfx950)
  a = v[0];
  b = v[1];
}

template <typename K, typename OFF, int BLOCK, int U, int HK>
__global__ __launch_bounds__(BLOCK) void k_probe_direct(const K *__restrict__ probe, uint32_t n, BinMap mp,
                                                        const OFF *__restrict__ offA, const K *__restrict__ keysA,
                                                        K *__restrict__ out, uint64_t capacity, K *__restrict__ heavy,
                                                        DirectState *__restrict__ st,
                                                        unsigned long long *__restrict__ res) {
  __shared__ uint32_t s_tmp[BLOCK / 64 + 1];
  __shared__ unsigned long long s_base;
  __shared__ uint32_t s_heavy;
  const uint32_t k0 = blockIdx.x * (BLOCK * U);
  const uint32_t cnt = min((uint32_t)(BLOCK * U), n - k0);
  const __amdgpu_buffer_rsrc_t rs = make_rsrc(probe + k0, cnt * (uint32_t)sizeof(K));
  K kr[U];
  OFF b0[U], b1[U];
  uint32_t m[U];
#pragma unroll
  for (int j = 0; j < U; j++) kr[j] = buf_load<K>(rs, threadIdx.x * (uint32_t)sizeof(K), j * BLOCK * (uint32_t)sizeof(K));
#pragma unroll
  for (int j = 0; j < U; j++) {
    const uint32_t l = bin_of<K, HK>(kr[j], mp);  // slots past cnt hold key 0: a valid bin
    load_pair(offA + l, b0[j], b1[j]);
  }
  uint32_t longest = 0, hm = 0;  // hm: slots whose key goes to the heavy list
#pragma unroll
  for (int j = 0; j < U; j++) {
    m[j] = 0;
    if (j * BLOCK + threadIdx.x >= cnt) b1[j] = b0[j];
    if (b1[j] - b0[j] > PROBE_BIN_LIMIT) {
      hm |= 1u << j;
      b1[j] = b0[j];
    }
    longest = max(longest, (uint32_t)(b1[j] - b0[j]));
  }
  // the U walks advance together, two keys of each bin per step
  for (uint32_t q = 0; q < longest; q += 2) {
    K v[U][2];
#pragma unroll
    for (int j = 0; j < U; j++)
#pragma unroll
      for (int i = 0; i < 2; i++) v[j][i] = b0[j] + q + i < b1[j] ? keysA[b0[j] + q + i] : (K)~kr[j];
#pragma unroll
    for (int j = 0; j < U; j++)
#pragma unroll
      for (int i = 0; i < 2; i++) m[j] += v[j][i] == kr[j] ? 1u : 0u;
  }
  uint32_t mine = 0;
#pragma unroll
  for (int j = 0; j < U; j++) mine += m[j];
  // one scan of both counts: at most 2^17 matches and 2^12 listed keys a workgroup
  static_assert(BLOCK * U * PROBE_BIN_LIMIT <= (1u << 17) && BLOCK * U < (1 << 14), "packed scan");
  uint32_t tot;
  const uint32_t ex = block_exclusive_sum<BLOCK, uint32_t>(mine | ((uint32_t)__popc(hm) << 18), s_tmp, tot);
  if (threadIdx.x == 0) {
    const uint32_t tm = tot & 0x3FFFFu, th = tot >> 18;
    s_base = tm ? atomicAdd(&st->cursor, (unsigned long long)tm) : 0ull;
    s_heavy = th ? atomicAdd(&st->heavy, th) : 0u;
  }
  __syncthreads();
  if (hm) {
    uint32_t w = s_heavy + (ex >> 18);
#pragma unroll
    for (int j = 0; j < U; j++)
      if ((hm >> j) & 1u) heavy[w++] = kr[j];
  }
  if (out != nullptr && mine && s_base < capacity) {
    unsigned long long w = s_base + (ex & 0x3FFFFu);
#pragma unroll
    for (int j = 0; j < U; j++)
      for (uint32_t r = 0; r < m[j]; r++, w++)
        if (w < capacity) out[w] = kr[j];
  }
  if (threadIdx.x == 0) {
    __threadfence();  // this workgroup's adds before its ticket
    if (atomicAdd(&st->ticket, 1u) == gridDim.x - 1) {
      __threadfence();
      res[0] = atomicExch(&st->cursor, 0ull);
      res[1] = atomicExch(&st->heavy, 0u);
      atomicExch(&st->ticket, 0u);
      __threadfence_system();
    }
  }
}

namespace {

template <typename K, typename OFF, int HK>
hipError_t launch_direct_u(const LaunchProbeDirect &p, hipStream_t st) {
  auto go = [&](auto kern, uint32_t block, uint32_t per) {
    hipLaunchKernelGGL(kern, dim3((p.n + per - 1) / per), dim3(block), 0, st, (const K *)p.probe, p.n, p.map,
                       (const OFF *)p.offA, (const K *)p.keysA, (K *)p.out, p.capacity, (K *)p.heavy,
                       (DirectState *)p.state, p.res);
    return hipGetLastError();
  };
  // few keys are spread over more, smaller workgroups; many take fewer
  // reservations of the shared cursor (one address: about 80 a microsecond)
  if (p.n <= 65536) return go(&k_probe_direct<K, OFF, 256, 1, HK>, 256, 256);
  if (p.n <= (1u << 18)) return go(&k_probe_direct<K, OFF, 256, 4, HK>, 256, 1024);
  return go(&k_probe_direct<K, OFF, 1024, 4, HK>, 1024, 4096);
}

template <typename K, typename OFF>
hipError_t launch_direct_hk(const LaunchProbeDirect &p, hipStream_t st) {
  return p.map.kind == 0 ? launch_direct_u<K, OFF, HK_MURMUR>(p, st) : launch_direct_u<K, OFF, HK_RMI>(p, st);
}

template <typename K, typename OFF, int BLOCK, int KPT, int HK>
hipError_t launch_one(const LaunchBuildOne &b, hipStream_t st) {
  // counters (u16 per bin), then the staged keys over them
  const uint32_t lds = (std::max<uint32_t>((uint32_t)((b.nbins + 1) / 2 * 4), b.n * (uint32_t)sizeof(K)) + 255u) & ~255u;
  hipLaunchKernelGGL((k_build_one<K, OFF, BLOCK, KPT, HK>), dim3(1), dim3(BLOCK), lds, st, (const K *)b.keys, (K *)b.csr,
                     (OFF *)b.off, b.n, b.bin_lo, b.nbins, b.map, lds);
  return hipGetLastError();
}

template <typename K, typename OFF, int HK>
hipError_t launch_one_size(const LaunchBuildOne &b, hipStream_t st) {
  if (b.n <= 1024 && b.nbins <= 4096) return launch_one<K, OFF, 256, 4, HK>(b, st);
  if (b.n <= 4096) return launch_one<K, OFF, 1024, 4, HK>(b, st);
  return launch_one<K, OFF, 1024, 16, HK>(b, st);
}

template <typename K, typename OFF>
hipError_t launch_one_hk(const LaunchBuildOne &b, hipStream_t st) {
  return b.map.kind == 0 ? launch_one_size<K, OFF, HK_MURMUR>(b, st) : launch_one_size<K, OFF, HK_RMI>(b, st);
}

template <typename F>
hipError_t max_lds(F *fn) {
  return hipFuncSetAttribute((const void *)fn, hipFuncAttributeMaxDynamicSharedMemorySize, 131072);
}

template <typename K, typename OFF, int HK>
hipError_t direct_lds() {
  hipError_t e = max_lds(&k_build_one<K, OFF, 1024, 4, HK>);
  if (e == hipSuccess) e = max_lds(&k_build_one<K, OFF, 1024, 16, HK>);
  return e;
}

}  // namespace

bool build_one_takes(uint64_t n, uint64_t nbins) {
  return n && n <= BUILD_ONE_KEYS && nbins <= 65535;
}

hipError_t launch_build_one(const LaunchBuildOne &b, hipStream_t st) {
  if (!build_one_takes(b.n, b.nbins) || b.map.kind > 1) return hipErrorInvalidValue;
  if (b.key_bytes == 4)
    return b.off_bytes == 4 ? launch_one_hk<uint32_t, uint32_t>(b, st) : launch_one_hk<uint32_t, uint64_t>(b, st);
  return b.off_bytes == 4 ? launch_one_hk<uint64_t, uint32_t>(b, st) : launch_one_hk<uint64_t, uint64_t>(b, st);
}

hipError_t launch_probe_direct(const LaunchProbeDirect &p, hipStream_t st) {
  if (!p.n || p.map.kind > 1) return hipErrorInvalidValue;
  if (p.key_bytes == 4)
    return p.off_bytes == 4 ? launch_direct_hk<uint32_t, uint32_t>(p, st) : launch_direct_hk<uint32_t, uint64_t>(p, st);
  return p.off_bytes == 4 ? launch_direct_hk<uint64_t, uint32_t>(p, st) : launch_direct_hk<uint64_t, uint64_t>(p, st);
}

hipError_t set_direct_kernel_attributes() {
  hipError_t e = hipSuccess;
  for (hipError_t x : {direct_lds<uint32_t, uint32_t, HK_MURMUR>(), direct_lds<uint32_t, uint64_t, HK_MURMUR>(),
                       direct_lds<uint64_t, uint32_t, HK_MURMUR>(), direct_lds<uint64_t, uint64_t, HK_MURMUR>(),
                       direct_lds<uint32_t, uint32_t, HK_RMI>(), direct_lds<uint32_t, uint64_t, HK_RMI>(),
                       direct_lds<uint64_t, uint32_t, HK_RMI>(), direct_lds<uint64_t, uint64_t, HK_RMI>()})
    if (x != hipSuccess) e = x;
  return e;
}

}  // namespace hg
