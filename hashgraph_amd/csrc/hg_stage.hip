// hg_stage.hip -- gfx950 kernels of the staged (host-resident) builds.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <algorithm>
#include "hg_common.hpp"
#include "hg_kernels.hpp"

namespace hg {

__global__ __launch_bounds__(256) void k_stage_count(const uint32_t *__restrict__ tot, uint32_t np,
                                                     unsigned long long *__restrict__ acc) {
  const uint32_t p = blockIdx.x * 256 + threadIdx.x;
  if (p < np) acc[p] += tot[p];
}

__global__ __launch_bounds__(256) void k_stage_shares(const uint32_t *__restrict__ bstart,
                                                      const uint32_t *__restrict__ tot,
                                                      const StageSlab *__restrict__ slabs, uint32_t ns,
                                                      unsigned long long *__restrict__ cur,
                                                      StageMove *__restrict__ mv) {
  const uint32_t s = blockIdx.x * 256 + threadIdx.x;
  if (s >= ns) return;
  const StageSlab sl = slabs[s];
  StageMove m;
  m.src = bstart[sl.p0];
  m.count = (uint64_t)bstart[sl.p1 - 1] + tot[sl.p1 - 1] - m.src;
  const uint64_t c = cur[s];
  m.dst = sl.pos + c;
  if (c + m.count > sl.count) {
    cur[ns] = 1;
    m.count = 0;
  }
  mv[s] = m;
  cur[s] = c + m.count;
}

// dst[0..n) = src[0..n) + add by blocks of 256 threads, this one the i-th of
// nblk: 16-byte stores, aligned at the destination.
template <typename T>
__device__ __forceinline__ void copy_out(T *__restrict__ dst, const T *__restrict__ src, uint64_t n, T add,
                                         uint32_t block, uint32_t nblk) {
  constexpr uint32_t V = 16 / sizeof(T);
  struct alignas(16) Vec {
    T v[V];
  };
  const uint64_t head = min(n, (uint64_t)((16 - ((uintptr_t)dst & 15)) & 15) / sizeof(T));
  const uint64_t nv = (n - head) / V, tail = head + nv * V;
  if (block == 0) {
    if (threadIdx.x < head) dst[threadIdx.x] = src[threadIdx.x] + add;
    if (threadIdx.x < n - tail) dst[tail + threadIdx.x] = src[tail + threadIdx.x] + add;
  }
  for (uint64_t i = (uint64_t)block * 256 + threadIdx.x; i < nv; i += (uint64_t)nblk * 256) {
    Vec r;
    __builtin_memcpy(&r, src + head + i * V, 16);  // element alignment is enough for the load
#pragma unroll
    for (uint32_t k = 0; k < V; k++) r.v[k] += add;
    *(Vec *)(dst + head + i * V) = r;
  }
}

// Block (x, s) writes the x-th part of share s.  Bound by the host link; a
// copy call a share took 20 us each (chunks of 5.5 MB to 28 slabs: 0.67 ms
// each, with the link moving for 0.11).
template <typename K>
__global__ __launch_bounds__(256) void k_stage_out(const K *__restrict__ keys, K *__restrict__ host,
                                                   const StageMove *__restrict__ mv) {
  const StageMove m = mv[blockIdx.y];
  copy_out<K>(host + m.dst, keys + m.src, m.count, (K)0, blockIdx.x, gridDim.x);
}

template <typename K, typename OFF>
__global__ __launch_bounds__(256) void k_stage_back(const K *__restrict__ keys, K *__restrict__ host_keys, uint64_t n,
                                                    const OFF *__restrict__ off, OFF *__restrict__ host_off,
                                                    uint64_t noff, OFF add) {
  copy_out<K>(host_keys, keys, n, (K)0, blockIdx.x, gridDim.x);
  copy_out<OFF>(host_off, off, noff, add, blockIdx.x, gridDim.x);
}

hipError_t launch_stage_count(const uint32_t *tot, uint32_t np, unsigned long long *acc, hipStream_t st) {
  if (!np) return hipSuccess;
  hipLaunchKernelGGL(k_stage_count, dim3((np + 255) / 256), dim3(256), 0, st, tot, np, acc);
  return hipGetLastError();
}

hipError_t launch_stage_shares(const uint32_t *bstart, const uint32_t *tot, const StageSlab *slabs, uint32_t ns,
                               unsigned long long *cur, StageMove *mv, hipStream_t st) {
  if (!ns) return hipSuccess;
  hipLaunchKernelGGL(k_stage_shares, dim3((ns + 255) / 256), dim3(256), 0, st, bstart, tot, slabs, ns, cur, mv);
  return hipGetLastError();
}

hipError_t launch_stage_out(const void *keys, void *host, int key_bytes, const StageMove *mv, uint32_t ns,
                            hipStream_t st) {
  if (!ns) return hipSuccess;
  const dim3 grid(std::max(1u, 256u / ns), ns);  // about a workgroup a CU: enough for the link
  if (key_bytes == 4)
    hipLaunchKernelGGL(k_stage_out<uint32_t>, grid, dim3(256), 0, st, (const uint32_t *)keys, (uint32_t *)host, mv);
  else
    hipLaunchKernelGGL(k_stage_out<uint64_t>, grid, dim3(256), 0, st, (const uint64_t *)keys, (uint64_t *)host, mv);
  return hipGetLastError();
}

hipError_t launch_stage_back(const void *keys, void *host_keys, int key_bytes, uint64_t n, const void *off,
                             void *host_off, int off_bytes, uint64_t noff, uint64_t add, hipStream_t st) {
  const auto go = [&](auto k, auto o) {
    using K = decltype(k);
    using OFF = decltype(o);
    hipLaunchKernelGGL((k_stage_back<K, OFF>), dim3(256), dim3(256), 0, st, (const K *)keys, (K *)host_keys, n,
                       (const OFF *)off, (OFF *)host_off, noff, (OFF)add);
    return hipGetLastError();
  };
  if (key_bytes == 4) return off_bytes == 4 ? go(uint32_t(), uint32_t()) : go(uint32_t(), uint64_t());
  return off_bytes == 4 ? go(uint64_t(), uint32_t()) : go(uint64_t(), uint64_t());
}

}  // namespace hg
