// hg_stage.hip -- gfx950 kernels of the staged (host-resident) builds.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <algorithm>
#include "hg_common.hpp"
#include "hg_device.hpp"
#include "hg_kernels.hpp"
#include "hg_scatter.hpp"

namespace hg {

__global__ __launch_bounds__(256) void k_stage_count(const uint32_t *__restrict__ tot, uint32_t np,
                                                     unsigned long long *__restrict__ acc) {
  const uint32_t p = blockIdx.x * 256 + threadIdx.x;
  if (p < np) acc[p] += tot[p];
}

// Number of the bounds b[1..n] (ascending, in LDS) that are <= bin.
__device__ __forceinline__ uint32_t slab_of(uint32_t bin, const uint32_t *b, uint32_t n) {
  uint32_t p = 0;
  for (uint32_t step = 1u << (31 - __clz(n)); step; step >>= 1) {
    const uint32_t q = p + step;
    if (q <= n && b[q] <= bin) p = q;
  }
  return p;
}

// A chunk is partitioned by slab: a few columns, so the narrow pass's shape
// (rows of keys to workgroups, one count matrix, three workgroups a CU) with a
// search of the slabs' bounds in place of a division.  1.4 M keys into 28
// slabs: 25 us where the pieces the slabs are made of (4096 columns) took 190.
constexpr int PB = 512;

template <typename K, int HK>
__global__ __launch_bounds__(PB) void k_stage_hist(const K *__restrict__ keys, uint32_t n, uint32_t per, BinMap map,
                                                   const uint32_t *__restrict__ bound, uint32_t ns,
                                                   uint32_t *__restrict__ cmat) {
  constexpr int U = scatter_tile_keys<K>(PB) / PB;
  __shared__ uint32_t s_cnt[NARROW_COLS], s_bound[NARROW_COLS];
  const uint32_t k0 = blockIdx.x * per, m = min(per, n - k0), b = threadIdx.x;
  if (b <= ns) {
    s_cnt[b] = 0;
    s_bound[b] = bound[b];
  }
  __syncthreads();
  for (uint32_t base = 0; base < m; base += PB * U) {
    const uint32_t cnt = min((uint32_t)(PB * U), m - base);
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(keys + k0 + base, cnt * (uint32_t)sizeof(K));
    K kr[U];
#pragma unroll
    for (int j = 0; j < U; j++) kr[j] = buf_load<K>(rs, b * (uint32_t)sizeof(K), j * PB * (uint32_t)sizeof(K));
#pragma unroll
    for (int j = 0; j < U; j++)
      if (j * PB + b < cnt) atomicAdd(&s_cnt[slab_of(bin_of<K, HK>(kr[j], map), s_bound, ns)], 1u);
  }
  __syncthreads();
  if (b <= ns) cmat[(uint64_t)blockIdx.x * (ns + 1) + b] = s_cnt[b];
}

// Workgroup 0 also takes the chunk's share of every slab from the totals.
template <typename K, int HK>
__global__ __launch_bounds__(PB) void k_stage_scatter(LaunchStagePart p, uint32_t per) {
  constexpr uint32_t T = scatter_tile_keys<K>(PB);
  __shared__ ScatterLds<K, PB> s;
  __shared__ uint32_t s_bound[NARROW_COLS];
  const uint32_t b = threadIdx.x, ns = p.ns;
  const uint32_t mine = b <= ns ? p.tot[b] : 0u;
  if (b <= ns) s_bound[b] = p.bound[b];
  uint32_t all;
  const uint32_t start = block_exclusive_sum<PB, uint32_t>(mine, s.tmp, all);
  if (blockIdx.x == 0 && b < ns) {
    const StageSlab sl = p.slabs[b];
    const uint64_t c = p.cur[b];
    StageMove m;
    m.src = start;
    m.dst = sl.pos + c;
    m.count = mine;
    if (c + mine > sl.count) {
      p.cur[ns] = 1;
      m.count = 0;
    }
    p.mv[b] = m;
    p.cur[b] = c + m.count;
  }
  uint32_t next = b <= ns ? start + p.cmat[(uint64_t)blockIdx.x * (ns + 1) + b] : 0u;
  const uint32_t k0 = blockIdx.x * per, n = min(per, p.n - k0);
  for (uint32_t base = 0; base < n; base += T)
    scatter_tile<K, PB, false>(p.keys, k0 + base, min(T, n - base), ns + 1, s, [&](uint32_t) { return (K *)p.out; },
                               [&](K key) { return slab_of(bin_of<K, HK>(key, p.map), s_bound, ns); },
                               [&](uint32_t c) {
                                 const uint32_t at = next;
                                 next += c;
                                 return at;
                               });
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

template <typename K, int HK>
static hipError_t launch_stage_part_t(const LaunchStagePart &p, hipStream_t st) {
  const uint32_t per = std::max<uint32_t>(2048, ((p.n + NARROW_ROWS - 1) / NARROW_ROWS + 1023) & ~1023u);
  const uint32_t rows = (p.n + per - 1) / per;
  hipLaunchKernelGGL((k_stage_hist<K, HK>), dim3(rows), dim3(PB), 0, st, (const K *)p.keys, p.n, per, p.map, p.bound,
                     p.ns, p.cmat);
  const hipError_t e = launch_narrow_scan(p.cmat, rows, p.ns + 1, p.tot, st);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((k_stage_scatter<K, HK>), dim3(rows), dim3(PB), 0, st, p, per);
  return hipGetLastError();
}

hipError_t launch_stage_part(const LaunchStagePart &p, hipStream_t st) {
  if (!p.n || p.n > (1u << 31) || !p.ns || p.ns >= NARROW_COLS || p.map.kind > 1) return hipErrorInvalidValue;
  if (p.key_bytes == 4)
    return p.map.kind == 0 ? launch_stage_part_t<uint32_t, HK_MURMUR>(p, st)
                           : launch_stage_part_t<uint32_t, HK_RMI>(p, st);
  return p.map.kind == 0 ? launch_stage_part_t<uint64_t, HK_MURMUR>(p, st)
                         : launch_stage_part_t<uint64_t, HK_RMI>(p, st);
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
