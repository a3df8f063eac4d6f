// hg_deep.hip -- gfx950 kernels of the two-step partition of a large table:
// up to DEEP_FINE buckets reached through about their square root of groups.
//
// One pass over thousands of buckets writes runs of a few keys (2^28 uint32
// keys over 9363 buckets: 3.5 keys a run, 2.6 times the bytes) from one
// workgroup a CU, whose counters alone fill half of its LDS.  Here every pass
// has at most about 200 columns: runs of 40 keys and more, three workgroups a
// CU.  The first step's histogram counts the buckets themselves and sums their
// counts to the groups', so the second step needs no histogram: a tile of it
// reserves its places in the buckets.  The buckets can then be small ones
// (8 K keys), which the final stage and the probe take several of to a CU.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <algorithm>
#include "hg_common.hpp"
#include "hg_device.hpp"
#include "hg_kernels.hpp"
#include "hg_scatter.hpp"

namespace hg {

constexpr int HB = 1024;        // threads of the histogram
constexpr int SB = 512;         // threads of the scatter steps
constexpr int SUM_COLS = 32;    // columns of a column-sum workgroup
constexpr uint32_t XCDS = 8;
constexpr uint32_t HOT_GRID = 768;  // three workgroups a CU
constexpr uint32_t XROWS = DEEP_ROWS / XCDS;  // key ranges of an XCD
static_assert(DEEP_ROWS % XCDS == 0 && DEEP_ROWS % (1024 / SUM_COLS) == 0 && DEEP_GROUPS <= SB, "two-step geometry");

// Counts of the buckets over key range blockIdx.x (a row of fmat) and of the
// groups (a row of cmat).  One workgroup a CU: its LDS holds a counter for
// every bucket and, behind them, a learned model of up to leaf_cap leaves
// (larger ones are read from global memory: 2^25 uint64 keys, 4096 leaves,
// 123 us that way and 81 from LDS).
template <typename K, int HK>
__global__ __launch_bounds__(HB) void k_deep_hist(const K *__restrict__ keys, DeepGeom g, uint32_t *__restrict__ cmat,
                                                  uint32_t *__restrict__ fmat, uint32_t leaf_cap) {
  constexpr int U = sizeof(K) == 4 ? 16 : 8;
  extern __shared__ __align__(16) uint32_t s_cnt[];
  for (uint32_t i = threadIdx.x; i < g.nfine; i += HB) s_cnt[i] = 0;
  RmiHeader h{};
  RmiLeaf *s_leaf = (RmiLeaf *)(s_cnt + ((g.nfine + 3) & ~3u));
  if constexpr (HK == HK_RMI) {
    h = *(const RmiHeader *)g.map.rmi;
    if (h.n_leaves <= leaf_cap) rmi_copy_leaves<HB>(g.map.rmi, s_leaf, 0, h.n_leaves);
  }
  __syncthreads();
  const uint64_t k0 = (uint64_t)blockIdx.x * g.per;
  const uint32_t n = (uint32_t)min((uint64_t)g.per, g.n - k0);
  for (uint32_t base = 0; base < n; base += HB * U) {
    const uint32_t cnt = min((uint32_t)(HB * U), n - base);
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(keys + k0 + base, cnt * (uint32_t)sizeof(K));
    K kr[U];
#pragma unroll
    for (int j = 0; j < U; j++) kr[j] = buf_load<K>(rs, threadIdx.x * (uint32_t)sizeof(K), j * HB * (uint32_t)sizeof(K));
    if (HK == HK_RMI && h.n_leaves <= leaf_cap) {
      const uint32_t nv = cnt > threadIdx.x ? (cnt - threadIdx.x + HB - 1) / HB : 0;
      rmi_window_bins<K, U>(kr, nv, h, s_leaf, 0, h.n_leaves, g.map.M,
                            [&](int, uint32_t bin) { atomicAdd(&s_cnt[divq(bin - g.bin_lo, g.fine)], 1u); });
      continue;
    }
#pragma unroll
    for (int j = 0; j < U; j++)
      if (j * HB + threadIdx.x < cnt) atomicAdd(&s_cnt[divq(bin_of<K, HK>(kr[j], g.map) - g.bin_lo, g.fine)], 1u);
  }
  __syncthreads();
  for (uint32_t s = threadIdx.x >> 6; s < g.ngroups; s += HB / 64) {  // a wave a group
    uint32_t v = 0;
    const uint32_t f1 = min(g.nfine, (s + 1) * g.group);
    for (uint32_t f = s * g.group + (threadIdx.x & 63); f < f1; f += 64) v += s_cnt[f];
    v = wave_inclusive_sum<uint32_t>(v);
    if ((threadIdx.x & 63) == 63) cmat[(uint64_t)blockIdx.x * g.ngroups + s] = v;
  }
  for (uint32_t i = threadIdx.x; i < g.nfine; i += HB) fmat[(uint64_t)blockIdx.x * g.nfine + i] = s_cnt[i];
}

// 32 columns of a count matrix, PER rows a thread in registers.  SCAN: the
// counts become exclusive sums down the column; else only its total is kept.
template <int PER, bool SCAN>
__device__ __forceinline__ void sum_columns(uint32_t *mat, uint32_t rows, uint32_t ncols, uint32_t block,
                                            uint32_t (*s_sum)[SUM_COLS], uint32_t *tot) {
  constexpr int CH = 1024 / SUM_COLS;
  const uint32_t c = threadIdx.x % SUM_COLS, ch = threadIdx.x / SUM_COLS;
  const uint32_t col = block * SUM_COLS + c, r0 = ch * PER;
  uint32_t v[PER], s = 0;
#pragma unroll
  for (int i = 0; i < PER; i++) v[i] = col < ncols && r0 + i < rows ? mat[(uint64_t)(r0 + i) * ncols + col] : 0u;
#pragma unroll
  for (int i = 0; i < PER; i++) s += v[i];
  s_sum[ch][c] = s;
  __syncthreads();
  if (col >= ncols || (!SCAN && ch != CH - 1)) return;
  uint32_t run = 0;
  for (uint32_t q = 0; q < ch; q++) run += s_sum[q][c];
  if (ch == CH - 1 && tot) tot[col] = run + s;
  if constexpr (SCAN) {
#pragma unroll
    for (int i = 0; i < PER; i++) {
      if (r0 + i < rows) mat[(uint64_t)(r0 + i) * ncols + col] = run;
      run += v[i];
    }
  }
}

// The first blocks: totals of the buckets' columns; the others: exclusive sums
// of the groups' columns.
__global__ __launch_bounds__(1024) void k_deep_sum(uint32_t *__restrict__ cmat, uint32_t rows, uint32_t ngroups,
                                                   uint32_t *__restrict__ fmat, uint32_t nfine,
                                                   uint32_t *__restrict__ ftot) {
  constexpr int PER = DEEP_ROWS * SUM_COLS / 1024;
  __shared__ uint32_t s_sum[1024 / SUM_COLS][SUM_COLS];
  const uint32_t nb = (nfine + SUM_COLS - 1) / SUM_COLS;
  if (blockIdx.x < nb)
    sum_columns<PER, false>(fmat, rows, nfine, blockIdx.x, s_sum, ftot);
  else
    sum_columns<PER, true>(cmat, rows, ngroups, blockIdx.x - nb, s_sum, nullptr);
}

// Starts of the buckets (fstart, nfine + 1), each XCD's first places in the
// groups (gstart) and the second step's chunks, group by group.  One workgroup.
__global__ __launch_bounds__(1024) void k_deep_starts(const uint32_t *__restrict__ ftot, DeepGeom g, uint32_t rows,
                                                      const uint32_t *__restrict__ cmat, uint32_t chunk_keys,
                                                      uint32_t *__restrict__ fstart, uint32_t *__restrict__ gstart,
                                                      DeepChunk *__restrict__ chunks, uint32_t *__restrict__ nchunks) {
  extern __shared__ __align__(16) uint32_t s_a[];  // nfine + 1
  __shared__ uint32_t s_tmp[1024 / 64 + 1];
  lds_fill<uint32_t, 1024, 8>(s_a, ftot, g.nfine);
  __syncthreads();
  const uint32_t tot = lds_exclusive_scan<1024>(s_a, g.nfine, s_tmp);
  if (threadIdx.x == 0) s_a[g.nfine] = tot;
  __syncthreads();
  for (uint32_t f = threadIdx.x; f <= g.nfine; f += 1024) fstart[f] = s_a[f];
  const uint32_t s = threadIdx.x;
  static_assert((DEEP_GROUPS & (DEEP_GROUPS - 1)) == 0, "the search below");
  uint32_t a = 0, e = 0;
  if (s < g.ngroups) {
    a = s_a[s * g.group];
    e = s_a[min(g.nfine, (s + 1) * g.group)];
  }
  if (s < g.ngroups)
    for (uint32_t x = 0; x < XCDS; x++)
      if (x * XROWS < rows) gstart[x * g.ngroups + s] = a + cmat[(uint64_t)x * XROWS * g.ngroups + s];
  const uint32_t nc = (uint32_t)(((uint64_t)(e - a) + chunk_keys - 1) / chunk_keys);
  // ordinary groups' chunks, then the hot ones', a thread a chunk (a hot key's
  // group may have most of them)
  __shared__ uint32_t s_c0[2][DEEP_GROUPS];
  const bool hot = e - a > g.n / g.ngroups * 2;
  uint32_t all[2];
  const uint32_t c0 = block_exclusive_sum<1024, uint32_t>(hot ? 0u : nc, s_tmp, all[0]);
  const uint32_t c1 = block_exclusive_sum<1024, uint32_t>(hot ? nc : 0u, s_tmp, all[1]);
  if (s < g.ngroups) {
    s_c0[0][s] = c0;
    s_c0[1][s] = c1;
  }
  if (s < 2) nchunks[s] = all[s];
  __syncthreads();
  for (uint32_t i = s; i < all[0] + all[1]; i += 1024) {
    const uint32_t h = i >= all[0], ci = h ? i - all[0] : i;
    uint32_t q = 0;  // last group whose first chunk is at most ci (groups without chunks precede it)
    for (uint32_t step = DEEP_GROUPS / 2; step; step >>= 1)
      if (q + step < g.ngroups && s_c0[h][q + step] <= ci) q += step;
    const uint32_t ga = s_a[q * g.group], ge = s_a[min(g.nfine, (q + 1) * g.group)];
    DeepChunk d;
    d.start = ga + (ci - s_c0[h][q]) * chunk_keys;
    d.count = min(chunk_keys, ge - d.start);
    d.group = q;
    d.pad = 0;
    chunks[i] = d;
  }
}

// First step: chunks of the keys into the groups; a tile reserves its places.
// XCD x takes the x-th eighth of the keys in order and writes one part of each
// group, so the tiles in flight on an XCD write next to each other: 2^28 uint32
// keys in 515 us (747 with a contiguous key range for each workgroup; a plain
// copy takes 410).
// The first workgroups also write the buckets' items and clear what the items'
// kernels need.
template <typename K, bool PACK, int HK>
__global__ __launch_bounds__(SB) void k_deep_first(const void *__restrict__ keys, DeepGeom g, uint32_t chunk_keys,
                                                   uint32_t *__restrict__ gstart,
                                                   const uint32_t *__restrict__ fstart, K *__restrict__ out,
                                                   FinItem *__restrict__ items, BinMap *__restrict__ maps,
                                                   unsigned long long *__restrict__ zero, uint32_t nzero,
                                                   unsigned int *__restrict__ zero_col) {
  constexpr uint32_t T = scatter_tile_keys<K>(SB);
  using IN = typename std::conditional<PACK, uint32_t, K>::type;
  __shared__ ScatterLds<K, SB> s;
  const uint32_t b = threadIdx.x;
  for (uint32_t f = blockIdx.x * SB + b; f < g.nfine; f += gridDim.x * SB) {
    FinItem it;
    const uint64_t lo = (uint64_t)f * g.fine.d;
    it.key_start = fstart[f];
    it.key_rel = 0;
    it.off_pos = lo;
    it.end_pos = f + 1 == g.nfine ? g.nbins : ~0ull;
    it.count = fstart[f + 1] - fstart[f];
    it.nbins = (uint32_t)min((uint64_t)g.fine.d, g.nbins - lo);
    it.bin_lo = (uint32_t)(g.bin_lo + lo);
    it.table = 0;
    items[f] = it;
    if (zero_col) zero_col[f] = 0;
  }
  if (blockIdx.x == 0) {
    if (b == 0) maps[0] = g.map;
    if (b < nzero) zero[b] = 0;
  }
  const uint32_t x = blockIdx.x % XCDS;
  const uint64_t share = (uint64_t)XROWS * g.per, end = min(g.n, (x + 1) * share);
  const uint64_t k0 = x * share + (uint64_t)(blockIdx.x / XCDS) * chunk_keys;
  if (k0 >= end) return;
  const uint32_t n = (uint32_t)min((uint64_t)chunk_keys, end - k0);
  for (uint32_t base = 0; base < n; base += T)
    scatter_tile<K, SB, PACK>(keys, k0 + base, min(T, n - base), g.ngroups, s, out,
                              [&](IN key) { return divq(bin_of<IN, HK>(key, g.map) - g.bin_lo, g.coarse); },
                              [&](uint32_t c) { return c ? atomicAdd(&gstart[x * g.ngroups + b], c) : 0u; });
}

// Second step: a chunk of one group into the group's buckets; every tile
// reserves its places (fstart ends as the buckets' ends).
template <typename K, int HK, bool HOT>
__device__ __forceinline__ void second_chunk(const K *__restrict__ keys, const DeepGeom &g, const DeepChunk &d,
                                             ScatterLds<K, SB> &s, uint32_t *__restrict__ fstart,
                                             K *__restrict__ out) {
  constexpr uint32_t T = scatter_tile_keys<K>(SB);
  const uint32_t f0 = d.group * g.group, ncols = min(g.group, g.nfine - f0);
  const uint32_t lo = g.bin_lo + f0 * g.fine.d;  // first bin of the group
  for (uint32_t base = 0; base < d.count; base += T)
    scatter_tile<K, SB, false, HOT>(keys, (uint64_t)d.start + base, min(T, d.count - base), ncols, s, out,
                                    [&](K key) { return divq(bin_of<K, HK>(key, g.map) - lo, g.fine); },
                                    [&](uint32_t c) { return c ? atomicAdd(&fstart[f0 + threadIdx.x], c) : 0u; });
}

// Consecutive chunks run on one XCD, so the runs of a bucket meet in its L2.
template <typename K, int HK>
__global__ __launch_bounds__(SB) void k_deep_second(const K *__restrict__ keys, DeepGeom g,
                                                    const DeepChunk *__restrict__ chunks,
                                                    const uint32_t *__restrict__ nchunks, uint32_t *__restrict__ fstart,
                                                    K *__restrict__ out) {
  __shared__ ScatterLds<K, SB> s;
  const uint32_t nc = nchunks[0];
  if (blockIdx.x >= nc) return;
  const uint32_t q = nc >> 3, r = nc & 7, x = blockIdx.x & 7;
  second_chunk<K, HK, false>(keys, g, chunks[x * q + min(x, r) + (blockIdx.x >> 3)], s, fstart, out);
}

// The chunks of groups with more than twice their share of the keys: one value
// fills most of them (a kernel of its own, since its registers would cost the
// other one a workgroup a CU).  Builds of 2^27 uint32 keys: Zipf(1.1) 2.02 ms
// without it, 1.88 with it, Zipf(1.3) 2.18 and 2.05; uniform keys pay a launch.
template <typename K, int HK>
__global__ __launch_bounds__(SB) void k_deep_hot(const K *__restrict__ keys, DeepGeom g,
                                                 const DeepChunk *__restrict__ chunks,
                                                 const uint32_t *__restrict__ nchunks, uint32_t *__restrict__ fstart,
                                                 K *__restrict__ out) {
  __shared__ ScatterLds<K, SB> s;
  const uint32_t n0 = nchunks[0], n1 = nchunks[1];
  for (uint32_t i = blockIdx.x; i < n1; i += gridDim.x)
    second_chunk<K, HK, true>(keys, g, chunks[n0 + i], s, fstart, out);
}

namespace {

// Keys of a scatter workgroup: four tiles, fewer where that would leave less
// than a few workgroups for each of the chip's 768 places.
uint32_t chunk_keys(uint64_t n, int key_bytes) {
  const uint64_t t = key_bytes == 4 ? scatter_tile_keys<uint32_t>(SB) : scatter_tile_keys<uint64_t>(SB);
  return (uint32_t)(t * std::min<uint64_t>(4, std::max<uint64_t>(1, n / (t * 3072))));
}

template <typename K, int HK>
hipError_t launch_deep_t(const LaunchDeep &p, bool scatter, hipStream_t st) {
  const DeepGeom &g = p.geom;
  const uint32_t chunk = chunk_keys(g.n, p.key_bytes);
  if (!scatter) {
    const size_t cnts = (size_t)((g.nfine + 3) & ~3u) * 4, room = (size_t)(DEEP_FINE + 1) * 4;
    const uint32_t leaf_cap =
        HK == HK_RMI && room > cnts ? (uint32_t)std::min<size_t>(4096, (room - cnts) / sizeof(RmiLeaf)) : 0;
    const size_t hlds = std::max((size_t)g.nfine * 4, leaf_cap ? cnts + leaf_cap * sizeof(RmiLeaf) : 0);
    if (p.pack)
      hipLaunchKernelGGL((k_deep_hist<uint32_t, HK>), dim3(p.rows), dim3(HB), hlds, st, (const uint32_t *)p.keys, g, p.cmat,
                         p.fmat, leaf_cap);
    else
      hipLaunchKernelGGL((k_deep_hist<K, HK>), dim3(p.rows), dim3(HB), hlds, st, (const K *)p.keys, g, p.cmat, p.fmat,
                         leaf_cap);
    hipLaunchKernelGGL(k_deep_sum, dim3((g.nfine + SUM_COLS - 1) / SUM_COLS + (g.ngroups + SUM_COLS - 1) / SUM_COLS),
                       dim3(1024), 0, st, p.cmat, p.rows, g.ngroups, p.fmat, g.nfine, p.ftot);
    hipLaunchKernelGGL(k_deep_starts, dim3(1), dim3(1024), ((size_t)g.nfine + 1) * 4, st, (const uint32_t *)p.ftot, g,
                       p.rows, (const uint32_t *)p.cmat, chunk, p.fstart, p.gstart, p.chunks, p.nchunks);
    return hipGetLastError();
  }
  auto first = &k_deep_first<K, false, HK>;
  if constexpr (sizeof(K) == 8 && HK == HK_MURMUR)
    if (p.pack) first = &k_deep_first<K, true, HK>;
  const uint64_t share = std::min<uint64_t>((uint64_t)XROWS * g.per, g.n);
  hipLaunchKernelGGL(first, dim3((uint32_t)((share + chunk - 1) / chunk) * XCDS), dim3(SB), 0, st, p.keys, g, chunk,
                     p.gstart, (const uint32_t *)p.fstart, (K *)p.mid, p.items, p.maps, p.zero, p.nzero, p.zero_col);
  hipLaunchKernelGGL((k_deep_second<K, HK>), dim3(deep_max_chunks(g, p.key_bytes)), dim3(SB), 0, st, (const K *)p.mid, g,
                     (const DeepChunk *)p.chunks, (const uint32_t *)p.nchunks, p.fstart, (K *)p.out);
  hipLaunchKernelGGL((k_deep_hot<K, HK>), dim3(HOT_GRID), dim3(SB), 0, st, (const K *)p.mid, g,
                     (const DeepChunk *)p.chunks, (const uint32_t *)p.nchunks, p.fstart, (K *)p.out);
  return hipGetLastError();
}

}  // namespace

uint32_t deep_max_chunks(const DeepGeom &g, int key_bytes) {
  return (uint32_t)(g.n / chunk_keys(g.n, key_bytes) + g.ngroups);
}

static hipError_t launch_deep(const LaunchDeep &p, bool scatter, hipStream_t st) {
  const DeepGeom &g = p.geom;
  if (!g.n || g.n >= (1ull << 32) || !g.nfine || g.nfine > DEEP_FINE || !g.group || g.group > (uint32_t)SB ||
      !g.ngroups || g.ngroups > DEEP_GROUPS || (uint64_t)g.ngroups * g.group < g.nfine ||
      (uint64_t)(g.ngroups - 1) * g.group >= g.nfine || !p.rows || p.rows > DEEP_ROWS ||
      (uint64_t)p.rows * g.per < g.n || (uint64_t)(p.rows - 1) * g.per >= g.n || p.nzero > (uint32_t)SB ||
      g.map.kind > 1 || (uint64_t)g.nfine * g.fine.d < g.nbins || (p.pack && (p.key_bytes != 8 || g.map.kind != 0)))
    return hipErrorInvalidValue;
  if (p.key_bytes == 4)
    return g.map.kind == 0 ? launch_deep_t<uint32_t, HK_MURMUR>(p, scatter, st)
                           : launch_deep_t<uint32_t, HK_RMI>(p, scatter, st);
  return g.map.kind == 0 ? launch_deep_t<uint64_t, HK_MURMUR>(p, scatter, st)
                         : launch_deep_t<uint64_t, HK_RMI>(p, scatter, st);
}

hipError_t launch_deep_count(const LaunchDeep &p, hipStream_t st) { return launch_deep(p, false, st); }
hipError_t launch_deep_scatter(const LaunchDeep &p, hipStream_t st) { return launch_deep(p, true, st); }

hipError_t set_deep_kernel_attributes() {
  const auto lds = [](const void *f) {
    return hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (DEEP_FINE + 1) * 4);
  };
  hipError_t e = hipSuccess;
  for (hipError_t x : {lds((const void *)&k_deep_hist<uint32_t, HK_MURMUR>),
                       lds((const void *)&k_deep_hist<uint64_t, HK_MURMUR>),
                       lds((const void *)&k_deep_hist<uint32_t, HK_RMI>),
                       lds((const void *)&k_deep_hist<uint64_t, HK_RMI>),
                       lds((const void *)&k_deep_starts)})
    if (x != hipSuccess) e = x;
  return e;
}

}  // namespace hg
