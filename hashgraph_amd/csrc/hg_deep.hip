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
// A hot value's bucket skips the groups: the histogram tells before any key moves.
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
static_assert(2 * DEEP_GROUPS <= SB, "a column a group and one for its hot bucket");
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
// groups and in the hot buckets (gstart, hstart) and the second step's chunks,
// group by group.  One workgroup.
// A group's largest bucket is hot when it has more keys than a group's share:
// hot holds its index in the group (NO_HOT: none).  Its keys never enter the
// group, so they are taken off the group's counts.
constexpr uint32_t NO_HOT = 255;
static_assert(DEEP_FINE <= (NO_HOT - 1) * (NO_HOT - 1), "a bucket's index in its group");
__global__ __launch_bounds__(1024) void k_deep_starts(const uint32_t *__restrict__ ftot, DeepGeom g, uint32_t rows,
                                                      const uint32_t *__restrict__ cmat,
                                                      const uint32_t *__restrict__ fmat, uint32_t chunk_keys,
                                                      uint32_t *__restrict__ fstart, uint32_t *__restrict__ gstart,
                                                      uint32_t *__restrict__ hot, uint32_t *__restrict__ hstart,
                                                      DeepChunk *__restrict__ chunks, uint32_t *__restrict__ nchunks) {
  extern __shared__ __align__(16) uint32_t s_a[];  // nfine + 1
  __shared__ uint32_t s_tmp[1024 / 64 + 1];
  __shared__ unsigned long long s_hot[DEEP_GROUPS];  // keys of the group's hot bucket << 32 | its index
  __shared__ uint32_t s_nhot;
  const uint32_t t = threadIdx.x;
  if (t < DEEP_GROUPS) s_hot[t] = 0;
  if (t == 0) s_nhot = 0;
  lds_fill<uint32_t, 1024, 8>(s_a, ftot, g.nfine);
  __syncthreads();
  const uint32_t tot = lds_exclusive_scan<1024>(s_a, g.nfine, s_tmp);
  if (t == 0) s_a[g.nfine] = tot;
  __syncthreads();
  const uint32_t share = (uint32_t)(g.n / g.ngroups);
  for (uint32_t f = t; f <= g.nfine; f += 1024) {
    const uint32_t at = s_a[f];
    fstart[f] = at;
    if (f < g.nfine && s_a[f + 1] - at > share)
      atomicMax(&s_hot[f / g.group], ((unsigned long long)(s_a[f + 1] - at) << 32) | (f % g.group));
  }
  __syncthreads();
  // a wave a group: the hot bucket's keys in each XCD's eighth of the rows
  for (uint32_t s = t / 64; s < g.ngroups; s += 1024 / 64) {
    const uint32_t lane = t & 63, c = (uint32_t)(s_hot[s] >> 32), b = c ? (uint32_t)s_hot[s] : NO_HOT;
    if (lane == 0) hot[s] = b;
    if (!c) continue;
    if (lane == 0) atomicAdd(&s_nhot, 1u);
    const uint32_t f = s * g.group + b;
    uint32_t before = 0;
    for (uint32_t x = 0; x < XCDS; x += 64 / XROWS) {
      const uint32_t r = x * XROWS + lane;
      uint32_t v = r < rows ? fmat[(uint64_t)r * g.nfine + f] : 0u;
      for (uint32_t d = XROWS / 2; d; d >>= 1) v += __shfl_xor(v, d, 64);
      for (uint32_t y = 0; y < 64 / XROWS; y++) {
        if (lane == 0) hstart[(x + y) * g.ngroups + s] = s_a[f] + before;
        before += __shfl(v, y * XROWS, 64);
      }
    }
  }
  __syncthreads();
  static_assert((DEEP_GROUPS & (DEEP_GROUPS - 1)) == 0 && 64 % XROWS == 0, "the search below, the sums above");
  __shared__ uint32_t s_n[DEEP_GROUPS], s_c0[DEEP_GROUPS];  // keys of a group without its hot bucket, its first chunk
  uint32_t nc = 0;
  if (t < g.ngroups) {
    const uint32_t a = s_a[t * g.group], e = s_a[min(g.nfine, (t + 1) * g.group)], c = (uint32_t)(s_hot[t] >> 32);
    for (uint32_t x = 0; x < XCDS; x++)
      if (x * XROWS < rows)
        gstart[x * g.ngroups + t] = a + cmat[(uint64_t)x * XROWS * g.ngroups + t] -
                                    (c ? hstart[x * g.ngroups + t] - hstart[t] : 0u);
    s_n[t] = e - a - c;
    nc = (uint32_t)(((uint64_t)s_n[t] + chunk_keys - 1) / chunk_keys);
  }
  uint32_t all;
  const uint32_t c0 = block_exclusive_sum<1024, uint32_t>(nc, s_tmp, all);
  if (t < g.ngroups) s_c0[t] = c0;
  if (t == 0) {
    nchunks[0] = all;
    nchunks[1] = s_nhot;
  }
  __syncthreads();
  for (uint32_t i = t; i < all; i += 1024) {  // a thread a chunk
    uint32_t q = 0;  // last group whose first chunk is at most i (groups without chunks precede it)
    for (uint32_t step = DEEP_GROUPS / 2; step; step >>= 1)
      if (q + step < g.ngroups && s_c0[q + step] <= i) q += step;
    DeepChunk d;
    d.start = s_a[q * g.group] + (i - s_c0[q]) * chunk_keys;
    d.count = min(chunk_keys, s_n[q] - (i - s_c0[q]) * chunk_keys);
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
// A group's hot bucket is a column of its own, whose keys go to their places in
// out at once and so are moved once instead of twice: 2^27 uint64 keys of
// Zipf(1.3) are built in 2.22 ms (2.60 with both steps for all of them, 2.35
// through the wide pass), half of them one value 1.83 (2.21, 2.05); uniform keys
// take the same 1.65.  Six waves a SIMD (80 registers): with four, 915 us of
// 2^27 uniform uint32 keys became 951.
// The first workgroups also write the buckets' items and clear what the items'
// kernels need.
template <typename K, bool PACK, int HK>
__global__ __launch_bounds__(SB, 6) void k_deep_first(const void *__restrict__ keys, DeepGeom g, uint32_t chunk_keys,
                                                   const uint32_t *__restrict__ nhot, const uint32_t *__restrict__ hot,
                                                   uint32_t *__restrict__ hstart, uint32_t *__restrict__ gstart,
                                                   const uint32_t *__restrict__ fstart, K *__restrict__ mid,
                                                   K *__restrict__ out, FinItem *__restrict__ items,
                                                   BinMap *__restrict__ maps, unsigned long long *__restrict__ zero,
                                                   uint32_t nzero, unsigned int *__restrict__ zero_col) {
  constexpr uint32_t T = scatter_tile_keys<K>(SB);
  using IN = typename std::conditional<PACK, uint32_t, K>::type;
  __shared__ ScatterLds<K, SB> s;
  __shared__ uint8_t s_hot[DEEP_GROUPS];  // (in bytes it leaves room for three workgroups a CU)
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
  if (*nhot == 0) {
    for (uint32_t base = 0; base < n; base += T)
      scatter_tile<K, SB, PACK>(keys, k0 + base, min(T, n - base), g.ngroups, s, [&](uint32_t) { return mid; },
                                [&](IN key) { return divq(bin_of<IN, HK>(key, g.map) - g.bin_lo, g.coarse); },
                                [&](uint32_t c) { return c ? atomicAdd(&gstart[x * g.ngroups + b], c) : 0u; });
    return;
  }
  if (b < g.ngroups) s_hot[b] = (uint8_t)hot[b];
  __syncthreads();
  const auto column = [&](IN key) {
    const uint32_t rel = bin_of<IN, HK>(key, g.map) - g.bin_lo, c = divq(rel, g.coarse);
    // a bucket of index NO_HOT lies in another group (past the tile's end: key
    // 0, whose bin may lie outside)
    return rel - (c * g.group + s_hot[min(c, DEEP_GROUPS - 1)]) * g.fine.d < g.fine.d ? c + g.ngroups : c;
  };
  uint32_t *const at = (b < g.ngroups ? gstart + b : hstart + (b - g.ngroups)) + x * g.ngroups;
  for (uint32_t base = 0; base < n; base += T)
    scatter_tile<K, SB, PACK>(keys, k0 + base, min(T, n - base), 2 * g.ngroups, s,
                              [&](uint32_t c) { return c < g.ngroups ? mid : out; }, column,
                              [&](uint32_t c) { return c ? atomicAdd(at, c) : 0u; });
}

// Second step: a chunk of one group into the group's buckets; every tile
// reserves its places (fstart ends as the buckets' ends).  Consecutive chunks
// run on one XCD, so the runs of a bucket meet in its L2.
template <typename K, int HK>
__global__ __launch_bounds__(SB) void k_deep_second(const K *__restrict__ keys, DeepGeom g,
                                                    const DeepChunk *__restrict__ chunks,
                                                    const uint32_t *__restrict__ nchunks, uint32_t *__restrict__ fstart,
                                                    K *__restrict__ out) {
  constexpr uint32_t T = scatter_tile_keys<K>(SB);
  __shared__ ScatterLds<K, SB> s;
  const uint32_t nc = nchunks[0];
  if (blockIdx.x >= nc) return;
  const uint32_t q = nc >> 3, r = nc & 7, x = blockIdx.x & 7;
  const DeepChunk d = chunks[x * q + min(x, r) + (blockIdx.x >> 3)];
  const uint32_t f0 = d.group * g.group, ncols = min(g.group, g.nfine - f0);
  const uint32_t lo = g.bin_lo + f0 * g.fine.d;  // first bin of the group
  for (uint32_t base = 0; base < d.count; base += T)
    scatter_tile<K, SB, false>(keys, (uint64_t)d.start + base, min(T, d.count - base), ncols, s,
                               [&](uint32_t) { return out; },
                               [&](K key) { return divq(bin_of<K, HK>(key, g.map) - lo, g.fine); },
                               [&](uint32_t c) { return c ? atomicAdd(&fstart[f0 + threadIdx.x], c) : 0u; });
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
                       p.rows, (const uint32_t *)p.cmat, (const uint32_t *)p.fmat, chunk, p.fstart, p.gstart, p.hot,
                       p.hstart, p.chunks, p.nchunks);
    return hipGetLastError();
  }
  const uint64_t share = std::min<uint64_t>((uint64_t)XROWS * g.per, g.n);
  auto first = &k_deep_first<K, false, HK>;
  if constexpr (sizeof(K) == 8 && HK == HK_MURMUR)
    if (p.pack) first = &k_deep_first<K, true, HK>;
  hipLaunchKernelGGL(first, dim3((uint32_t)((share + chunk - 1) / chunk) * XCDS), dim3(SB), 0, st, p.keys, g, chunk,
                     (const uint32_t *)(p.nchunks + 1), (const uint32_t *)p.hot, p.hstart, p.gstart,
                     (const uint32_t *)p.fstart, (K *)p.mid, (K *)p.out, p.items, p.maps, p.zero, p.nzero, p.zero_col);
  hipLaunchKernelGGL((k_deep_second<K, HK>), dim3(deep_max_chunks(g, p.key_bytes)), dim3(SB), 0, st, (const K *)p.mid, g,
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
