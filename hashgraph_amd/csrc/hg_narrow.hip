// hg_narrow.hip -- gfx950 kernels of the narrow partition pass: one table cut
// into at most NARROW_COLS buckets.
//
// The wide pass (hg_kernels.hip) serves thousands of buckets and many
// segments: 32 K-key rounds, one workgroup per CU, host-built descriptors and
// a count matrix of tiles x buckets.  A table of a few million keys has
// neither the tiles to fill the chip that way nor the buckets to need it.
// Here each of up to NARROW_ROWS workgroups takes one contiguous range of the
// keys, its counts are one row of a small matrix, and every kernel takes its
// geometry from its arguments, so a build is hist, column scan, scatter and
// final stage, with no upload.  2^20 uint32 keys: 35 us a build, 78 us through
// the wide pass; below about 2^21 keys the time is launches and each kernel's
// own latency, above it the scatter's and the final stage's LDS phases.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>
#include "hg_common.hpp"
#include "hg_device.hpp"
#include "hg_kernels.hpp"
#include "hg_scatter.hpp"

namespace hg {

constexpr int NB = 512;        // threads of the hist and scatter workgroups (>= NARROW_COLS)
constexpr int SCAN_COLS = 32;  // columns of a column-scan workgroup
constexpr int SCAN_PER = 16;   // rows of one of its threads
static_assert(NARROW_COLS <= NB && NARROW_ROWS == 1024 / SCAN_COLS * SCAN_PER, "narrow geometry");

// Bucket counts of key range g: row g of cmat (ncols words).
template <typename K, int HK>
__global__ __launch_bounds__(NB) void k_narrow_hist(const K *__restrict__ keys, NarrowGeom g, uint32_t *__restrict__ cmat) {
  constexpr int U = sizeof(K) == 4 ? 16 : 8;
  __shared__ uint32_t s_cnt[NARROW_COLS];
  const uint64_t k0 = (uint64_t)blockIdx.x * g.per;
  const uint32_t n = (uint32_t)min((uint64_t)g.per, g.n - k0);
  if (threadIdx.x < g.ncols) s_cnt[threadIdx.x] = 0;
  __syncthreads();
  for (uint32_t base = 0; base < n; base += NB * U) {
    const uint32_t cnt = min((uint32_t)(NB * U), n - base);
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(keys + k0 + base, cnt * (uint32_t)sizeof(K));
    K kr[U];
#pragma unroll
    for (int j = 0; j < U; j++) kr[j] = buf_load<K>(rs, threadIdx.x * (uint32_t)sizeof(K), j * NB * (uint32_t)sizeof(K));
#pragma unroll
    for (int j = 0; j < U; j++)
      if (j * NB + threadIdx.x < cnt) atomicAdd(&s_cnt[divq(bin_of<K, HK>(kr[j], g.map) - g.bin_lo, g.div)], 1u);
  }
  __syncthreads();
  if (threadIdx.x < g.ncols) cmat[(uint64_t)blockIdx.x * g.ncols + threadIdx.x] = s_cnt[threadIdx.x];
}

// Columns [32 b, 32 b + 32) of the count matrix: counts become exclusive sums
// down the column, the column's total goes to tot.  Each thread holds 16 rows
// of one column in registers, so the matrix is read and written once.
__global__ __launch_bounds__(1024) void k_narrow_scan(uint32_t *__restrict__ cmat, uint32_t rows, uint32_t ncols,
                                                      uint32_t *__restrict__ tot) {
  constexpr int CH = 1024 / SCAN_COLS;
  __shared__ uint32_t s_sum[CH][SCAN_COLS];
  const uint32_t c = threadIdx.x % SCAN_COLS, ch = threadIdx.x / SCAN_COLS;
  const uint32_t col = blockIdx.x * SCAN_COLS + c, r0 = ch * SCAN_PER;
  uint32_t v[SCAN_PER], s = 0;
#pragma unroll
  for (int i = 0; i < SCAN_PER; i++) v[i] = col < ncols && r0 + i < rows ? cmat[(uint64_t)(r0 + i) * ncols + col] : 0u;
#pragma unroll
  for (int i = 0; i < SCAN_PER; i++) s += v[i];
  s_sum[ch][c] = s;
  __syncthreads();
  uint32_t run = 0;
  for (uint32_t q = 0; q < ch; q++) run += s_sum[q][c];
  if (col >= ncols) return;
  if (ch == CH - 1) tot[col] = run + s;
#pragma unroll
  for (int i = 0; i < SCAN_PER; i++) {
    if (r0 + i < rows) cmat[(uint64_t)(r0 + i) * ncols + col] = run;
    run += v[i];
  }
}

// Scatter of key range g, tile by tile (scatter_tile); thread b carries bucket
// b's next place in a register.  Workgroup 0 also writes the final stage's items.
// PACK: the keys are 32-bit and the output 8-byte records (position << 32 | key).
template <typename K, int HK, bool PACK>
__global__ __launch_bounds__(NB) void k_narrow_scatter(const void *__restrict__ keys, NarrowGeom g,
                                                       const uint32_t *__restrict__ cmat,
                                                       const uint32_t *__restrict__ tot, K *__restrict__ out,
                                                       FinItem *__restrict__ items, BinMap *__restrict__ maps,
                                                       unsigned long long *__restrict__ zero, uint32_t nzero,
                                                       unsigned int *__restrict__ zero_col) {
  constexpr uint32_t T = scatter_tile_keys<K>(NB);
  using IN = typename std::conditional<PACK, uint32_t, K>::type;
  __shared__ ScatterLds<K, NB> s;
  const uint32_t b = threadIdx.x;
  const bool col = b < g.ncols;
  const uint32_t mine = col ? tot[b] : 0u;
  uint32_t all;
  const uint32_t start = block_exclusive_sum<NB, uint32_t>(mine, s.tmp, all);
  if (blockIdx.x == 0) {
    if (col) {
      FinItem it;
      const uint64_t lo = (uint64_t)b * g.div.d;
      it.key_start = start;
      it.key_rel = 0;
      it.off_pos = lo;
      it.end_pos = b + 1 == g.ncols ? g.nbins : ~0ull;
      it.count = mine;
      it.nbins = (uint32_t)min((uint64_t)g.div.d, g.nbins - lo);
      it.bin_lo = (uint32_t)(g.bin_lo + lo);
      it.table = 0;
      items[b] = it;
      if (zero_col) zero_col[b] = 0;
    }
    if (b == 0) maps[0] = g.map;
    if (b < nzero) zero[b] = 0;
  }
  uint32_t next = col ? start + cmat[(uint64_t)blockIdx.x * g.ncols + b] : 0u;
  const uint64_t k0 = (uint64_t)blockIdx.x * g.per;
  const uint32_t n = (uint32_t)min((uint64_t)g.per, g.n - k0);
  for (uint32_t base = 0; base < n; base += T)
    scatter_tile<K, NB, PACK>(keys, k0 + base, min(T, n - base), g.ncols, s, [&](uint32_t) { return out; },
                              [&](IN key) { return divq(bin_of<IN, HK>(key, g.map) - g.bin_lo, g.div); },
                              [&](uint32_t c) {
                                const uint32_t at = next;
                                next += c;
                                return at;
                              });
}

hipError_t launch_narrow_scan(uint32_t *cmat, uint32_t rows, uint32_t ncols, uint32_t *tot, hipStream_t st) {
  if (!rows || rows > NARROW_ROWS || !ncols || ncols > NARROW_COLS) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_narrow_scan, dim3((ncols + SCAN_COLS - 1) / SCAN_COLS), dim3(1024), 0, st, cmat, rows, ncols,
                     tot);
  return hipGetLastError();
}

namespace {

template <typename K, int HK>
hipError_t launch_narrow_t(const LaunchNarrow &p, hipStream_t st) {
  const NarrowGeom &g = p.geom;
  if (p.pack)
    hipLaunchKernelGGL((k_narrow_hist<uint32_t, HK>), dim3(p.rows), dim3(NB), 0, st, (const uint32_t *)p.keys, g, p.cmat);
  else
    hipLaunchKernelGGL((k_narrow_hist<K, HK>), dim3(p.rows), dim3(NB), 0, st, (const K *)p.keys, g, p.cmat);
  const hipError_t e = launch_narrow_scan(p.cmat, p.rows, g.ncols, p.tot, st);
  if (e != hipSuccess) return e;
  auto kern = &k_narrow_scatter<K, HK, false>;
  if constexpr (sizeof(K) == 8 && HK == HK_MURMUR)
    if (p.pack) kern = &k_narrow_scatter<K, HK, true>;
  hipLaunchKernelGGL(kern, dim3(p.rows), dim3(NB), 0, st, p.keys, g, (const uint32_t *)p.cmat,
                     (const uint32_t *)p.tot, (K *)p.out, p.items, p.maps, p.zero, p.nzero,
                     p.zero_col);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_narrow(const LaunchNarrow &p, hipStream_t st) {
  const NarrowGeom &g = p.geom;
  if (!g.ncols || g.ncols > NARROW_COLS || !p.rows || p.rows > NARROW_ROWS || !g.n || p.nzero > (uint32_t)NB ||
      (uint64_t)p.rows * g.per < g.n || (uint64_t)(p.rows - 1) * g.per >= g.n || g.map.kind > 1 ||
      (p.pack && (p.key_bytes != 8 || g.map.kind != 0)))
    return hipErrorInvalidValue;
  if (p.key_bytes == 4)
    return g.map.kind == 0 ? launch_narrow_t<uint32_t, HK_MURMUR>(p, st) : launch_narrow_t<uint32_t, HK_RMI>(p, st);
  return g.map.kind == 0 ? launch_narrow_t<uint64_t, HK_MURMUR>(p, st) : launch_narrow_t<uint64_t, HK_RMI>(p, st);
}

}  // namespace hg
