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

namespace {

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

bool build_one_takes(uint64_t n, uint64_t nbins, int key_bytes) {
  (void)key_bytes;
  return n && n <= BUILD_ONE_KEYS && nbins <= 65535;
}

hipError_t launch_build_one(const LaunchBuildOne &b, hipStream_t st) {
  if (!build_one_takes(b.n, b.nbins, b.key_bytes) || b.map.kind > 1) return hipErrorInvalidValue;
  if (b.key_bytes == 4)
    return b.off_bytes == 4 ? launch_one_hk<uint32_t, uint32_t>(b, st) : launch_one_hk<uint32_t, uint64_t>(b, st);
  return b.off_bytes == 4 ? launch_one_hk<uint64_t, uint32_t>(b, st) : launch_one_hk<uint64_t, uint64_t>(b, st);
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
