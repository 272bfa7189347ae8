// host_cpu.cc -- the host CPU's distance kernel sets and filter counts (host-only code).
//
// vdb picks its distance kernels from the CPU it runs on (src/distance/cpu_features.cc:
// 19-21, 40-48): scalar always, AVX2 with AVX2 + FMA, AVX-512 with AVX-512F on top.  The GPU
// reproduces the arithmetic order of whichever set a vdb process on this host would use.
#include <cstddef>
#include <cstdint>

namespace vdbg {

// 0 = scalar, 1 = avx2, 2 = avx512.
int BestHostKernelSet() {
  __builtin_cpu_init();
  const bool avx2 = __builtin_cpu_supports("avx2") && __builtin_cpu_supports("fma");
  if (avx2 && __builtin_cpu_supports("avx512f")) return 2;
  return avx2 ? 1 : 0;
}

namespace {

inline __attribute__((always_inline)) size_t Count(const uint64_t* w, size_t rows) {
  size_t n = 0;
  for (size_t i = 0; i < rows / 64; ++i) n += size_t(__builtin_popcountll(w[i]));
  if (rows % 64)
    n += size_t(__builtin_popcountll(w[rows / 64] & ((uint64_t(1) << (rows % 64)) - 1)));
  return n;
}
__attribute__((target("popcnt"))) size_t CountPopcnt(const uint64_t* w, size_t rows) {
  return Count(w, rows);
}

}  // namespace

// The set bits among the first `rows` of w (1M rows: 5 us with the popcnt instruction).
size_t CountRows(const uint64_t* w, size_t rows) {
  __builtin_cpu_init();
  if (__builtin_cpu_supports("popcnt")) return CountPopcnt(w, rows);
  return Count(w, rows);
}

}  // namespace vdbg
