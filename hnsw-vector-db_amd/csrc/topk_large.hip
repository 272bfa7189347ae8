// topk_large.hip -- top-k beyond what one wavefront keeps in registers.
//
// The wave top-k of the scans holds up to 256 keys.  vdb allows k up to 10,000
// (src/engine/collection_impl.cc:26, 1038-1039), IVF-PQ's default rerank depth is
// max(10 k, 100) (src/index/quant/ivf_pq.cc:16-19) and nprobe may reach nlist.  For those
// sizes every candidate is scored into a per-query array of 64-bit keys
//   key = order-preserving bits of the distance << 32 | row id
// (-0 folded into +0, so equal distances tie on the id as Neighbor::operator< does,
// include/vdb/types.h:23-25), the arrays are sorted by a segmented radix sort, and the first
// k keys of each query are the reference's TopK(k).sorted().
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <vector>

#include "vdbg_device.h"
#include "vdbg_internal.h"

namespace vdbg {

__global__ void k_unpack_keys(const uint64_t* __restrict__ keys, const int* __restrict__ off,
                              int nseg, int K, uint32_t* __restrict__ out_ids,
                              float* __restrict__ out_d) {
  const size_t t = blockIdx.x * size_t(blockDim.x) + threadIdx.x;
  if (t >= size_t(nseg) * K) return;
  const int q = int(t / K), i = int(t - size_t(q) * K);
  const int at = off[q] + i;
  const uint64_t key = at < off[q + 1] ? keys[at] : kNoKey;
  if (key == kNoKey) {
    out_ids[t] = kNoId;
    out_d[t] = __builtin_inff();
  } else {
    out_ids[t] = uint32_t(key);
    out_d[t] = key_dist(key);
  }
}

// The K smallest of each query's keys, sorted, by one block per query: the keys (at most
// kBlockSortKeys, kNoKey for none) go to LDS, padded to a power of two, through a bitonic
// sort.  Layers of stride at most 64 stay inside one wave's 128 consecutive keys (thread i
// takes the i-th pair), so only wider ones need a block barrier: 10 of 66 at 2,048 keys.
// Bound: LDS (two reads and two writes of 8 bytes per key and layer).  It replaces the
// device-wide segmented radix sort where a query's keys fit the LDS: 61 queries of 118,385
// keys took 3.7 ms there, 61 of about 1,300 admitted keys take 20 us here.
__global__ __launch_bounds__(1024) void k_sort_keys(SortKeysArgs a) {
  extern __shared__ uint64_t sk[];
  const int q = blockIdx.x;
  const int tid = threadIdx.x, nt = blockDim.x;
  const uint32_t n = a.counts != nullptr ? a.counts[q] : a.stride;
  if (n > a.stride) {  // overflowed: the caller answers this query another way
    if (tid == 0) a.fb_list[atomicAdd(a.fb_count, 1u)] = uint32_t(q);
    return;
  }
  uint32_t P = 2;
  while (P < n) P <<= 1;
  const uint64_t* src = a.keys + size_t(q) * a.stride;
  for (uint32_t i = tid; i < P; i += nt) sk[i] = i < n ? src[i] : kNoKey;
  __syncthreads();
  for (uint32_t size = 2; size <= P; size <<= 1)
    for (uint32_t j = size >> 1; j > 0; j >>= 1) {
      for (uint32_t i = tid; i < P / 2; i += nt) {
        const uint32_t lo = 2 * i - (i & (j - 1)), hi = lo + j;
        const uint64_t x = sk[lo], y = sk[hi];
        if ((x > y) == ((lo & size) == 0)) {
          sk[lo] = y;
          sk[hi] = x;
        }
      }
      // the next layer crosses waves when its stride (or this one's) is above 64
      const uint32_t next = j > 1 ? j >> 1 : size;
      if (j > kWave || next > kWave) {
        __syncthreads();
      } else {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      }
    }
  __syncthreads();
  for (int i = tid; i < a.K; i += nt) {
    const uint64_t key = uint32_t(i) < P ? sk[i] : kNoKey;
    a.out_ids[size_t(q) * a.K + i] = key == kNoKey ? kNoId : uint32_t(key);
    a.out_d[size_t(q) * a.K + i] = key == kNoKey ? __builtin_inff() : key_dist(key);
  }
  if (a.T != nullptr && tid == 0) {
    // every row outside the keys has GEMM value > T, so an exact distance above
    // T + shift - eb: certified when the K-th is at most that
    const uint64_t key = uint32_t(a.K) <= P ? sk[a.K - 1] : kNoKey;
    const double dk = key == kNoKey ? double(__builtin_inff()) : double(key_dist(key));
    const double lower = (double(a.T[q]) + double(a.shift[q])) - double(a.eb[q]);
    if (!(dk <= lower) || a.force_fallback) a.fb_list[atomicAdd(a.fb_count, 1u)] = uint32_t(q);
  }
}

int SortKeysTopK(Ctx* c, const SortKeysArgs& a, int nq, hipStream_t s) {
  if (nq == 0 || a.K == 0) return kOk;
  uint32_t P = 128;
  while (P < a.stride) P <<= 1;
  if (P > kBlockSortKeys) return SetError(kInternal, "block sort: too many keys per query");
  const size_t lds = size_t(P) * sizeof(uint64_t);
  if (lds > 65536)  // (the default limit of dynamic LDS)
    VDBG_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(k_sort_keys),
                                 hipFuncAttributeMaxDynamicSharedMemorySize,
                                 int(kBlockSortKeys * sizeof(uint64_t))));
  ProfScope ps(c, "sort_keys", s);
  k_sort_keys<<<dim3(unsigned(nq)), std::min<uint32_t>(1024, P / 2), lds, s>>>(a);
  VDBG_HIP(hipGetLastError());
  return kOk;
}

int SortSegmentsTopK(Ctx* c, uint64_t* keys, uint64_t* keys_alt, const int* off_dev, int nseg,
                     int total, int K, uint32_t* out_ids, float* out_d, hipStream_t s) {
  if (nseg == 0) return kOk;
  if (total > 0) {
    size_t tmp_bytes = 0;
    VDBG_HIP(hipcub::DeviceSegmentedRadixSort::SortKeys(nullptr, tmp_bytes, keys, keys_alt, total,
                                                        nseg, off_dev, off_dev + 1, 0, 64, s));
    void* tmp = nullptr;
    VDBG_HIP(hipMallocAsync(&tmp, tmp_bytes + 16, s));
    {
      ProfScope ps(c, "segmented_sort", s);
      VDBG_HIP(hipcub::DeviceSegmentedRadixSort::SortKeys(tmp, tmp_bytes, keys, keys_alt, total,
                                                          nseg, off_dev, off_dev + 1, 0, 64, s));
    }
    (void)hipFreeAsync(tmp, s);
  }
  const size_t n = size_t(nseg) * K;
  k_unpack_keys<<<dim3(unsigned((n + 255) / 256)), 256, 0, s>>>(keys_alt, off_dev, nseg, K,
                                                                  out_ids, out_d);
  VDBG_HIP(hipGetLastError());
  return kOk;
}

// Exact distance of every (query, row) pair of a chunk of queries; disallowed rows get kNoKey.
template <class Scorer>
__global__ __launch_bounds__(256) void k_score_all(const float* __restrict__ Q, int pd,
                                                   uint32_t N, const uint64_t* __restrict__ allow,
                                                   Scorer sc, uint64_t* __restrict__ keys) {
  const uint32_t r = blockIdx.x * 256 + threadIdx.x;
  const int qi = blockIdx.y;
  if (r >= N) return;
  uint64_t key = kNoKey;
  if (row_allowed(allow, r)) key = dist_key(sc(Q + size_t(qi) * pd, r), r);
  keys[size_t(qi) * N + r] = key;
}

__global__ void k_seg_offsets(int* off, int nseg, int len) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i <= nseg) off[i] = i * len;
}

template <class Scorer>
static int ExactAllT(Ctx* c, const ScanSource& src, const Scorer& sc, const float* Q, size_t nq,
                     size_t kk, const uint64_t* allow, uint32_t* out_ids, float* out_d,
                     hipStream_t s) {
  const uint32_t N = src.N;
  const int spd = ScorePd(src);
  // queries per chunk: at most 256 MiB of keys and fewer than 2^31 keys
  size_t chunk = std::max<size_t>(1, (size_t(256) << 20) / (size_t(N) * 8));
  chunk = std::min({chunk, nq, size_t(65535)});  // queries run on grid.y
  uint64_t* keys = nullptr;
  int* off = nullptr;
  const size_t nk = chunk * N;
  VDBG_HIP(hipMallocAsync(reinterpret_cast<void**>(&keys), nk * 16 + 16, s));
  VDBG_HIP(hipMallocAsync(reinterpret_cast<void**>(&off), (chunk + 1) * sizeof(int), s));
  int rc = kOk;
  for (size_t q0 = 0; q0 < nq && rc == kOk; q0 += chunk) {
    const int nc = int(std::min(chunk, nq - q0));
    {
      ProfScope ps(c, "exact_all", s);
      k_score_all<Scorer><<<dim3((N + 255) / 256, nc), 256, 0, s>>>(Q + q0 * spd, spd, N, allow,
                                                                       sc, keys);
    }
    if (hipGetLastError() != hipSuccess) {
      rc = SetError(kInternal, "exact-all launch");
      break;
    }
    if (N <= kBlockSortKeys) {
      rc = SortKeysTopK(c, SortKeysArgs{keys, N, int(kk), out_ids + q0 * kk, out_d + q0 * kk}, nc,
                        s);
      continue;
    }
    k_seg_offsets<<<dim3(unsigned((nc + 256) / 256)), 256, 0, s>>>(off, nc, int(N));
    rc = SortSegmentsTopK(c, keys, keys + nk, off, nc, int(size_t(nc) * N), int(kk),
                          out_ids + q0 * kk, out_d + q0 * kk, s);
  }
  (void)hipStreamSynchronize(s);
  (void)hipFreeAsync(keys, s);
  (void)hipFreeAsync(off, s);
  return rc;
}

int ExactScanAll(Ctx* c, const ScanSource& src, const float* Q, size_t nq, size_t kk,
                 const uint64_t* allow, uint32_t* out_ids, float* out_d, hipStream_t s) {
  if (nq == 0 || kk == 0) return kOk;
  if (kk > (size_t(1) << 30)) return SetError(kInvalidArgument, "too many results per query");
  if (src.kind == 0)
    return ExactAllT(c, src, FlatScorer{src.X, src.pd, src.metric, c->kset, src.Xmap}, Q, nq, kk, allow,
                     out_ids, out_d, s);
  if (src.kind == 2)
    return ExactAllT(c, src, PqScorer{src.C, src.pq_m}, Q, nq, kk, allow, out_ids, out_d, s);
  return ExactAllT(c, src, Sq8Scorer{src.C, src.vmin, src.scale, src.pd, src.metric, c->kset}, Q,
                   nq, kk, allow, out_ids, out_d, s);
}

// The listed queries' rows of w floats, gathered.
__global__ void k_gather_queries(const float* __restrict__ Q, int w,
                                 const uint32_t* __restrict__ list, float* __restrict__ y) {
  const float* src = Q + size_t(list[blockIdx.x]) * w;
  float* dst = y + size_t(blockIdx.x) * w;
  for (int i = threadIdx.x; i < w; i += blockDim.x) dst[i] = src[i];
}
// Their results, back to their places.
__global__ void k_scatter_results(const uint32_t* __restrict__ ids, const float* __restrict__ d,
                                  size_t kk, const uint32_t* __restrict__ list,
                                  uint32_t* __restrict__ out_ids, float* __restrict__ out_d) {
  const size_t from = size_t(blockIdx.x) * kk, to = size_t(list[blockIdx.x]) * kk;
  for (size_t i = threadIdx.x; i < kk; i += blockDim.x) {
    out_ids[to + i] = ids[from + i];
    out_d[to + i] = d[from + i];
  }
}

int ExactScanAllListed(Ctx* c, const ScanSource& src, const float* Q, size_t nq,
                       const uint32_t* list, size_t n, size_t kk, const uint64_t* allow,
                       uint32_t* out_ids, float* out_d, hipStream_t s) {
  if (n == 0 || kk == 0) return kOk;
  if (n == nq) return ExactScanAll(c, src, Q, nq, kk, allow, out_ids, out_d, s);
  // parts of at most 64 MiB of gathered queries and as many of results
  const size_t w = size_t(ScorePd(src));
  const size_t part = std::min(n, std::max<size_t>(1, (size_t(64) << 20) / (4 * (w + 2 * kk))));
  char* buf = nullptr;
  VDBG_HIP(hipMallocAsync(reinterpret_cast<void**>(&buf), part * (w + 2 * kk) * 4, s));
  float* q = reinterpret_cast<float*>(buf);
  uint32_t* ids = reinterpret_cast<uint32_t*>(q + part * w);
  float* d = reinterpret_cast<float*>(ids + part * kk);
  int rc = kOk;
  for (size_t i = 0; i < n && rc == kOk; i += part) {
    const size_t m = std::min(part, n - i);
    k_gather_queries<<<dim3(unsigned(m)), 256, 0, s>>>(Q, int(w), list + i, q);
    rc = ExactScanAll(c, src, q, m, kk, allow, ids, d, s);
    if (rc != kOk) break;
    k_scatter_results<<<dim3(unsigned(m)), 256, 0, s>>>(ids, d, kk, list + i, out_ids, out_d);
    if (hipGetLastError() != hipSuccess) rc = SetError(kInternal, "listed scan");
  }
  (void)hipFreeAsync(buf, s);
  return rc;
}

// Rerank (src/index/index.cc:89-95) for depths beyond the wave kernel: exact distances of
// the depth candidates per query, sorted, the first k.
__global__ void k_rerank_keys(const float* __restrict__ X, const float* __restrict__ Q, int pd,
                              int metric, int kset, const uint32_t* __restrict__ cand, int depth,
                              int nq, uint64_t* __restrict__ keys) {
  const size_t t = blockIdx.x * size_t(blockDim.x) + threadIdx.x;
  if (t >= size_t(nq) * depth) return;
  const size_t q = t / depth;
  const uint32_t id = cand[t];
  keys[t] = id == kNoId ? kNoKey
                        : dist_key(metric_exact_k(kset, metric, Q + q * pd, X + size_t(id) * pd, pd),
                                   id);
}

int RerankLarge(Ctx* c, const float* X, int pd, int metric, const float* Q, size_t nq,
                const uint32_t* cand, size_t depth, size_t k, uint32_t* out_ids, float* out_d,
                hipStream_t s) {
  if (nq == 0 || k == 0) return kOk;
  size_t chunk = std::max<size_t>(1, (size_t(256) << 20) / (depth * 8));
  chunk = std::min(chunk, nq);
  uint64_t* keys = nullptr;
  int* off = nullptr;
  const size_t nk = chunk * depth;
  VDBG_HIP(hipMallocAsync(reinterpret_cast<void**>(&keys), nk * 16 + 16, s));
  VDBG_HIP(hipMallocAsync(reinterpret_cast<void**>(&off), (chunk + 1) * sizeof(int), s));
  int rc = kOk;
  for (size_t q0 = 0; q0 < nq && rc == kOk; q0 += chunk) {
    const int nc = int(std::min(chunk, nq - q0));
    const size_t n = size_t(nc) * depth;
    {
      ProfScope ps(c, "rerank", s);
      k_rerank_keys<<<dim3(unsigned((n + 255) / 256)), 256, 0, s>>>(
          X, Q + q0 * pd, pd, metric, c->kset, cand + q0 * depth, int(depth), nc, keys);
    }
    if (hipGetLastError() != hipSuccess) {
      rc = SetError(kInternal, "rerank launch");
      break;
    }
    if (depth <= kBlockSortKeys) {
      rc = SortKeysTopK(c, SortKeysArgs{keys, uint32_t(depth), int(k), out_ids + q0 * k,
                                        out_d + q0 * k}, nc, s);
      continue;
    }
    k_seg_offsets<<<dim3(unsigned((nc + 256) / 256)), 256, 0, s>>>(off, nc, int(depth));
    rc = SortSegmentsTopK(c, keys, keys + nk, off, nc, int(n), int(k), out_ids + q0 * k,
                          out_d + q0 * k, s);
  }
  (void)hipStreamSynchronize(s);
  (void)hipFreeAsync(keys, s);
  (void)hipFreeAsync(off, s);
  return rc;
}

}  // namespace vdbg
