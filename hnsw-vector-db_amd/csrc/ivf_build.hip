// ivf_build.hip -- index construction on the GPU: AssignNearest, Lloyd's k-means, the
// product quantizer's training and the IVF-PQ build.
//
// The reference's construction (src/index/quant/kmeans.cc, pq.cc:14-41, ivf_pq.cc:102-149)
// is reproduced exactly: the seeded std::mt19937_64 draws (subsample, initialisation, empty
// cluster noise) stay on the host with the same standard-library distributions; every
// distance and assignment runs on the GPU with the reference's arithmetic (AVX-512 order for
// padded rows, L2SqAny otherwise, first minimum wins); centroid sums are fp64 over each
// cluster's members in row order (a stable radix sort by cluster, then one thread per
// (cluster, dim)), which is the order of the reference's single loop.
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <limits>
#include <numeric>
#include <random>
#include <vector>

#include "vdbg_device.h"
#include "vdbg_internal.h"

namespace vdbg {

int InstallIvf(Ctx* c, IvfIndex* x, hipStream_t s);
void FreeIvf(IvfIndex* x);
int PqEncode(Ctx* c, const float* X, uint32_t n, int pd, int dim, const float* coarse,
             const uint32_t* assign, const float* cen, int m, int dsub, uint8_t* codes,
             hipStream_t s);

namespace {

// ---------------------------------------------------------------- host distances

// l2_sq_avx512 (src/distance/avx512.cc:19-33) lane by lane, for the k-means++ pass.
float HostL2Avx512(const float* a, const float* b, size_t d) {
  float acc0[16] = {0}, acc1[16] = {0};
  size_t i = 0;
  for (; i + 32 <= d; i += 32) {
    for (int l = 0; l < 16; ++l) {
      const float d0 = a[i + l] - b[i + l];
      acc0[l] = std::fma(d0, d0, acc0[l]);
    }
    for (int l = 0; l < 16; ++l) {
      const float d1 = a[i + 16 + l] - b[i + 16 + l];
      acc1[l] = std::fma(d1, d1, acc1[l]);
    }
  }
  if (i < d)
    for (int l = 0; l < 16; ++l) {
      const float d0 = a[i + l] - b[i + l];
      acc0[l] = std::fma(d0, d0, acc0[l]);
    }
  float v[16], t3[8], t6[4];
  for (int l = 0; l < 16; ++l) v[l] = acc0[l] + acc1[l];
  for (int l = 0; l < 8; ++l) t3[l] = v[8 + l] + v[l];
  for (int l = 0; l < 4; ++l) t6[l] = t3[4 + l] + t3[l];
  return (t6[0] + t6[2]) + (t6[1] + t6[3]);
}

// L2SqAny (src/distance/scalar.cc:43-60).
float HostL2Any(const float* a, const float* b, size_t d) {
  float s0 = 0, s1 = 0, s2 = 0, s3 = 0;
  size_t i = 0;
  for (; i + 4 <= d; i += 4) {
    const float t0 = a[i] - b[i], t1 = a[i + 1] - b[i + 1];
    const float t2 = a[i + 2] - b[i + 2], t3 = a[i + 3] - b[i + 3];
    s0 += t0 * t0;
    s1 += t1 * t1;
    s2 += t2 * t2;
    s3 += t3 * t3;
  }
  for (; i < d; ++i) {
    const float t = a[i] - b[i];
    s0 += t * t;
  }
  return (s0 + s1) + (s2 + s3);
}

// l2_sq_avx2 (src/distance/avx2.cc:26-35) and l2_sq_scalar (scalar.cc:8-15).
float HostL2Avx2(const float* a, const float* b, size_t d) {
  float acc0[8] = {0}, acc1[8] = {0};
  for (size_t i = 0; i < d; i += 16)
    for (int l = 0; l < 8; ++l) {
      const float d0 = a[i + l] - b[i + l];
      acc0[l] = std::fma(d0, d0, acc0[l]);
      const float d1 = a[i + 8 + l] - b[i + 8 + l];
      acc1[l] = std::fma(d1, d1, acc1[l]);
    }
  float v[8], h[4];
  for (int l = 0; l < 8; ++l) v[l] = acc0[l] + acc1[l];
  for (int l = 0; l < 4; ++l) h[l] = v[l] + v[4 + l];
  return (h[0] + h[1]) + (h[2] + h[3]);
}
float HostL2Scalar(const float* a, const float* b, size_t d) {
  float s = 0.f;
  for (size_t i = 0; i < d; ++i) {
    const float t = a[i] - b[i];
    s += t * t;
  }
  return s;
}
float HostL2Kset(int kset, const float* a, const float* b, size_t d) {
  return kset == 2 ? HostL2Avx512(a, b, d) : kset == 1 ? HostL2Avx2(a, b, d) : HostL2Scalar(a, b, d);
}

// PickL2 (src/index/quant/kmeans.cc:16-19): the kernel set's L2 when rows are padded.
bool SimdL2(size_t d, size_t stride) { return d % 16 == 0 && stride % 16 == 0; }

}  // namespace

// ---------------------------------------------------------------- device kernels

template <int D>
__device__ __forceinline__ float l2any_fixed(const float* a, const float* b, int d) {
  const int dd = D > 0 ? D : d;
  float s0 = 0.f, s1 = 0.f, s2 = 0.f, s3 = 0.f;
  int i = 0;
#pragma unroll
  for (; i + 4 <= dd; i += 4) {
    const float t0 = a[i] - b[i], t1 = a[i + 1] - b[i + 1];
    const float t2 = a[i + 2] - b[i + 2], t3 = a[i + 3] - b[i + 3];
    s0 += t0 * t0;
    s1 += t1 * t1;
    s2 += t2 * t2;
    s3 += t3 * t3;
  }
  for (; i < dd; ++i) {
    const float t = a[i] - b[i];
    s0 += t * t;
  }
  return (s0 + s1) + (s2 + s3);
}

// AssignNearest with L2SqAny (kmeans.cc:23-55 when rows are not padded): one thread per
// point, the first centroid with the smallest distance.  Centroids staged in LDS.
template <int D>
__global__ __launch_bounds__(256) void k_assign_any(const float* __restrict__ x, uint32_t n, int d,
                                                    int stride, const float* __restrict__ cen,
                                                    int k, uint32_t* __restrict__ assign,
                                                    float* __restrict__ dist) {
  extern __shared__ float cs[];
  for (int i = threadIdx.x; i < k * d; i += blockDim.x) cs[i] = cen[i];
  __syncthreads();
  const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  float xr[D > 0 ? D : 64];
  const int dd = D > 0 ? D : d;
  for (int i = 0; i < dd; ++i) xr[i] = x[size_t(p) * stride + i];
  float best = __builtin_inff();
  uint32_t arg = 0;
  for (int c = 0; c < k; ++c) {
    const float v = l2any_fixed<D>(xr, cs + c * dd, dd);
    if (v < best) {
      best = v;
      arg = uint32_t(c);
    }
  }
  assign[p] = arg;
  if (dist != nullptr) dist[p] = best;
}

// The same for rows too wide to stage (d > 64): rows and centroids read where they lie.
__global__ __launch_bounds__(256) void k_assign_wide(const float* __restrict__ x, uint32_t n,
                                                     int d, int stride,
                                                     const float* __restrict__ cen, int k,
                                                     uint32_t* __restrict__ assign,
                                                     float* __restrict__ dist) {
  const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  const float* xr = x + size_t(p) * stride;
  float best = __builtin_inff();
  uint32_t arg = 0;
  for (int c = 0; c < k; ++c) {
    const float v = l2sq_any(xr, cen + size_t(c) * d, d);
    if (v < best) {
      best = v;
      arg = uint32_t(c);
    }
  }
  assign[p] = arg;
  if (dist != nullptr) dist[p] = best;
}

// v[i] = i mod per (per: the points of one set)
__global__ void k_iota(uint32_t* v, uint32_t n, uint32_t per) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) v[i] = i % per;
}

__global__ void k_histogram(const uint32_t* __restrict__ a, uint32_t n, uint32_t* __restrict__ counts) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) atomicAdd(&counts[a[i]], 1u);
}

// off[c] = the first place of a cluster id >= c among the sorted ids (c in [0, k]).
__global__ void k_offsets(const uint32_t* __restrict__ sorted, uint32_t n, uint32_t k,
                          uint32_t* __restrict__ off) {
  const uint32_t c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c > k) return;
  uint32_t lo = 0, hi = n;
  while (lo < hi) {
    const uint32_t mid = (lo + hi) >> 1;
    if (sorted[mid] < c) lo = mid + 1; else hi = mid;
  }
  off[c] = lo;
}

// AssignNearest with L2SqAny of several point sets at once (grid.y), one thread per point, a
// set's centroids in LDS: key = set * k + the first centroid with the smallest distance.
template <int D>
__global__ __launch_bounds__(256) void k_assign_sets(const float* __restrict__ x, uint32_t n,
                                                     int d, const float* __restrict__ cen, int k,
                                                     uint32_t* __restrict__ key) {
  extern __shared__ float cs[];
  const size_t set = blockIdx.y;
  for (int i = threadIdx.x; i < k * d; i += blockDim.x) cs[i] = cen[set * k * d + i];
  __syncthreads();
  const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  const float* xp = x + (set * n + p) * d;
  float xr[D > 0 ? D : 64];
  const int dd = D > 0 ? D : d;
  for (int i = 0; i < dd; ++i) xr[i] = xp[i];
  float best = __builtin_inff();
  uint32_t arg = 0;
#pragma unroll 2
  for (int c = 0; c < k; ++c) {
    const float v = l2any_fixed<D>(xr, cs + c * dd, dd);
    if (v < best) {
      best = v;
      arg = uint32_t(c);
    }
  }
  key[set * n + p] = uint32_t(set * k) + arg;
}

// k-means++ (kmeans.cc:92-120) of several point sets of n points at once, two launches a pick:
// k_pp_dist lowers every point's distance to its nearest pick, k_pp_pick (one block a set)
// finds the next pick as the reference's loop does.  The host has drawn each set's first pick
// and its canonical variates r (t = r total is what uniform_real_distribution(0, total) gives).
//
// That loop adds the n floats into one double in index order, and both the total and the pick
// depend on every rounding of it.  While the sum stays in one binade [2^e, 2^(e+1)) its quantum
// is u = 2^(e-52) and adding x adds exactly u rint(x / u), whatever the sum is, unless x / u
// lies halfway between integers (the even neighbour then depends on the sum) or the sum
// leaves the binade.  So a tile of points is summed in parallel in units of u (integers below
// 2^53, exact in double and associative); at the first point that ties or leaves the binade
// the block adds that point as the reference does and goes on behind it with the new quantum.
// A sum of 65,536 squares crosses about 16 binades, six of them in the first 64 points, which
// every thread adds one by one.  Every tile start and every point added by itself is a mark
// (position, sum), so the pick is searched in one stretch between marks.
//
// fail: a set with a non-finite distance, a total that is not positive, or more marks than
// are kept; the host then runs the reference's loop itself.
// Bound: one block a set, the latency of about 27 block scans a pick (66 us; 132 us with 1,024
// threads of four points, whose scans cross 16 waves).  16 sets of 65,536 points of 8 dims, 255
// picks each: 18.6 ms, where the host's loop took 700 ms.
constexpr int kPpThreads = 256, kPpPer = 16, kPpTile = kPpThreads * kPpPer, kPpMarks = 512;
constexpr int kPpHead = 64;
struct PpArgs {
  const float* x;         // set j's points at x + j xset, `stride` floats apart
  size_t xset;
  uint32_t n, n4;         // n4: mind's set stride (a multiple of 4)
  int d, stride, k, q, simd, kset;
  const uint32_t* first;  // [sets]
  const double* r;        // [sets][k - 1]
  float* mind;            // [sets][n4]
  float* cen;             // [sets][k][d]
  int* fail;              // [sets]
};

// Distances to pick q - 1 (the first pick itself is written here, q = 1); grid.y the set.
template <int D>
__global__ __launch_bounds__(256) void k_pp_dist(PpArgs a) {
  const int d = D > 0 ? D : a.d;
  const size_t set = blockIdx.y;
  const float* x = a.x + set * a.xset;
  const float* last =
      a.q == 1 ? x + size_t(a.first[set]) * a.stride : a.cen + (set * a.k + a.q - 1) * d;
  if (a.q == 1 && blockIdx.x == 0)
    for (int i = threadIdx.x; i < d; i += blockDim.x) a.cen[set * a.k * d + i] = last[i];
  float* mind = a.mind + set * a.n4;
  auto put = [&](uint32_t p, float dist) {
    const float old = a.q == 1 ? __builtin_inff() : mind[p];
    const float v = dist < old ? dist : old;
    mind[p] = v;
    if (!(v < __builtin_inff())) a.fail[set] = 1;
  };
  if (D == 0 && a.simd && a.kset == kKsetAvx512) {  // eight lanes a point, two points a group
    const uint32_t p = (blockIdx.x * 4 + (threadIdx.x >> 6)) * 16 + (lane_id() >> 3) * 2;
    const float* const xs[2] = {x + size_t(min(p, a.n - 1)) * a.stride,
                                x + size_t(min(p + 1, a.n - 1)) * a.stride};
    float v[2];
    metric_exact_g8n<2>(0, last, xs, d, v);
    if ((lane_id() & 7) < 2) {
      const uint32_t pp = p + (lane_id() & 1);
      if (pp < a.n) put(pp, (lane_id() & 1) ? v[1] : v[0]);
    }
    return;
  }
  const uint32_t p = blockIdx.x * 256 + threadIdx.x;
  if (p >= a.n) return;
  float c[D > 0 ? D : 1], xr[D > 0 ? D : 1];
  if constexpr (D > 0) {
    for (int i = 0; i < D; ++i) {
      c[i] = last[i];
      xr[i] = x[size_t(p) * a.stride + i];
    }
    put(p, l2any_fixed<D>(xr, c, D));
  } else {
    put(p, a.simd ? metric_exact_k(a.kset, 0, x + size_t(p) * a.stride, last, d)
                  : l2sq_any(x + size_t(p) * a.stride, last, d));
  }
}

// v of lane - n (0 below it) for n = 1, 2, 4, 8 inside the lane's row of 16 (DPP row_shr).
template <int N>
__device__ __forceinline__ double row_shr(double v) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const int lo = __builtin_amdgcn_update_dpp(0, int(uint32_t(b)), 0x110 + N, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_update_dpp(0, int(uint32_t(b >> 32)), 0x110 + N, 0xF, 0xF, true);
  return __builtin_bit_cast(double, uint64_t(uint32_t(lo)) | (uint64_t(uint32_t(hi)) << 32));
}
__device__ __forceinline__ double lane_of(double v, int l) {  // v of lane l (a constant)
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  return __builtin_bit_cast(
      double, uint64_t(uint32_t(__builtin_amdgcn_readlane(int(uint32_t(b)), l))) |
                  (uint64_t(uint32_t(__builtin_amdgcn_readlane(int(uint32_t(b >> 32)), l))) << 32));
}

__global__ __launch_bounds__(kPpThreads) void k_pp_pick(PpArgs a) {
  constexpr int W = kPpThreads / 64;
  __shared__ double s_wave[W];
  __shared__ int s_alone[W];
  __shared__ float s_head[kPpHead];
  __shared__ uint32_t s_hit;         // first point of the tile that ties or leaves the binade
  __shared__ double s_before, s_at;  // the sum (in u) before it, and its value
  __shared__ uint32_t s_pos[kPpMarks];
  __shared__ double s_acc[kPpMarks];
  __shared__ uint32_t s_pick;
  const int tid = threadIdx.x, wave = tid >> 6, lane = lane_id();
  const size_t set = blockIdx.x;
  if (a.fail[set] != 0) return;  // (block-uniform: written by earlier launches only)
  const float* mind = a.mind + set * a.n4;
  const double kTop = 9007199254740992.0;  // 2^53
  // the units of value v under scale = 1 / u, and whether it must be added by itself
  auto units = [&](float v, double scale, bool zero, bool& alone) {
    const double y = double(v) * scale, r = rint(y);
    alone = zero ? v != 0.f : fabs(y - r) == 0.5;
    return zero ? 0.0 : r;
  };
  // exclusive block prefix of v, and the block's sum (each exact up to the first point that
  // leaves the binade, and at least 2^53 behind it)
  // (any: whether some thread passed alone)
  auto block_scan = [&](double v, bool alone, double& sum, bool& any) {
    double incl = v;  // inside each row of 16 lanes
    incl += row_shr<1>(incl);
    incl += row_shr<2>(incl);
    incl += row_shr<4>(incl);
    incl += row_shr<8>(incl);
    const double t0 = lane_of(incl, 15), t1 = t0 + lane_of(incl, 31), t2 = t1 + lane_of(incl, 47);
    const double before = lane < 16 ? 0.0 : lane < 32 ? t0 : lane < 48 ? t1 : t2;
    const double excl = before + row_shr<1>(incl);
    __syncthreads();  // (s_wave's last readers are done)
    const bool one = __ballot(alone) != 0;
    if (lane == kWave - 1) {
      s_wave[wave] = before + incl;
      s_alone[wave] = one ? 1 : 0;
    }
    __syncthreads();
    double base = 0.0;
    sum = 0.0;
    any = false;
#pragma unroll
    for (int w = 0; w < W; ++w) {
      const double x = s_wave[w];
      base += w < wave ? x : 0.0;
      sum += x;
      any |= s_alone[w] != 0;
    }
    return base + excl;
  };
  double acc = 0.0;
  int marks = 0;
  auto mark = [&](uint32_t pos) {
    if (tid == 0 && marks < kPpMarks) {
      s_pos[marks] = pos;
      s_acc[marks] = acc;
    }
    ++marks;
  };
  auto load = [&](uint32_t p0, float (&v)[kPpPer]) {
#pragma unroll
    for (int e = 0; e < kPpPer; e += 4) {
      float4 f = make_float4(0.f, 0.f, 0.f, 0.f);
      if (p0 + e < a.n4) f = *reinterpret_cast<const float4*>(mind + p0 + e);
      v[e] = f.x;
      v[e + 1] = f.y;
      v[e + 2] = f.z;
      v[e + 3] = f.w;
    }
  };
  // the scale of the binade sum `from` lies in (1 / u), and u
  auto quantum = [&](double from, double& scale, double& u) {
    int ex = 0;
    (void)frexp(from, &ex);
    scale = ldexp(1.0, 53 - ex);
    u = ldexp(1.0, ex - 53);
  };
  // the head's points one by one (the sum would leave its binade at every second of them)
  if (tid < kPpHead) s_head[tid] = mind[tid];
  float nxt[kPpPer];
  load(tid * kPpPer, nxt);
  mark(0);
  __syncthreads();
#pragma unroll 16
  for (int i = 0; i < kPpHead; ++i) acc += double(s_head[i]);
  for (uint32_t base = 0; base < a.n; base += kPpTile) {
    const uint32_t p0 = base + tid * kPpPer;
    float v[kPpPer];
#pragma unroll
    for (int e = 0; e < kPpPer; ++e) v[e] = nxt[e];  // (zero past the set's points)
    load(p0 + kPpTile, nxt);  // the next tile's, while this one is summed
    uint32_t pos = max(base, uint32_t(kPpHead));  // points before it are in acc
    mark(pos);
    for (;;) {  // (pos grows every round: at most kPpTile rounds)
      const bool zero = acc == 0.0;
      double scale, u;
      quantum(acc, scale, u);
      const double A = acc * scale;
      double mine = 0.0;
      bool alone = false;
#pragma unroll
      for (int e = 0; e < kPpPer; ++e) {
        bool al;
        const double y = units(v[e], scale, zero, al);
        const bool in = p0 + e >= pos;
        mine += in ? y : 0.0;
        alone |= al && in;
      }
      if (tid == 0) s_hit = 0xffffffffu;
      double sum;
      bool any;
      double run = A + block_scan(mine, alone, sum, any);
      if (!any && A + sum < kTop) {  // (block-uniform)
        acc = (A + sum) * u;
        break;
      }
      if (alone || run + mine >= kTop) {
#pragma unroll
        for (int e = 0; e < kPpPer; ++e) {
          if (p0 + e < pos) continue;
          bool al;
          const double y = units(v[e], scale, zero, al);
          if (al || run + y >= kTop) {
            atomicMin(&s_hit, p0 + e);
            break;
          }
          run += y;
        }
      }
      __syncthreads();
      const uint32_t hit = s_hit;
      if (hit >= p0 && hit < p0 + kPpPer) {  // (run stopped in front of it)
        s_before = run;
#pragma unroll
        for (int e = 0; e < kPpPer; ++e)
          if (hit == p0 + e) s_at = double(v[e]);
      }
      __syncthreads();
      acc = s_before * u + s_at;
      pos = hit + 1;
      mark(pos);
      if (marks > kPpMarks) break;
    }
    if (marks > kPpMarks) break;
  }
  __syncthreads();
  if (marks > kPpMarks || !(acc > 0.0) || !(acc < double(__builtin_inff()))) {
    if (tid == 0) a.fail[set] = 1;
    return;  // (block-uniform)
  }
  // the first point whose sum reaches t, in the stretch behind the last mark below t
  const double t = a.r[set * (a.k - 1) + (a.q - 1)] * acc;
  if (tid == 0) s_pick = 0xffffffffu;
  int mk = 0;
  while (mk + 1 < marks && s_acc[mk + 1] < t) ++mk;
  const uint32_t lo = s_pos[mk], hi = mk + 1 < marks ? s_pos[mk + 1] : a.n;
  if (mk == 0) {  // in the head
    double run = 0.0;
    uint32_t at = kPpHead - 1;
    for (int i = 0; i < kPpHead; ++i) {
      run += double(s_head[i]);
      if (run >= t) {
        at = uint32_t(i);
        break;
      }
    }
    __syncthreads();
    if (tid == 0) s_pick = at;
  } else {
    const double from = s_acc[mk];
    const bool zero = from == 0.0;
    double scale, u;
    quantum(from, scale, u);
    // (a stretch lies inside one tile; one that a point by itself ends holds that point last)
    const uint32_t p0 = lo / kPpTile * kPpTile + tid * kPpPer;
    float v[kPpPer];
    load(p0, v);
    double mine = 0.0;
    bool al;
#pragma unroll
    for (int e = 0; e < kPpPer; ++e) {
      if (p0 + e < lo || p0 + e >= hi) v[e] = 0.f;
      mine += units(v[e], scale, zero, al);
    }
    double sum;
    bool any;
    double run = from * scale + block_scan(mine, false, sum, any);
#pragma unroll
    for (int e = 0; e < kPpPer; ++e) {
      run += units(v[e], scale, zero, al);
      if (p0 + e >= lo && p0 + e < hi && run * u >= t) {
        atomicMin(&s_pick, p0 + e);
        break;
      }
    }
  }
  __syncthreads();
  // none inside: the point by itself that ends the stretch reached t (behind the last mark
  // the reference's loop ends on the last point)
  const uint32_t pick = s_pick != 0xffffffffu ? s_pick : hi - 1;
  const float* xp = a.x + set * a.xset + size_t(pick) * a.stride;
  for (int i = tid; i < a.d; i += kPpThreads) a.cen[(set * a.k + a.q) * a.d + i] = xp[i];
}

// Centroid update (kmeans.cc:146-158): fp64 sums of each cluster's members in row order,
// float(sum * (1.0 / count)) for non-empty clusters.  grid = clusters, threads over dims;
// clusters come in sets of `per` (a set per point set, xset floats apart).  Bound: the latency
// of one chain of dependent adds per (cluster, dim); with one member's load at a time behind
// each add it took 100 us for 256 clusters of 256 points.
__global__ void k_centroid_update(const float* __restrict__ x, int d, int stride, int per,
                                  size_t xset, const uint32_t* __restrict__ order,
                                  const uint32_t* __restrict__ off, float* __restrict__ cen) {
  const int c = blockIdx.x;
  const uint32_t b = off[c], e = off[c + 1];
  if (b == e) return;
  const double inv = 1.0 / double(e - b);
  x += size_t(c / per) * xset;
  for (int j = threadIdx.x; j < d; j += blockDim.x) {
    double s = 0.0;
    uint32_t t = b;
    for (; t + 16 <= e; t += 16) {  // sixteen members' loads in flight, added in row order
      float v[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) v[i] = x[size_t(order[t + i]) * stride + j];
#pragma unroll
      for (int i = 0; i < 16; ++i) s += double(v[i]);
    }
    for (; t < e; ++t) s += double(x[size_t(order[t]) * stride + j]);
    cen[size_t(c) * d + j] = float(s * inv);
  }
}

__global__ void k_gather_rows(const float* __restrict__ x, int stride, const uint32_t* __restrict__ idx,
                              uint32_t n, int d, int xo, float* __restrict__ out) {
  const size_t t = blockIdx.x * size_t(blockDim.x) + threadIdx.x;
  if (t >= size_t(n) * d) return;
  const size_t r = t / d, j = t - r * d;
  out[t] = x[size_t(idx[r]) * stride + xo + j];
}

// Residuals x - coarse[assign] over the real dims (ivf_pq.cc:116-124, 128-139).
__global__ void k_residuals(const float* __restrict__ X, int pd, int dim,
                            const float* __restrict__ coarse, const uint32_t* __restrict__ assign,
                            const uint32_t* __restrict__ rows, uint32_t nrows, float* __restrict__ out) {
  const size_t t = blockIdx.x * size_t(blockDim.x) + threadIdx.x;
  if (t >= size_t(nrows) * dim) return;
  const size_t r = t / dim, j = t - r * dim;
  const uint32_t i = rows[r];
  out[t] = X[size_t(i) * pd + j] - coarse[size_t(assign[i]) * pd + j];
}

__global__ void k_gather_codes(const uint8_t* __restrict__ all, const uint32_t* __restrict__ order,
                               uint32_t n, int m, uint8_t* __restrict__ out) {
  const size_t t = blockIdx.x * size_t(blockDim.x) + threadIdx.x;
  if (t >= size_t(n) * m) return;
  const size_t r = t / m, j = t - r * m;
  out[t] = all[size_t(order[r]) * m + j];
}

// ---------------------------------------------------------------- host orchestration

struct DevBuf {
  void* p = nullptr;
  hipStream_t s = nullptr;
  ~DevBuf() {
    if (p) (void)hipFreeAsync(p, s);
  }
  template <class T>
  T* get() const {
    return static_cast<T*>(p);
  }
};

static int Alloc(DevBuf* b, size_t bytes, hipStream_t s) {
  b->s = s;
  VDBG_HIP(hipMallocAsync(&b->p, std::max<size_t>(bytes, 16), s));
  return kOk;
}

// AssignNearest (kmeans.cc:23-55): x is n rows of d floats at `stride`, centroids k x d
// (device).  Padded rows go through the exact scan with k = 1 (AVX-512 order, ties to the
// lowest index); other shapes through L2SqAny.
int AssignNearestGpu(Ctx* c, const float* x, size_t n, size_t d, size_t stride, const float* cen,
                     size_t k, uint32_t* assign, float* dist, hipStream_t s) {
  if (n == 0) return kOk;
  if (SimdL2(d, stride)) {
    if (stride != d) return SetError(kNotSupported, "AssignNearest: padded rows need stride == d");
    vdbg_dataset* cds = nullptr;
    VDBG_RETURN_IF_ERROR(vdbg_dataset_create_device(c->handle, cen, k, d, d, 0, &cds));
    DevBuf dd;
    int rc = dist ? kOk : Alloc(&dd, n * sizeof(float), s);
    if (rc == kOk) rc = RunScan(c, &cds->d.src, x, n, 1, nullptr, assign, dist ? dist : dd.get<float>(), s);
    if (rc == kOk) rc = hipStreamSynchronize(s) == hipSuccess ? kOk : SetError(kInternal, "sync");
    vdbg_dataset_destroy(cds);
    return rc;
  }
  const size_t lds = k * d * sizeof(float);
  ProfScope ps(c, "assign_any", s);
  const dim3 grid(unsigned((n + 255) / 256));
  if (d > 64 || lds > 64 * 1024) {
    k_assign_wide<<<grid, 256, 0, s>>>(x, uint32_t(n), int(d), int(stride), cen, int(k), assign,
                                       dist);
    VDBG_HIP(hipGetLastError());
    return kOk;
  }
#define VDBG_ASSIGN(DD) k_assign_any<DD><<<grid, 256, lds, s>>>(x, uint32_t(n), int(d), int(stride), cen, int(k), assign, dist)
  switch (d) {
    case 4: VDBG_ASSIGN(4); break;
    case 8: VDBG_ASSIGN(8); break;
    case 12: VDBG_ASSIGN(12); break;
    case 24: VDBG_ASSIGN(24); break;
    default: VDBG_ASSIGN(0); break;
  }
#undef VDBG_ASSIGN
  VDBG_HIP(hipGetLastError());
  return kOk;
}

struct KMeansOpts {
  size_t iters = 25;
  uint64_t seed = 1234;
  size_t max_points = 256;
  bool kmeanspp = true;
};

struct KMeansInfo {
  double inertia = 0;
  size_t train_points = 0, empty_reseeds = 0, iterations = 0;
};

// k-means++ initialisation of `sets` point sets on the device (k_pp_dist, k_pp_pick): x + j xset
// holds set j's n points `stride` apart, dcen receives [sets][k][d], and each set's generator is
// advanced by the draws the reference makes.  *failed: a set needs the host's loop (no
// generator is advanced then).
int KMeansPPGpu(Ctx* c, const float* x, size_t xset, size_t sets, size_t n, size_t d, size_t stride,
                size_t k, std::vector<std::mt19937_64>* rngs, float* dcen, bool* failed,
                hipStream_t s) {
  std::vector<std::mt19937_64> drawn = *rngs;
  std::vector<uint32_t> first(sets);
  std::vector<double> r(sets * std::max<size_t>(1, k - 1));
  for (size_t j = 0; j < sets; ++j) {
    std::uniform_int_distribution<size_t> u0(0, n - 1);
    first[j] = uint32_t(u0(drawn[j]));
    std::uniform_real_distribution<double> u(0.0, 1.0);
    for (size_t q = 0; q + 1 < k; ++q) r[j * (k - 1) + q] = u(drawn[j]);
  }
  const size_t n4 = (n + 3) / 4 * 4;
  DevBuf df, dr, dm, dfail;
  VDBG_RETURN_IF_ERROR(Alloc(&df, sets * 4, s));
  VDBG_RETURN_IF_ERROR(Alloc(&dr, r.size() * 8, s));
  VDBG_RETURN_IF_ERROR(Alloc(&dm, sets * n4 * 4, s));
  VDBG_RETURN_IF_ERROR(Alloc(&dfail, sets * 4, s));
  VDBG_HIP(hipMemcpyAsync(df.p, first.data(), sets * 4, hipMemcpyHostToDevice, s));
  VDBG_HIP(hipMemcpyAsync(dr.p, r.data(), r.size() * 8, hipMemcpyHostToDevice, s));
  VDBG_RETURN_IF_ERROR(Fill32(dfail.p, 0, sets, s));
  VDBG_RETURN_IF_ERROR(Fill32(dm.p, 0, sets * n4, s));  // (the padding after each set's points)
  PpArgs a{x, xset, uint32_t(n), uint32_t(n4), int(d), int(stride), int(k), 1,
           SimdL2(d, stride) ? 1 : 0, c->kset, df.get<uint32_t>(), dr.get<double>(),
           dm.get<float>(), dcen, dfail.get<int>()};
  const bool group = a.simd && c->kset == kKsetAvx512;
  const dim3 grid(unsigned(group ? (n + 63) / 64 : (n + 255) / 256), unsigned(sets));
  {
    ProfScope ps(c, "kmeanspp", s);
    for (size_t q = 1; q < std::max<size_t>(k, 2); ++q) {
      a.q = int(q);
      if (a.simd) k_pp_dist<0><<<grid, 256, 0, s>>>(a);
      else if (d == 4) k_pp_dist<4><<<grid, 256, 0, s>>>(a);
      else if (d == 8) k_pp_dist<8><<<grid, 256, 0, s>>>(a);
      else if (d == 12) k_pp_dist<12><<<grid, 256, 0, s>>>(a);
      else k_pp_dist<0><<<grid, 256, 0, s>>>(a);
      if (q < k) k_pp_pick<<<dim3(unsigned(sets)), kPpThreads, 0, s>>>(a);
    }
    VDBG_HIP(hipGetLastError());
  }
  std::vector<int> fail(sets);
  VDBG_HIP(hipMemcpyAsync(fail.data(), dfail.p, sets * 4, hipMemcpyDeviceToHost, s));
  VDBG_HIP(hipStreamSynchronize(s));
  *failed = std::any_of(fail.begin(), fail.end(), [](int f) { return f != 0; });
  if (!*failed) *rngs = std::move(drawn);
  return kOk;
}
// Where the device pass is the faster one.  It takes two launches a pick for all sets, 28 us and
// 0.6 ns a point; the host's loop, a set at a time, 2.9 ns a point or 0.24 a dim where that is
// more, 1.1 a dim in the kernel sets' order (a whole call of 64 picks, host / device in ms:
// 4,096 x 8 1.2 / 2.4, 12,288 x 8 2.7 / 3.0, 16,384 x 8 3.4 / 3.2, 65,536 x 8 13.4 / 5.3, 4,096 x
// 24 2.0 / 2.5, 8,192 x 24 3.7 / 2.9, 4,096 x 32 9.8 / 2.7).  One block's marks cover kPpMarks
// tiles at most.
bool KMeansPPOnGpu(size_t n, size_t d, size_t stride, size_t sets) {
  if (n < 4096 || n > size_t(kPpTile) * (kPpMarks / 2)) return false;
  const double host =
      SimdL2(d, stride) ? 1.1e-3 * double(d) : std::max(2.9e-3, 0.24e-3 * double(d));
  return host * double(n) * double(sets) > 28.0 + 0.6e-3 * double(n);
}

// The empty clusters of one iteration (kmeans.cc:159-172): the largest split in two with a
// symmetric perturbation.  cen: k x d on the host.
void SplitLargest(float* cen, size_t k, size_t d, const uint32_t* cnt, std::mt19937_64& rng,
                  size_t* reseeds) {
  constexpr float kEps = 1.0f / 1024.0f;
  std::vector<size_t> counts(cnt, cnt + k);
  for (size_t q = 0; q < k; ++q) {
    if (counts[q] != 0) continue;
    const size_t big =
        static_cast<size_t>(std::max_element(counts.begin(), counts.end()) - counts.begin());
    std::uniform_real_distribution<float> noise(-1.f, 1.f);
    for (size_t j = 0; j < d; ++j) {
      const float v = cen[big * d + j];
      const float delta = kEps * (std::fabs(v) + 1e-3f) * noise(rng);
      cen[q * d + j] = v + delta;
      cen[big * d + j] = v - delta;
    }
    counts[q] = counts[big] / 2;
    counts[big] -= counts[q];
    ++*reseeds;
  }
}

unsigned UpdateThreads(size_t d) { return unsigned(std::min<size_t>(256, (d + 63) / 64 * 64)); }

// KMeans (kmeans.cc:57-174) over n device rows of d floats at `stride`.
int KMeansGpu(Ctx* c, const float* data, size_t n, size_t d, size_t stride, size_t k,
              const KMeansOpts& o, std::vector<float>* centroids, KMeansInfo* info, hipStream_t s) {
  if (k == 0 || d == 0) return SetError(kInvalidArgument, "k-means needs k > 0 and d > 0");
  if (n == 0) return SetError(kInvalidArgument, "k-means needs training points");
  centroids->assign(k * d, 0.f);
  std::mt19937_64 rng(o.seed);
  KMeansInfo st;

  // Fewer points than centroids: the points themselves, with duplicates.
  if (n <= k) {
    std::vector<float> rows(n * stride);
    VDBG_HIP(hipMemcpyAsync(rows.data(), data, n * stride * sizeof(float), hipMemcpyDeviceToHost, s));
    VDBG_HIP(hipStreamSynchronize(s));
    for (size_t q = 0; q < k; ++q)
      std::memcpy(centroids->data() + q * d, rows.data() + (q % n) * stride, d * sizeof(float));
    st.train_points = n;
    if (info) *info = st;
    return kOk;
  }

  // Subsample to k * max_points rows: partial Fisher-Yates, then sorted.
  const size_t m = std::min(n, k * std::max<size_t>(1, o.max_points));
  DevBuf sample;
  const float* x = data;
  size_t xs = stride;
  if (m < n) {
    std::vector<size_t> idx(n);
    std::iota(idx.begin(), idx.end(), 0);
    for (size_t i = 0; i < m; ++i) {
      std::uniform_int_distribution<size_t> u(i, n - 1);
      std::swap(idx[i], idx[u(rng)]);
    }
    std::sort(idx.begin(), idx.begin() + static_cast<std::ptrdiff_t>(m));
    std::vector<uint32_t> idx32(idx.begin(), idx.begin() + static_cast<std::ptrdiff_t>(m));
    DevBuf di;
    VDBG_RETURN_IF_ERROR(Alloc(&di, m * 4, s));
    VDBG_RETURN_IF_ERROR(Alloc(&sample, m * d * sizeof(float), s));
    VDBG_HIP(hipMemcpyAsync(di.p, idx32.data(), m * 4, hipMemcpyHostToDevice, s));
    k_gather_rows<<<dim3(unsigned((m * d + 255) / 256)), 256, 0, s>>>(
        data, int(stride), di.get<uint32_t>(), uint32_t(m), int(d), 0, sample.get<float>());
    VDBG_HIP(hipGetLastError());
    VDBG_HIP(hipStreamSynchronize(s));
    x = sample.get<float>();
    xs = d;
  }
  const bool simd = SimdL2(d, xs);
  auto fn = [&](const float* a, const float* b) {
    return simd ? HostL2Kset(c->kset, a, b, d) : HostL2Any(a, b, d);
  };

  // Initialisation.
  float* cen = centroids->data();
  const bool use_pp = o.kmeanspp && static_cast<double>(k) * static_cast<double>(m) <= 2.0e7;
  bool host_pp = use_pp;
  if (use_pp && KMeansPPOnGpu(m, d, xs, 1)) {
    DevBuf dc;
    VDBG_RETURN_IF_ERROR(Alloc(&dc, k * d * sizeof(float), s));
    std::vector<std::mt19937_64> rngs{rng};
    VDBG_RETURN_IF_ERROR(KMeansPPGpu(c, x, 0, 1, m, d, xs, k, &rngs, dc.get<float>(), &host_pp, s));
    if (!host_pp) {
      rng = rngs[0];
      VDBG_HIP(hipMemcpyAsync(cen, dc.p, k * d * sizeof(float), hipMemcpyDeviceToHost, s));
      VDBG_HIP(hipStreamSynchronize(s));
    }
  }
  if (host_pp) {
    std::vector<float> xh(m * xs);
    VDBG_HIP(hipMemcpyAsync(xh.data(), x, m * xs * sizeof(float), hipMemcpyDeviceToHost, s));
    VDBG_HIP(hipStreamSynchronize(s));
    std::vector<float> mind(m, std::numeric_limits<float>::infinity());
    std::uniform_int_distribution<size_t> u0(0, m - 1);
    const size_t first = u0(rng);
    std::memcpy(cen, xh.data() + first * xs, d * sizeof(float));
    for (size_t q = 1; q < k; ++q) {
      const float* last = cen + (q - 1) * d;
      double total = 0;
      for (size_t i = 0; i < m; ++i) {
        mind[i] = std::min(mind[i], fn(xh.data() + i * xs, last));
        total += mind[i];
      }
      size_t pick = 0;
      if (total > 0) {
        std::uniform_real_distribution<double> ur(0.0, total);
        const double t = ur(rng);
        double acc = 0;
        for (pick = 0; pick + 1 < m; ++pick) {
          acc += mind[pick];
          if (acc >= t) break;
        }
      } else {
        pick = u0(rng);
      }
      std::memcpy(cen + q * d, xh.data() + pick * xs, d * sizeof(float));
    }
  } else if (!use_pp) {
    std::vector<size_t> idx(m);
    std::iota(idx.begin(), idx.end(), 0);
    std::vector<uint32_t> rows(k);
    for (size_t q = 0; q < k; ++q) {
      std::uniform_int_distribution<size_t> u(q, m - 1);
      std::swap(idx[q], idx[u(rng)]);
      rows[q] = uint32_t(idx[q]);
    }
    DevBuf dr, dc;
    VDBG_RETURN_IF_ERROR(Alloc(&dr, k * 4, s));
    VDBG_RETURN_IF_ERROR(Alloc(&dc, k * d * sizeof(float), s));
    VDBG_HIP(hipMemcpyAsync(dr.p, rows.data(), k * 4, hipMemcpyHostToDevice, s));
    k_gather_rows<<<dim3(unsigned((k * d + 255) / 256)), 256, 0, s>>>(
        x, int(xs), dr.get<uint32_t>(), uint32_t(k), int(d), 0, dc.get<float>());
    VDBG_HIP(hipGetLastError());
    VDBG_HIP(hipMemcpyAsync(cen, dc.p, k * d * sizeof(float), hipMemcpyDeviceToHost, s));
    VDBG_HIP(hipStreamSynchronize(s));
  }

  // Lloyd iterations.
  DevBuf dcen, assign, dist, keys_out, vals_in, vals_out, off, tmp;
  VDBG_RETURN_IF_ERROR(Alloc(&dcen, k * d * sizeof(float), s));
  VDBG_RETURN_IF_ERROR(Alloc(&assign, m * 4, s));
  VDBG_RETURN_IF_ERROR(Alloc(&dist, m * 4, s));
  VDBG_RETURN_IF_ERROR(Alloc(&keys_out, m * 4, s));
  VDBG_RETURN_IF_ERROR(Alloc(&vals_in, m * 4, s));
  VDBG_RETURN_IF_ERROR(Alloc(&vals_out, m * 4, s));
  VDBG_RETURN_IF_ERROR(Alloc(&off, (k + 1) * 4, s));
  int end_bit = 1;
  while ((size_t(1) << end_bit) < k) ++end_bit;
  size_t tmp_bytes = 0;
  VDBG_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, tmp_bytes, assign.get<uint32_t>(),
                                              keys_out.get<uint32_t>(), vals_in.get<uint32_t>(),
                                              vals_out.get<uint32_t>(), int(m), 0, end_bit, s));
  VDBG_RETURN_IF_ERROR(Alloc(&tmp, tmp_bytes, s));
  k_iota<<<dim3(unsigned((m + 255) / 256)), 256, 0, s>>>(vals_in.get<uint32_t>(), uint32_t(m),
                                                         uint32_t(m));
  VDBG_HIP(hipGetLastError());
  std::vector<uint32_t> cnt(k), offh(k + 1);
  st.train_points = m;
  VDBG_HIP(hipMemcpyAsync(dcen.p, cen, k * d * sizeof(float), hipMemcpyHostToDevice, s));
  for (size_t it = 0; it < o.iters; ++it) {
    VDBG_RETURN_IF_ERROR(AssignNearestGpu(c, x, m, d, xs, dcen.get<float>(), k,
                                          assign.get<uint32_t>(), dist.get<float>(), s));
    VDBG_HIP(hipcub::DeviceRadixSort::SortPairs(tmp.p, tmp_bytes, assign.get<uint32_t>(),
                                                keys_out.get<uint32_t>(), vals_in.get<uint32_t>(),
                                                vals_out.get<uint32_t>(), int(m), 0, end_bit, s));
    k_offsets<<<dim3(unsigned(k / 256 + 1)), 256, 0, s>>>(keys_out.get<uint32_t>(), uint32_t(m),
                                                          uint32_t(k), off.get<uint32_t>());
    k_centroid_update<<<dim3(unsigned(k)), UpdateThreads(d), 0, s>>>(
        x, int(d), int(xs), int(k), 0, vals_out.get<uint32_t>(), off.get<uint32_t>(),
        dcen.get<float>());
    VDBG_HIP(hipGetLastError());
    VDBG_HIP(hipMemcpyAsync(offh.data(), off.p, (k + 1) * 4, hipMemcpyDeviceToHost, s));
    VDBG_HIP(hipMemcpyAsync(cen, dcen.p, k * d * sizeof(float), hipMemcpyDeviceToHost, s));
    VDBG_HIP(hipStreamSynchronize(s));
    size_t empty = 0;
    for (size_t q = 0; q < k; ++q) {
      cnt[q] = offh[q + 1] - offh[q];
      empty += cnt[q] == 0 ? 1 : 0;
    }
    if (empty > 0) {
      SplitLargest(cen, k, d, cnt.data(), rng, &st.empty_reseeds);
      VDBG_HIP(hipMemcpyAsync(dcen.p, cen, k * d * sizeof(float), hipMemcpyHostToDevice, s));
    }
    st.iterations = it + 1;
  }
  if (info != nullptr && o.iters > 0) {  // the last assignment's distances, summed in row order
    std::vector<float> disth(m);
    VDBG_HIP(hipMemcpyAsync(disth.data(), dist.p, m * 4, hipMemcpyDeviceToHost, s));
    VDBG_HIP(hipStreamSynchronize(s));
    for (size_t i = 0; i < m; ++i) st.inertia += disth[i];
  }
  if (info) *info = st;
  VDBG_HIP(hipStreamSynchronize(s));  // (copies from this call's host arrays have completed)
  return kOk;
}

// Lloyd iterations of m sub-quantizers at once (PqTrainGpu): x [m][n][d] training sub-vectors,
// dcen [m][256][d] initial centroids, both on the device, distances in L2SqAny order.  One
// assignment, one stable sort by (set, cluster), one update and one small copy back an
// iteration, where a set at a time took the same launches and two waits each.
int LloydSets(Ctx* c, const float* x, size_t m, size_t n, size_t d, float* dcen, size_t iters,
              std::vector<std::mt19937_64>* rngs, hipStream_t s) {
  constexpr size_t k = 256;
  const size_t total = m * n;
  DevBuf key, skey, vals, order, off, tmp;
  VDBG_RETURN_IF_ERROR(Alloc(&key, total * 4, s));
  VDBG_RETURN_IF_ERROR(Alloc(&skey, total * 4, s));
  VDBG_RETURN_IF_ERROR(Alloc(&vals, total * 4, s));
  VDBG_RETURN_IF_ERROR(Alloc(&order, total * 4, s));
  VDBG_RETURN_IF_ERROR(Alloc(&off, (m * k + 1) * 4, s));
  int end_bit = 8;
  while ((size_t(1) << end_bit) < m * k) ++end_bit;
  size_t tmp_bytes = 0;
  VDBG_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, tmp_bytes, key.get<uint32_t>(),
                                              skey.get<uint32_t>(), vals.get<uint32_t>(),
                                              order.get<uint32_t>(), int(total), 0, end_bit, s));
  VDBG_RETURN_IF_ERROR(Alloc(&tmp, tmp_bytes, s));
  k_iota<<<dim3(unsigned((total + 255) / 256)), 256, 0, s>>>(vals.get<uint32_t>(), uint32_t(total),
                                                             uint32_t(n));
  const dim3 grid(unsigned((n + 255) / 256), unsigned(m));
  const size_t lds = k * d * sizeof(float);
  std::vector<uint32_t> offh(m * k + 1), cnt(k);
  std::vector<float> cen;
  for (size_t it = 0; it < iters; ++it) {
    {
      ProfScope ps(c, "assign_any", s);
      uint32_t* kp = key.get<uint32_t>();
#define VDBG_SETS(DD) k_assign_sets<DD><<<grid, 256, lds, s>>>(x, uint32_t(n), int(d), dcen, int(k), kp)
      switch (d) {
        case 4: VDBG_SETS(4); break;
        case 8: VDBG_SETS(8); break;
        case 12: VDBG_SETS(12); break;
        case 24: VDBG_SETS(24); break;
        default: VDBG_SETS(0); break;
      }
#undef VDBG_SETS
    }
    VDBG_HIP(hipcub::DeviceRadixSort::SortPairs(tmp.p, tmp_bytes, key.get<uint32_t>(),
                                                skey.get<uint32_t>(), vals.get<uint32_t>(),
                                                order.get<uint32_t>(), int(total), 0, end_bit, s));
    k_offsets<<<dim3(unsigned(m * k / 256 + 1)), 256, 0, s>>>(
        skey.get<uint32_t>(), uint32_t(total), uint32_t(m * k), off.get<uint32_t>());
    k_centroid_update<<<dim3(unsigned(m * k)), UpdateThreads(d), 0, s>>>(
        x, int(d), int(d), int(k), n * d, order.get<uint32_t>(), off.get<uint32_t>(), dcen);
    VDBG_HIP(hipGetLastError());
    VDBG_HIP(hipMemcpyAsync(offh.data(), off.p, offh.size() * 4, hipMemcpyDeviceToHost, s));
    VDBG_HIP(hipStreamSynchronize(s));
    bool empty = false;
    for (size_t q = 0; q < m * k; ++q) empty |= offh[q + 1] == offh[q];
    if (!empty) continue;
    cen.resize(m * k * d);
    VDBG_HIP(hipMemcpyAsync(cen.data(), dcen, cen.size() * 4, hipMemcpyDeviceToHost, s));
    VDBG_HIP(hipStreamSynchronize(s));
    for (size_t j = 0; j < m; ++j) {
      for (size_t q = 0; q < k; ++q) cnt[q] = offh[j * k + q + 1] - offh[j * k + q];
      size_t reseeds = 0;
      SplitLargest(cen.data() + j * k * d, k, d, cnt.data(), (*rngs)[j], &reseeds);
    }
    VDBG_HIP(hipMemcpyAsync(dcen, cen.data(), cen.size() * 4, hipMemcpyHostToDevice, s));
    VDBG_HIP(hipStreamSynchronize(s));
  }
  return kOk;
}

// ProductQuantizer::train (src/index/quant/pq.cc:14-41) on n device rows at `stride`.
int PqTrainGpu(Ctx* c, const float* data, size_t n, size_t stride, size_t dim, size_t m,
               const KMeansOpts& opts, std::vector<float>* centroids, hipStream_t s) {
  if (m == 0 || dim % m != 0)
    return SetError(kInvalidArgument, "pq_m must divide the dimension (dim " + std::to_string(dim) +
                                          ", m " + std::to_string(m) + ")");
  const size_t dsub = dim / m;
  centroids->assign(m * 256 * dsub, 0.f);
  const size_t cap = std::min(n, size_t(256) * std::max<size_t>(1, opts.max_points));
  const size_t step = std::max<size_t>(1, n / std::max<size_t>(1, cap));
  std::vector<uint32_t> rows;
  for (size_t i = 0, taken = 0; i < n && taken < cap; i += step, ++taken) rows.push_back(uint32_t(i));
  DevBuf dr, sub;
  VDBG_RETURN_IF_ERROR(Alloc(&dr, rows.size() * 4, s));
  VDBG_HIP(hipMemcpyAsync(dr.p, rows.data(), rows.size() * 4, hipMemcpyHostToDevice, s));
  // All m sub-quantizers at once: narrow sub-vectors of enough points to initialise on the
  // device, whose training sets fit 1 GiB and whose (set, row) pairs a 32-bit sort takes.
  const size_t np = rows.size();
  if (opts.kmeanspp && KMeansPPOnGpu(np, dsub, dsub, m) && 256.0 * double(np) <= 2.0e7 &&
      dsub <= 64 &&
      !SimdL2(dsub, dsub) && np * dim * 4 <= (size_t(1) << 30) && m * np < (size_t(1) << 31) &&
      m <= 65535) {
    VDBG_RETURN_IF_ERROR(Alloc(&sub, m * np * dsub * sizeof(float), s));
    for (size_t j = 0; j < m; ++j)
      k_gather_rows<<<dim3(unsigned((np * dsub + 255) / 256)), 256, 0, s>>>(
          data, int(stride), dr.get<uint32_t>(), uint32_t(np), int(dsub), int(j * dsub),
          sub.get<float>() + j * np * dsub);
    VDBG_HIP(hipGetLastError());
    std::vector<std::mt19937_64> rngs;
    for (size_t j = 0; j < m; ++j) rngs.emplace_back(opts.seed + j * 7919);
    DevBuf dcen;
    VDBG_RETURN_IF_ERROR(Alloc(&dcen, centroids->size() * sizeof(float), s));
    bool failed = false;
    VDBG_RETURN_IF_ERROR(KMeansPPGpu(c, sub.get<float>(), np * dsub, m, np, dsub, dsub, 256, &rngs,
                                     dcen.get<float>(), &failed, s));
    if (!failed) {
      VDBG_RETURN_IF_ERROR(LloydSets(c, sub.get<float>(), m, np, dsub, dcen.get<float>(),
                                     opts.iters, &rngs, s));
      VDBG_HIP(hipMemcpyAsync(centroids->data(), dcen.p, centroids->size() * sizeof(float),
                              hipMemcpyDeviceToHost, s));
      VDBG_HIP(hipStreamSynchronize(s));
      return kOk;
    }
  } else {
    VDBG_RETURN_IF_ERROR(Alloc(&sub, rows.size() * dsub * sizeof(float), s));
  }
  std::vector<float> cen;
  for (size_t j = 0; j < m; ++j) {
    k_gather_rows<<<dim3(unsigned((rows.size() * dsub + 255) / 256)), 256, 0, s>>>(
        data, int(stride), dr.get<uint32_t>(), uint32_t(rows.size()), int(dsub), int(j * dsub),
        sub.get<float>());
    VDBG_HIP(hipGetLastError());
    KMeansOpts o = opts;
    o.seed = opts.seed + j * 7919;
    VDBG_RETURN_IF_ERROR(KMeansGpu(c, sub.get<float>(), rows.size(), dsub, dsub, 256, o, &cen,
                                   nullptr, s));
    std::memcpy(centroids->data() + j * 256 * dsub, cen.data(), 256 * dsub * sizeof(float));
  }
  return kOk;
}

// ProductQuantizer::train with IndexOptions' k-means settings (MakeKMeansOptions,
// ivf_pq.cc:21-26), for callers outside this file (PqFlatIndex::build).
int PqTrainRows(Ctx* c, const float* data, size_t n, size_t stride, size_t dim, size_t m,
                uint64_t seed, size_t max_points, size_t iters, std::vector<float>* centroids,
                hipStream_t s) {
  KMeansOpts ko;
  ko.seed = seed;
  ko.max_points = max_points;
  ko.iters = iters;
  return PqTrainGpu(c, data, n, stride, dim, m, ko, centroids, s);
}

// IvfPqIndex::build (ivf_pq.cc:102-149).
int IvfBuildGpu(Ctx* c, IvfIndex* x, size_t nlist_req, size_t m, uint64_t seed, size_t max_points,
                size_t iters, hipStream_t s) {
  Dataset* ds = x->ds;
  const size_t n = ds->n, pd = ds->pd, d = ds->dim;
  if (m == 0 || d % m != 0) return SetError(kInvalidArgument, "pq_m must divide the dimension");
  x->pd = int(pd);
  x->dim = int(d);
  x->m = int(m);
  x->dsub = int(d / m);
  x->metric = ds->metric;
  if (n == 0) {
    x->nlist = 0;
    x->off_h.assign(1, 0);
    return kOk;
  }
  // Small segments get fewer lists (FAISS warns below 39 training points per centroid).
  const size_t nlist = std::clamp<size_t>(nlist_req, 1, std::max<size_t>(1, n / 39));
  x->nlist = int(nlist);
  KMeansOpts ko;
  ko.seed = seed;
  ko.max_points = max_points;
  ko.iters = iters;
  VDBG_RETURN_IF_ERROR(KMeansGpu(c, ds->rows, n, pd, pd, nlist, ko, &x->coarse_h, nullptr, s));

  DevBuf dcoarse, assign;
  VDBG_RETURN_IF_ERROR(Alloc(&dcoarse, nlist * pd * sizeof(float), s));
  VDBG_RETURN_IF_ERROR(Alloc(&assign, n * 4, s));
  VDBG_HIP(hipMemcpyAsync(dcoarse.p, x->coarse_h.data(), nlist * pd * sizeof(float),
                          hipMemcpyHostToDevice, s));
  VDBG_RETURN_IF_ERROR(AssignNearestGpu(c, ds->rows, n, pd, pd, dcoarse.get<float>(), nlist,
                                        assign.get<uint32_t>(), nullptr, s));

  // Train PQ on residuals of a strided sample (<= 65,536 rows).
  constexpr size_t kMaxPqTrainRows = 65536;
  const size_t step = std::max<size_t>(1, n / kMaxPqTrainRows);
  std::vector<uint32_t> rows;
  for (size_t i = 0; i < n; i += step) rows.push_back(uint32_t(i));
  DevBuf drows, res;
  VDBG_RETURN_IF_ERROR(Alloc(&drows, rows.size() * 4, s));
  VDBG_RETURN_IF_ERROR(Alloc(&res, rows.size() * d * sizeof(float), s));
  VDBG_HIP(hipMemcpyAsync(drows.p, rows.data(), rows.size() * 4, hipMemcpyHostToDevice, s));
  k_residuals<<<dim3(unsigned((rows.size() * d + 255) / 256)), 256, 0, s>>>(
      ds->rows, int(pd), int(d), dcoarse.get<float>(), assign.get<uint32_t>(),
      drows.get<uint32_t>(), uint32_t(rows.size()), res.get<float>());
  VDBG_HIP(hipGetLastError());
  VDBG_RETURN_IF_ERROR(PqTrainGpu(c, res.get<float>(), rows.size(), d, d, m, ko, &x->cen_h, s));

  // Encode every row's residual, then the lists: ids ascending within a list.
  DevBuf dcen, all, order_in, order_out, keys_out, counts, tmp;
  VDBG_RETURN_IF_ERROR(Alloc(&dcen, x->cen_h.size() * sizeof(float), s));
  VDBG_RETURN_IF_ERROR(Alloc(&all, n * m, s));
  VDBG_HIP(hipMemcpyAsync(dcen.p, x->cen_h.data(), x->cen_h.size() * sizeof(float),
                          hipMemcpyHostToDevice, s));
  VDBG_RETURN_IF_ERROR(PqEncode(c, ds->rows, uint32_t(n), int(pd), int(d), dcoarse.get<float>(),
                                assign.get<uint32_t>(), dcen.get<float>(), int(m), int(d / m),
                                all.get<uint8_t>(), s));
  VDBG_RETURN_IF_ERROR(Alloc(&order_in, n * 4, s));
  VDBG_RETURN_IF_ERROR(Alloc(&keys_out, n * 4, s));
  VDBG_RETURN_IF_ERROR(Alloc(&counts, nlist * 4, s));
  VDBG_HIP(hipMalloc(reinterpret_cast<void**>(&x->ids), n * 4));
  VDBG_HIP(hipMalloc(reinterpret_cast<void**>(&x->codes), n * m));
  k_iota<<<dim3(unsigned((n + 255) / 256)), 256, 0, s>>>(order_in.get<uint32_t>(), uint32_t(n),
                                                         uint32_t(n));
  VDBG_HIP(hipMemsetAsync(counts.p, 0, nlist * 4, s));
  k_histogram<<<dim3(unsigned((n + 255) / 256)), 256, 0, s>>>(assign.get<uint32_t>(), uint32_t(n),
                                                              counts.get<uint32_t>());
  int end_bit = 1;
  while ((size_t(1) << end_bit) < nlist) ++end_bit;
  size_t tmp_bytes = 0;
  VDBG_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, tmp_bytes, assign.get<uint32_t>(),
                                              keys_out.get<uint32_t>(), order_in.get<uint32_t>(),
                                              x->ids, int(n), 0, end_bit, s));
  VDBG_RETURN_IF_ERROR(Alloc(&tmp, tmp_bytes, s));
  VDBG_HIP(hipcub::DeviceRadixSort::SortPairs(tmp.p, tmp_bytes, assign.get<uint32_t>(),
                                              keys_out.get<uint32_t>(), order_in.get<uint32_t>(),
                                              x->ids, int(n), 0, end_bit, s));
  k_gather_codes<<<dim3(unsigned((n * m + 255) / 256)), 256, 0, s>>>(all.get<uint8_t>(), x->ids,
                                                                     uint32_t(n), int(m), x->codes);
  VDBG_HIP(hipGetLastError());
  std::vector<uint32_t> cnt(nlist);
  VDBG_HIP(hipMemcpyAsync(cnt.data(), counts.p, nlist * 4, hipMemcpyDeviceToHost, s));
  VDBG_HIP(hipStreamSynchronize(s));
  x->off_h.assign(nlist + 1, 0);
  for (size_t l = 0; l < nlist; ++l) x->off_h[l + 1] = x->off_h[l] + cnt[l];
  return InstallIvf(c, x, s);
}

}  // namespace vdbg

using namespace vdbg;

extern "C" {

int vdbg_kmeans(vdbg_ctx* ctx, const float* data, size_t n, size_t d, size_t stride, size_t k,
                size_t iters, uint64_t seed, size_t max_points_per_centroid, int kmeanspp,
                float* centroids_out, double* inertia, size_t* empty_reseeds) {
  if (ctx == nullptr || (n > 0 && data == nullptr) || centroids_out == nullptr || stride < d)
    return SetError(kInvalidArgument, "bad argument");
  Ctx* c = &ctx->c;
  std::lock_guard<std::recursive_mutex> g(c->mu);
  VDBG_HIP(hipSetDevice(c->device));
  hipStream_t s = c->stream;
  DevBuf dd;
  VDBG_RETURN_IF_ERROR(Alloc(&dd, std::max<size_t>(1, n * stride) * sizeof(float), s));
  if (n > 0)
    VDBG_HIP(hipMemcpyAsync(dd.p, data, n * stride * sizeof(float), hipMemcpyHostToDevice, s));
  KMeansOpts o;
  o.iters = iters;
  o.seed = seed;
  o.max_points = max_points_per_centroid;
  o.kmeanspp = kmeanspp != 0;
  std::vector<float> cen;
  KMeansInfo info;
  VDBG_RETURN_IF_ERROR(KMeansGpu(c, dd.get<float>(), n, d, stride, k, o, &cen, &info, s));
  std::memcpy(centroids_out, cen.data(), cen.size() * sizeof(float));
  if (inertia) *inertia = info.inertia;
  if (empty_reseeds) *empty_reseeds = info.empty_reseeds;
  return kOk;
}

int vdbg_assign_nearest(vdbg_ctx* ctx, const float* data, size_t n, size_t d, size_t stride,
                        const float* centroids, size_t k, uint32_t* assign, float* dist) {
  if (ctx == nullptr || (n > 0 && (data == nullptr || assign == nullptr)) || centroids == nullptr ||
      stride < d || k == 0)
    return SetError(kInvalidArgument, "bad argument");
  Ctx* c = &ctx->c;
  std::lock_guard<std::recursive_mutex> g(c->mu);
  VDBG_HIP(hipSetDevice(c->device));
  hipStream_t s = c->stream;
  if (n == 0) return kOk;
  DevBuf dd, dc, da, dist_d;
  VDBG_RETURN_IF_ERROR(Alloc(&dd, n * stride * sizeof(float), s));
  VDBG_RETURN_IF_ERROR(Alloc(&dc, k * d * sizeof(float), s));
  VDBG_RETURN_IF_ERROR(Alloc(&da, n * 4, s));
  VDBG_RETURN_IF_ERROR(Alloc(&dist_d, n * 4, s));
  VDBG_HIP(hipMemcpyAsync(dd.p, data, n * stride * sizeof(float), hipMemcpyHostToDevice, s));
  VDBG_HIP(hipMemcpyAsync(dc.p, centroids, k * d * sizeof(float), hipMemcpyHostToDevice, s));
  VDBG_RETURN_IF_ERROR(AssignNearestGpu(c, dd.get<float>(), n, d, stride, dc.get<float>(), k,
                                        da.get<uint32_t>(), dist_d.get<float>(), s));
  VDBG_HIP(hipMemcpyAsync(assign, da.p, n * 4, hipMemcpyDeviceToHost, s));
  if (dist) VDBG_HIP(hipMemcpyAsync(dist, dist_d.p, n * 4, hipMemcpyDeviceToHost, s));
  VDBG_HIP(hipStreamSynchronize(s));
  return kOk;
}

int vdbg_ivfpq_build(vdbg_dataset* ds, size_t nlist, size_t pq_m, uint64_t seed,
                     size_t max_train_points_per_centroid, size_t kmeans_iters, vdbg_ivfpq** out) {
  if (ds == nullptr || out == nullptr) return SetError(kInvalidArgument, "null argument");
  Ctx* c = ds->d.ctx;
  std::lock_guard<std::recursive_mutex> g(c->mu);
  VDBG_HIP(hipSetDevice(c->device));
  auto* h = new (std::nothrow) vdbg_ivfpq;
  if (h == nullptr) return SetError(kResourceExhausted, "out of host memory");
  h->x.ds = &ds->d;
  int rc = IvfBuildGpu(c, &h->x, nlist, pq_m, seed, max_train_points_per_centroid, kmeans_iters,
                       c->stream);
  if (rc != kOk) {
    FreeIvf(&h->x);
    delete h;
    return rc;
  }
  ++ds->d.live_indexes;
  *out = h;
  return kOk;
}

}  // extern "C"
