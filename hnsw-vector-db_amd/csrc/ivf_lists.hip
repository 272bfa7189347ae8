// ivf_lists.hip -- the IVF-PQ scan of a large batch by list, on fp16 MFMA.
//
// A code of list l scores E = offset + sum_j fl(term2[l][j][c_j] + qtab[j][c_j]) (ivf_pq.cc:
// 203-214), which up to rounding is offset + rowsum - 2 q.r: rowsum the row's term-2 sum (kept
// per row, k_ivf_rowsum) and r the residual its code decodes to.  Scanned by query, every
// (query, row) pair costs m random reads of the query's table (k_ivf_scan_rs, bound by LDS bank
// conflicts).  Here the batch's (query, probe) pairs are grouped by list, and a list's decoded
// residuals (held as fp16 halves r 2^e, 2 pd bytes a row) are multiplied with the queries that
// probe it:
//   k_lists_group .. the (query, probe) pairs of a set grouped by list (block histograms in LDS,
//                    column sums, a scan, a scatter): the seeds' nearest probes, then all
//                    that can hold a candidate;
//   k_ivf_lists<1>   the seeds: values of the first rows of each query's nearest lists;
//   k_ivf_seed_kth   the R-th smallest seed a: T = a + 2 eb, eb bounding |value - E|;
//   k_ivf_lists<0>   every row with value <= T of the lists that can hold one, to the query's
//                    candidates;
//   k_ivf_pick       per query, a_R the R-th smallest candidate value: values below a_R - 2 eb
//                    are of the top R and above a_R + 2 eb are not, whatever their exact scores;
//                    the rest are scored exactly (all of them when the scores are returned).
// At least R rows have E <= a + eb, so the top R by (E, id) have values <= T.  A list whose rows
// all lie farther than that, by |q - c - r| >= |q - c| - max |r|, is left out for the query.
// Queries without a finite bound or with more candidates than their buffer are scanned by
// k_ivf_scan_listed (queued for every batch on a bounded grid that runs the few the device
// listed).
#include <algorithm>
#include <cmath>
#include <cstring>

#include "gemm.h"
#include "vdbg_device.h"
#include "vdbg_internal.h"

namespace vdbg {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int kKsub = 256;
constexpr int kLq = 128;        // queries of a work item (32 a wave)
constexpr int kLrows = 64;      // rows of a stage
constexpr int kSeeds = 256;     // seeds of a (query, list): the minima of 1 or 4 rows each
constexpr int kSeedLists = 4;   // nearest lists that give seeds
constexpr int kCap = 1024;      // candidates of a query
constexpr int kStage = 768;     // candidates a wave stages before they are stored
constexpr size_t kListsQueries = 65536;  // queries of one pass, at most,
constexpr size_t kListsBytes = size_t(1) << 30;  // and its scratch per query times their number
constexpr int kListBlocks = 768;  // persistent blocks (three a CU)
constexpr int kHistBlocks = 256;
constexpr int kMaxLists = 16384;  // LDS histogram words

// ---------------------------------------------------------------- the decoded residuals

// fp16(r 2^e) of every CSR row's decoded residual, zero in the padding, and each list's largest
// |r|^2 (float bits).  One wave per row, once per index.
__global__ __launch_bounds__(256) void k_ivf_decode16(const uint8_t* __restrict__ codes,
                                                      const float* __restrict__ cen,
                                                      const uint32_t* __restrict__ off, int nlist,
                                                      uint32_t n, int m, int dsub, int pd, int e,
                                                      uint16_t* __restrict__ y,
                                                      uint32_t* __restrict__ list_norm) {
  const int wave = threadIdx.x >> 6, lane = lane_id();
  const size_t r = size_t(blockIdx.x) * 4 + wave;
  if (r >= n) return;
  float sum = 0.f;
  for (int i = lane; i < pd; i += kWave) {
    float v = 0.f;
    if (i < m * dsub) {
      const int j = i / dsub;
      v = cen[(size_t(j) * kKsub + codes[r * m + j]) * dsub + (i - j * dsub)];
    }
    y[r * pd + i] = __builtin_bit_cast(uint16_t, _Float16(ldexpf(v, e)));
    sum = fmaf(v, v, sum);
  }
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
  int lo = 0, hi = nlist;  // off[lo] <= r < off[hi]
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (off[mid] <= r) lo = mid; else hi = mid;
  }
  if (lane == 0) atomicMax(&list_norm[lo], __float_as_uint(sum));
}

int IvfMakeDecoded(Ctx* c, IvfIndex* x, hipStream_t s) {
  const size_t n = x->off_h.empty() ? 0 : x->off_h.back();
  const size_t pd = size_t(x->pd);
  if (n == 0 || pd % 16 != 0 || pd > 128 || x->nlist > kMaxLists || x->rowsum == nullptr) return kOk;
  float ma = 0.f;
  for (const float v : x->cen_h) {
    if (!(std::fabs(v) <= 3.0e38f)) return kOk;
    ma = std::max(ma, std::fabs(v));
  }
  int e = 0;  // the largest magnitude in [2^14, 2^15)
  if (ma > 0.f) {
    int ex = 0;
    (void)std::frexp(ma, &ex);
    e = 15 - ex;
  }
  const size_t nl = size_t(x->nlist);
  size_t mem_free = 0, mem_all = 0;
  if (hipMemGetInfo(&mem_free, &mem_all) != hipSuccess || n * pd * sizeof(uint16_t) > mem_free / 4)
    return kOk;  // short of memory: the scan by query serves every batch
  if (hipMalloc(reinterpret_cast<void**>(&x->res16), n * pd * sizeof(uint16_t)) != hipSuccess ||
      hipMalloc(reinterpret_cast<void**>(&x->list_rad), nl * sizeof(float)) != hipSuccess) {
    (void)hipGetLastError();
    (void)hipFree(x->res16);
    x->res16 = nullptr;
    return kOk;
  }
  std::vector<float> rad(nl), t2(nl);
  int rc = Fill32(x->list_rad, 0, nl, s);
  if (rc == kOk) {
    k_ivf_decode16<<<dim3(unsigned((n + 3) / 4)), 256, 0, s>>>(
        x->codes, x->cen, x->off, x->nlist, uint32_t(n), x->m, x->dsub, int(pd), e, x->res16,
        reinterpret_cast<uint32_t*>(x->list_rad));
    VDBG_HIP(hipGetLastError());
    VDBG_HIP(hipMemcpyAsync(rad.data(), x->list_rad, nl * 4, hipMemcpyDeviceToHost, s));
    VDBG_HIP(hipMemcpyAsync(t2.data(), x->t2abs, nl * 4, hipMemcpyDeviceToHost, s));
    VDBG_HIP(hipStreamSynchronize(s));
  }
  double rn = 0.0, t2max = 0.0;
  for (size_t l = 0; l < nl; ++l) {
    rad[l] = float(std::sqrt(double(rad[l])) * (1.0 + 1e-4));
    rn = std::max(rn, double(rad[l]));
    if (!(t2[l] <= 1e30f)) t2max = __builtin_inf();
    t2max = std::max(t2max, double(t2[l]));
  }
  if (rc == kOk) {
    VDBG_HIP(hipMemcpyAsync(x->list_rad, rad.data(), nl * 4, hipMemcpyHostToDevice, s));
    VDBG_HIP(hipStreamSynchronize(s));
  }
  // per-subspace and coarse centroid norms (they bound the tables and the offsets)
  double cn = 0.0, cc = 0.0;
  for (int j = 0; j < x->m; ++j) {
    double mx = 0.0;
    for (int k = 0; k < kKsub; ++k) {
      const float* v = x->cen_h.data() + (size_t(j) * kKsub + k) * x->dsub;
      double q = 0.0;
      for (int i = 0; i < x->dsub; ++i) q += double(v[i]) * v[i];
      mx = std::max(mx, q);
    }
    cn += mx;
  }
  for (int l = 0; l < x->nlist; ++l) {
    const float* v = x->coarse_h.data() + size_t(l) * pd;
    double q = 0.0;
    for (size_t i = 0; i < pd; ++i) q += double(v[i]) * v[i];
    cc = std::max(cc, q);
  }
  x->res_exp = e;
  x->res_max = ma;
  x->res_norm = rn;
  x->t2_max = t2max;
  x->cen_norm = std::sqrt(cn) * (1.0 + 1e-6);
  x->coarse_norm = std::sqrt(cc) * (1.0 + 1e-6);
  if (rc != kOk || !(x->res_norm < 1e19) || !(x->coarse_norm < 1e19) || !(t2max < 1e30)) {
    (void)hipFree(x->res16);
    x->res16 = nullptr;
  }
  return rc;
}

// ---------------------------------------------------------------- queries

struct LPrepArgs {
  const float* Q;
  int nq, pd, dsub, m;
  int e;            // the residuals' scale exponent
  float rmax;       // their largest component
  double rn, cn, cc, t2;  // largest |r|, sqrt(sum_j max |C_j|^2), largest |coarse|, t2abs
  uint16_t* Q16;
  float* Qf;
  float* eb;
  float* slack;     // beyond eb: |E - the real |q - c - r|^2|
  int* ovf;
  uint32_t* cnt;    // zeroed
  uint32_t* fb_count;
};

// One wave per query: q 2^sc as fp16 (largest magnitude in [2^14, 2^15)), the factor taking the
// product back, and eb.  With u = 2^-24 and P = sum_i |q_i r_i| <= |q| max|r|:
//   value: 2 (2^-10 + 2^-22) P for the halves (each within 2^-11 of its value), fp16 values
//          below the normal range (2^-14 of a unit each), pd u 2P for the fp32 sum;
//   E:     2 (dsub + 3) u P for the table entries' own dots; 2^-19 S for the rest of E and for
//          rowsum and its sum with the offset (k_ivf_scan_rs's bound, S = offset + sum |term2| +
//          sum |qtab| <= (|q| + cc)^2 + max t2abs + 2 |q| cn);
//   E from the real |q - c - r|^2: besides, the roundings of the coarse distance and of the
//          term-2 entries, (pd + 32) u of (|q| + cc)^2 and (dsub + 32) u of (cn + cc)^2 each.
__global__ __launch_bounds__(256) void k_lists_prep(LPrepArgs a) {
  const int q = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (q >= a.nq) return;
  const int lane = lane_id();
  const float* v = a.Q + size_t(q) * a.pd;
  float s = 0.f, ma = 0.f;
  float x[2] = {0.f, 0.f};  // pd <= 128
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int i = t * kWave + lane;
    if (i < a.pd) x[t] = v[i];
    s = fmaf(x[t], x[t], s);
    // (a NaN survives as a NaN norm)
    ma = fmaxf(ma, fabsf(x[t]));
  }
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) {
    s += __shfl_xor(s, o);
    ma = fmaxf(ma, __shfl_xor(ma, o));
  }
  int sc = 0;
  if (ma > 0.f && ma <= 3.0e38f) {
    int ex = 0;
    (void)frexpf(ma, &ex);
    sc = 15 - ex;
  }
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int i = t * kWave + lane;
    if (i < a.pd)
      a.Q16[size_t(q) * a.pd + i] = __builtin_bit_cast(uint16_t, _Float16(ldexpf(x[t], sc)));
  }
  if (lane == 0) {
    const double u = 1.0 / 16777216.0;
    const double nq = sqrt(double(s)) * (1.0 + 1e-5), P = nq * a.rn;
    const double S = (nq + a.cc) * (nq + a.cc) + a.t2 + 2.0 * nq * a.cn;
    const double sub = 4.0 * a.pd * ldexp(1.0, -14) *
                       (ldexp(double(ma), -a.e) + ldexp(double(a.rmax), -sc));
    const double eb = 2.0 * P * (ldexp(1.0, -10) + ldexp(1.0, -21) + (a.pd + a.dsub + 32.0) * u) +
                      sub + ldexp(1.0, -18) * S;
    a.Qf[q] = ldexpf(-2.f, -sc - a.e);
    a.eb[q] = float(eb * 1.001);
    a.slack[q] = float(eb + 2.0 * (a.pd + 32) * u *
                                ((nq + a.cc) * (nq + a.cc) + (a.cn + a.cc) * (a.cn + a.cc)));
    a.cnt[q] = 0;
    if (q == 0) *a.fb_count = 0;
    // no bound (NaN, infinities), or a factor outside the normal range: scanned by query
    a.ovf[q] = float(eb) < __builtin_inff() && abs(sc + a.e) <= 120 ? 0 : 1;
  }
}

// ---------------------------------------------------------------- pairs by list

// The pairs (q, p < np) grouped by list.  Block b takes queries [b per, (b + 1) per).  Counts stay
// in LDS and the blocks' counts are summed by column, so no pair waits on a global atomic; 1,024
// threads a block, since each pair is a chain of three loads (640,000 and 40,000 pairs, both
// passes: 32 us, 51 with 256 threads).
struct GroupArgs {
  const uint32_t* probe;  // [nq][nprobe]
  const float* probe_d;
  int nq, nprobe, np;
  uint32_t nlist;
  const float* Tp;        // nullable: leave out the lists whose rows all lie beyond it,
  const float* rad;       //           by their largest |r|,
  const int* ovf;         //           and the queries scanned by query
  uint32_t* hist;         // [kHistBlocks][nlist]: counts, then each block's first place
  uint32_t* total;        // [nlist]
  uint32_t* ent_off;      // [nlist + 1]
  const float* Qf;
  const float* T;         // nullable (the seeds)
  uint4* entry;           // by list: q * nprobe + p, and the floats offset, T - offset, Qf
  const uint32_t* off;    // CSR
  uint4* items;           // first row, row end, first entry, entries (at most kLq)
  uint32_t* nitems;
  uint32_t max_items;
};

template <bool SCATTER>
__global__ __launch_bounds__(1024) void k_lists_group(GroupArgs a) {
  extern __shared__ uint32_t cnt[];
  uint32_t* hist = a.hist + size_t(blockIdx.x) * a.nlist;
  for (uint32_t l = threadIdx.x; l < a.nlist; l += 1024)
    cnt[l] = SCATTER ? a.ent_off[l] + hist[l] : 0u;
  __syncthreads();
  const int per = (a.nq + kHistBlocks - 1) / kHistBlocks;
  const int q0 = blockIdx.x * per, q1 = min(a.nq, q0 + per);
  const int n = max(0, q1 - q0) * a.np;
  for (int t = threadIdx.x; t < n; t += 1024) {
    const int qi = t / a.np, p = t - qi * a.np, q = q0 + qi;
    const uint32_t e = uint32_t(q) * uint32_t(a.nprobe) + uint32_t(p);
    const uint32_t l = a.probe[e];
    if (l >= a.nlist) continue;  // no list: nothing to scan
    if (a.Tp != nullptr) {
      if (a.ovf[q] != 0) continue;
      // the coarse distance is the real |q - c|^2 to (pd + 2) u, so its root to 2^-17
      const float d = sqrtf(a.probe_d[e]) * (1.f - 0x1p-16f) - a.rad[l];
      if (d > 0.f && d * d * (1.f - 0x1p-20f) > a.Tp[q]) continue;
    }
    const uint32_t pos = atomicAdd(&cnt[l], 1u);
    if (SCATTER) {
      const float po = a.probe_d[e];
      float T = 0.f;
      if (a.T != nullptr) {
        // value - offset <= T - offset, the roundings of both sides (u of |T| + |offset|) in the
        // 2^-19 S of the bound's E side given away once more
        const float Tq = a.T[q];
        T = (Tq - po) + 0x1p-20f * (fabsf(Tq) + fabsf(po));
      }
      a.entry[pos] = make_uint4(e, __float_as_uint(po), __float_as_uint(T),
                                __float_as_uint(a.Qf[q]));
    }
  }
  if (SCATTER) return;
  __syncthreads();
  for (uint32_t l = threadIdx.x; l < a.nlist; l += 1024) hist[l] = cnt[l];
}

// Each list's counts of the blocks become the blocks' first places in the list.
__global__ __launch_bounds__(256) void k_lists_columns(GroupArgs a) {
  __shared__ uint32_t part[8][32];
  const uint32_t l = blockIdx.x * 32 + (threadIdx.x & 31);
  const int g = threadIdx.x >> 5;  // blocks [32 g, 32 g + 32)
  static_assert(kHistBlocks == 256, "eight groups of 32 blocks");
  uint32_t* h = a.hist + size_t(g) * 32 * a.nlist + l;
  uint32_t v[32], run = 0;
  if (l < a.nlist) {
#pragma unroll
    for (int b = 0; b < 32; ++b) v[b] = h[size_t(b) * a.nlist];
#pragma unroll
    for (int b = 0; b < 32; ++b) run += v[b];
  }
  part[g][threadIdx.x & 31] = run;
  __syncthreads();
  if (l >= a.nlist) return;
  uint32_t at = 0;
  for (int i = 0; i < g; ++i) at += part[i][threadIdx.x & 31];
#pragma unroll
  for (int b = 0; b < 32; ++b) {
    h[size_t(b) * a.nlist] = at;
    at += v[b];
  }
  if (g == 7) a.total[l] = at;
}

// One block: the lists' first entries, and the work items.
__global__ __launch_bounds__(1024) void k_lists_scan(GroupArgs a) {
  __shared__ uint32_t w_n[16], w_i[16];
  const int tid = threadIdx.x, wave = tid >> 6, lane = lane_id();
  const uint32_t per = (a.nlist + 1023) / 1024;
  const uint32_t l0 = min(a.nlist, tid * per), l1 = min(a.nlist, l0 + per);
  uint32_t n = 0, it = 0;
  for (uint32_t l = l0; l < l1; ++l) {
    n += a.total[l];
    it += (a.total[l] + kLq - 1) / kLq;
  }
  uint32_t in = n, ii = it;
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    const uint32_t x = __shfl_up(in, o), z = __shfl_up(ii, o);
    if (lane >= o) {
      in += x;
      ii += z;
    }
  }
  if (lane == kWave - 1) {
    w_n[wave] = in;
    w_i[wave] = ii;
  }
  __syncthreads();
  uint32_t bn = in - n, bi = ii - it;
  for (int w = 0; w < wave; ++w) {
    bn += w_n[w];
    bi += w_i[w];
  }
  for (uint32_t l = l0; l < l1; ++l) {
    const uint32_t c = a.total[l];
    a.ent_off[l] = bn;
    const uint32_t r0 = a.off[l], r1 = a.off[l + 1];
    for (uint32_t t = 0; t < c; t += kLq)
      if (bi < a.max_items)
        a.items[bi++] = make_uint4(r0, r1, bn + t, min(c - t, uint32_t(kLq)));
    bn += c;
  }
  if (tid == 1023) {
    a.ent_off[a.nlist] = bn;
    *a.nitems = bi;
  }
}

// ---------------------------------------------------------------- the contraction

struct ListArgs {
  const uint16_t* R16;     // [CSR rows][PD]
  const float* rowsum;
  const uint16_t* Q16;     // [nq][PD]
  const uint4* entry;
  const uint4* items;
  const uint32_t* nitems;
  int nprobe, s;
  uint2* cand;             // MODE 0: [nq][cap] (value, CSR row)
  uint8_t* cand_p;         // and its probe
  uint32_t* cnt;           // [nq] candidates found (past cap: not stored)
  uint32_t cap;
  float* seed;             // MODE 1: [nq][s][kSeeds]
  int seed_rows;           // rows per seed: 1 or 4
};

// Orders this wave's LDS accesses.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Block = 4 waves x 32 pairs of one list against the list's rows, 64 rows a stage through LDS,
// the next stage's rows loading while one is multiplied.  v_mfma_f32_32x32x16_f16 as in k_gemm16 with the
// operands exchanged: lane l holds dims 8 (l / 32) .. + 7 of each 16-dim block of pair l % 32's
// query (in registers) and of row l % 32 (from LDS); its outputs are row l % 32 of pairs
// 8 (r / 4) + 4 (l / 32) + r % 4.  A pair that has candidates in a list has many, so a ballot
// over the rows finds most registers empty and takes a pair's candidates at once (with the rows
// in the registers almost every register held one).
// Candidates are staged in LDS per wave, so a pair updates its query's counter once (an update
// per candidate past a short stage: 410 us, so: 182).
// The blocks stride over the items; those of one list are consecutive and go to one XCD, so its
// L2 holds the rows.  10,000 queries, nprobe 64 of 4,096 lists of 1M x 128: 182 us for 204M
// padded products (52 GFLOP, and 256 MB of rows, 55 us of HBM), the seeds 70 us, which read the
// same rows; between items the blocks wait on the entries and queries.
template <int PD, int MODE>
__global__ __launch_bounds__(256, 3) void k_ivf_lists(ListArgs a) {
  constexpr int NKB = PD / 16, STR = PD + 8, VPR = PD / 8, VPT = kLrows * VPR;
  constexpr int VT = (VPT + 255) / 256;
  constexpr int kSt = MODE == 0 ? kStage : 1;
  __shared__ __attribute__((aligned(16))) uint16_t xs[kLrows * STR];
  __shared__ float rs[kLrows];
  __shared__ uint2 st[4][kSt];     // (value - offset, row)
  __shared__ uint8_t st_q[4][kSt];   // the wave's pair
  __shared__ uint16_t st_at[4][kSt]; // its place among the pair's
  __shared__ __attribute__((aligned(16))) uint32_t st_n[4][32];  // candidates (seeds: the slots)
  __shared__ __attribute__((aligned(16))) float s_T[4][32], s_qf[4][32];
  const uint32_t nit = *a.nitems, per = (nit + 7) / 8;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, j = lane & 31, h = lane >> 5;
  const uint32_t i0 = (blockIdx.x & 7) * per, i1 = min(nit, i0 + per);
  for (uint32_t item = i0 + (blockIdx.x >> 3); item < i1; item += gridDim.x / 8) {
    const uint4 it = a.items[item];
    const uint32_t r0 = it.x;
    const uint32_t r1 = MODE == 0 ? it.y : min(it.y, r0 + uint32_t(kSeeds * a.seed_rows));
    // (the seeds' slots past the list's end are written too, as NaN)
    const int ntiles = MODE == 0 ? int((r1 - r0 + kLrows - 1) / kLrows)
                                 : kSeeds * a.seed_rows / kLrows;
    u32x4 v[VT];
    float vn = 0.f;
    auto load = [&](int tile) {
      const uint32_t base = r0 + uint32_t(tile) * kLrows;
      const uint32_t last = r1 > 0 ? r1 - 1 : 0;  // (the index holds at least one row)
#pragma unroll
      for (int i = 0; i < VT; ++i) {
        const int f = min(tid + 256 * i, VPT - 1);
        const uint32_t row = min(base + uint32_t(f / VPR), last);
        v[i] = *reinterpret_cast<const u32x4*>(a.R16 + size_t(row) * PD + (f % VPR) * 8);
      }
      const uint32_t rr = base + uint32_t(tid & (kLrows - 1));
      vn = rr < r1 ? a.rowsum[rr] : __builtin_nanf("");
    };
    auto store = [&]() {
#pragma unroll
      for (int i = 0; i < VT; ++i) {
        const int f = tid + 256 * i;
        if (VPT % 256 == 0 || f < VPT)
          *reinterpret_cast<u32x4*>(&xs[(f / VPR) * STR + (f % VPR) * 8]) = v[i];
      }
      if (tid < kLrows) rs[tid] = vn;
    };
    load(0);
    const uint32_t t = uint32_t(wave * 32 + j);
    const bool live = t < it.w;
    const uint4 en = a.entry[it.z + min(t, it.w - 1)];
    const uint32_t q = en.x / uint32_t(a.nprobe);
    const int p = int(en.x - q * uint32_t(a.nprobe));
    const float po = __uint_as_float(en.y);
    half8 qv[NKB];
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb)
      qv[kb] = *reinterpret_cast<const half8*>(a.Q16 + size_t(q) * PD + kb * 16 + h * 8);
    if (h == 0) {  // (a tile's missing pairs take no row)
      s_T[wave][j] = MODE == 1 ? po : live ? __uint_as_float(en.z) : -__builtin_inff();
      s_qf[wave][j] = __uint_as_float(en.w);
      st_n[wave][j] = MODE == 0 ? 0u : live ? (q * a.s + p) * kSeeds : 0xffffffffu;
    }
    uint32_t staged = 0;  // this wave's candidates
    // one counter update per pair, then the staged candidates to their places
    auto flush = [&]() {
      wave_sync();
      const uint32_t n = staged;
      for (uint32_t i = lane; i < n; i += kWave)
        st_at[wave][i] = uint16_t(__hip_atomic_fetch_add(
            &st_n[wave][st_q[wave][i]], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT));
      wave_sync();
      uint32_t first = 0;
      if (h == 0) {
        const uint32_t mine = st_n[wave][j];
        if (mine != 0) first = atomicAdd(&a.cnt[q], mine);
        st_n[wave][j] = 0;
      }
      for (uint32_t b = 0; b < n; b += kWave) {
        const uint32_t i = min(b + lane, n - 1);
        const int src = st_q[wave][i];
        const uint2 c = st[wave][i];
        const uint32_t at = __shfl(first, src) + st_at[wave][i];
        const uint32_t qs = __shfl(q, src);
        const int ps = __shfl(p, src);
        const float of = __shfl(po, src);
        if (b + lane < n && at < a.cap) {
          a.cand[size_t(qs) * a.cap + at] =
              make_uint2(__float_as_uint(of + __uint_as_float(c.x)), c.y);
          a.cand_p[size_t(qs) * a.cap + at] = uint8_t(ps);
        }
      }
      wave_sync();
      staged = 0;
    };
    for (int tile = 0; tile < ntiles; ++tile) {
      __syncthreads();  // the previous stage is no longer read
      store();
      __syncthreads();
      if (tile + 1 < ntiles) load(tile + 1);
#pragma unroll
      for (int half = 0; half < kLrows / 64; ++half) {
        v16f acc[2] = {};
        const uint16_t* x0 = &xs[(half * 64 + j) * STR + h * 8];
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb) {
          const half8 u0 = *reinterpret_cast<const half8*>(x0 + kb * 16);
          const half8 u1 = *reinterpret_cast<const half8*>(x0 + 32 * STR + kb * 16);
          acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(qv[kb], u0, acc[0], 0, 0, 0);
          acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(qv[kb], u1, acc[1], 0, 0, 0);
        }
        const uint32_t row0 = r0 + uint32_t(tile) * kLrows + half * 64 + j;
        const float rs0 = rs[half * 64 + j], rs1 = rs[half * 64 + 32 + j];
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          __builtin_amdgcn_sched_barrier(0);  // (32 values and their terms at once would spill)
          if (MODE == 0 && staged > uint32_t(kStage - 512)) flush();  // four pairs' 64 rows and halves
          const v4f qf = *reinterpret_cast<const v4f*>(&s_qf[wave][8 * g + 4 * h]);
          const v4f T = *reinterpret_cast<const v4f*>(&s_T[wave][8 * g + 4 * h]);
          u32x4 so = {};
          if constexpr (MODE == 1) so = *reinterpret_cast<const u32x4*>(&st_n[wave][8 * g + 4 * h]);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float v0 = fmaf(qf[e], acc[0][4 * g + e], rs0);
            const float v1 = fmaf(qf[e], acc[1][4 * g + e], rs1);
            if constexpr (MODE == 0) {
              const uint64_t b0 = __builtin_amdgcn_ballot_w64(v0 <= T[e]);
              const uint64_t b1 = __builtin_amdgcn_ballot_w64(v1 <= T[e]);
              if ((b0 | b1) == 0) continue;
              auto take = [&](uint64_t b, float val, uint32_t row) {
                if ((b >> lane) & 1) {
                  int sq = 4 * h;  // (opaque: 16 invariant indices and addresses would spill)
                  asm volatile("" : "+v"(sq));
                  sq += 8 * g + e;
                  const uint32_t pos =
                      staged + __builtin_amdgcn_mbcnt_hi(
                                   uint32_t(b >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(b), 0u));
                  st[wave][pos] = make_uint2(__float_as_uint(val), row);
                  st_q[wave][pos] = uint8_t(sq);
                }
                staged += __popcll(b);
              };
              take(b0, v0, row0);
              take(b1, v1, row0 + 32);
            } else {
              const uint32_t at = uint32_t(tile) * kLrows + half * 64;
              const bool on = so[e] != 0xffffffffu;
              float* o = a.seed + so[e];
              const float of = T[e];
              if (a.seed_rows == 1) {
                if (on) o[at + j] = of + v0;
                if (on) o[at + 32 + j] = of + v1;
              } else {  // (fminf skips NaN: rows past the list's end)
                float m = of + fminf(v0, v1);
                m = fminf(m, __shfl_xor(m, 1));
                if (on && (j & 1) == 0) o[at / 4 + j / 2] = m;
              }
            }
          }
        }
      }
    }
    if (MODE == 0 && staged != 0) flush();
  }
}

// ---------------------------------------------------------------- threshold

__device__ __forceinline__ uint32_t list_enc(float f) {  // order-preserving, NaN last
  const uint32_t b = __float_as_uint(f);
  return f != f ? 0xffffffffu : (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ __forceinline__ float list_dec(uint32_t e) {
  return __uint_as_float((e & 0x80000000u) ? (e & 0x7fffffffu) : ~e);
}

// The rank-th smallest of the wave's 64 V keys: the top 16 bits by radix select (its upper end,
// when round is set: at least rank keys lie at or below it), or all 32.
template <int V>
__device__ __forceinline__ uint32_t wave_kth(const uint32_t (&key)[V], int rank, int low_bit) {
  uint32_t ans = 0;
  for (int bit = 31; bit >= low_bit; --bit) {
    const uint32_t t = ans | ((1u << bit) - 1u);
    int c = 0;
#pragma unroll
    for (int v = 0; v < V; ++v) c += __popcll(__ballot(key[v] <= t));
    if (c < rank) ans |= 1u << bit;
  }
  return ans;
}

// T = a + 2 eb, a the R-th smallest seed (to its upper 20 bits, rounded up: an upper bound is
// as good).  One wave per query.
__global__ __launch_bounds__(256) void k_ivf_seed_kth(const float* __restrict__ seed, int nq, int rank, const float* __restrict__ eb,
                                                      const float* __restrict__ slack,
                                                      float* __restrict__ T,
                                                      float* __restrict__ Tp) {
  const int q = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (q >= nq) return;
  constexpr int V = kSeedLists * kSeeds / kWave;
  const float* g = seed + size_t(q) * (kSeedLists * kSeeds);
  uint32_t key[V];
#pragma unroll
  for (int v = 0; v < V; ++v) key[v] = list_enc(g[v * kWave + lane_id()]);
  constexpr int kLow = 12;
  const uint32_t k = wave_kth<V>(key, rank, kLow) | ((1u << kLow) - 1u);
  if (lane_id() == 0) {
    const float a = list_dec(k);
    T[q] = a < __builtin_inff() ? a + 2.f * eb[q] : __builtin_inff();
    Tp[q] = T[q] + slack[q];
  }
}

// ---------------------------------------------------------------- the top R

struct PickArgs {
  const float* Q;
  int pd, dsub, m, nq, nprobe, R;
  uint32_t nlist;
  const float* cen;
  const float* term2;
  const uint8_t* codes;
  const uint32_t* off;
  const uint32_t* ids;
  const uint32_t* probe;
  const float* probe_d;
  const uint2* cand;
  const uint8_t* cand_p;
  const uint32_t* cnt;
  uint32_t cap;
  const int* ovf;
  const float* eb;
  int scores;             // the scores are returned: every candidate is scored
  uint32_t* out_ids;      // [nq][R]
  float* out_d;
  uint64_t* dc;           // nullable
  uint64_t dc_base;
  int count_top;
  uint32_t* fb_list;
  uint32_t* fb_count;
};

// sum_j fl(term2 + qtab), the reference's four accumulators over j mod 4.  M subspaces of D dims
// compiled in (M 0: both at run time), one or two code words a turn, at most 128 floats of
// centroids in flight (unrolled whole it spills at six waves a SIMD).  4,000 queries, 32 of 512 lists of
// 200,000 rows, scores returned, against the run-time loop: m 16 x 4 dims 181 -> 151 us, 8 x 16
// 166 -> 121, 8 x 8 123 -> 105, 4 x 32 141 -> 117, 4 x 8 79 -> 73.
template <int M, int D>
__device__ __forceinline__ float pick_score(const PickArgs& a, const float* qv,
                                            const float* __restrict__ t2,
                                            const uint8_t* __restrict__ cd) {
  float s[4] = {0.f, 0.f, 0.f, 0.f};
  if constexpr (M != 0) {
    constexpr int W = D <= 8 && M >= 8 ? 2 : 1;  // words of four codes a turn
    uint32_t codes[M / 4];  // (a row's codes start on a multiple of M bytes: one load)
    __builtin_memcpy(codes, __builtin_assume_aligned(cd, M), M);
#pragma unroll 1
    for (int j0 = 0; j0 < M / 4; j0 += W) {
      uint32_t w[W];
#pragma unroll
      for (int i = 0; i < W; ++i) {
        w[i] = codes[i];
#pragma unroll
        for (int t = i; t + W < M / 4; t += W) codes[t] = codes[t + W];  // (the next turn's)
      }
#pragma unroll
      for (int i = 0; i < 4 * W; ++i) {
        const int j = 4 * j0 + i, c = int((w[i >> 2] >> (8 * (i & 3))) & 0xffu);
        const v4f* q = reinterpret_cast<const v4f*>(qv + j * D);
        const v4f* y = reinterpret_cast<const v4f*>(a.cen + (j * kKsub + c) * D);
        v4f d = q[0] * y[0];  // dot_any's four accumulators
#pragma unroll
        for (int e = 1; e < D / 4; ++e) d += q[e] * y[e];
        s[i & 3] += t2[j * kKsub + c] + (-((d[0] + d[1]) + (d[2] + d[3]))) * 2.f;
      }
    }
  } else {
#pragma unroll 1
    for (int j = 0; j < a.m; j += 4) {
      const uint32_t w = *reinterpret_cast<const uint32_t*>(cd + j);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int c = int((w >> (8 * i)) & 0xffu);
        const float dot = dot_any(qv + (j + i) * a.dsub,
                                  a.cen + (size_t(j + i) * kKsub + c) * a.dsub, a.dsub);
        s[i] += t2[(j + i) * kKsub + c] + (-dot) * 2.f;
      }
    }
  }
  return (s[0] + s[1]) + (s[2] + s[3]);
}

// The top R of a query's total <= 64 V candidates.
template <int E, int V, int M, int D>
__device__ __forceinline__ void pick_query(const PickArgs& a, int q, uint32_t total,
                                           uint32_t* st_row, uint8_t* st_p, float* qv) {
  const int lane = lane_id();
  uint32_t key[V], row[V];
  uint8_t sp[V];
#pragma unroll
  for (int v = 0; v < V; ++v) {
    key[v] = 0xffffffffu;
    row[v] = kNoId;
    sp[v] = 0;
    const uint32_t g = v * kWave + lane;
    if (g < total) {
      const uint2 c = a.cand[size_t(q) * a.cap + g];
      sp[v] = a.cand_p[size_t(q) * a.cap + g];
      key[v] = list_enc(__uint_as_float(c.x));
      row[v] = c.y;
    }
  }
  uint32_t* oi = a.out_ids + size_t(q) * a.R;
  float* od = a.out_d + size_t(q) * a.R;
  // sure members below lo, sure non-members above hi
  float lo = -__builtin_inff(), hi = __builtin_inff();
  if (!a.scores) {
    if (total <= uint32_t(a.R)) {
      lo = __builtin_inff();
    } else {
      constexpr int kLow = 12;  // a_R to its upper 20 bits: between ar0 and ar1
      const uint32_t k = wave_kth<V>(key, a.R, kLow);
      const float ar0 = list_dec(k), ar1 = list_dec(k | ((1u << kLow) - 1u));
      const float eb = a.eb[q];
      lo = (ar0 - 2.f * eb) - 0x1p-20f * fabsf(ar0);
      hi = (ar1 + 2.f * eb) + 0x1p-20f * fabsf(ar1);
    }
  }
  for (int i = lane; i < a.pd; i += kWave) qv[i] = a.Q[size_t(q) * a.pd + i];
  int sure = 0, staged = 0;
#pragma unroll
  for (int v = 0; v < V; ++v) {
    const float val = list_dec(key[v]);
    const bool have = row[v] != kNoId;
    const bool in = have && val < lo, test = have && !in && val <= hi;
    const uint64_t bi = __ballot(in), bt = __ballot(test);
    if (in) oi[sure + __popcll(bi & ((1ull << lane) - 1ull))] = a.ids[row[v]];
    if (test) {
      const int at = staged + __popcll(bt & ((1ull << lane) - 1ull));
      st_row[at] = row[v];
      st_p[at] = sp[v];
    }
    sure += __popcll(bi);
    staged += __popcll(bt);
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  WaveTopK<E> top;
  top.init();
  for (int b = 0; b < staged; b += kWave) {
    float d = __builtin_inff();
    uint32_t id = kNoId;
    if (b + lane < staged) {
      int z = 0;  // (opaque: the query would be held in 128 registers)
      asm volatile("" : "+v"(z));
      const uint32_t r = st_row[b + lane];
      const size_t pq = size_t(q) * a.nprobe + st_p[b + lane];
      const float* t2 = a.term2 + size_t(a.probe[pq]) * a.m * kKsub;
      const uint8_t* cd = a.codes + size_t(r) * a.m;
      id = a.ids[r];
      const float sum = pick_score<M, D>(a, qv + z, t2, cd);
      d = a.probe_d[pq] + sum;
    }
    top.insert(d, id);
  }
  int valid = 0;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int g = e * kWave + lane;
    if (sure + g < a.R) {
      oi[sure + g] = top.k.id[e];
      od[sure + g] = top.k.d[e];
    }
    valid += __popcll(__ballot(top.k.id[e] != kNoId && sure + g < a.R));
  }
  if (a.dc != nullptr) {
    uint64_t scanned = 0;
    for (int p = lane; p < a.nprobe; p += kWave) {
      const uint32_t l = a.probe[size_t(q) * a.nprobe + p];
      if (l < a.nlist) scanned += a.off[l + 1] - a.off[l];
    }
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) scanned += __shfl_xor(scanned, o);
    if (lane == 0) a.dc[q] = a.dc_base + scanned + (a.count_top ? uint64_t(sure + valid) : 0);
  }
}

// One wave per query.  Bound: a chain of gathers (candidates, codes, centroids and term-2
// entries of the band's rows), hidden by waves, so the registers are held to six a SIMD: 84 us per
// 10,000 queries of 182 candidates (94 at four).
template <int E, int M, int D>
__global__ __launch_bounds__(256, 6) void k_ivf_pick(PickArgs a) {
  __shared__ uint32_t st_row[4][kCap];
  __shared__ uint8_t st_p[4][kCap];
  __shared__ __attribute__((aligned(16))) float qv[4][128];
  const int wave = threadIdx.x >> 6;
  const int q = blockIdx.x * 4 + wave;
  if (q >= a.nq) return;
  const uint32_t total = a.cnt[q];
  if (a.ovf[q] != 0 || total > a.cap) {
    if (lane_id() == 0) a.fb_list[atomicAdd(a.fb_count, 1u)] = uint32_t(q);
    return;
  }
  if (total <= 4 * kWave) pick_query<E, 4, M, D>(a, q, total, st_row[wave], st_p[wave], qv[wave]);
  else pick_query<E, kCap / kWave, M, D>(a, q, total, st_row[wave], st_p[wave], qv[wave]);
}

// ---------------------------------------------------------------- host

// Batches whose (query, row) products pay for the path's fixed costs: about 60 us of launches and
// two passes over the residuals (2 x 256 bytes a row of 128 dims), against some 2.6 us less per
// million products than the scan by query.  Measured by query / by list in us (whole searches,
// nprobe 64 of 4,096 lists of 1M rows): 2,000 queries 308 / 362, 5,000 565 / 518, 10,000
// 1,038 / 694; (64 of 1,024, 200k) 4,000 queries 515 / 286; (16 of 256, 100k x 96) 1,000 queries
// 142 / 194, 3,000 250 / 242; (32 of 128, 50k x 64) 1,000 138 / 156, 3,000 267 / 197.  A row filter
// stays with the scan by query: the few rows it leaves would not bound the rest.
bool IvfListsEligible(const IvfIndex& x, size_t nq, size_t nprobe, size_t R) {
  if (x.res16 == nullptr || x.nlist <= 0 || nprobe < kSeedLists || nprobe > 256 || R > 256)
    return false;
  const double rows = x.off_h.back(), scanned = double(nprobe) * rows / x.nlist;
  // at least four times the depth scanned, so that the seeds bound the rest
  return scanned >= 4.0 * double(R) && double(nq) * scanned >= 12e6 + 50.0 * rows;
}

static size_t Al(size_t b) { return (b + 255) & ~size_t(255); }

// Scratch of one query, and the queries of one pass (the scratch of all stays bounded: at 128
// padded dims 14.6 KB a query at nprobe 64, 17.7 KB at 256).
static size_t QueryBytes(const IvfIndex& x, size_t nprobe) {
  return size_t(x.pd) * 2 + 8 * 4 + nprobe * 16 + kCap * 9 + kSeedLists * kSeeds * 4;
}
static size_t ListsPass(const IvfIndex& x, size_t nq, size_t nprobe) {
  return std::min({nq, kListsQueries, kListsBytes / QueryBytes(x, nprobe)});
}

size_t IvfListsScratch(const IvfIndex& x, size_t all, size_t nprobe) {
  const size_t nl = size_t(x.nlist), nq = ListsPass(x, all, nprobe), pairs = nq * nprobe;
  return Al(nq * size_t(x.pd) * 2) + 8 * Al(nq * 4) + Al(kHistBlocks * nl * 4) + Al(nl * 4) +
         Al((nl + 1) * 4) + Al(pairs * 16) + Al((pairs / kLq + nl + 1) * 16) + 2 * 256 +
         Al(nq * kCap * 8) + Al(nq * kCap) + Al(nq * kSeedLists * kSeeds * 4);
}

template <int MODE>
static int launch_lists(int pd, hipStream_t s, const ListArgs& a) {
  switch (pd) {
#define VDBG_L(P) \
  case P: k_ivf_lists<P, MODE><<<dim3(kListBlocks), 256, 0, s>>>(a); break;
    VDBG_L(16) VDBG_L(32) VDBG_L(48) VDBG_L(64) VDBG_L(80) VDBG_L(96) VDBG_L(112) VDBG_L(128)
#undef VDBG_L
    default: return SetError(kInternal, "ivf lists: padded dim");
  }
  VDBG_HIP(hipGetLastError());
  return kOk;
}

template <int E>
static void launch_pick(unsigned grid, hipStream_t s, const PickArgs& a) {
#define VDBG_P(MM, DD) \
  if (a.m == MM && a.dsub == DD) return k_ivf_pick<E, MM, DD><<<dim3(grid), 256, 0, s>>>(a)
  VDBG_P(16, 8);
  VDBG_P(16, 4);
  VDBG_P(8, 16);
  VDBG_P(8, 12);
  VDBG_P(8, 8);
  VDBG_P(8, 4);
  VDBG_P(4, 32);
  VDBG_P(4, 24);
  VDBG_P(4, 16);
  VDBG_P(4, 8);
  VDBG_P(4, 4);
#undef VDBG_P
  k_ivf_pick<E, 0, 0><<<dim3(grid), 256, 0, s>>>(a);
}

static int GroupPairs(hipStream_t s, const GroupArgs& g) {
  const unsigned lds = g.nlist * 4;
  k_lists_group<false><<<dim3(kHistBlocks), 1024, lds, s>>>(g);
  k_lists_columns<<<dim3((g.nlist + 31) / 32), 256, 0, s>>>(g);
  k_lists_scan<<<1, 1024, 0, s>>>(g);
  k_lists_group<true><<<dim3(kHistBlocks), 1024, lds, s>>>(g);
  VDBG_HIP(hipGetLastError());
  return kOk;
}

static int ListsOnePass(Ctx* c, const IvfIndex& x, const IvfScanArgs& a, hipStream_t s,
                        void* scratch) {
  const size_t nq = size_t(a.nq), nprobe = size_t(a.nprobe), nl = size_t(x.nlist), pd = size_t(x.pd);
  char* p = static_cast<char*>(scratch);
  auto take = [&](size_t b) {
    char* r = p;
    p += Al(b);
    return r;
  };
  uint16_t* Q16 = reinterpret_cast<uint16_t*>(take(nq * pd * 2));
  float* Qf = reinterpret_cast<float*>(take(nq * 4));
  float* eb = reinterpret_cast<float*>(take(nq * 4));
  float* slack = reinterpret_cast<float*>(take(nq * 4));
  float* T = reinterpret_cast<float*>(take(nq * 4));
  float* Tp = reinterpret_cast<float*>(take(nq * 4));
  int* ovf = reinterpret_cast<int*>(take(nq * 4));
  uint32_t* cnt = reinterpret_cast<uint32_t*>(take(nq * 4));
  uint32_t* fb_list = reinterpret_cast<uint32_t*>(take(nq * 4));
  GroupArgs g{};
  g.probe = a.probe;
  g.probe_d = a.probe_d;
  g.nq = a.nq;
  g.nprobe = a.nprobe;
  g.nlist = uint32_t(nl);
  g.Qf = Qf;
  g.off = x.off;
  g.rad = x.list_rad;
  g.ovf = ovf;
  g.max_items = uint32_t(nq * nprobe / kLq + nl + 1);
  g.hist = reinterpret_cast<uint32_t*>(take(kHistBlocks * nl * 4));
  g.total = reinterpret_cast<uint32_t*>(take(nl * 4));
  g.ent_off = reinterpret_cast<uint32_t*>(take((nl + 1) * 4));
  g.entry = reinterpret_cast<uint4*>(take(nq * nprobe * 16));
  g.items = reinterpret_cast<uint4*>(take(size_t(g.max_items) * 16));
  g.nitems = reinterpret_cast<uint32_t*>(take(4));
  uint32_t* fb_count = reinterpret_cast<uint32_t*>(take(4));
  const size_t cap = kCap;
  uint2* cand = reinterpret_cast<uint2*>(take(nq * cap * 8));
  uint8_t* cand_p = reinterpret_cast<uint8_t*>(take(nq * cap));
  float* seed = reinterpret_cast<float*>(take(nq * kSeedLists * kSeeds * 4));
  const unsigned g4 = unsigned((nq + 3) / 4);
  // lists longer than the seeds' slots give minima of 4 rows (their R-th smallest is an upper
  // bound too)
  const int seed_rows = double(x.off_h.back()) / x.nlist > kSeeds ? 4 : 1;
  ListArgs la{x.res16, x.rowsum, Q16, g.entry, g.items, g.nitems, a.nprobe, kSeedLists, cand,
              cand_p, cnt, uint32_t(cap), seed, seed_rows};
  {
    ProfScope ps(c, "ivf_seed", s);
    LPrepArgs pa{a.Q, a.nq, x.pd, x.dsub, x.m, x.res_exp, x.res_max, x.res_norm, x.cen_norm,
                 x.coarse_norm, x.t2_max, Q16, Qf, eb, slack, ovf, cnt, fb_count};
    k_lists_prep<<<dim3(g4), 256, 0, s>>>(pa);
    g.np = kSeedLists;  // nprobe >= 4
    VDBG_RETURN_IF_ERROR(GroupPairs(s, g));
    VDBG_RETURN_IF_ERROR(launch_lists<1>(x.pd, s, la));
    k_ivf_seed_kth<<<dim3(g4), 256, 0, s>>>(seed, a.nq, a.R, eb, slack, T, Tp);
    VDBG_HIP(hipGetLastError());
  }
  {
    ProfScope ps(c, "ivf_scan", s);
    g.np = a.nprobe;
    g.Tp = Tp;
    g.T = T;
    VDBG_RETURN_IF_ERROR(GroupPairs(s, g));
    VDBG_RETURN_IF_ERROR(launch_lists<0>(x.pd, s, la));
  }
  {
    ProfScope ps(c, "ivf_pick", s);
    PickArgs pk{a.Q, x.pd, x.dsub, x.m, a.nq, a.nprobe, a.R, uint32_t(x.nlist), x.cen, x.term2,
                x.codes, x.off, x.ids, a.probe, a.probe_d, cand, cand_p, cnt, uint32_t(cap), ovf,
                eb, a.count_top ? 0 : 1, a.out_ids, a.out_d, a.dc, a.dc_base, a.count_top,
                fb_list, fb_count};
    if (a.R <= 64) launch_pick<1>(g4, s, pk);
    else if (a.R <= 128) launch_pick<2>(g4, s, pk);
    else launch_pick<4>(g4, s, pk);
    VDBG_HIP(hipGetLastError());
  }
  return IvfScanListed(c, a, fb_list, fb_count, s);
}

int IvfScanLists(Ctx* c, const IvfIndex& x, const IvfScanArgs& a, hipStream_t s, void* scratch) {
  const size_t pass = ListsPass(x, size_t(a.nq), size_t(a.nprobe));
  for (size_t q0 = 0; q0 < size_t(a.nq); q0 += pass) {
    IvfScanArgs b = a;
    b.nq = int(std::min(pass, size_t(a.nq) - q0));
    b.Q = a.Q + q0 * a.pd;
    b.probe = a.probe + q0 * a.nprobe;
    b.probe_d = a.probe_d + q0 * a.nprobe;
    b.out_ids = a.out_ids + q0 * a.R;
    b.out_d = a.out_d + q0 * a.R;
    if (a.dc != nullptr) b.dc = a.dc + q0;
    VDBG_RETURN_IF_ERROR(ListsOnePass(c, x, b, s, scratch));
  }
  return kOk;
}

}  // namespace vdbg
