// pqflat.hip -- PqFlatIndex (src/index/quant/ivf_pq.h:12-36, ivf_pq.cc:41-98) on gfx950.
//
// Every row's PQ code is scored by ADC against the query's table, the max(depth, k) best
// by (ADC, id) kept, then FinishSearch (:28-36): the float Rerank of those candidates, or
// with depth 0 the best k by ADC.  Per query:
//   table[j][c] = L2SqAny(q_j, C_j[c])  (L2)  or  -DotAny(q_j, C_j[c])  (inner product,
//                 cosine)                                  ProductQuantizer::compute_table
//   adc(code)   = four accumulators over j mod 4           pq.h:36-46
//   depth       = rerank < 0 ? max(10 k, 100) : rerank     RerankDepth, ivf_pq.cc:16-19
//   distance_computations = rows (+ the candidates reranked)
// The tables are built on the device ([nq][m x 256] floats).  Over at least 1,024 rows,
// where the padded dim has a GEMM kernel, the scan is the flat path's ranking
// GEMM over the rows the codes decode to (fp16 halves, gemm16.hip SPLIT 3: the ADC is the
// distance to the decoded row up to its rounding, which the query's bound takes in); every
// candidate it admits is then scored by ADC from the query's table, certified against the
// admission threshold, and re-scanned code by code when that fails.  Small batches over few
// rows or under a selective filter (PqScoreFew, PqScoreFiltered), and widths without a kernel,
// score every allowed code instead (row splits with a wave top-k each, then a merge; a sort
// beyond 240 results).
//
// Bound: MFMA (2 n pd flop per query; 890 TFLOP/s at 1M x 128, 2,000 queries).  Scoring every
// code is bound by its m table reads a row instead: the batch of 2,000 queries over 1M codes
// of 16 bytes took 26.1 ms that way and takes 0.74 ms ranked (the GEMM 0.57).  The decoded
// rows cost 2 pd + 4 bytes a row of device memory.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "gemm.h"
#include "vdbg_device.h"
#include "vdbg_internal.h"

namespace vdbg {
namespace {

constexpr int kKsub = 256;
constexpr size_t kRankRows = 1024;  // the ranking GEMM path's fewest rows (RunScan)

// compute_table (pq.cc:63-73) for nq queries: one thread per (query, subspace, centroid).
__global__ void k_pq_tables(const float* __restrict__ Q, int pd, int nq,
                            const float* __restrict__ cen, int m, int dsub, int l2,
                            float* __restrict__ T) {
  const size_t t = blockIdx.x * size_t(blockDim.x) + threadIdx.x;
  const size_t ts = size_t(m) * kKsub;
  if (t >= size_t(nq) * ts) return;
  const size_t q = t / ts;
  const int e = int(t - q * ts);
  const int j = e / kKsub;
  const float* qs = Q + q * pd + size_t(j) * dsub;
  const float* cc = cen + size_t(e) * dsub;
  T[t] = l2 ? l2sq_any(qs, cc, dsub) : -dot_any(qs, cc, dsub);
}

// The rows the codes decode to, for the ranking GEMM (gemm16.hip SPLIT 3): fp16(v 2^e) of
// each decoded value, zero in the padding, the row's fp32 norm and the largest norm (float
// bits).  One wave per row; writes 2 pd bytes a row, once per index.
__global__ __launch_bounds__(256) void k_pq_decode16(const uint8_t* __restrict__ codes,
                                                     const float* __restrict__ cen, uint32_t n,
                                                     int m, int dsub, int pd, int e,
                                                     uint16_t* __restrict__ y,
                                                     float* __restrict__ norm,
                                                     uint32_t* __restrict__ max_norm) {
  __shared__ float s_max[4];
  const int wave = threadIdx.x >> 6, lane = lane_id();
  const size_t r = size_t(blockIdx.x) * 4 + wave;
  float sum = 0.f;
  if (r < n) {
    for (int i = lane; i < pd; i += kWave) {
      float v = 0.f;
      if (i < m * dsub) {
        const int j = i / dsub;
        v = cen[(size_t(j) * kKsub + codes[r * m + j]) * dsub + (i - j * dsub)];
      }
      y[r * pd + i] = __builtin_bit_cast(uint16_t, _Float16(ldexpf(v, e)));
      sum = fmaf(v, v, sum);
    }
  }
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
  if (lane == 0) {
    if (r < n) norm[r] = sum;
    s_max[wave] = r < n ? sum : 0.f;
  }
  __syncthreads();
  if (threadIdx.x == 0)
    atomicMax(max_norm, __float_as_uint(fmaxf(fmaxf(s_max[0], s_max[1]),
                                              fmaxf(s_max[2], s_max[3]))));
}

// distance_computations of PqFlatIndex::search: every row, plus the candidates handed to
// Rerank (ivf_pq.cc:76-79).
__global__ void k_pqflat_dc(const uint32_t* __restrict__ cand, int kk, int nq, uint64_t rows,
                            int reranked, uint64_t* __restrict__ dc) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= nq) return;
  uint64_t v = rows;
  if (reranked)
    for (int i = 0; i < kk; ++i) v += cand[size_t(q) * kk + i] != kNoId ? 1 : 0;
  dc[q] = v;
}

// A device buffer released on the stream when the call ends.
struct Tmp {
  void* p = nullptr;
  hipStream_t s = nullptr;
  ~Tmp() {
    if (p != nullptr) (void)hipFreeAsync(p, s);
  }
};

// Whether scoring every allowed code takes less than the ranking GEMM over every row.  Each side
// of the lines was timed with host calls, in us.
//
// Few rows: below 25 rows for each of the depth the ranking's threshold admits most of them
// (ranked / scored at depth 100, m 16 x 8 dims: 2,000 rows 118 / 81 for 1 query and 317 / 237 for
// 2,000; 3,000 rows 96 / 82 and 209 / 272; at depth 240: 4,000 rows 440 / 423 for 2,000 queries,
// 6,000 rows 294 / 503).  Above that small batches score while the table reads cost less than the
// ranking's launches do beyond the scoring's (depth 10: 4,000 rows 88 / 69 for 1 query, 98 / 112
// for 500; 12,000 rows 86 / 83 for 16, 90 / 94 for 64; depth 100: 4,000 rows 121 / 103 for 64,
// 142 / 154 for 500, 20,000 rows 125 / 126 for 64; depth 240: 6,000 rows 135 / 146 for 1).  From 8
// queries on the ranking takes about 12 us more at depths up to 100, none at 240.
bool PqScoreFew(size_t rows, int m, size_t nq, size_t kk) {
  const double n = double(rows), q = double(nq), k = double(kk);
  if (n < 25.0 * k) return true;
  const double reads = n * (6e-4 + q * 1e-6 * std::max(13, m));
  return reads < 20.0 - 0.16 * k + (nq >= 8 && kk <= 100 ? 12.0 : 0.0) + (rows < 3000 ? 25.0 : 0.0);
}
// A selective filter (at most a sixteenth of the rows, past which the fits below fail): the scan
// of the codes skips what it leaves out.  Both sides as fitted, within 15%.  Ranked / scored at
// depth 100, 1M x 128, m 16: 0.2% allowed 188 / 119 for 1 query, 195 / 173 for 16, 200 / 220
// for 32, and 2% 194 / 209 for 1; 100,000 rows: 2% 131 / 114 for 1, 144 / 133 for 16, 148 / 156
// for 32; 200,000 x 384, m 48: 2% 190 / 169 for 8, 193 / 202 for 16.  `spent`: what the choice
// itself costs (counting the filter's rows on the device).
bool PqScoreFiltered(size_t rows, size_t pd, int m, size_t nq, size_t allowed, double spent) {
  const double n = double(rows), q = double(nq), a = double(allowed);
  if (16 * a > n) return false;
  const double score = 85.0 + 3e-5 * n + 4.5e-3 * a +
                       q * (0.06 + 2e-6 * n + 4e-4 * a * (16.0 + m) / 32.0);
  const double rank = 110.0 + 6.2e-7 * n * double(pd) + 0.25 * std::min(q, 64.0) +
                      q * (0.05 + 2e-7 * n);
  return score + spent + 8.0 < rank;
}
constexpr double kCountUs = 10.0;  // CountAllowed

// allowed: the rows a filter allows, where the caller knows (-1: not).
int PqFlatSearch(PqFlatIndex* x, const float* Q, size_t nq, size_t k, int rerank,
                 const uint64_t* allow, int64_t allowed, uint32_t* out_ids, float* out_d,
                 uint64_t* dc, hipStream_t s) {
  Dataset* ds = x->ds;
  Ctx* c = ds->ctx;
  const size_t n = ds->n;
  if (nq == 0) return kOk;
  if (n == 0 || k == 0) {  // ivf_pq.cc:62: nothing searched, nothing counted
    if (k > 0) {
      ScanSource none;
      VDBG_RETURN_IF_ERROR(ScoreScan(c, none, Q, nq, k, nullptr, out_ids, out_d, s));
    }
    if (dc != nullptr) VDBG_HIP(hipMemsetAsync(dc, 0, nq * 8, s));
    return kOk;
  }
  const size_t depth = rerank < 0 ? std::max<size_t>(10 * k, 100) : size_t(rerank);
  const size_t kk = std::max(depth, k);
  const size_t ts = size_t(x->m) * kKsub;
  // the scan keeps at most n candidates, as a TopK of any capacity over n rows does (depth
  // may exceed vdb's largest k: max(10 k, 100) at k = 10,000)
  const size_t keep = std::min(kk, std::max<size_t>(n, k));
  const bool can_rank = x->src.X16 != nullptr && x->src.N == n && c->fp16_gemm && kk <= 10000;
  bool ranked = can_rank && (kk > 240 || !PqScoreFew(n, x->m, nq, kk));
  if (ranked && allow != nullptr && kk <= 240) {
    if (allowed < 0 && PqScoreFiltered(n, ds->pd, x->m, nq, 0, kCountUs)) {
      // (a captured stream cannot be read from: it ranks)
      hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
      if (hipStreamIsCapturing(s, &cap) != hipSuccess) (void)hipGetLastError();
      if (cap == hipStreamCaptureStatusNone) {
        uint32_t count = 0;
        VDBG_RETURN_IF_ERROR(CountAllowed(c, allow, uint32_t(n), &count, s, nullptr));
        allowed = count;
      }
    }
    if (allowed >= 0) ranked = !PqScoreFiltered(n, ds->pd, x->m, nq, size_t(allowed), 0.0);
  }
  Tmp tables;  // the tables, and the candidates handed to the rerank
  tables.s = s;
  const size_t tb = (nq * ts * sizeof(float) + 255) / 256 * 256;
  const size_t cb = depth == 0 ? 0 : (nq * keep * 4 + 255) / 256 * 256;
  VDBG_HIP(ScratchAlloc(c, &tables.p, tb + 2 * cb, s));
  {
    ProfScope ps(c, "pq_tables", s);
    const size_t total = nq * ts;
    k_pq_tables<<<dim3(unsigned((total + 255) / 256)), 256, 0, s>>>(
        Q, int(ds->pd), int(nq), x->cen, x->m, x->dsub, ds->metric == 0 ? 1 : 0,
        static_cast<float*>(tables.p));
    VDBG_HIP(hipGetLastError());
  }
  const float* T = static_cast<const float*>(tables.p);
  ScanSource src;
  src.kind = 2;
  src.C = x->codes;
  src.pq_m = x->m;
  src.N = uint32_t(n);
  src.pd = int(ds->pd);
  src.metric = ds->metric;
  // the kk best by (ADC, id): the ranking GEMM over the decoded rows and the ADC of the few
  // codes it admits, or the ADC of every allowed code
  auto scan = [&](size_t kk, uint32_t* ids, float* d) {
    if (ranked) {
      VDBG_RETURN_IF_ERROR(BuildSample(c, &x->src, s));
      ScanSource rs = x->src;
      rs.pq_tables = T;
      return RunScan(c, &rs, Q, nq, kk, allow, ids, d, s);
    }
    return ScoreScan(c, src, T, nq, kk, allow, ids, d, s);
  };
  if (depth == 0) {
    VDBG_RETURN_IF_ERROR(scan(k, out_ids, out_d));
    if (dc != nullptr)
      k_pqflat_dc<<<dim3(unsigned((nq + 255) / 256)), 256, 0, s>>>(out_ids, int(k), int(nq), n, 0,
                                                                   dc);
    VDBG_HIP(hipGetLastError());
    return kOk;
  }
  uint32_t* cand = reinterpret_cast<uint32_t*>(static_cast<char*>(tables.p) + tb);
  float* cand_d = reinterpret_cast<float*>(static_cast<char*>(tables.p) + tb + cb);
  VDBG_RETURN_IF_ERROR(scan(keep, cand, cand_d));
  VDBG_RETURN_IF_ERROR(Rerank(c, ds->rows, int(ds->pd), ds->metric, Q, nq, cand, keep, k, out_ids,
                              out_d, s, &ds->src));
  if (dc != nullptr)
    k_pqflat_dc<<<dim3(unsigned((nq + 255) / 256)), 256, 0, s>>>(cand, int(keep), int(nq), n, 1,
                                                                 dc);
  VDBG_HIP(hipGetLastError());
  return kOk;
}

void FreePqFlat(PqFlatIndex* x) {
  FreeSample(&x->src);
  x->src = ScanSource{};
  (void)hipFree(x->dec16);
  (void)hipFree(x->dec_norm);
  x->dec16 = nullptr;
  x->dec_norm = nullptr;
  (void)hipFree(x->cen);
  (void)hipFree(x->codes);
  x->cen = nullptr;
  x->codes = nullptr;
}

// Makes the decoded rows the ranking GEMM reads (the codes are in place).  Without them, for
// padded dims with no GEMM kernel, segments below the GEMM path's 1,024 rows, non-finite
// codebooks or where they would take more than a quarter of the free memory (they are 2 pd / m
// times the codes, and later segments need room), searches score every code.
int MakeDecoded(Ctx* c, PqFlatIndex* x, hipStream_t s) {
  const size_t n = x->ds->n, pd = x->ds->pd;
  if (n < kRankRows || !GemmSupported(pd)) return kOk;
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
  size_t mem_free = 0, mem_all = 0;
  if (hipMemGetInfo(&mem_free, &mem_all) != hipSuccess ||
      n * (pd * sizeof(uint16_t) + sizeof(float)) > mem_free / 4) {
    (void)hipGetLastError();
    return kOk;
  }
  uint32_t* max_norm = nullptr;
  const bool got =
      hipMalloc(reinterpret_cast<void**>(&x->dec16), n * pd * sizeof(uint16_t)) == hipSuccess &&
      hipMalloc(reinterpret_cast<void**>(&x->dec_norm), n * sizeof(float)) == hipSuccess &&
      hipMalloc(reinterpret_cast<void**>(&max_norm), 256) == hipSuccess;
  auto drop = [&]() {
    (void)hipFree(x->dec16);
    (void)hipFree(x->dec_norm);
    (void)hipFree(max_norm);
    x->dec16 = nullptr;
    x->dec_norm = nullptr;
  };
  if (!got) {
    (void)hipGetLastError();
    drop();
    return kOk;
  }
  uint32_t bits = 0;
  int rc = Fill32(max_norm, 0, 1, s);
  if (rc == kOk) {
    k_pq_decode16<<<dim3(unsigned((n + 3) / 4)), 256, 0, s>>>(x->codes, x->cen, uint32_t(n), x->m,
                                                               x->dsub, int(pd), e, x->dec16,
                                                               x->dec_norm, max_norm);
    if (hipGetLastError() != hipSuccess) rc = SetError(kInternal, "pq decode");
  }
  if (rc == kOk) rc = ReadWords(c, max_norm, 1, s, &bits);
  float xn = 0.f;
  std::memcpy(&xn, &bits, 4);
  if (rc != kOk || !(xn <= 3.0e38f)) {
    (void)hipStreamSynchronize(s);
    drop();
    return rc;
  }
  (void)hipFree(max_norm);
  ScanSource& src = x->src;
  src.kind = 2;
  src.C = x->codes;
  src.pq_m = x->m;
  src.X16 = x->dec16;
  src.x16_exp = e;
  src.x16_approx = 1;
  src.rn = x->dec_norm;
  src.N = uint32_t(n);
  src.pd = int(pd);
  src.metric = x->ds->metric;
  src.stats.max_abs = ma;
  src.stats.xn_max = xn;
  src.stats.all_int = 0;  // the ranking is never exact: ADC sums in its own order
  src.rmag = xn;
  return kOk;
}

// Uploads the codebook (and codes, when given on the host) of an index over ds.
int InstallPqFlat(Ctx* c, PqFlatIndex* x, const uint8_t* codes_h, hipStream_t s) {
  const size_t n = x->ds->n;
  if (!x->cen_h.empty()) {
    VDBG_HIP(hipMalloc(reinterpret_cast<void**>(&x->cen), x->cen_h.size() * sizeof(float)));
    VDBG_HIP(hipMemcpyAsync(x->cen, x->cen_h.data(), x->cen_h.size() * sizeof(float),
                            hipMemcpyHostToDevice, s));
  }
  if (n > 0 && x->codes == nullptr) {
    VDBG_HIP(hipMalloc(reinterpret_cast<void**>(&x->codes), n * x->m));
    if (codes_h != nullptr)
      VDBG_HIP(hipMemcpyAsync(x->codes, codes_h, n * x->m, hipMemcpyHostToDevice, s));
  }
  VDBG_HIP(hipStreamSynchronize(s));
  return kOk;
}

}  // namespace

int PqFlatSearchDevice(vdbg_pqflat* ix, const float* queries, size_t nq, size_t k, int rerank,
                       const uint64_t* allow_words, int64_t allowed, uint32_t* out_ids,
                       float* out_dists, uint64_t* dist_comps, void* stream) {
  if (ix == nullptr) return SetError(kInvalidArgument, "null index");
  if (nq > 0 && k > 0 && (queries == nullptr || out_ids == nullptr || out_dists == nullptr))
    return SetError(kInvalidArgument, "null pointer");
  if (k > 10000) return SetError(kInvalidArgument, "k must be in 1..10000");
  Ctx* c = ix->p.ds->ctx;
  std::lock_guard<std::recursive_mutex> g(c->mu);
  VDBG_HIP(hipSetDevice(c->device));
  hipStream_t s = stream ? static_cast<hipStream_t>(stream) : c->stream;
  return PqFlatSearch(&ix->p, queries, nq, k, rerank, allow_words, allowed, out_ids, out_dists,
                      dist_comps, s);
}

}  // namespace vdbg

using namespace vdbg;

extern "C" {

int vdbg_pqflat_build(vdbg_dataset* ds, size_t pq_m, uint64_t seed,
                      size_t max_points_per_centroid, size_t kmeans_iters, vdbg_pqflat** out) {
  if (ds == nullptr || out == nullptr) return SetError(kInvalidArgument, "null argument");
  Dataset& d = ds->d;
  if (pq_m == 0 || d.dim % pq_m != 0)
    return SetError(kInvalidArgument, "pq_m must divide the dimension");  // index.cc:27-29
  Ctx* c = d.ctx;
  std::lock_guard<std::recursive_mutex> g(c->mu);
  VDBG_HIP(hipSetDevice(c->device));
  hipStream_t s = c->stream;
  auto* h = new (std::nothrow) vdbg_pqflat;
  if (h == nullptr) return SetError(kResourceExhausted, "out of host memory");
  PqFlatIndex& x = h->p;
  x.ds = &d;
  x.m = int(pq_m);
  x.dsub = int(d.dim / pq_m);
  auto fail = [&](int rc) {
    FreePqFlat(&x);
    delete h;
    return rc;
  };
  // PqFlatIndex::build (ivf_pq.cc:45-57): nothing is trained over no rows
  if (d.n > 0) {
    int rc = PqTrainRows(c, d.rows, d.n, d.pd, d.dim, pq_m, seed, max_points_per_centroid,
                         kmeans_iters, &x.cen_h, s);
    if (rc != kOk) return fail(rc);
    x.trained = true;
  }
  int rc = InstallPqFlat(c, &x, nullptr, s);
  if (rc != kOk) return fail(rc);
  if (d.n > 0) {
    rc = PqEncode(c, d.rows, uint32_t(d.n), int(d.pd), int(d.dim), nullptr, nullptr, x.cen, x.m,
                  x.dsub, x.codes, s);
    if (rc != kOk) return fail(rc);
    if (hipStreamSynchronize(s) != hipSuccess) return fail(SetError(kInternal, "pq encode"));
    rc = MakeDecoded(c, &x, s);
    if (rc != kOk) return fail(rc);
  }
  ++d.live_indexes;
  *out = h;
  return kOk;
}

// LoadIndex of a VDBPQFL1 file (index.cc:38-87, 76-77) and PqFlatIndex::load (ivf_pq.cc:
// 89-98): u64 rows, the ProductQuantizer (pq.cc:75-92: u32 dim, u32 m, centroids), then rows
// x m code bytes.
int vdbg_pqflat_load(vdbg_dataset* ds, const void* file, size_t len, vdbg_pqflat** out) {
  if (ds == nullptr || out == nullptr || (file == nullptr && len > 0))
    return SetError(kInvalidArgument, "null argument");
  const auto* b = static_cast<const uint8_t*>(file);
  if (len < 12) return SetError(VDBG_CORRUPTION, "index file too short");
  uint32_t stored;
  std::memcpy(&stored, b + len - 4, 4);
  if (Crc32c(b, len - 4) != stored) return SetError(VDBG_CORRUPTION, "index file checksum mismatch");
  if (std::memcmp(b, "VDBPQFL1", 8) != 0)
    return SetError(VDBG_CORRUPTION, "not a pq-flat index file (magic VDBPQFL1)");
  const uint8_t* p = b + 8;
  size_t left = len - 12;
  auto take = [&](void* dst, size_t n) {
    if (left < n) return false;
    if (dst != nullptr && n > 0) std::memcpy(dst, p, n);
    p += n;
    left -= n;
    return true;
  };
  Dataset& d = ds->d;
  uint64_t n = 0;
  uint32_t dim = 0, m = 0;
  const char* mismatch = "pq index does not match the segment";
  if (!take(&n, 8) || n != d.n || !take(&dim, 4) || !take(&m, 4) || m == 0 || dim % m != 0)
    return SetError(VDBG_CORRUPTION, mismatch);
  const size_t dsub = dim / m;
  std::vector<float> cen(size_t(m) * kKsub * dsub);
  if (!take(cen.data(), cen.size() * sizeof(float)) || dim != d.dim)
    return SetError(VDBG_CORRUPTION, mismatch);
  const uint8_t* codes = p;
  if (!take(nullptr, size_t(n) * m)) return SetError(VDBG_CORRUPTION, "truncated pq codes");
  Ctx* c = d.ctx;
  std::lock_guard<std::recursive_mutex> g(c->mu);
  VDBG_HIP(hipSetDevice(c->device));
  auto* h = new (std::nothrow) vdbg_pqflat;
  if (h == nullptr) return SetError(kResourceExhausted, "out of host memory");
  PqFlatIndex& x = h->p;
  x.ds = &d;
  x.m = int(m);
  x.dsub = int(dsub);
  x.cen_h = std::move(cen);
  x.trained = true;
  int rc = InstallPqFlat(c, &x, codes, c->stream);
  if (rc == kOk) rc = MakeDecoded(c, &x, c->stream);
  if (rc != kOk) {
    FreePqFlat(&x);
    delete h;
    return rc;
  }
  ++d.live_indexes;
  *out = h;
  return kOk;
}

// PqFlatIndex::save (ivf_pq.cc:81-87) through WriteIndexFile (index.cc:40-46).
int vdbg_pqflat_save(vdbg_pqflat* ix, void* buf, size_t cap, size_t* len) {
  if (ix == nullptr || len == nullptr) return SetError(kInvalidArgument, "null argument");
  PqFlatIndex& x = ix->p;
  Dataset& d = *x.ds;
  const size_t n = d.n;
  std::string out("VDBPQFL1");
  auto put = [&](const void* v, size_t bytes) {
    out.append(static_cast<const char*>(v), bytes);
  };
  const uint64_t rows = n;
  const uint32_t dim = uint32_t(d.dim), m = uint32_t(x.m);
  put(&rows, 8);
  put(&dim, 4);
  put(&m, 4);
  put(x.cen_h.data(), x.cen_h.size() * sizeof(float));
  const size_t at = out.size();
  out.resize(at + n * x.m);
  if (n > 0) {
    Ctx* c = d.ctx;
    std::lock_guard<std::recursive_mutex> g(c->mu);
    VDBG_HIP(hipSetDevice(c->device));
    VDBG_HIP(hipMemcpyAsync(&out[at], x.codes, n * x.m, hipMemcpyDeviceToHost, c->stream));
    VDBG_HIP(hipStreamSynchronize(c->stream));
  }
  const uint32_t crc = Crc32c(out.data(), out.size());
  put(&crc, 4);
  *len = out.size();
  if (buf != nullptr) {
    if (cap < out.size()) return SetError(kResourceExhausted, "buffer too small for the index file");
    std::memcpy(buf, out.data(), out.size());
  }
  return kOk;
}

int vdbg_pqflat_destroy(vdbg_pqflat* ix) {
  if (ix == nullptr) return kOk;
  Ctx* c = ix->p.ds->ctx;
  std::lock_guard<std::recursive_mutex> g(c->mu);
  (void)hipSetDevice(c->device);
  (void)hipDeviceSynchronize();
  --ix->p.ds->live_indexes;
  FreePqFlat(&ix->p);
  delete ix;
  return kOk;
}

int vdbg_pqflat_info(vdbg_pqflat* ix, size_t* m, float* centroids_out) {
  if (ix == nullptr || m == nullptr) return SetError(kInvalidArgument, "null argument");
  *m = size_t(ix->p.m);
  if (centroids_out != nullptr && !ix->p.cen_h.empty())
    std::memcpy(centroids_out, ix->p.cen_h.data(), ix->p.cen_h.size() * sizeof(float));
  return kOk;
}

int vdbg_pqflat_codes(vdbg_pqflat* ix, uint8_t* codes_out) {
  if (ix == nullptr || codes_out == nullptr) return SetError(kInvalidArgument, "null argument");
  const size_t bytes = ix->p.ds->n * size_t(ix->p.m);
  if (bytes == 0) return kOk;
  Ctx* c = ix->p.ds->ctx;
  std::lock_guard<std::recursive_mutex> g(c->mu);
  VDBG_HIP(hipSetDevice(c->device));
  VDBG_HIP(hipMemcpyAsync(codes_out, ix->p.codes, bytes, hipMemcpyDeviceToHost, c->stream));
  VDBG_HIP(hipStreamSynchronize(c->stream));
  return kOk;
}

int vdbg_pqflat_search_device(vdbg_pqflat* ix, const float* queries, size_t nq, size_t k,
                              int rerank, const uint64_t* allow_words, uint32_t* out_ids,
                              float* out_dists, uint64_t* dist_comps, void* stream) {
  return PqFlatSearchDevice(ix, queries, nq, k, rerank, allow_words, -1, out_ids, out_dists,
                            dist_comps, stream);
}

int vdbg_pqflat_search_host(vdbg_pqflat* ix, const float* queries, size_t nq, size_t k,
                            int rerank, const uint64_t* allow_words, uint32_t* out_ids,
                            float* out_dists, uint64_t* dist_comps) {
  if (ix == nullptr) return SetError(kInvalidArgument, "null index");
  if (nq == 0 || k == 0) {
    if (dist_comps != nullptr) std::fill(dist_comps, dist_comps + nq, uint64_t(0));
    return kOk;
  }
  if (queries == nullptr || out_ids == nullptr || out_dists == nullptr)
    return SetError(kInvalidArgument, "null pointer");
  if (k > 10000) return SetError(kInvalidArgument, "k must be in 1..10000");
  Dataset& d = *ix->p.ds;
  Ctx* c = d.ctx;
  std::lock_guard<std::recursive_mutex> g(c->mu);
  VDBG_HIP(hipSetDevice(c->device));
  const int64_t allowed = allow_words != nullptr ? int64_t(CountRows(allow_words, d.n)) : -1;
  return StageHost(c, d.n, d.pd, queries, nq, k, allow_words, out_ids, out_dists, dist_comps,
                   [&](const float* dq, const uint64_t* dm, uint32_t* di, float* dd,
                       uint64_t* ddc, hipStream_t st) {
                     return PqFlatSearch(&ix->p, dq, nq, k, rerank, dm, allowed, di, dd, ddc, st);
                   });
}

}  // extern "C"
