// Tile-scheduler metadata kernel: balanced split-KV partition.
//
// The reference chooses ONE split count per launch on the host
// (src/flag_attn/paged.py:52-67, src/flag_attn/split_kv.py:248-276), so a
// batch of skewed lengths leaves CUs idle.  Here the work of every sequence
// (its 64-token blocks plus a fixed per-sequence overhead) is laid end to end
// in a "cost line" of length W, cut into num_parts equal shares, and each cut
// is mapped back to a (sequence, block) position.  One work-group, one part
// per thread: three block scans, two binary searches per part and closed-form
// divisions for the rest.
//
// Spec (integer arithmetic throughout):
//   nb[b] = ceil(len_b / 64)          (dense; topk > 0: ceil(topk / 64))
//   c[b]  = nb[b] > 0 ? nb[b] + overhead : 0
//   C, G  = exclusive prefix sums of c and nb;  W = C[B], NB = G[B]
//   x_p   = ceil(p * W / P) for p in [0, P]
//   gs_p  = NB if x_p >= W, else G[b] + max(0, x_p - C[b] - overhead) with
//           b the sequence whose cost interval [C[b], C[b+1]) holds x_p
//   part p covers global blocks [gs_p, gs_{p+1}); the segments of sequence b
//   are the non-empty parts that intersect [G[b], G[b+1]).
#include "fa_common.h"
#include "fa_wave.h"

namespace fa {
namespace {

// One part per thread (P <= threads) and at most four sequences per thread
// (B <= 4 * threads): 1024 threads cover every valid call, and 256 threads
// (fewer waves in every scan) the calls with P <= 256 and B <= 1024.
constexpr int kMetaThreadsMax = 1024;
constexpr int kMetaThreadsSmall = 256;
constexpr int kMaxB = FA_MLA_MAX_BATCH;
constexpr int kMaxP = FA_MLA_MAX_PARTS;
static_assert(kMaxP <= kMetaThreadsMax && kMaxB <= 4 * kMetaThreadsMax, "one block covers a call");

__device__ inline long long wave_scan(long long x) { return wave_incl_scan64(x); }
__device__ inline int wave_scan(int x) { return wave_incl_scan(x); }

// Inclusive prefix sums over the work-group of a value of type I and a 32-bit value
// (one pair per thread): DPP scans inside each wave (no LDS round trips), then
// the totals of the waves before this one read back from LDS (broadcast reads;
// two barriers; `shv` / `sh32` are free again on return).  Returns the total of k.
template <typename I, int kWaves>
__device__ int block_incl_scan2(I& v, int& k, I* shv, int* sh32) {
  const int lane = threadIdx.x & 63, w = wave_id();
  v = wave_scan(v);
  k = wave_incl_scan(k);
  if (lane == 63) {
    shv[w] = v;
    sh32[w] = k;
  }
  __syncthreads();
  I bv = 0;
  int bk = 0, total = 0;
#pragma unroll
  for (int i = 0; i < kWaves; ++i) {
    const int ki = sh32[i];
    if (i < w) {  // uniform
      bv += shv[i];
      bk += ki;
    }
    total += ki;
  }
  __syncthreads();
  v += bv;
  k += bk;
  return total;
}

// block_incl_scan2 of a 32-bit value alone.
template <int kWaves>
__device__ void block_incl_scan(int& k, int* sh32) {
  const int lane = threadIdx.x & 63, w = wave_id();
  k = wave_incl_scan(k);
  if (lane == 63) sh32[w] = k;
  __syncthreads();
  int bk = 0;
#pragma unroll
  for (int i = 0; i < kWaves - 1; ++i) {
    if (i < w) bk += sh32[i];  // uniform
  }
  __syncthreads();
  k += bk;
}

// Largest i in [0, n) with a[i] <= x (a non-decreasing, a[0] <= x).  An 8-way search:
// the answer lies in [lo, hi) with a[lo] <= x; each round probes lo + k * step for
// k = 1..7 (seven independent LDS reads, one latency per round instead of one per
// halving), and the probes that pass form a prefix.  n <= 64 takes two rounds.
template <typename I>
__device__ int last_le(const I* a, int n, I x) {
  int lo = 0, hi = n;
  while (hi - lo > 1) {
    const int step = (hi - lo + 7) >> 3;
    int cnt = 0;
#pragma unroll
    for (int k = 1; k < 8; ++k) {
      const int p = lo + k * step;
      const I v = a[p < hi ? p : hi - 1];
      cnt += (p < hi && v <= x) ? 1 : 0;
    }
    lo += cnt * step;
    hi = min(hi, lo + step);
  }
  return lo;
}

// floor(a / b) for 0 <= a < 2^48, b > 0, given rb = 1.0 / b: the double-precision
// estimate a * rb is within 2^48 * 2^-52 of a / b, so one integer correction step
// makes it exact (a stays below 2^48 here: P * W with P <= 2^10 and W <= 4096 *
// (2^25 + 4)).  The divisors P and W are the same for every part, so each thread
// divides once per divisor and multiplies per quotient.
__device__ inline long long floor_div(long long a, long long b, double rb) {
  long long q = static_cast<long long>(static_cast<double>(a) * rb);
  while (q * b > a) --q;
  while ((q + 1) * b <= a) ++q;
  return q;
}

// Cuts of the cost line, x_p = ceil(p W / P), and the last part whose cut is <= c.
// 64-bit: both divisions by double estimates.
template <typename I>
struct Cuts;
template <>
struct Cuts<long long> {
  long long W;
  int P;
  double rP, rW;
  __device__ Cuts(long long w, int p)
      : W(w), P(p), rP(1.0 / static_cast<double>(p)), rW(1.0 / static_cast<double>(w > 0 ? w : 1)) {}
  __device__ long long at(int p) const {
    // x_P = W exactly: no division for the last cut (with P = threads it is the one
    // part a thread would otherwise take second)
    return p == P ? W : floor_div(static_cast<long long>(p) * W + P - 1, P, rP);
  }
  __device__ int last_at_or_before(long long c) const {
    return static_cast<int>(floor_div(c * P, W, rW));
  }
};
// 32-bit (W < 2^30, P <= 2^10): W = wq P + wr gives x_p = p wq + ceil(p wr / P), whose
// dividend stays below 2^21: exact from a float estimate and one correction; the part of a
// position c comes from the float estimate c P / W (below 2^10, so within 1) and the cuts
// beside it.
template <>
struct Cuts<int> {
  int W, P, wq, wr;
  float rP, rW;
  __device__ Cuts(int w, int p) : W(w), P(p), wq(w / p), wr(w - w / p * p) {
    rP = 1.f / static_cast<float>(p);
    rW = static_cast<float>(p) / static_cast<float>(w > 0 ? w : 1);
  }
  __device__ int at(int p) const {
    const int n = p * wr + P - 1;
    int q = static_cast<int>(static_cast<float>(n) * rP);
    if (q * P > n) --q;
    if ((q + 1) * P <= n) ++q;
    return p * wq + q;
  }
  __device__ int last_at_or_before(int c) const {
    int q = min(static_cast<int>(static_cast<float>(c) * rW), P);
    if (at(q) > c) --q;
    if (q < P && at(q + 1) <= c) ++q;
    return q;
  }
};

// The partition, in block-count type I (see the file comment): C, G, gs are prefix arrays in
// LDS, ginc / kinc this thread's inclusive sums of blocks and of non-empty sequences.
template <typename I, int kMetaThreads>
__device__ void partition(const int (&nbs)[4], int b0, int b1, I ginc, I gsum, int kinc, int ksum,
                          int B, int P, int overhead, int32_t* __restrict__ md,
                          int32_t* __restrict__ num_splits, I* C, I* G, I* gs, int* pf, int* pl,
                          int* owner, int* E, int* sh32) {
  constexpr int kMetaWaves = kMetaThreads / 64;
  const int t = threadIdx.x;
  // 1. G and C[b] = G[b] + overhead * (non-empty sequences before b)
  {
    I gg = ginc - gsum;
    int kk = kinc - ksum;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (b0 + i < b1) {
        G[b0 + i] = gg;
        C[b0 + i] = gg + static_cast<I>(overhead) * kk;
        gg += nbs[i];
        kk += nbs[i] > 0;
      }
    }
    if (t == kMetaThreads - 1) {
      G[B] = ginc;
      C[B] = ginc + static_cast<I>(overhead) * kinc;
    }
  }
  __syncthreads();
  const I W = C[B];
  const I NB = G[B];
  const Cuts<I> cuts(W, P);

  // 2. part starts x_p = ceil(p W / P) on the cost line -> global blocks; and
  //    per sequence, the parts that hold its first and last block, in closed
  //    form: gs_p <= G[b] exactly when x_p <= C[b] + overhead, and
  //    gs_p < G[b+1] exactly when x_p < C[b+1], and x_p grows with p.
  for (int p = t; p <= P; p += kMetaThreads) {
    const I x = cuts.at(p);
    I v;
    int own;
    if (x >= W) {
      v = NB;
      own = B;
    } else {
      own = last_le(C, B, x);
      const I o = x - C[own] - overhead;
      v = G[own] + (o > 0 ? o : 0);
    }
    gs[p] = v;
    owner[p] = own;
  }
  for (int b = b0; b < b1; ++b) {
    if (G[b + 1] > G[b]) {
      pf[b] = cuts.last_at_or_before(C[b] + overhead);
      pl[b] = cuts.last_at_or_before(C[b + 1] - 1);
    }
  }
  __syncthreads();

  // 3. E[p] = number of empty parts in [0, p).
  {
    const int cnt = (t < P && gs[t] == gs[t + 1]) ? 1 : 0;
    int inc = cnt;
    block_incl_scan<kMetaWaves>(inc, sh32);
    if (t < P) E[t] = inc - cnt;
    if (t == kMetaThreads - 1) E[P] = inc;
  }
  __syncthreads();

  // 4. per-part descriptors: a non-empty part starts in the sequence whose
  //    cost interval holds its x_p.
  if (t < P) {
    const I g0 = gs[t], g1 = gs[t + 1];
    int4* m = reinterpret_cast<int4*>(md + static_cast<long long>(t) * kMdStride);
    if (g0 == g1) {
      m[0] = make_int4(0, 0, 0, 0);
      m[1] = make_int4(0, 0, static_cast<int32_t>(g0), 0);
    } else {
      const int bb = owner[t];
      const int eb = last_le(G, B, static_cast<I>(g1 - 1));
      const int f = pf[bb];
      m[0] = make_int4(bb, static_cast<int32_t>(g0 - G[bb]), eb, static_cast<int32_t>(g1 - G[eb]));
      m[1] = make_int4((t - f) - (E[t] - E[f]), static_cast<int32_t>(g1 - g0),
                       static_cast<int32_t>(g0), 0);
    }
  }

  // 5. segments per sequence (non-empty parts from pf[b] to pl[b]) ->
  //    exclusive prefix num_splits[B+1].
  {
    int segs[4];
    int sum = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int b = b0 + i;
      segs[i] = b < b1 && nbs[i] > 0 ? (pl[b] - pf[b] + 1) - (E[pl[b]] - E[pf[b]]) : 0;
      sum += segs[i];
    }
    int inc = sum;
    block_incl_scan<kMetaWaves>(inc, sh32);
    int acc = inc - sum;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (b0 + i < b1) num_splits[b0 + i] = acc;
      acc += segs[i];
    }
    if (t == kMetaThreads - 1) num_splits[B] = inc;
  }
}

// The 32-bit partition runs when no sequence has 2^17 blocks (8.4M tokens) and the overhead
// is at most 2^16, which keeps every sum below 2^30; the count of longer sequences rides in
// the upper half of the non-empty count's scan.  Time per call in a replayed graph, 256 parts,
// 64 bits / 32: 2 sequences 3.9 / 3.7 us, 64 4.3 / 4.0, 300 5.7 / 4.8 (what is left is the
// chain of scans, searches and barriers).
constexpr int kBigBlocks = 1 << 17;
constexpr int kBigOverhead = 1 << 16;

template <int kMetaThreads>
__global__ __launch_bounds__(kMetaThreads) void mla_metadata_kernel(
    const int32_t* __restrict__ lens, int B, int topk, int P, int overhead,
    int32_t* __restrict__ md, int32_t* __restrict__ num_splits) {
  __shared__ long long C[kMaxB + 1];  // exclusive prefix of the cost
  __shared__ long long G[kMaxB + 1];  // exclusive prefix of the blocks
  __shared__ int pf[kMaxB];           // part holding the first block of sequence b
  __shared__ int pl[kMaxB];           // part holding its last block
  __shared__ long long gs[kMaxP + 1];  // first global block of part p
  __shared__ int owner[kMaxP + 1];     // sequence whose cost interval holds x_p
  __shared__ int E[kMaxP + 1];         // empty parts in [0, p)
  constexpr int kMetaWaves = kMetaThreads / 64;
  __shared__ long long sh64[kMetaWaves];
  __shared__ int sh32[kMetaWaves];

  const int t = threadIdx.x;
  const int ipt = cdiv(B, kMetaThreads);  // sequences per thread (<= 4)
  const int b0 = min(B, t * ipt), b1 = min(B, b0 + ipt);
  int nbs[4];
  int gsum = 0, ksum = 0;  // at most 4 * 2^25
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    // topk > 0: every sequence has topk slots
    const int len = b0 + i < b1 ? (topk > 0 ? topk : lens[b0 + i]) : 0;
    nbs[i] = len > 0 ? (len >> 6) + ((len & 63) != 0) : 0;
    gsum += nbs[i];
    ksum += (nbs[i] > 0) + ((nbs[i] >= kBigBlocks) << 16);
  }
  static_assert(kPage == 64, "blocks by shifts");
  int ginc = gsum, kinc = ksum;
  const int total = block_incl_scan2<int, kMetaWaves>(ginc, kinc, reinterpret_cast<int*>(sh64), sh32);
  const bool big = (total >> 16) != 0 || overhead > kBigOverhead;  // uniform
  if (!big) {
    partition<int, kMetaThreads>(nbs, b0, b1, ginc, gsum, kinc, ksum, B, P, overhead, md,
                                 num_splits, reinterpret_cast<int*>(C), reinterpret_cast<int*>(G),
                                 reinterpret_cast<int*>(gs), pf, pl, owner, E, sh32);
  } else {
    long long ginc64 = gsum;
    ksum &= 0xFFFF;
    int kinc64 = ksum;
    block_incl_scan2<long long, kMetaWaves>(ginc64, kinc64, sh64, sh32);
    partition<long long, kMetaThreads>(nbs, b0, b1, ginc64, gsum, kinc64, ksum, B, P, overhead,
                                       md, num_splits, C, G, gs, pf, pl, owner, E, sh32);
  }
}

// Sparse: every sequence has T = ceil(topk / 64) blocks and costs nothing more, so W = NB =
// B T and the values have closed forms: a part's cut is its first block, and the first and
// last parts of a sequence come from the cuts.  Parts are empty only when P > W; then every
// other part holds one block, and x_p parts before part p are not empty.  A sequence start
// j T is also a part's start exactly when (P j mod B) T < P; the segments before sequence b
// are the parts that start before b T plus one for every start in between that splits a
// part -- the one scan here.  Time per call in a replayed graph, general
// partition / this: 64 sequences of top-2,048, 256 parts 4.15 / 2.09 us.
template <int kMetaThreads>
__global__ __launch_bounds__(kMetaThreads) void mla_metadata_uniform_kernel(
    int B, int T, int P, int32_t* __restrict__ md, int32_t* __restrict__ num_splits) {
  constexpr int kMetaWaves = kMetaThreads / 64;
  __shared__ int sh32[kMetaWaves];
  const int t = threadIdx.x;
  const int W = B * T;  // < 2^30 (host)
  const Cuts<int> cuts(W, P);
  auto used_before = [&](int p) { return P <= W ? p : cuts.at(p); };  // non-empty parts in [0, p)
  if (t < P) {
    const int g0 = cuts.at(t), g1 = cuts.at(t + 1);
    int4* m = reinterpret_cast<int4*>(md + static_cast<long long>(t) * kMdStride);
    if (g0 == g1) {
      m[0] = make_int4(0, 0, 0, 0);
      m[1] = make_int4(0, 0, g0, 0);
    } else {
      const int bb = g0 / T, eb = (g1 - 1) / T;
      const int f = cuts.last_at_or_before(bb * T);
      m[0] = make_int4(bb, g0 - bb * T, eb, g1 - eb * T);
      m[1] = make_int4(used_before(t) - used_before(f), g1 - g0, g0, 0);
    }
  }
  const int ipt = cdiv(B, kMetaThreads);  // <= 4
  const int b0 = min(B, t * ipt), b1 = min(B, b0 + ipt);
  int cut[4], sum = 0;  // starts that split a part
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int j = b0 + i;
    cut[i] = j < b1 && j > 0 && static_cast<int>(static_cast<unsigned int>(P * j) % B) * T >= P;
    sum += cut[i];
  }
  int inc = sum;
  block_incl_scan<kMetaWaves>(inc, sh32);
  int acc = inc - sum;  // of the starts before b0
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int b = b0 + i;
    if (b < b1)
      num_splits[b] = b == 0 ? 0 : used_before(cuts.last_at_or_before(b * T - 1) + 1) + acc;
    acc += cut[i];
  }
  if (t == kMetaThreads - 1)
    num_splits[B] = used_before(cuts.last_at_or_before(W - 1) + 1) + inc;
}

}  // namespace
}  // namespace fa

extern "C" int fa_mla_get_metadata(const int32_t* cache_seqlens, int32_t batch, int32_t topk,
                                   int32_t num_parts, int32_t fixed_overhead, int32_t* tile_md,
                                   int32_t* num_splits, void* stream) {
  FA_CHECK_ARG(batch >= 1 && batch <= FA_MLA_MAX_BATCH, "batch %d outside [1, %d]", batch,
               FA_MLA_MAX_BATCH);
  FA_CHECK_ARG(num_parts >= 1 && num_parts <= FA_MLA_MAX_PARTS,
               "num_parts %d outside [1, %d]", num_parts, FA_MLA_MAX_PARTS);
  FA_CHECK_ARG(fixed_overhead >= 0, "fixed_overhead %d < 0", fixed_overhead);
  FA_CHECK_ARG(topk >= 0, "topk %d < 0", topk);
  FA_CHECK_ARG(topk > 0 || cache_seqlens != nullptr, "cache_seqlens is NULL");
  FA_CHECK_ARG(tile_md != nullptr && num_splits != nullptr, "output pointer is NULL");
  FA_CHECK_ARG(reinterpret_cast<uintptr_t>(tile_md) % 16 == 0, "tile_md is not 16-byte aligned");
  const bool small = num_parts <= fa::kMetaThreadsSmall && batch <= 4 * fa::kMetaThreadsSmall;
  const dim3 threads(small ? fa::kMetaThreadsSmall : fa::kMetaThreadsMax);
  const hipStream_t s = static_cast<hipStream_t>(stream);
  const long long t = (static_cast<long long>(topk) + fa::kPage - 1) / fa::kPage;
  if (topk > 0 && fixed_overhead == 0 && batch * t < (1ll << 30)) {
    hipLaunchKernelGGL(small ? fa::mla_metadata_uniform_kernel<fa::kMetaThreadsSmall>
                             : fa::mla_metadata_uniform_kernel<fa::kMetaThreadsMax>,
                       dim3(1), threads, 0, s, batch, static_cast<int>(t), num_parts, tile_md,
                       num_splits);
  } else {
    hipLaunchKernelGGL(small ? fa::mla_metadata_kernel<fa::kMetaThreadsSmall>
                             : fa::mla_metadata_kernel<fa::kMetaThreadsMax>,
                       dim3(1), threads, 0, s, cache_seqlens, batch, topk, num_parts,
                       fixed_overhead, tile_md, num_splits);
  }
  FA_CHECK_HIP(hipGetLastError());
  return FA_OK;
}
