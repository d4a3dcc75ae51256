// Attention of many query rows per KV head over contiguous K/V (chunked and whole
// prefill, speculative verification) for gfx950: fp16 or bf16, head dim 64, 128, 256.
//
// The decode kernels (fa_gqa_decode.hip) give a work-group 16 query rows, and every block
// of 16 rows streams the whole K and V: with thousands of rows that is bound by the L2 and
// by VALU work per tile, not by the matrix cores.  Here a work-group = 4 waves = 128 query
// rows of one (sequence, KV head), 32 per wave, which share every K/V tile through LDS;
// two work-groups (of independent phase) per CU, so that one wave of a SIMD runs MFMAs
// while the other runs its softmax.
//
// A query row is a (query position, query head of the group) pair, positions outermost:
// the rows of a work-group then span as few positions as possible, so a causal work-group
// stops at the last key its rows see and only its last tiles need masks.
//
// Per tile of 64 keys (32 at head dim 256, where the O accumulators leave fewer
// registers) and wave, all MFMA 32x32x16, fp32 accumulation:
//   S^T[keys, 32 rows] = K Q^T: K (A operand) by ds_read_b128, Q^T (B) in VGPRs for the
//     whole kernel;
//   softmax: a lane holds half of one row's scores (lane % 32 = row, the other half is 32
//     lanes away), so the row max is in-lane plus one lane swap, and the row sum stays
//     in-lane until the end.  The reference that P is relative to follows each tile's
//     maximum, down as well as up (kFall), and the accumulators are rescaled at every tile:
//     the largest P of a tile is then a power of two, and rounding it to 16 bits costs nothing.
//     With one running maximum instead (rescaling only where some row has a new one) a long
//     row has few such keys: 2% faster, but bf16 error against 64 bits 2.26e-3 instead of
//     2.09e-3 at the first shape below, where the 16-row kernel (a reference per 32-key tile
//     and wave) has 2.20e-3.  Over few keys the tile's halves take a reference each
//     (kHalvesKeys).
//   O^T[D, 32 rows] += V^T P^T: P^T (B) is the lane's own scores rounded to 16 bits (the
//     k order only has to agree between A and B: lane half g holds keys 16s + 4g..+3 and
//     16s + 8 + 4g..+3 of k-step s), V^T (A) by the transposing ds_read_b64_tr_b16.
// Tiles go HBM/L2 -> LDS without VGPR staging, double-buffered: tile t+1 is requested when
// every wave is done with tile t-1, and has the whole of step t to land.  K operands are
// read one k-step ahead of their MFMAs (2% at D = 128, 8% at D = 256 causal).
//
// Measured (bf16, wall time per call, 16-row kernel -> this one): 2,048 new positions behind
// 1,901, B = 2, 32 heads of 8 KV heads, D = 128, causal: 1578 -> 213 us (0.92 PFLOP/s; a
// large bf16 matrix product reaches 1.4 here, and the socket's power limit bounds both);
// 8 positions x group 8 over 2,000 keys, B = 8: 45 -> 23 us;
// 5 positions x group 4 over 4,000 keys, B = 8: 59 -> 26 us.
//
// LDS layouts (16-byte chunk c of token row r): K at chunk c ^ fk(r), so that the 16 rows
// of a quarter wave's reads at one chunk cover 256 distinct bytes; V at pair (c / 2) ^
// fv(r), so that the 4 rows x 2 dim halves of a transposing read's half wave do.
//
// Reference lineage: _fwd_kernel (src/flag_attn/flash.py:348-500): online softmax, causal
// bottom-right alignment, (o, L) outputs.
#include "fa_common.h"
#include "fa_prefill.h"
#include "fa_wave.h"

namespace fa {
namespace {

constexpr int kPWaves = 4;
constexpr int kPThreads = 64 * kPWaves;
constexpr int kPWaveRows = 32;
static_assert(kPWaves * kPWaveRows == kPrefillRows, "rows per work-group");
// A row's reference is the rounded product of its largest score and the scale; the fused
// multiply-add of the exponents does not round that product, which leaves the largest
// exponent at the rounding error instead of a whole number: up to 2^-15 for references below
// 2^10 (P still rounds to a power of two), but +-32 at 2^30.  Past this reference the scores
// are scaled in a pass of their own.
constexpr float kFusedScale = 1024.f;
// How far below a row's running maximum (log2 units) the maximum that P follows may fall.
// Error at the first shape above 2.11e-3 at 2, 2.090e-3 at 4 and at 8.  In bf16 the reference
// lies kFall above that maximum (the largest P of a tile is 2^-4, as exact as 1), so never
// below the running one, and the sums of any finite V stay as far from overflow as with it.
// fp16 keeps 1: its P would lose bits below 2^-14, and its V is at most 2^16.
constexpr float kFall = 4.f;
// Up to this many keys that a row sees on average, the 32-key halves of a 64-key tile take a
// reference each.  bf16 error against 64 bits, 16-row kernel / tile / halves: 300 keys
// 2.056e-3 / 2.115e-3 / 2.042e-3, 300 x 300 causal 1.900e-3 / 1.924e-3 / 1.894e-3, 1,024 x
// 1,024 causal 1.946e-3 / 1.963e-3 / 1.924e-3; at 2,100 keys 2.087e-3 / 2.076e-3 / 2.015e-3,
// 3,000 x 3,000 causal 1.987e-3 / 1.985e-3 / 1.942e-3.  The second rescale costs 5 .. 9%
// (1,024 x 1,024 37.4 -> 40.7 us), so it stays off where the tile's maximum is enough.
constexpr int kHalvesKeys = 1536;

template <typename T>
struct PVec {
  typedef T v8 __attribute__((ext_vector_type(8)));
  typedef T v4 __attribute__((ext_vector_type(4)));
};

__device__ inline floatx16 mfma_32x32x16(PVec<__bf16>::v8 a, PVec<__bf16>::v8 b, floatx16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}
__device__ inline floatx16 mfma_32x32x16(PVec<_Float16>::v8 a, PVec<_Float16>::v8 b, floatx16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

template <typename T>
__device__ inline typename PVec<T>::v4 lds_tr_read4(const unsigned char* p) {
  typedef short shortx4 __attribute__((ext_vector_type(4)));
  const shortx4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((FA_LDS shortx4*)(p));
  return __builtin_bit_cast(typename PVec<T>::v4, v);
}

// 16 bytes per lane from base + off (32-bit lane offset, uniform base) into LDS.
__device__ inline void lds_dma16_off(const unsigned char* base, unsigned int off, FA_LDS void* lds) {
  const unsigned m0 = __builtin_amdgcn_readfirstlane(
      static_cast<unsigned>(reinterpret_cast<__SIZE_TYPE__>(lds)));
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
               :
               : "v"(off), "s"(base), "s"(m0)
               : "memory", "m0");
}

// Chunk (K) and chunk-pair (V) swizzles of token row r, C chunks per row.
template <int C>
__device__ inline int fk(int r) {
  return C >= 16 ? (r & 15) : ((r >> 1) & 7);  // C = 8: two rows per 256 bytes
}
template <int C>
__device__ inline int fv(int r) {
  return C >= 16 ? (((r & 3) << 1) | ((r >> 2) & 1)) : ((r & 2) | ((r >> 2) & 1));
}

template <typename T, int D, bool kHalves>
__global__ __launch_bounds__(kPThreads, 2) void gqa_prefill_kernel(const fa_gqa_decode_args a,
                                                                  const int n_rb,
                                                                  const int fits) {
  typedef typename PVec<T>::v8 T8;
  typedef typename PVec<T>::v4 T4;
  constexpr int C = D / 8;               // 16-byte chunks per row
  constexpr int kRowB = 2 * D;           // bytes per token row
  constexpr int kTok = D <= 128 ? 64 : 32;  // keys per tile
  constexpr int kSub = kTok / 32;        // 32-key sub-tiles of S^T
  constexpr int kParts = kHalves ? kSub : 1;  // softmax references per tile
  constexpr int kPer = kSub / kParts;    // sub-tiles of each
  constexpr int kTileB = kTok * kRowB;
  constexpr int kCopies = kTileB / 1024 / kPWaves;  // 1 KB copies per wave, of K and of V
  constexpr int kRowsPerCopy = 1024 / kRowB;
  constexpr int kKSteps = D / 16;        // MFMA k-steps of QK
  constexpr int kDimTiles = D / 32;      // 32-dim tiles of O^T
  static_assert(kCopies * kPWaves * 1024 == kTileB, "whole copies per wave");
  // [K, V][tile parity]; the epilogue stages each wave's 32 output rows over them
  __shared__ __attribute__((aligned(16))) unsigned char bufs[4 * kTileB];
  static_assert(4 * kTileB >= kPrefillRows * kRowB, "output staging fits the tile buffers");

  // Work-group -> ((sequence, KV head) pair, row block).  Work-groups are dealt round-robin
  // over 8 XCDs.  Pairs in multiples of 8: each XCD takes whole pairs one after the other,
  // so a pair's K/V stays in one L2.  Otherwise pairs vary fastest.  Either way the last
  // row blocks (the longest under a causal mask) go first, and the shortest last; but when
  // everything is resident at once (fits), the second half goes up again, so that a CU's
  // two work-groups are a long and a short one.
  const int group = a.h_q / a.h_kv;
  const int rows_total = group * a.m;
  const int pairs = a.batch * a.h_kv;
  const int split = blockIdx.y;
  const int wg = blockIdx.x;
  int pair, rb;
  if ((pairs & 7) == 0) {
    const int k = wg >> 3, i = k % n_rb;
    pair = (wg & 7) * (pairs >> 3) + k / n_rb;
    rb = n_rb - 1 - i;
    if (fits && i >= n_rb / 2) rb = i - n_rb / 2;  // n_rb - 1 .. ceil(n_rb / 2), then 0 ..
  } else {
    pair = wg % pairs;
    rb = n_rb - 1 - wg / pairs;
  }
  const int b = pair / a.h_kv;
  const int hk = pair - b * a.h_kv;

  const int wave = wave_id();
  const int lane = threadIdx.x & 63;
  const int g = lane >> 5, c32 = lane & 31;

  const int seqlen = a.seqlens ? sload(a.seqlens + b) : a.n;
  const int t0 = split * a.split_tokens;
  const int t1 = min(t0 + a.split_tokens, seqlen);
  // keys visible to a row of position mm: [0, seqlen - m + 1 + mm) causal, all otherwise
  auto limit_of = [&](int row) -> int {
    return a.causal ? min(seqlen - a.m + 1 + row / group, t1) : t1;
  };
  const int row0 = rb * kPrefillRows;
  const int wg_lim = limit_of(min(row0 + kPrefillRows, rows_total) - 1);
  const int ntiles = wg_lim > t0 ? cdiv(wg_lim - t0, kTok) : 0;
  // this wave's rows (past the end: the last row again, not stored)
  const int wrow0 = row0 + kPWaveRows * wave;
  const int wave_min = limit_of(min(wrow0, rows_total - 1));
  const int wave_max = limit_of(min(wrow0 + kPWaveRows, rows_total) - 1);
  const bool wave_on = wrow0 < rows_total;
  const int row = min(wrow0 + c32, rows_total - 1);
  const int mm = row / group, jj = row - mm * group;
  const int lim = limit_of(row);

  const float ninf = -__builtin_inff();
  // The scale is applied inside the exponent, after the mask and the maximum.  That needs a
  // positive one: a negative one turns the order of the scores, and 0 times a masked -inf is
  // NaN.  Otherwise the scores are scaled before either (prescale).
  const bool prescale = !(a.scale > 0.f);  // uniform
  const float scale_log2 = prescale ? 1.f : a.scale * kLog2e;

  const unsigned char* const kp = static_cast<const unsigned char*>(a.k) +
                                  2 * (b * a.k_stride_0 + hk * a.k_stride_h);
  const unsigned char* const vp = static_cast<const unsigned char*>(a.v) +
                                  2 * (b * a.v_stride_0 + hk * a.v_stride_h);
  // Copy i of this wave: tile rows of 1 KB piece kCopies * wave + i; the lane's source chunk
  // undoes the swizzle of its LDS slot.  Offsets fit 32 bits (checked on the host).
  const unsigned int k_tb = static_cast<unsigned int>(2 * a.k_stride_t);
  const unsigned int v_tb = static_cast<unsigned int>(2 * a.v_stride_t);
  const int crow = lane / C, cslot = lane % C;
  unsigned int koff[kCopies], voff[kCopies];
#pragma unroll
  for (int i = 0; i < kCopies; ++i) {
    const int r = (kCopies * wave + i) * kRowsPerCopy + crow;
    koff[i] = r * k_tb + 16 * (cslot ^ fk<C>(r));
    voff[i] = r * v_tb + 16 * (cslot ^ (fv<C>(r) << 1));
  }
  auto issue = [&](int u, int buf) {
    const int start = t0 + kTok * u;
    const unsigned char* const ks = kp + static_cast<long long>(start) * k_tb;
    const unsigned char* const vs = vp + static_cast<long long>(start) * v_tb;
    unsigned char* const kd = bufs + buf * kTileB + kCopies * wave * 1024;
    unsigned char* const vd = bufs + (2 + buf) * kTileB + kCopies * wave * 1024;
    if (start + kTok <= t1) {  // uniform
#pragma unroll
      for (int i = 0; i < kCopies; ++i) lds_dma16_off(ks, koff[i], (FA_LDS void*)(kd + 1024 * i));
#pragma unroll
      for (int i = 0; i < kCopies; ++i) lds_dma16_off(vs, voff[i], (FA_LDS void*)(vd + 1024 * i));
    } else {  // rows past the split's end repeat its last row (masked)
      const int last = t1 - 1 - start;
#pragma unroll
      for (int i = 0; i < kCopies; ++i) {
        const int r = (kCopies * wave + i) * kRowsPerCopy + crow;
        const unsigned int back = r > last ? r - last : 0;
        lds_dma16_off(ks, koff[i] - back * k_tb, (FA_LDS void*)(kd + 1024 * i));
        lds_dma16_off(vs, voff[i] - back * v_tb, (FA_LDS void*)(vd + 1024 * i));
      }
    }
  };

  // Q^T operand: row c32, dims 16kk + 8g..+7
  T8 qf[kKSteps];
  {
    const T* const qrow = static_cast<const T*>(a.q) + b * a.q_stride_b +
                          (hk * group + jj) * a.q_stride_h + mm * a.q_stride_m + 8 * g;
#pragma unroll
    for (int kk = 0; kk < kKSteps; ++kk) qf[kk] = *reinterpret_cast<const T8*>(qrow + 16 * kk);
  }

  floatx16 acc[kDimTiles];
#pragma unroll
  for (int dt = 0; dt < kDimTiles; ++dt) acc[dt] = floatx16{};
  float mref = ninf, mrun = ninf, lsum = 0.f;

  // lane offsets of the LDS reads
  const int kbase = c32 * kRowB + 16 * (g ^ fk<C>(c32));  // chunk 2kk + g: xor 32 kk
  const int h16 = lane >> 4, e = (lane & 15) >> 2, qd = lane & 3;
  const int vtok = 4 * g + e;  // token within 8
  constexpr int kVBases = kDimTiles < 4 ? kDimTiles : 4;  // fv < 8: dt + 4 is 256 bytes on
  int vbase[kVBases];
#pragma unroll
  for (int dt = 0; dt < kVBases; ++dt)
    vbase[dt] = vtok * kRowB + 32 * ((2 * dt + (h16 & 1)) ^ fv<C>(vtok)) + 16 * (qd >> 1) +
                8 * (qd & 1);

  if (ntiles > 0) issue(0, 0);
  for (int u = 0; u < ntiles; ++u) {
    const int buf = u & 1;
    const int start = t0 + kTok * u;
    wait_vmem<0>();  // this wave's copies of tile u (requested one step ago)
    barrier();       // everyone's; and everyone is done with tile u-1
    if (u + 1 < ntiles) issue(u + 1, buf ^ 1);
    if (!wave_on || start >= wave_max) continue;  // uniform: no row of the wave sees a key here
    const unsigned char* const kb = bufs + buf * kTileB;
    const unsigned char* const vb = bufs + (2 + buf) * kTileB;

    // K operands one k-step ahead of their MFMAs (the fences keep them there)
    floatx16 s[kSub];
    T8 ka[2][kSub];
    auto k_read = [&](int kk, int tt) -> T8 {
      return *reinterpret_cast<const T8*>(kb + 32 * tt * kRowB + (kbase ^ (32 * kk)));
    };
#pragma unroll
    for (int tt = 0; tt < kSub; ++tt) {
      s[tt] = floatx16{};
      ka[0][tt] = k_read(0, tt);
    }
#pragma unroll
    for (int kk = 0; kk < kKSteps; ++kk) {
      if (kk + 1 < kKSteps) {
#pragma unroll
        for (int tt = 0; tt < kSub; ++tt) ka[(kk + 1) & 1][tt] = k_read(kk + 1, tt);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int tt = 0; tt < kSub; ++tt) s[tt] = mfma_32x32x16(ka[kk & 1][tt], qf[kk], s[tt]);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (prescale) {
#pragma unroll
      for (int tt = 0; tt < kSub; ++tt)
#pragma unroll
        for (int i = 0; i < 16; ++i) s[tt][i] *= a.scale * kLog2e;
    }
    if (start + kTok > wave_min) {  // uniform: some row does not see the whole tile
      const int left = lim - start - 4 * g;
#pragma unroll
      for (int tt = 0; tt < kSub; ++tt)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int j = 32 * tt + 8 * (i >> 2) + (i & 3);  // + 4g: the key of s[tt][i]
          s[tt][i] = j < left ? s[tt][i] : ninf;
        }
    }
    // softmax and PV of the tile, or of its 32-key halves one after the other
#pragma unroll
    for (int part = 0; part < kParts; ++part) {
      const int tt0 = part * kPer;
      float mx = s[tt0][0];
#pragma unroll
      for (int tt = tt0; tt < tt0 + kPer; ++tt)
#pragma unroll
        for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[tt][i]);
      mx = max_xor32(mx) * scale_log2;
      mrun = fmaxf(mrun, mx);
      const float m_new =
          __is_same(T, __bf16) ? fmaxf(mx + kFall, mrun) : fmaxf(mx, mrun - kFall);
      const float alpha = m_new == ninf ? 1.f : __builtin_amdgcn_exp2f(mref - m_new);
      lsum *= alpha;
      mref = m_new;
#pragma unroll
      for (int dt = 0; dt < kDimTiles; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[dt][i] *= alpha;
      const float nm = mref == ninf ? 0.f : -mref;
      float c = scale_log2;
      if (__ballot(fabsf(nm) > kFusedScale) != 0ull) {  // uniform
#pragma unroll
        for (int tt = tt0; tt < tt0 + kPer; ++tt)
#pragma unroll
          for (int i = 0; i < 16; ++i) s[tt][i] *= c;
        c = 1.f;
      }
      T8 pb[2 * kPer];
      float ps = 0.f;
#pragma unroll
      for (int ss = 0; ss < 2 * kPer; ++ss)
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const float p = __builtin_amdgcn_exp2f(
              __builtin_fmaf(s[tt0 + (ss >> 1)][8 * (ss & 1) + i], c, nm));
          ps += p;
          pb[ss][i] = static_cast<T>(p);
        }
      lsum += ps;
#pragma unroll
      for (int ss = 0; ss < 2 * kPer; ++ss)
#pragma unroll
        for (int dt = 0; dt < kDimTiles; ++dt) {
          const unsigned char* const p = vb + 16 * (2 * tt0 + ss) * kRowB + 256 * (dt >> 2) + vbase[dt & 3];
          const T4 lo = lds_tr_read4<T>(p);
          const T4 hi = lds_tr_read4<T>(p + 8 * kRowB);
          const T8 va = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
          acc[dt] = mfma_32x32x16(va, pb[ss], acc[dt]);
        }
    }
  }
  wait_vmem<0>();
  barrier();  // the tile buffers are free
  if (!wave_on) return;

  const float l = sum_xor32(lsum);
  const bool some = l > 0.f;  // else no visible key: out 0, lse -inf
  const float inv = some ? 1.f / l : 0.f;
  const float lse = some ? (mref + log2f(l)) * kLn2 : ninf;
  const int h = hk * group + jj;
  const long long orow = (static_cast<long long>(b) * a.h_q + h) * a.m + mm;
  const bool mine = wrow0 + c32 < rows_total;
  if (a.o_part != nullptr) {
    if (mine) {
      const long long prow = orow * a.num_splits + split;
      float* const op = a.o_part + prow * D + 4 * g;
#pragma unroll
      for (int dt = 0; dt < kDimTiles; ++dt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          floatx4 w;
#pragma unroll
          for (int x = 0; x < 4; ++x) w[x] = some ? acc[dt][4 * i + x] * inv : 0.f;
          *reinterpret_cast<floatx4*>(op + 32 * dt + 8 * i) = w;
        }
      if (g == 0) a.lse_part[prow] = lse;
    }
    return;
  }
  if (mine && g == 0 && a.lse) a.lse[orow] = lse;
  // whole output rows through LDS (the wave's own 32 rows): 16 bytes per lane and store
  unsigned char* const st = bufs + wave * kPWaveRows * kRowB;
#pragma unroll
  for (int dt = 0; dt < kDimTiles; ++dt)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      T4 w;
#pragma unroll
      for (int x = 0; x < 4; ++x) w[x] = static_cast<T>(some ? acc[dt][4 * i + x] * inv : 0.f);
      *reinterpret_cast<T4*>(st + c32 * kRowB + 16 * ((4 * dt + i) ^ (c32 & 7)) + 8 * g) = w;
    }
  asm volatile("" ::: "memory");
  wait_lds();
  asm volatile("" ::: "memory");
#pragma unroll
  for (int i = 0; i < kPWaveRows * kRowB / 1024; ++i) {
    const int r = i * kRowsPerCopy + crow;
    const int rr = wrow0 + r;
    const T8 v = *reinterpret_cast<const T8*>(st + r * kRowB + 16 * (cslot ^ (r & 7)));
    if (rr < rows_total) {
      const int m2 = rr / group, j2 = rr - m2 * group;
      T* const op = static_cast<T*>(a.out) + b * a.o_stride_b + (hk * group + j2) * a.o_stride_h +
                    m2 * a.o_stride_m;
      *reinterpret_cast<T8*>(op + 8 * cslot) = v;
    }
  }
}

template <typename T>
void launch_prefill_t(const fa_gqa_decode_args* a, hipStream_t stream) {
  const int n_rb = cdiv((a->h_q / a->h_kv) * a->m, kPrefillRows);
  const dim3 grid(static_cast<unsigned>(a->batch * a->h_kv * n_rb),
                  static_cast<unsigned>(a->num_splits));
  // resident work-groups: 2 per CU (LDS), 4 at head dim 64 (VGPRs), 256 CUs
  const int fits = a->causal && a->num_splits == 1 && grid.x <= (a->d == 64 ? 1024u : 512u);
  // device lengths are not known here: halves
  const bool halves = a->seqlens || a->n - (a->causal ? a->m / 2 : 0) <= kHalvesKeys;
  if (a->d == 64)
    hipLaunchKernelGGL((halves ? gqa_prefill_kernel<T, 64, true> : gqa_prefill_kernel<T, 64, false>),
                       grid, dim3(kPThreads), 0, stream, *a, n_rb, fits);
  else if (a->d == 128)
    hipLaunchKernelGGL((halves ? gqa_prefill_kernel<T, 128, true> : gqa_prefill_kernel<T, 128, false>),
                       grid, dim3(kPThreads), 0, stream, *a, n_rb, fits);
  else
    hipLaunchKernelGGL((gqa_prefill_kernel<T, 256, false>), grid, dim3(kPThreads), 0, stream, *a,
                       n_rb, fits);
}

}  // namespace

bool prefill_takes(const fa_gqa_decode_args* a) {
  const long long rows = static_cast<long long>(a->h_q / a->h_kv) * a->m;
  if (a->block_table != nullptr || rows <= kPrefillMinRows) return false;
  if (a->d != 64 && a->d != 128 && a->d != 256) return false;
  // few keys: the 16-row kernel, if it has few work-groups
  const long long wg16 = static_cast<long long>(a->batch) * a->h_kv * ((rows + 15) / 16);
  if (a->num_splits == 1 && !a->seqlens && a->n > few_keys_min(a->d) && a->n <= kFewKeysMax &&
      wg16 <= few_keys_wgs(a->d))
    return false;
  // 32-bit lane offsets inside a tile (64 rows)
  if (a->k_stride_t < 0 || a->v_stride_t < 0 || a->k_stride_t >= (1ll << 23) ||
      a->v_stride_t >= (1ll << 23))
    return false;
  // 16-byte output stores
  if ((reinterpret_cast<uintptr_t>(a->out) & 15) != 0 || a->o_stride_b % 8 != 0 ||
      a->o_stride_h % 8 != 0 || a->o_stride_m % 8 != 0)
    return false;
  // row numbers, work-groups and pairs in 32 bits
  const long long n_rb = (rows + kPrefillRows - 1) / kPrefillRows;
  return rows < (1ll << 30) && static_cast<long long>(a->batch) * a->h_kv * n_rb < (1ll << 30);
}

int launch_prefill(const fa_gqa_decode_args* a, void* stream) {
  const hipStream_t s = static_cast<hipStream_t>(stream);
  if (a->dtype == 1)
    launch_prefill_t<__bf16>(a, s);
  else
    launch_prefill_t<_Float16>(a, s);
  FA_CHECK_HIP(hipGetLastError());
  return FA_OK;
}

}  // namespace fa
