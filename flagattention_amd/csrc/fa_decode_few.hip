// MLA decode of few query rows per KV stream (up to 32) for gfx950: dense paged, sparse
// top-k bf16, sparse fp8 -- 16 or 32 heads (one rank of a tensor-parallel model), or fewer
// heads with several query tokens.
//
// The 128-row kernel (fa_decode.hip) multiplies 128 rows whatever the call holds: at 16
// rows it spends 8x the matrix work and its per-tile chain (QK -> softmax -> P -> barrier ->
// PV) bounds the launch, not the cache stream.  Here a work-group is again 4 waves and one
// scheduler part, but holds 16 NR rows (NR = 1 or 2), which leaves the stream of tiles as
// the bound, and the step is arranged to keep it busy:
//   * four tile buffers (144 KB of LDS): two tiles in flight behind the two in use;
//   * one barrier per tile.  Step t waits for this wave's copies of tile t+1, meets the
//     barrier (tile t+1 and S(t) are then complete, buffer t-1 is free), requests tile t+3,
//     and runs softmax(t), PV(t) and QK(t+1) without another;
//   * QK split by keys and, NR = 1, by k-steps (NR = 2: by row tiles): wave w takes 16 of
//     the tile's 32 keys and the even or odd half of the 18 k-steps (or one row tile), and
//     leaves its piece of S in LDS, two slots by tile parity;
//   * every wave reads all of S (4 KB) and runs the same softmax for all rows -- the same
//     bits in every wave, cheaper than exchanging P behind a second barrier -- and keeps
//     P^T in the registers that PV takes it from;
//   * PV split by value dims: wave w owns dims 128w..128w+127 of every row.
// Softmax reference: the row max of the first tile in which the row sees a key, as in the
// 128-row kernel (scores up to 2^64 above it only make P > 1).  Past that the accumulators
// are rescaled in place.  Only then does the row maximum cross lanes.
// Tile layout, fp8 conversion (in place, by the wave that loaded each row-group), masks,
// scheduling and outputs are those of the 128-row kernel.
//
// Measured (config: 64 sequences of 4,096..8,192 tokens, 16 heads, bf16): decode kernel
// 109 -> 74 us (6.2 TB/s of cache), 32 heads 109 -> 82 us; two sequences of 256 and 384
// tokens 14.9 -> 7.3 us; sparse top-2,048 of 64 sequences, 16 heads, 43 -> 30 us (bf16) and
// 46 -> 31 us (fp8).
//
// All tile loads are inline asm with explicit vmcnt counts, so the compiler must have no
// vector-memory load of its own in flight: Q goes through LDS (the last tile buffer, free
// until the first step's request), page ids are scalar loads, row ids go through LDS.
#include "fa_common.h"
#include "fa_mla_tile.h"
#include "fa_wave.h"

namespace fa {
namespace {

constexpr int kFewRing = 4;                  // tile buffers
constexpr int kFewDimTiles = kDv / 4 / 16;   // 16-dim tiles of O^T per wave
constexpr float kHeadroom = 64.f;            // log2: how far a score may pass its row's reference

// Source of masked gather rows; never written.
__device__ __attribute__((aligned(16))) unsigned char g_few_zero[kRowBytes];

// 16 bytes per lane of a buffer resource into LDS; the pages are read once (nt).  Lanes
// past the resource's size read zeros.
__device__ inline void buf_lds16_nt(uintx4 rsrc, unsigned int voff, unsigned int soff,
                                    FA_LDS void* lds) {
  const unsigned m0 = __builtin_amdgcn_readfirstlane(
      static_cast<unsigned>(reinterpret_cast<__SIZE_TYPE__>(lds)));
  asm volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen nt lds"
               :
               : "v"(voff), "s"(rsrc), "s"(soff), "s"(m0)
               : "memory", "m0");
}

template <int kMode, int NR, bool kFold>
__global__ __launch_bounds__(kThreads, 2) void mla_decode_few_kernel(const fa_mla_decode_args a,
                                                                     int num_m_blocks) {
  __shared__ __attribute__((aligned(16))) unsigned char tiles[kFewRing * kTileBytes];
  // S pieces: [tile parity][k-step half or row tile][16-key half][lane]
  __shared__ floatx4 sx[2][2][2][64];
  // sparse: the segment's translated row ids (kFold), or each wave's ring of tile row lists
  __shared__ int32_t row_list[kFold ? kFoldTopk : 1];
  __shared__ int32_t row_ring[kMode == kDense || kFold ? 1 : 4][kFold ? 1 : kFewRing][64];

  // XCD-aware work-group -> (part, query token), as in the 128-row kernel
  const int wg = blockIdx.x;
  int part, mb;
  if ((a.num_parts & 7) == 0) {
    const int x = wg & 7, k = wg >> 3;
    mb = k % num_m_blocks;
    part = x * (a.num_parts >> 3) + k / num_m_blocks;
  } else {
    part = wg / num_m_blocks;
    mb = wg - part * num_m_blocks;
  }
  const int32_t* md = a.tile_md + part * kMdStride;
  if (sload(md + 5) == 0) return;
  const int b_begin = sload(md + 0), blk_begin = sload(md + 1);
  const int b_end = sload(md + 2), blk_end = sload(md + 3);
  const int first_local = sload(md + 4);

  const int wave = wave_id(), lane = threadIdx.x & 63;
  const int G = lane >> 4, i16 = lane & 15;
  const int lrow = lane >> 3;
  const int sub = wave & 1, hi = wave >> 1;  // this wave's piece of QK

  // Row rho -> (query token, head): dense rows are the flattened (s, h) pairs, sparse ones
  // the heads of query token mb.
  const int rows_total = a.s_q * a.h_q;
  const int rows_here = kMode == kDense ? rows_total : a.h_q;
  auto row_token = [&](int rho) -> int { return kMode == kDense ? rho / a.h_q : mb; };

  const float scale_log2 = a.softmax_scale * kLog2e;
  const float ninf = -__builtin_inff();
  const int topk_pad = (a.topk + kPage - 1) / kPage * kPage;
  const long long row_stride = a.kv_row_stride, block_stride = a.kv_block_stride;
  const unsigned char* const kv = static_cast<const unsigned char*>(a.kv);
  const bf16* const q = static_cast<const bf16*>(a.q);

  // LDS read offsets: K operand (token 16 sub + i16, chunk 4 kq + G) by k-step parity, V^T
  // operand by dim tile % 4 (see fa_decode.hip)
  int koff[2], voff[4];
#pragma unroll
  for (int par = 0; par < 2; ++par)
    koff[par] = ((i16 >> 3) + 2 * sub) * kRowGroupBytes + 128 * (i16 & 7) +
                16 * ((4 * par + G) ^ (i16 & 7));
  {
    const int e = i16 >> 2, qd = i16 & 3;
    const int rr = 4 * (G & 1) + e;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
      voff[dt] = ((G >> 1) * kChunkGroups + 2 * wave) * kBlockBytes +
                 16 * (rr * 8 + ((2 * dt + (qd >> 1)) ^ rr)) + 8 * (qd & 1);
  }
  // dense copies: lane offset inside a half page
  const unsigned int page_voff =
      __umul24(static_cast<unsigned int>(8 * wave + lrow), static_cast<unsigned int>(row_stride)) +
      static_cast<unsigned int>(16 * ((lane & 7) ^ lrow));
  constexpr int kCopies = kMode == kSparseFp8 ? kFp8Copies : kCopiesPerWave;

  // metadata of another call must not drive accesses out of bounds
  const int b_last = b_end < a.batch ? b_end : a.batch - 1;
  const int max_split = a.batch + a.num_parts;
  for (int b = b_begin < 0 ? 0 : b_begin; b <= b_last; ++b) {
    const int seqlen = sload(a.cache_seqlens + b);
    const int nblk_seq = (kMode == kDense) ? (seqlen > 0 ? (seqlen + kPage - 1) / kPage : 0)
                                           : topk_pad / kPage;
    const int blk_lo = (b == b_begin) ? blk_begin : 0;
    const int blk_hi = (b == b_end && blk_end < nblk_seq) ? blk_end : nblk_seq;
    if (blk_lo < 0 || blk_hi <= blk_lo) continue;
    const int tok_lo = blk_lo * kPage;
    const int tok_hi = min(blk_hi * kPage, kMode == kDense ? seqlen : a.topk);
    const int ntiles = (tok_hi - tok_lo + kTileRows - 1) / kTileRows;  // >= 1
    const int split_local = (b == b_begin) ? first_local : 0;
    const int ns0 = sload(a.num_splits + b);
    const int nsplit = sload(a.num_splits + b + 1) - ns0;
    const bool split_ok = ns0 >= 0 && split_local >= 0 && ns0 + split_local < max_split;
    // keys a row may see, relative to the segment (dense, bottom-right causal)
    int lim[NR];
#pragma unroll
    for (int rt = 0; rt < NR; ++rt) {
      const int s = row_token(min(16 * rt + i16, rows_here - 1));
      lim[rt] = ((kMode == kDense && a.causal) ? seqlen - a.s_q + 1 + s : seqlen) - tok_lo;
    }
    const int causal_from =
        (kMode == kDense && a.causal) ? (seqlen - a.s_q + 1 - tok_lo) / kTileRows : ntiles;
    const int32_t* const bt = a.block_table + static_cast<long long>(b) * a.bt_stride_b;
    const int32_t* const srows =
        kMode == kDense ? nullptr
                        : a.sparse_rows + (static_cast<long long>(b) * a.s_q + mb) * topk_pad;

    // ---- tile requests (every tile < ntiles, in order; kCopies loads per wave each) ----
    auto load_page = [&](int u) -> int {  // scalar; clamped into the table row
      return sload(bt + min(blk_lo + (u >> 1), a.max_blocks_per_seq - 1));
    };
    int page_next = -1;
    auto request_rows = [&](int u) {  // sparse: tile u's row list into this wave's ring
      if constexpr (kFold) return;
      lds_dma4(srows + tok_lo + kTileRows * u + (lane & 31),
               (FA_LDS void*)(&row_ring[wave][u & 3][0]));
    };
    // Requests tile u; returns its key mask (bit j: key j may be used).
    auto request = [&](int u) -> unsigned int {
      unsigned char* const dst = tiles + (u & 3) * kTileBytes + wave * kRowGroupBytes;
      if constexpr (kMode == kDense) {
        const int blk = blk_lo + (u >> 1), half = u & 1;
        const int page = page_next;
        if (half == 1 && u + 1 < ntiles) page_next = load_page(u + 1);
        const bool ok = blk < a.max_blocks_per_seq && page >= 0 && page < a.num_kv_blocks;
        const int start = blk * kPage + kTileRows * half;
        const int nrows = ok ? max(0, min(seqlen - start, kTileRows)) : 0;
        const unsigned long long base = reinterpret_cast<unsigned long long>(
            uniform(kv + (ok ? page : 0) * block_stride + kTileRows * half * row_stride));
        uintx4 rs;
        rs[0] = static_cast<unsigned int>(base);
        rs[1] = static_cast<unsigned int>(base >> 32) & 0xFFFFu;
        rs[2] = static_cast<unsigned int>(uniform(nrows * static_cast<int>(row_stride)));
        rs[3] = 0x00020000u;
#pragma unroll
        for (int c = 0; c < kCopies; ++c)
          buf_lds16_nt(rs, page_voff, 128 * c, (FA_LDS void*)(dst + c * kBlockBytes));
        return nrows >= kTileRows ? ~0u : ((1u << nrows) - 1u);
      } else {
        const int32_t* const ring = kFold ? row_list + kTileRows * u : row_ring[wave][u & 3];
        const int32_t rm = ring[lane & 31], r = ring[8 * wave + lrow];
        const unsigned int rr = static_cast<unsigned int>(r < 0 ? 0 : r);
        const unsigned char* src =
            kv + static_cast<unsigned long long>(rr >> 6) * static_cast<unsigned int>(block_stride) +
            __umul24(rr & 63u, static_cast<unsigned int>(row_stride));
        src = r >= 0 ? src : g_few_zero;
        if constexpr (kMode == kSparseBf16) {
          src += 16 * ((lane & 7) ^ lrow);
#pragma unroll
          for (int c = 0; c < kCopies; ++c)
            lds_dma16(src + 128 * c, (FA_LDS void*)(dst + c * kBlockBytes));
        } else {  // raw fp8 row: four code blocks, the scales, the rope chunks
          const int l8 = lane & 7;
#pragma unroll
          for (int c = 0; c < 4; ++c)
            lds_dma16(src + 128 * c + 16 * l8, (FA_LDS void*)(dst + c * kBlockBytes));
          lds_dma16(src + 512, (FA_LDS void*)(dst + kFp8ScaleOff));
          lds_dma16(src + 528 + 16 * (l8 ^ lrow), (FA_LDS void*)(dst + 8 * kBlockBytes));
        }
        return static_cast<unsigned int>(__ballot(rm >= 0));
      }
    };

    // ---- prologue: Q (into the last buffer), tiles 0..2 ----
    // Q^T operands of 1 KB, row tile rt, k-step kq at slot 18 rt + kq: lane (G, i16) row
    // 16 rt + i16, dims 32 kq + 8 G..+7.  Spread over the waves; rows past the last one
    // read zeros.
    unsigned char* const qbuf = tiles + (kFewRing - 1) * kTileBytes;
    static_assert(NR * kQkSteps * kBlockBytes <= kTileBytes, "Q fits one tile buffer");
    auto load_q = [&] {
      constexpr int kOps = NR * kQkSteps, kPerWave = (kOps + 3) / 4;
#pragma unroll
      for (int i = 0; i < kPerWave; ++i) {
        const int j = min(4 * i + wave, kOps - 1);
        const int rt = j / kQkSteps, kq = j - rt * kQkSteps;
        const int rho = 16 * rt + i16;
        const int s = row_token(min(rho, rows_here - 1));
        const int h = kMode == kDense ? rho - s * a.h_q : rho;
        const unsigned char* src =
            rho < rows_here ? reinterpret_cast<const unsigned char*>(
                                  q + b * a.q_stride_b + s * a.q_stride_s + h * a.q_stride_h +
                                  32 * kq + 8 * G)
                            : g_few_zero;
        lds_dma16(src, (FA_LDS void*)(qbuf + j * kBlockBytes));
      }
    };
    if constexpr (!kFold) load_q();
    unsigned int vm[4] = {0u, 0u, 0u, 0u};  // key masks of tiles t .. t+3
    if constexpr (kMode == kDense) {
      page_next = load_page(0);
    } else if constexpr (kFold) {
      fold_rows(a, b, mb, seqlen, tok_lo, ntiles * kTileRows, wave, row_list, load_q);
      wait_vmem<0>();
      asm volatile("" ::: "memory");
      barrier();
      asm volatile("" ::: "memory");
    } else {
      for (int u = 0; u < min(ntiles, 4); ++u) request_rows(u);
      wait_vmem<0>();
      __builtin_amdgcn_sched_barrier(0);
      asm volatile("" ::: "memory");
    }
    vm[0] = request(0);
    if (ntiles > 1) vm[1] = request(1);
    if (ntiles > 2) vm[2] = request(2);
    if (ntiles > 2) {
      wait_vmem<2 * kCopies>();
    } else if (ntiles > 1) {
      wait_vmem<kCopies>();
    } else {
      wait_vmem<0>();
    }
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
    if constexpr (kMode == kSparseFp8) dequant_fp8_rowgroup(tiles, wave);
    asm volatile("" ::: "memory");
    barrier();
    asm volatile("" ::: "memory");

    // this wave's Q operands: k-steps 2j + hi of row tile 0, or all of row tile hi
    constexpr int kNq = NR == 1 ? kQkSteps / 2 : kQkSteps;
    bf16x8 qf[kNq];
#pragma unroll
    for (int j = 0; j < kNq; ++j) {
      const int slot = NR == 1 ? 2 * j + hi : kQkSteps * hi + j;
      qf[j] = *reinterpret_cast<const bf16x8*>(qbuf + slot * kBlockBytes + 16 * lane);
    }

    // S piece of tile u -> slot u % 2 (two accumulator chains)
    auto qk = [&](int u) {
      const unsigned char* const kb = tiles + (u & 3) * kTileBytes;
      floatx4 s0 = floatx4{}, s1 = floatx4{};
#pragma unroll
      for (int j = 0; j < kNq; ++j) {
        bf16x8 k;
        if constexpr (NR == 1) {
          k = *reinterpret_cast<const bf16x8*>(kb + koff[hi] + j * kBlockBytes);
        } else {
          k = *reinterpret_cast<const bf16x8*>(kb + koff[j & 1] + (j >> 1) * kBlockBytes);
        }
        if (j & 1)
          s1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k, qf[j], s1, 0, 0, 0);
        else
          s0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k, qf[j], s0, 0, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) s0[i] += s1[i];
      sx[u & 1][hi][sub][lane] = s0;
    };

    floatx4 acc[kFewDimTiles][NR];
#pragma unroll
    for (int dt = 0; dt < kFewDimTiles; ++dt)
#pragma unroll
      for (int rt = 0; rt < NR; ++rt) acc[dt][rt] = floatx4{};
    float mref[NR], lsum[NR];
#pragma unroll
    for (int rt = 0; rt < NR; ++rt) {
      mref[rt] = ninf;
      lsum[rt] = 0.f;
    }

    qk(0);
    for (int t = 0; t < ntiles; ++t) {
      // this wave's copies of tile t+1 (and the row ids of tile t+3) have landed
      if (t + 2 < ntiles) {
        wait_vmem<kCopies>();
      } else {
        wait_vmem<0>();
      }
      __builtin_amdgcn_sched_barrier(0);
      asm volatile("" ::: "memory");
      if constexpr (kMode == kSparseFp8) {
        if (t + 1 < ntiles) dequant_fp8_rowgroup(tiles + ((t + 1) & 3) * kTileBytes, wave);
      }
      asm volatile("" ::: "memory");
      barrier();  // tile t+1 and S(t) complete; everyone is done with PV(t-1)
      asm volatile("" ::: "memory");
      if (t + 3 < ntiles) {
        if constexpr (kMode != kDense) {
          if (t + 4 < ntiles) request_rows(t + 4);  // ahead of the copies: one wait covers it
        }
        vm[3] = request(t + 3);
      }
      __builtin_amdgcn_sched_barrier(0);

      // softmax(t), all rows: row 16 rt + i16, keys 16 x + 4 G + i
      float sv[NR][8];
#pragma unroll
      for (int rt = 0; rt < NR; ++rt) {
        const float nmu = mref[rt] == ninf ? 0.f : -mref[rt];
#pragma unroll
        for (int x = 0; x < 2; ++x) {
          floatx4 s = sx[t & 1][NR == 1 ? 0 : rt][x][lane];
          if constexpr (NR == 1) {
            const floatx4 o = sx[t & 1][1][x][lane];
#pragma unroll
            for (int i = 0; i < 4; ++i) s[i] += o[i];
          }
#pragma unroll
          for (int i = 0; i < 4; ++i)
            sv[rt][4 * x + i] = __builtin_fmaf(s[i], scale_log2, nmu);
        }
      }
      if (vm[0] != ~0u || t >= causal_from) {  // uniform: not every key counts
        const unsigned int vmg = vm[0] >> (4 * G);
#pragma unroll
        for (int rt = 0; rt < NR; ++rt) {
          // sparse: slot positions are not token positions, only the mask applies
          const int left = kMode == kDense ? lim[rt] - kTileRows * t - 4 * G : kTileRows;
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            const int c = 16 * (i >> 2) + (i & 3);
            sv[rt][i] = (((vmg >> c) & 1u) && c < left) ? sv[rt][i] : ninf;
          }
        }
      }
      // V^T operands of PV(t): dims 128 wave.. of every row
      const unsigned char* const vb = tiles + (t & 3) * kTileBytes;
      bf16x8 va[kFewDimTiles];
#pragma unroll
      for (int dt = 0; dt < kFewDimTiles; ++dt) {
        const unsigned char* const p = vb + voff[dt & 3] + (dt >> 2) * kBlockBytes;
        const bf16x4 l4 = lds_read_tr4(p);
        const bf16x4 h4 = lds_read_tr4(p + 2 * kRowGroupBytes);
        va[dt] = __builtin_shufflevector(l4, h4, 0, 1, 2, 3, 4, 5, 6, 7);
      }
      // QK(t+1), in one block with the maxima so that the two overlap (past the last tile
      // it multiplies an old buffer, and its S is never read)
      qk(t + 1);
      float mx[NR];
      bool up = false;
#pragma unroll
      for (int rt = 0; rt < NR; ++rt) {
        mx[rt] = sv[rt][0];
#pragma unroll
        for (int i = 1; i < 8; ++i) mx[rt] = fmaxf(mx[rt], sv[rt][i]);
        up = up || mx[rt] > (mref[rt] == ninf ? ninf : kHeadroom);
      }
      if (__ballot(up) != 0ull) {  // uniform; a row's first keys, or scores 2^64 apart
#pragma unroll
        for (int rt = 0; rt < NR; ++rt) {
          const float old = mref[rt];
          const float m = max_xor32(max_xor16(mx[rt])) + (old == ninf ? 0.f : old);
          const float m_new = fmaxf(old, m);
          const float alpha = old == ninf ? 1.f : __builtin_amdgcn_exp2f(old - m_new);
          const float shift = m_new == ninf ? 0.f : m_new - (old == ninf ? 0.f : old);
          mref[rt] = m_new;
          lsum[rt] *= alpha;
#pragma unroll
          for (int i = 0; i < 8; ++i) sv[rt][i] -= shift;
#pragma unroll
          for (int dt = 0; dt < kFewDimTiles; ++dt)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[dt][rt][i] *= alpha;
        }
      }
      bf16x8 pb[NR];
#pragma unroll
      for (int rt = 0; rt < NR; ++rt) {
        float ps = 0.f;
        uintx4 w;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          sv[rt][i] = __builtin_amdgcn_exp2f(sv[rt][i]);
          ps += sv[rt][i];
        }
        lsum[rt] += ps;
#pragma unroll
        for (int j = 0; j < 4; ++j) w[j] = pack_bf16x2(sv[rt][2 * j], sv[rt][2 * j + 1]);
        pb[rt] = __builtin_bit_cast(bf16x8, w);
      }
#pragma unroll
      for (int dt = 0; dt < kFewDimTiles; ++dt)
#pragma unroll
        for (int rt = 0; rt < NR; ++rt)
          acc[dt][rt] =
              __builtin_amdgcn_mfma_f32_16x16x32_bf16(va[dt], pb[rt], acc[dt][rt], 0, 0, 0);
      vm[0] = vm[1];
      vm[1] = vm[2];
      vm[2] = vm[3];
    }

    // ---- outputs: lane (G, i16): row 16 rt + i16, dims 128 wave + 16 dt + 4 G..+3 ----
    const long long pbase = static_cast<long long>(ns0 + split_local) * rows_total;
    if (nsplit == 1 || split_ok) {  // uniform
#pragma unroll
      for (int rt = 0; rt < NR; ++rt) {
        const float l = sum_xor32(sum_xor16(lsum[rt]));
        const float inv = l > 0.f ? 1.f / l : 0.f;
        const float lse = l > 0.f ? (mref[rt] + log2f(l)) * kLn2 : ninf;
        const int rho = 16 * rt + i16;
        if (rho < rows_here) {
          const int s = row_token(rho);
          const int h = kMode == kDense ? rho - s * a.h_q : rho;
          bf16* const op =
              (nsplit == 1
                   ? static_cast<bf16*>(a.out) +
                         ((static_cast<long long>(b) * a.s_q + s) * a.h_q + h) * kDv
                   : static_cast<bf16*>(a.o_accum) + (pbase + s * a.h_q + h) * kDv) +
              128 * wave + 4 * G;
#pragma unroll
          for (int dt = 0; dt < kFewDimTiles; ++dt) {
            uintx2 w;
            w[0] = pack_bf16x2(acc[dt][rt][0] * inv, acc[dt][rt][1] * inv);
            w[1] = pack_bf16x2(acc[dt][rt][2] * inv, acc[dt][rt][3] * inv);
            *reinterpret_cast<uintx2*>(op + 16 * dt) = w;
          }
          if (wave == 0 && G == 0) {
            if (nsplit == 1)
              a.lse[(static_cast<long long>(b) * a.h_q + h) * a.s_q + s] = lse;
            else
              a.lse_accum[pbase + s * a.h_q + h] = lse;
          }
        }
      }
    }
    barrier();  // the tile buffers are reused by the next sequence
  }
}

template <int kMode, bool kFold>
void launch_few(const fa_mla_decode_args* a, hipStream_t stream) {
  const int rows = kMode == kDense ? a->s_q * a->h_q : a->h_q;
  const int num_m_blocks = kMode == kDense ? 1 : a->s_q;
  const dim3 grid(static_cast<unsigned>(a->num_parts * num_m_blocks));
  if (rows <= 16)
    hipLaunchKernelGGL((mla_decode_few_kernel<kMode, 1, kFold>), grid, dim3(kThreads), 0, stream, *a,
                       num_m_blocks);
  else
    hipLaunchKernelGGL((mla_decode_few_kernel<kMode, 2, kFold>), grid, dim3(kThreads), 0, stream, *a,
                       num_m_blocks);
}

}  // namespace

int launch_decode_few(const fa_mla_decode_args* a, int mode, bool fold, hipStream_t stream) {
  if (mode == kDense)
    launch_few<kDense, false>(a, stream);
  else if (mode == kSparseBf16)
    fold ? launch_few<kSparseBf16, true>(a, stream) : launch_few<kSparseBf16, false>(a, stream);
  else
    fold ? launch_few<kSparseFp8, true>(a, stream) : launch_few<kSparseFp8, false>(a, stream);
  FA_CHECK_HIP(hipGetLastError());
  return FA_OK;
}

}  // namespace fa
