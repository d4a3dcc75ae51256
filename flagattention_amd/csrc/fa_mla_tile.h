// Tile geometry and fp8 row conversion shared by the MLA decode kernels (fa_decode.hip:
// 128 query rows per work-group; fa_decode_few.hip: up to 32).
//
// LDS tile layout: the 32 x 72 grid of 16-byte chunks (row r, logical chunk k) is stored as
// 4 row-groups x 9 chunk-groups of 1 KB blocks; block (r/8, k/8) holds slot
// (r%8)*8 + ((k%8) ^ (r%8)).
#pragma once

#include "fa_common.h"
#include "fa_wave.h"

namespace fa {

constexpr int kThreads = 256;                    // 4 waves, one per SIMD
constexpr int kTileRows = 32;                    // tokens per pipeline tile
constexpr int kRowBytes = kDqk * 2;              // 1152 B: one bf16 cache row
constexpr int kChunkGroups = kRowBytes / 128;    // 9 groups of 8 chunks per row
constexpr int kBlockBytes = 1024;                // 8 rows x 8 chunks
constexpr int kRowGroupBytes = kChunkGroups * kBlockBytes;  // 9216
constexpr int kTileBytes = kTileRows * kRowBytes;  // 36864 B per LDS tile
constexpr int kFp8RowBytes = FA_MLA_FP8_ROW_BYTES;  // 656
constexpr int kQkSteps = kDqk / 32;              // 18 MFMA k-steps of QK
constexpr int kCopiesPerWave = kChunkGroups;     // 9 wave-wide copies per tile

enum Mode { kDense = 0, kSparseBf16 = 1, kSparseFp8 = 2 };

// fp8-e4m3 (OCP "fn") pair -> two floats, using the gfx950 converter.
template <bool kHi>
__device__ inline floatx2 fp8x2_to_f32(unsigned int word) {
  return __builtin_amdgcn_cvt_pk_f32_fp8(word, kHi);
}

__device__ inline unsigned int pack_bf16x2(float a, float b) {
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  floatx2 f;
  f[0] = a;
  f[1] = b;
  return __builtin_bit_cast(unsigned int, __builtin_convertvector(f, bf16x2));  // one v_cvt_pk_bf16_f32
}

// fp8 tiles reach LDS raw, one row-group (8 tile rows) per wave, inside the
// row-group's own 9 KB of the bf16 tile buffer:
//   [0, 4096)      codes: block G (1 KB) holds codes 128G..128G+127 of the 8
//                  rows, slot 8r + c = row r, 16-byte chunk c
//   [4096, 5120)   the four fp32 scales of row r at 4096 + 128r (the copy
//                  lanes of a row all load them; slot 8r is the one read)
//   [8192, 9216)   the rope dims, already in the bf16 layout (chunk-group 8)
// and the wave that loaded them turns the codes into bf16 blocks 0..7 in
// place.  Those overlap the raw bytes, so every read of the row-group comes
// before its first write; no other wave touches the row-group meanwhile.
constexpr int kFp8Copies = 6;          // wave-wide 16-byte copies per row-group
constexpr int kFp8ScaleOff = 4096;

// The conversion in two parts, so that a step can spread it over its MFMAs:
// fp8_load reads this lane's 64 codes and their scale (all the row-group's
// reads, before any write), fp8_store<I, H> converts and writes one 16-byte
// bf16 chunk of them (8 calls cover the lane).  Addresses are rebuilt from a
// fresh lane id: kept live across the loop they would be spilled, and each
// reload would stall the conversion.
struct Fp8Codes {
  uintx4 code[4];
  float scale;
  int base;  // byte offset of the lane's row r, chunk-group e in the row-group
  int r;     // row of the lane in the row-group (the chunk swizzle)
  int eh;    // e / 2: the lane's rotation of its four pieces
};
__device__ inline Fp8Codes fp8_load(const unsigned char* buf, int wave) {
  const int lane = fresh_lane();
  const int r = lane >> 3, e = lane & 7;  // row r of the group, codes 64e..64e+63
  const unsigned char* rg = buf + wave * kRowGroupBytes;
  const unsigned char* src = rg + 1024 * (e >> 1) + 16 * (8 * r + 4 * (e & 1));
  // Lane (r, e) takes its four 16-code pieces in the order m = (i + e/2) % 4: the
  // reads of one instruction then fall in 16 different bank groups per 16 lanes, and
  // its writes in 8 (2-way) instead of 2 (8-way).
  const int rot = e >> 1;
  Fp8Codes c;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    c.code[i] = *reinterpret_cast<const uintx4*>(src + 16 * ((i + rot) & 3));
  c.scale = *reinterpret_cast<const float*>(rg + kFp8ScaleOff + 128 * r + 4 * (e >> 1));
  c.base = (kChunkGroups * wave + e) * kBlockBytes + 128 * r;  // tile_off(8 wave + r, 8 e)
  c.r = r;
  c.eh = rot;
  return c;
}
// Byte offset of piece I, half H of the lane: tile_off(8 wave + r, 8 e + 2 m + H).
template <int I, int H>
__device__ inline int fp8_store_off(const Fp8Codes& c) {
  return c.base + 16 * ((2 * ((I + c.eh) & 3) + H) ^ c.r);
}
template <int I, int H>  // piece I of the four, half H: 8 codes -> one 16-byte bf16 chunk
__device__ inline void fp8_store(unsigned char* buf, const Fp8Codes& c) {
  const unsigned int w0 = c.code[I][2 * H], w1 = c.code[I][2 * H + 1];
  floatx2 a = fp8x2_to_f32<false>(w0), b = fp8x2_to_f32<true>(w0);
  floatx2 d = fp8x2_to_f32<false>(w1), f = fp8x2_to_f32<true>(w1);
  uintx4 o;
  o[0] = pack_bf16x2(a[0] * c.scale, a[1] * c.scale);
  o[1] = pack_bf16x2(b[0] * c.scale, b[1] * c.scale);
  o[2] = pack_bf16x2(d[0] * c.scale, d[1] * c.scale);
  o[3] = pack_bf16x2(f[0] * c.scale, f[1] * c.scale);
  *reinterpret_cast<uintx4*>(buf + fp8_store_off<I, H>(c)) = o;
}
__device__ inline void dequant_fp8_rowgroup(unsigned char* buf, int wave) {
  const Fp8Codes c = fp8_load(buf, wave);
  static_for<8>([&](auto pt) {
    constexpr int P = decltype(pt)::value;
    fp8_store<P / 2, P % 2>(buf, c);
  });
}

// Sparse index translation inside the decode (topk <= FA_MLA_FOLD_TOPK): at the start of a
// segment the work-group turns its index slots into physical cache rows, -1 where masked, in
// an LDS list (the arithmetic of mla_sparse_rows_kernel).  512 slots at a time, two per
// thread.  Against a launch of its own in front of the decode (3.8 us and its gap): sparse
// top-2,048 steps of 64 sequences, bf16, 67.4 -> 64.7 us, of 128, fp8, 106.4 -> 104.3 (the
// decode itself 1 us longer).  The limit is the LDS that the 32-row kernel's tiles leave
// (8 KB).  between() is called once, after the first page lookups have been issued and before
// they are waited for, so that the caller's own loads overlap them.
constexpr int kFoldTopk = FA_MLA_FOLD_TOPK;
template <typename F>
__device__ inline void fold_rows(const fa_mla_decode_args& a, int b, int s, int seqlen, int tok_lo,
                                 int nslots, int wave, int32_t* list, F&& between) {
  const int32_t* const row = a.indices + b * a.idx_stride_b + s * a.idx_stride_s;
  const int32_t* const bt = a.block_table + static_cast<long long>(b) * a.bt_stride_b;
  auto part = [&](int k0, auto&& mid) {
    const int tid = 64 * wave + fresh_lane();  // rebuilt: kept, it is spilled
    int32_t idx[2], page[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int k = k0 + kThreads * i + tid;
      idx[i] = k < nslots && tok_lo + k < a.topk ? row[tok_lo + k] : -1;
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const bool ok = idx[i] >= 0 && idx[i] < seqlen && (idx[i] >> 6) < a.max_blocks_per_seq;
      page[i] = ok ? bt[idx[i] >> 6] : -1;
    }
    mid();
    const int tid2 = 64 * wave + fresh_lane();
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int k = k0 + kThreads * i + tid2;
      if (k < nslots)
        list[k] = page[i] >= 0 && page[i] < a.num_kv_blocks ? page[i] * kPage + (idx[i] & 63) : -1;
    }
  };
  part(0, between);
  for (int k0 = 2 * kThreads; k0 < nslots; k0 += 2 * kThreads) part(k0, [] {});
}

// Decode of up to kFewRowsMax query rows per KV stream (fa_decode_few.hip).
constexpr int kFewRowsMax = 32;
int launch_decode_few(const fa_mla_decode_args* a, int mode, bool fold, hipStream_t stream);

}  // namespace fa
