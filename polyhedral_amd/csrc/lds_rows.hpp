// Rows of [N, D] tensors (2-byte types, D = 64 or 128) staged in LDS by LDS DMA for 32x32x16
// MFMAs: where a row's 16-byte units sit, and the two ways they are read.
//
// A DMA instruction writes 64 consecutive 16-byte units, so the rows are stored unpadded and
// one XOR swizzle of the 16-byte units serves both ways a tile is read (unit u of row r sits
// at u ^ swz(r)):
//  * D = 128 (256-byte rows): 4 (r % 4) + (r / 4) % 4.  The 16 rows of a 16-byte row read
//    land on 16 different units of the 256-byte bank window, and the 4 rows of a transposed
//    read on 4 different 64-byte groups;
//  * D = 64 (128-byte rows, two to a bank window): with x = (r / 2) % 8, 4 (x % 2) + x / 2.
//    The 8 row pairs of a row read land on 8 different units, and the two rows of one
//    parity that a transposed read touches (x differing in its lowest bit) on different
//    halves of the row.
#pragma once

#include "attn_kernel.hpp"

namespace pa {

template <int D>
struct Rows {
  static constexpr int ROW = 2 * D;             // bytes of a row
  static constexpr int UPR = D / 8;             // 16-byte units of a row
  static constexpr int RPI = 64 / UPR;          // rows a DMA instruction moves
  static constexpr int NI = 16 / RPI;           // instructions for 16 rows
  // (period 16)
  __device__ static int swz(int r) {
    return D == 128 ? 4 * (r & 3) + ((r >> 2) & 3) : 4 * ((r >> 1) & 1) + ((r >> 2) & 3);
  }
};

typedef const __attribute__((address_space(3))) f32x4 lds_f4;
typedef __attribute__((address_space(3))) f32x4 lds_f4w;
typedef __attribute__((address_space(3))) u32x4 lds_u4w;
typedef const __attribute__((address_space(4))) int32_t cint;

// Per-lane LDS geometry of the reads of 32 staged rows (offsets of stage, tile and chunk are
// immediates on top of these).  With 256-byte rows, units 8 apart and blocks 2 apart differ
// in address bit 7 alone, so the upper half of the addresses is the lower half with that
// bit flipped: one VALU operation at the read instead of eight registers held through
// the loop.
template <int D>
struct TileReads {
  static constexpr int NR = D == 128 ? 4 : D / 16, NT = 2;
  lds_cptr row_[NR];     // 16-byte row reads: row m, unit 2 kc + G
  lds_cptr tr_[NT][2];   // transposed reads of block db: rows 4 G + j16 / 4 (+8)
  // (volatile, or the flips would be hoisted out of the loop into registers again)
  __device__ __forceinline__ static lds_cptr flip(lds_cptr p) {
    uint32_t x;
    asm volatile("v_xor_b32 %0, 0x80, %1" : "=v"(x) : "v"((uint32_t)(uintptr_t)p));
    return (lds_cptr)(uintptr_t)x;
  }
  __device__ __forceinline__ lds_cptr row(int kc) const { return kc < NR ? row_[kc] : flip(row_[kc - NR]); }
  __device__ __forceinline__ lds_cptr tr(int db, int s) const { return db < NT ? tr_[db][s] : flip(tr_[db - NT][s]); }
};

template <int D>
__device__ __forceinline__ TileReads<D> tile_reads(lds_cptr lds, int lane) {
  TileReads<D> t;
  const int m = lane & 31, G = lane >> 5, j16 = lane & 15, h16 = (lane >> 4) & 1;
#pragma unroll
  for (int kc = 0; kc < TileReads<D>::NR; ++kc) {
    t.row_[kc] = lds + m * Rows<D>::ROW + 16 * ((2 * kc + G) ^ Rows<D>::swz(m));
    // (opaque, so each address stays whole in one register)
    asm volatile("" : "+v"(t.row_[kc]));
  }
#pragma unroll
  for (int db = 0; db < TileReads<D>::NT; ++db)
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int R = 4 * G + (j16 >> 2) + 8 * s;
      const int u = 4 * db + 2 * h16 + ((j16 & 3) >> 1);
      t.tr_[db][s] = lds + R * Rows<D>::ROW + 16 * (u ^ Rows<D>::swz(R)) + 8 * (j16 & 1);
      asm volatile("" : "+v"(t.tr_[db][s]));
    }
  return t;
}

// Maximum that gives NaN when either side is NaN: one instruction (v_maximum3_f32) on scores
// straight from an MFMA, where fmaxf, which gives the other side, needs one more per score to
// quiet signalling NaNs.  A row with a NaN score is NaN either way, by its probabilities.
__device__ __forceinline__ float nan_max(float x, float y) { return __builtin_elementwise_maximum(x, y); }
// Over lanes l and l ^ 32, as row_max.
__device__ __forceinline__ float row_nan_max(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(int, x), __builtin_bit_cast(int, x), false, false);
  return nan_max(__builtin_bit_cast(float, (int)r[0]), __builtin_bit_cast(float, (int)r[1]));
}

// A operand X^T of 16 rows of a staged tile at byte offset `off` (stage + tile + first row):
// the transposed product's fragment for block db of D.
template <typename T, int D>
__device__ __forceinline__ typename Mma<T>::frag tr_frag(const TileReads<D>& t, int db, int off) {
  const s16x4 x1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(t.tr(db, 0) + off));
  const s16x4 x2 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(t.tr(db, 1) + off));
  const uint4 vx = {__builtin_bit_cast(uint2, x1).x, __builtin_bit_cast(uint2, x1).y, __builtin_bit_cast(uint2, x2).x,
                    __builtin_bit_cast(uint2, x2).y};
  return __builtin_bit_cast(typename Mma<T>::frag, vx);
}

// Byte offsets of the lanes of the NI DMA instructions that move 16 rows `pitch` bytes apart:
// instruction i writes rows RPI i + l / UPR, lane l unit l % UPR, fetching the unit the
// swizzle stores there.
template <int D>
__device__ __forceinline__ void dma_offsets(uint32_t* dvoff, int64_t pitch, int lane) {
  const int r = lane / Rows<D>::UPR, u = lane % Rows<D>::UPR;
#pragma unroll
  for (int i = 0; i < Rows<D>::NI; ++i)
    dvoff[i] = (uint32_t)(r * pitch) + 16u * (uint32_t)(u ^ Rows<D>::swz(Rows<D>::RPI * i + r));
}

}  // namespace pa
