// fp32 products on the 16-bit matrix instruction for the backward kernels (split3 / mfma_split in common.h:
// three bf16 parts per operand, six partial products per product, fp32 accumulation; this GPU multiplies
// bf16 sixteen times as fast as fp32).  Operand layouts are those of the 16-bit kernels: a tile of 32 rows
// is kept in LDS as three 16-bit planes [row][d], read by rows (16 bytes at d = 16 s + 8 g of row
// swap_bits_2_3(l32): with that row order the registers 0..7 / 8..15 of an accumulator column are the rows
// 8g .. 8g+7 of the tile's first / second half, and, split and packed, are the B operand of the next product
// as they stand) and by transposing reads (row 8g + j16/4, +4, +16; columns 32 dt + 16 half + 4 (j16 % 4)).
// Logits are kept in units of log2 (Q is multiplied by scale * log2(e) before its split, lse by log2(e)), the
// exponential is v_exp_f32.
#pragma once

#include "flash_bwd.h"

namespace axl {

template <int D>
struct TileF32x {
  static constexpr int TILE = 32;
  static constexpr int STRIDE = D * 2;      // bytes per row of a tile plane: unpadded, 16-byte chunks swizzled
                                            // (tile_swizzle: free of bank conflicts for both kinds of read)
  static constexpr int PLANE = TILE * STRIDE;
  static constexpr int TENSOR = 3 * PLANE;
  static constexpr int LD4(int nt) { return TILE * (D / 4) / nt; }   // float4 loads per thread of a workgroup of nt
};

__device__ __forceinline__ float bias_at(const AuxArgs& x, const char* row, int col) {
  if (x.bias_f32) return *(const float*)(row + (int64_t)col * 4);
  return (float)*(const __bf16*)(row + (int64_t)col * 2);
}

// This thread's part of a 32 x D tile, split, into the tile's three planes.
template <int D, int NT>
__device__ __forceinline__ void tile_deposit_split(char* planes, const float4 (&x)[TileF32x<D>::LD4(NT)], int tid) {
  using Tile = TileF32x<D>;
#pragma unroll
  for (int i = 0; i < Tile::LD4(NT); i++) {
    const int e = tid + i * NT, row = e / (D / 4), c4 = e % (D / 4);
    const Split3x2 lo2 = split3(x[i].x, x[i].y), hi2 = split3(x[i].z, x[i].w);
#pragma unroll
    for (int p = 0; p < 3; p++) {
      union { bf16x2 h[2]; uint2 u; } w;
      w.h[0] = lo2.part[p]; w.h[1] = hi2.part[p];
      *(uint2*)(planes + p * Tile::PLANE + row * Tile::STRIDE + (((c4 >> 1) ^ tile_swizzle<D>(row)) << 4) + (c4 & 1) * 8) = w.u;
    }
  }
}
// Per-lane read offsets into a tile plane.
template <int D>
struct TileReadOffsets {
  int row_base, row_xor;          // row read: row swap_bits_2_3(l32), chunk (2 ks + g) ^ swizzle
  int tr_base[2], tr_xor[2];      // transposing read: rows 8 g + j16 / 4 and + 4, byte column (16 half + 4 (j16 % 4)) * 2 + 64 dt
  int tr_col;
  __device__ __forceinline__ void init(int lane) {
    using Tile = TileF32x<D>;
    const int l32 = lane & 31, g = lane >> 5, j16 = lane & 15, half = (lane >> 4) & 1;
    const int row = swap_bits_2_3(l32);
    row_base = row * Tile::STRIDE;
    row_xor = (16 * g) ^ (tile_swizzle<D>(row) << 4);
    const int t_row = 8 * g + (j16 >> 2), col = (16 * half + 4 * (j16 & 3)) * 2;
    tr_col = col & ~15;
    tr_base[0] = t_row * Tile::STRIDE + (col & 15);
    tr_base[1] = tr_base[0] + 4 * Tile::STRIDE;
    tr_xor[0] = tile_swizzle<D>(t_row) << 4;
    tr_xor[1] = tile_swizzle<D>(t_row + 4) << 4;
  }
};
// Row-read operand (A) of k-step `ks` from a tile's planes.
template <int D>
__device__ __forceinline__ void read_rows(bf16x8 (&f)[3], const char* planes, const TileReadOffsets<D>& o, int ks) {
#pragma unroll
  for (int p = 0; p < 3; p++) f[p] = *(const bf16x8*)(planes + p * TileF32x<D>::PLANE + o.row_base + ((32 * ks) ^ o.row_xor));
}
// Transposed operand (A) for the tile's rows 16 kk + 8 g .. + 7 and columns 32 dt + l32.
template <int D>
__device__ __forceinline__ void read_transposed(bf16x8 (&f)[3], const char* planes, const TileReadOffsets<D>& o, int kk,
                                                int dt) {
  using Tile = TileF32x<D>;
#pragma unroll
  for (int p = 0; p < 3; p++) {
    union { bf16x8 v; shortx4 hlf[2]; } u;
    const char* at = planes + p * Tile::PLANE + 16 * kk * Tile::STRIDE;   // rows + 16: the same swizzle
    u.hlf[0] = lds_read_tr16(at + o.tr_base[0] + ((o.tr_col + 64 * dt) ^ o.tr_xor[0]));
    u.hlf[1] = lds_read_tr16(at + o.tr_base[1] + ((o.tr_col + 64 * dt) ^ o.tr_xor[1]));
    f[p] = u.v;
  }
}
// Registers 8 kk .. 8 kk + 7 of an accumulator column, split: the B operand of the next product.
__device__ __forceinline__ void split_column(bf16x8 (&f)[3], const floatx16& acc, int kk) {
  float x[8];
#pragma unroll
  for (int j = 0; j < 8; j++) x[j] = acc[8 * kk + j];
  Split3x8 sp;
  split3x8(x, sp);
#pragma unroll
  for (int p = 0; p < 3; p++) f[p] = sp.part[p].v;
}

}  // namespace axl
