// bf16 LDS tiles of the MFMA kernels: layout, fragment addressing and direct global -> LDS staging.
#pragma once

#include "pnfx_common.h"

namespace pnfx {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Row of a 16-row MFMA block (block index blk, row r) inside its 64-row/key tile.
// Blocks 2t and 2t+1 interleave in groups of four so that lane group a (= r / 4) ends up
// holding rows 32t + 8a .. 32t + 8a + 7 across the pair.
__device__ __forceinline__ int perm_row(int blk, int r) {
  return 32 * (blk >> 1) + 8 * (r >> 2) + 4 * (blk & 1) + (r & 3);
}

__device__ __forceinline__ bf16x8 ld16(const bf16* p) { return *reinterpret_cast<const bf16x8*>(p); }

// LDS tiles are unpadded and XOR-swizzled on the 16-byte chunk index of each row, with
// swizzles linear over GF(2) in the row bits.  They were chosen by measuring the LDS
// bank-conflict counter for every access pattern of the kernels (a b128 read is conflict
// free when each 16-lane group reads 16 consecutive tile rows at chunks g ^ swz(row)):
//  * tiles are row-major [rows][DK] and store logical row R at slot slot_of(R), which places
//    the 16 rows of an MFMA fragment (rows perm_row(blk, 0..15)) in consecutive slots
//    16 blk .. 16 blk + 15;
//  * the transposed operands (V^T, K^T, Q^T, dO^T) are read from the same row-major tiles
//    with ds_read_tr16_b64, which transposes 16-bit elements across each 16-lane group.
// Linearity lets a fragment's swizzle split into a per-lane part and a compile-time part.
__device__ __forceinline__ constexpr int parity6(int x) { return __builtin_popcount(x & 63) & 1; }
__device__ __forceinline__ constexpr int swz_cols(int d) {
  return parity6(d & 18) | (parity6(d & 39) << 1) | (parity6(d & 12) << 2);
}
// Row-major tiles: 64-column rows use swz_cols; 128-column rows (16 chunks) a 4-bit swizzle.
template <int DK>
__device__ __forceinline__ constexpr int swz_rt(int slot) {
  return DK == 128 ? (parity6(slot & 46) | (parity6(slot & 10) << 1) | (parity6(slot & 28) << 2) |
                      (parity6(slot & 13) << 3))
                   : swz_cols(slot) & (DK / 8 - 1);
}
// Slot of logical row R: rows perm_row(blk, r) -> 16 blk + r.
__device__ __forceinline__ constexpr int slot_of(int R) {
  return 16 * (2 * (R >> 5) + ((R >> 2) & 1)) + 4 * ((R >> 3) & 3) + (R & 3);
}

// Element offset of 16-byte chunk `chunk` of logical row `row` in a row-major tile of DK
// columns.
template <int DK>
__device__ __forceinline__ int rt_off(int row, int chunk) {
  const int slot = slot_of(row);
  return slot * DK + ((chunk ^ swz_rt<DK>(slot)) << 3);
}
// Fragment addressing with the lane part hoisted.  A row-major fragment reads logical row
// perm_row(blk, r16), i.e. slot 16 blk + r16 (disjoint bits), at chunk g + 4*ks:
//   offset = 16 blk DK + r16 DK + (((g ^ swz(r16)) ^ (4 ks ^ swz(16 blk))) << 3).
struct FragLane {
  int rbase;  // lane part of the element offset
  int x;      // lane part of the chunk index (XOR-combined with the constant part)
};
template <int DK>
__device__ __forceinline__ FragLane rt_lane(int r16, int g) {
  return FragLane{r16 * DK, g ^ swz_rt<DK>(r16)};
}
template <int DK>
__device__ __forceinline__ int rt_frag(const FragLane& fl, int blk, int ks) {
  const int cc = (4 * ks) ^ swz_rt<DK>(16 * blk);
  return 16 * blk * DK + fl.rbase + ((fl.x ^ cc) << 3);
}

// Transposed fragment X^T[16 db + r16][rows 32 hf + 8 g + t], t = 0..7 (the A operand of the
// second GEMM: V^T, K^T, Q^T or dO^T) from a row-major tile, as two ds_read_tr16_b64.  In
// each 16-lane group, lane 4 e + q addresses row 32 hf + 8 g + 4 u + e at columns
// 16 db + 4 q .. + 3 (u = 0, 1 for the two reads), and lane r16 = 4 q' + r' receives
// column 16 db + r16 of the four rows addressed by lanes 4 e + q'.  Row 32 hf + 8 g + 4 u + e
// sits in slot 16 (2 hf + u) + 4 g + e.
template <int DK>
__device__ __forceinline__ FragLane tr_lane(int lane) {
  const int g = lane >> 4, e = (lane >> 2) & 3, q = lane & 3;
  const int sl = 4 * g + e;
  return FragLane{sl * DK + 4 * (q & 1), (q >> 1) ^ swz_rt<DK>(sl)};
}
__device__ __forceinline__ bf16x4 ld_tr(const bf16* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4bf16((__attribute__((address_space(3))) bf16x4*)(p));
}
template <int DK>
__device__ __forceinline__ bf16x8 tr_frag(const bf16* tile, const FragLane& fl, int hf, int db) {
  bf16x4 h[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int sc = 16 * (2 * hf + u);
    const int cc = (2 * db) ^ swz_rt<DK>(sc);
    h[u] = ld_tr(tile + sc * DK + fl.rbase + ((fl.x ^ cc) << 3));
  }
  return __builtin_shufflevector(h[0], h[1], 0, 1, 2, 3, 4, 5, 6, 7);
}

// Columns of an LDS tile row for head size D: at least the 32 of one MFMA k-step, and a power of two
// for the swizzle (at D = 96 the last quarter of each row is neither filled nor read).
constexpr int tile_cols(int D) { return D < 32 ? 32 : D == 96 ? 128 : D; }
// k-steps of 32 columns of a product over the head dimension.
constexpr int k_steps(int D) { return D < 32 ? 1 : D / 32; }

// Direct global -> LDS staging of a 64-row tile (rows row0 .. row0 + 63 of an [N, D] bf16
// slice with row stride sn) into the swizzled row-major layout, with global_load_lds_dwordx4:
// no register staging and no LDS store instructions.  Each such load writes 16 bytes per
// lane to LDS at (wave-uniform base) + 16 * lane, so a wave fills 64 consecutive chunks; each
// lane loads the global chunk that belongs at its position (the layout is a permutation of
// the tile's chunks).  The per-lane row and column are fixed at construction.  Rows >= N
// re-load row N - 1 and the padding chunks of D < DK re-load a real chunk of the row: both
// only ever meet masked scores or zero MFMA operands, so any finite value serves.  The
// caller waits for the loads (vmcnt) before the barrier that publishes the tile.
// Direct global -> LDS copy of 16 bytes per lane (lane l lands at dst + 8 l).  (The builtin
// sits in a plain function: called directly from a class template's member, it kept the
// host pass from emitting some of the kernels' launch stubs.)
__device__ __forceinline__ void lds_dma16(const bf16* src, bf16* dst) {
  __builtin_amdgcn_global_load_lds(src, dst, 16, 0, 0);
}
__device__ __forceinline__ int row_of_slot(int s) {  // inverse of slot_of
  return (s & 32) | ((s & 12) << 1) | ((s >> 2) & 4) | (s & 3);
}
// `d` <= D: the columns that the rows hold; chunks past them re-load the row's last one.  ZERO: they are
// left alone instead, and clear_tail makes them 0 once.
template <int D, int DK, bool ZERO = false>
struct TileDma {
  static constexpr int CPR = DK / 8;      // 16-byte chunks per tile row
  static constexpr int NI = 64 * CPR / 256;  // loads per thread
  static constexpr bool PART = D > 32 && D < DK;  // chunks past D are left alone
  static constexpr bool SKIP = PART || ZERO;      // some chunks (col D here) are
  int row[NI], col[NI];
  unsigned off[NI];  // byte offset of the lane's chunks from the tile's first row
  __device__ __forceinline__ TileDma(int w, int lane, int64_t sn, int d = D) {
#pragma unroll
    for (int j = 0; j < NI; ++j) {
      const int L = (4 * j + w) * 64 + lane;  // chunk index in the tile
      const int slot = L / CPR, pos = L % CPR;
      const int ch = pos ^ swz_rt<DK>(slot);
      row[j] = row_of_slot(slot);
      if (ZERO) col[j] = 8 * ch < d ? 8 * ch : D;
      else col[j] = d == D ? 8 * (PART ? ch : ch % (D / 8)) : min(8 * ch, PART && ch >= D / 8 ? D : d - 8);
      off[j] = (unsigned)(2 * (row[j] * sn + col[j]));
    }
  }
  // Before the first load into `tile`; published with it.
  __device__ __forceinline__ void clear_tail(bf16* tile, int w, int lane) const {
#pragma unroll
    for (int j = 0; j < NI; ++j)
      if (col[j] >= D) *reinterpret_cast<bf16x8*>(tile + (4 * j + w) * 512 + 8 * lane) = zero_bf16x8();
  }
  // A whole tile (row0 + 64 <= N) is a wave-uniform base plus 32-bit lane offsets, which the
  // load takes as scalar base + vector offset: no per-load address arithmetic.
  __device__ __forceinline__ void load(const bf16* src, int64_t sn, int row0, int N, bf16* tile,
                                       int w, int d_last = D - 8) const {
    if (row0 + 64 <= N) {
      const char* base = reinterpret_cast<const char*>(src + (int64_t)row0 * sn);
#pragma unroll
      for (int j = 0; j < NI; ++j)
        if (!SKIP || col[j] < D)
          lds_dma16(reinterpret_cast<const bf16*>(base + off[j]), tile + (4 * j + w) * 512);
    } else {
      load_clamped(src, sn, row0, N, tile, w, d_last);
    }
  }
  // Any tile, from the row and column alone (fewer registers held across the loop, more
  // address arithmetic per load).
  __device__ __forceinline__ void load_clamped(const bf16* src, int64_t sn, int row0, int N,
                                               bf16* tile, int w, int d_last = D - 8) const {
#pragma unroll
    for (int j = 0; j < NI; ++j) {
      const int r = min(row0 + row[j], N - 1);
      if (!SKIP || col[j] < D)
        lds_dma16(src + (int64_t)r * sn + min(col[j], d_last), tile + (4 * j + w) * 512);
    }
  }
};
// Wait for this wave's outstanding global loads (including direct-to-LDS ones).
__device__ __forceinline__ void wait_vmem() { __builtin_amdgcn_s_waitcnt(0x0F70); }

}  // namespace
}  // namespace pnfx
