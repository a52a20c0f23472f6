// Flash pn_fir_tau attention for fp32 tensors (the reference's TF32-off parity path) on the
// MFMA units: scores on v_mfma_f64_16x16x4_f64, the other products on v_mfma_f32_16x16x4_f32.
//
// Math (src/triton_pnfirtau.py:313-621): s = fma(q.k, scale, -tau), u = relu(s), P = u^10,
// Z = sum P + 1e-12, M = max u, Nmax = #(u == M); O = (sum P v) gate / Z.  Nothing is
// rounded below fp32.  The score's dot product q.k is formed in fp64 (the fp32 inputs'
// products are exact there) and rounded to fp32 once: u^9 in the gradient multiplies the
// score's relative error by nine, and an fp32 sum of the d products, where they cancel, put
// single gradient elements past 1e-5 of the tensor's scale on random inputs.
//
// MFMA mapping.  Lane l = 16 g + r of a wave holds A[row r][k-slot g] and B[k-slot g][col r].  A
// dot product over the head dimension runs D/4 chained MFMAs; in step 4 j + e k-slot g carries
// head column 16 j + 4 g + e, in every kernel, so that one 16-byte LDS read feeds four steps.  The
// fp32 MFMA returns D[4 g + i][r] in register i, the fp64 MFMA D[g + 4 i][r].  The forward and the
// dQ kernel form S^T = K Q^T (K as A, Q as B); the dK/dV kernel forms S = Q K^T.  The fp64 MFMA's A
// rows are taken in the 4x4-transposed order perm4(r), so that its register i, like the fp32
// MFMA's, belongs to row 4 g + i of the 16-row block.  On gfx950 the fp64 MFMA is bitwise
// transpose-symmetric (swapping the A and B values gives exactly the transposed result), so every
// kernel recomputes the forward's scores bit for bit and the backward's peak-tie test u == M sees
// the forward's ties.  The score registers feed the second product directly: register i is
// k-slot g of MFMA i, i.e. rows i, 4 + i, 8 + i, 12 + i of the block.  Its A operand, a column
// slice of the same rows, takes head columns 4 r .. 4 r + 3 of a row for the four 16-column output
// blocks at once (one 16-byte read); the lane's results of a row are then 16 contiguous bytes.
//
// Work split.  A workgroup owns 32 query rows (forward, dQ) or 32 keys (dK/dV) as two 16-row
// groups and streams the other operand through LDS in tiles of 64 rows; the four 16-row blocks of
// a tile go to different waves (see Cfg), whose partial sums are added in a fixed order at the end
// (or, for dQ's row constants, between its sweeps).  Tiles go straight from global memory into one
// of two LDS buffers while the other is computed from.
//
// Bound: the matrix pipe, by the fp64 scores (a v_mfma_f64_16x16x4_f64 occupies it for 64 cycles, a
// v_mfma_f32_16x16x4_f32 for 32): per 16 x 16 block of scores at D = 64, 1536 cycles in the
// forward, 3584 in dQ (two sweeps), 2560 in dK/dV, about 0.21 ms for a step at B=1 H=8 N=2048
// d=64.  Measured there: forward 125 -> 75 us, dQ 258 -> 189, dK/dV 183 -> 139, the step 570 -> 385,
// against kernels that staged tiles through registers by single floats under per-element range
// tests and read the second products' operands from LDS one float at a time.  The matrix pipe is
// busy for about half of the time: at this size the longest causal block alone takes most of the
// kernel, at one or two waves per SIMD (B=8 H=8 N=1024: 1198 -> 697 us, 60 %).  Removing the tile
// loads and barriers from the forward's loop (timing only) gains 5 %.
#include "flash.h"

namespace pnfx {
namespace {

constexpr int TB = 64;   // rows per LDS tile
constexpr int RB = 32;   // rows (forward, dQ) or keys (dK/dV) per workgroup: two 16-row groups
// A wave takes QB of the row groups and one 16-row block of every tile.  QB = 1 (eight waves) is the
// faster form in the forward and at D <= 32; in the gradients at D = 64 one wave for both groups
// (four waves) is: a tile element is read from LDS and widened to fp64 once for both (the widening
// takes the matrix unit's fp64 datapath for 16 cycles beside the MFMA's 64) and the two MFMA
// chains are independent; forward + backward at B=8 H=8 N=1024 d=64 0.70 against 0.74 ms.  MINW:
// waves per SIMD that the registers must allow, so that two workgroups share a CU (D = 128: one,
// whose tiles fill the LDS; there the wave's own operand of the scores stays in fp32 and is
// widened at each use, which the registers force).
template <int D, bool BWD>
struct Cfg {
  static constexpr int QB = BWD && D == 64 ? 2 : 1, NW = 8 / QB, NT = 64 * NW;
  static constexpr int MINW = D == 128 ? 2 : NW / 2;
};
template <int D>
using FwdCfg = Cfg<D, false>;
template <int D>
using BwdCfg = Cfg<D, true>;
template <bool WIDE>  // the wave's operand of the scores: fp64 registers or fp32
struct Score { typedef double type; };
template <>
struct Score<false> { typedef float type; };
template <int D>
using score_t = typename Score<(D <= 64)>::type;
// Key tiles of one sequence with a tile mask
constexpr int kMaxTiles = kF32MaskMaxN / TB;

__device__ __forceinline__ float pow10f_(float u) {
  const float u2 = u * u;
  const float u4 = u2 * u2;
  return u4 * u4 * u2;
}

typedef double f64x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ int perm4(int r) { return 4 * (r & 3) + (r >> 2); }

__device__ __forceinline__ void wait_vmem() { __builtin_amdgcn_s_waitcnt(0x0F70); }

// Direct global -> LDS copies of 16 / 4 bytes per lane (lane l lands at dst + 4 l / dst + l).
__device__ __forceinline__ void lds_dma16(const float* src, float* dst) {
  __builtin_amdgcn_global_load_lds(src, dst, 16, 0, 0);
}
__device__ __forceinline__ void lds_dma4(const float* src, float* dst) {
  __builtin_amdgcn_global_load_lds(src, dst, 4, 0, 0);
}

// The 32-row (or 32-key) block and the (b, h) slice of this workgroup in a 1-D grid of nb * BH
// workgroups.  Every slice's blocks go in the same order, one block of each slice at a time, the
// longest first, so that none starts last and runs alone (heavy_last_index: the last block is the
// longest, as in the query-parallel kernels under a causal mask; in the key-parallel kernel block 0
// is).  A grid that is resident all at once, two workgroups per CU (`fold`), has no order in time:
// there the second half goes shortest first, which puts it beside the first half's longest
// (forward at B=1 H=8 N=2048 d=64: 95 -> 78 us).
constexpr int kResident = 512;
__device__ __forceinline__ void block_of(int nb, int BH, bool fold, bool heavy_last_index, int& blk,
                                         int& bh) {
  int j = blockIdx.x / BH;
  bh = blockIdx.x % BH;
  const int half = (nb + 1) / 2;
  if (fold && nb * BH <= kResident && j >= half) j = nb - 1 - (j - half);
  blk = heavy_last_index ? nb - 1 - j : j;
}

// LDS tiles hold 64 unpadded rows of D floats, the 16-byte chunks of row R at positions
// chunk ^ swz(R): 16 lanes reading one chunk of 16 rows (the dot products) or 16 chunks of one row
// (the second products) then touch every bank once.
template <int D>
__device__ __forceinline__ constexpr int swz(int row) {
  return D >= 64 ? row & 15 : D == 32 ? (row >> 1) & 7 : (row >> 2) & 3;
}
template <int D>
__device__ __forceinline__ f32x4 ld_chunk(const float* tile, int row, int chunk) {
  return *reinterpret_cast<const f32x4*>(tile + row * D + ((chunk ^ swz<D>(row)) << 2));
}

// Staging of a 64-row tile (rows row0 .. row0 + 63 of an [N, D] slice with row stride sn), without
// registers; rows past N repeat row N - 1.  The layout is a permutation of the tile's chunks, so
// each lane loads what belongs at its place of a contiguous 1 KB run: its chunk is the same in
// every run of a tile (the runs' rows differ by multiples of 16), so that a whole tile takes scalar
// bases and one 32-bit lane offset.  VEC: rows of whole 16-byte chunks, 64 rows within 4 GB;
// others go by single floats.
template <int D, bool VEC, int NW>
struct TileDma {
  static constexpr int NT = 64 * NW, CPR = D / 4, RPI = NT / CPR;  // chunks a row, rows a run
  static constexpr int NI = VEC ? (TB + RPI - 1) / RPI : TB * D / NT;
  int row, col;
  unsigned off;
  __device__ __forceinline__ TileDma(int w, int lane, int64_t sn) {
    const int L = w * 64 + lane;
    row = L / CPR;
    col = 4 * ((L % CPR) ^ swz<D>(row));
    off = (unsigned)(4 * (row * sn + col));
  }
  __device__ __forceinline__ void load(const float* src, int64_t sn, int row0, int N, float* tile,
                                       int w, int lane) const {
    if constexpr (VEC) {
      if (TB < RPI && w * 64 >= TB * CPR) return;  // D = 16: the first four waves cover the tile
      if (row0 + TB <= N) {
#pragma unroll
        for (int j = 0; j < NI; ++j) {
          const char* base = reinterpret_cast<const char*>(src + (int64_t)(row0 + RPI * j) * sn);
          lds_dma16(reinterpret_cast<const float*>(base + off), tile + 4 * (NW * j + w) * 64);
        }
      } else {
#pragma unroll
        for (int j = 0; j < NI; ++j)
          lds_dma16(src + (int64_t)min(row0 + RPI * j + row, N - 1) * sn + col,
                    tile + 4 * (NW * j + w) * 64);
      }
    } else {
      // one float per lane and run; a run's rows lie RPF below the run before
      constexpr int RPF = NT / D;
      const int L = w * 64 + lane, r0 = L / D, c = L % D;
      const float* rows = src + (int64_t)(row0 + r0) * sn + (c & 3);
      if (row0 + TB <= N) {
#pragma unroll 4
        for (int j = 0; j < NI; ++j) {
          const int r = r0 + RPF * j;
          lds_dma4(rows + 4 * ((c >> 2) ^ swz<D>(r)), tile + (NW * j + w) * 64);
          rows += RPF * sn;
        }
      } else {
#pragma unroll 1
        for (int j = 0; j < NI; ++j) {
          const int r = r0 + RPF * j;
          lds_dma4(src + (int64_t)min(row0 + r, N - 1) * sn + 4 * ((c >> 2) ^ swz<D>(r)) + (c & 3),
                   tile + (NW * j + w) * 64);
        }
      }
    }
  }
};

// The lane's head columns (16 j + 4 g + e) of one row of global memory, zero if the row is absent.
template <int D, bool VEC, typename T>
__device__ __forceinline__ void load_row(T (&dst)[D / 4], const float* row, bool ok, int g) {
#pragma unroll
  for (int j = 0; j < D / 16; ++j) {
    f32x4 x = f32x4{0.f, 0.f, 0.f, 0.f};
    const float* p = row + 16 * j + 4 * g;
    if (ok) {
      if (VEC) x = *reinterpret_cast<const f32x4*>(p);
      else x = f32x4{p[0], p[1], p[2], p[3]};
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) dst[4 * j + e] = (T)x[e];
  }
}

// The wave's operand of the scores: fp64 as it is; fp32 widened where it is used (the empty asm
// hides that it does not change over the key loop, so that the compiler does not keep the doubles).
__device__ __forceinline__ double widen(double x) { return x; }
__device__ __forceinline__ double widen(float x) {
  asm volatile("" : "+v"(x));
  return (double)x;
}

// Dot products of one 16-row block (rows row0 ..) of a tile with the lane's operands b[qb]:
// register i is row 4 g + i.  fp64 sums rounded once (the scores), or fp32.
template <int D, int QB, typename T>
__device__ __forceinline__ void dot64(const float* tile, int row0, int r, int g,
                                      const T (&b)[QB][D / 4], f32x4 (&out)[QB]) {
  const int row = row0 + perm4(r);
  f32x4 a[D / 16];
#pragma unroll
  for (int j = 0; j < D / 16; ++j) a[j] = ld_chunk<D>(tile, row, 4 * j + g);
  f64x4 acc[QB];
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) acc[qb] = f64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int j = 0; j < D / 16; ++j)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const double ae = (double)a[j][e];
#pragma unroll
      for (int qb = 0; qb < QB; ++qb)
        acc[qb] = __builtin_amdgcn_mfma_f64_16x16x4f64(ae, widen(b[qb][4 * j + e]), acc[qb], 0, 0, 0);
    }
#pragma unroll
  for (int qb = 0; qb < QB; ++qb)
    out[qb] = f32x4{(float)acc[qb][0], (float)acc[qb][1], (float)acc[qb][2], (float)acc[qb][3]};
}
template <int D, int QB>
__device__ __forceinline__ void dot32(const float* tile, int row0, int r, int g,
                                      const float (&b)[QB][D / 4], f32x4 (&out)[QB]) {
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) out[qb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < D / 16; ++j) {
    const f32x4 a = ld_chunk<D>(tile, row0 + r, 4 * j + g);
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) out[qb] = mfma4(a[e], b[qb][4 * j + e], out[qb]);
  }
}

// acc[db] += X^T B for one row of X per lane group: the lane's A operands of all D/16 output blocks
// are VW consecutive columns (two such runs at D = 128), read at once.  Output block db row rho is
// head column out_col(db, rho).
template <int D>
struct Cols {
  static constexpr int DB = D / 16, VW = DB < 4 ? DB : 4;
  __device__ static __forceinline__ int out_col(int db, int rho) {
    return 16 * VW * (db / VW) + VW * rho + db % VW;
  }
};
template <int D>
__device__ __forceinline__ void ld_cols(const float* tile, int row, int r, bool tail, bool ok,
                                        float (&x)[D / 16]) {
  constexpr int DB = Cols<D>::DB, VW = Cols<D>::VW;
  typedef float vec __attribute__((ext_vector_type(VW)));
#pragma unroll
  for (int h = 0; h < DB / VW; ++h) {
    const int c = VW * r + 16 * VW * h;  // first column
    const float* p = tile + row * D + (((c >> 2) ^ swz<D>(row)) << 2) + (c & 3);
    if constexpr (VW == 1) {
      x[h] = p[0];
    } else {
      const vec v = *reinterpret_cast<const vec*>(p);
#pragma unroll
      for (int e = 0; e < VW; ++e) x[VW * h + e] = v[e];
    }
  }
  if (tail) {  // the rows past N repeat the last one, which may not be finite: 0 there
#pragma unroll
    for (int e = 0; e < DB; ++e) x[e] = ok ? x[e] : 0.f;
  }
}
template <int D, int QB>
__device__ __forceinline__ void add_outer(const float (&x)[D / 16], const float (&b)[QB],
                                          f32x4 (&acc)[QB][D / 16]) {
#pragma unroll
  for (int db = 0; db < D / 16; ++db)
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) acc[qb][db] = mfma4(x[db], b[qb], acc[qb][db]);
}

// The lane's results of one output row: registers 4 g + i of every output block.
template <int D, bool VEC>
__device__ __forceinline__ void store_row(float* row, const f32x4 (&acc)[D / 16], int g) {
  constexpr int DB = Cols<D>::DB, VW = Cols<D>::VW;
#pragma unroll
  for (int h = 0; h < DB / VW; ++h)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float* p = row + Cols<D>::out_col(VW * h, 4 * g + i);
      if (VW == 4 && VEC) {
        *reinterpret_cast<f32x4*>(p) = f32x4{acc[VW * h][i], acc[VW * h + 1 % VW][i],
                                             acc[VW * h + 2 % VW][i], acc[VW * h + 3 % VW][i]};
      } else {
#pragma unroll
        for (int e = 0; e < VW; ++e) p[e] = acc[VW * h + e][i];
      }
    }
}

// Lane-wise sums handed from one wave to another through LDS.
template <int QB, int DB>
__device__ __forceinline__ void put_acc(float* xs, const f32x4 (&acc)[QB][DB]) {
#pragma unroll
  for (int qb = 0; qb < QB; ++qb)
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int i = 0; i < 4; ++i) xs[(4 * (DB * qb + db) + i) * 64] = acc[qb][db][i];
}
template <int QB, int DB>
__device__ __forceinline__ void add_acc(const float* xs, f32x4 (&acc)[QB][DB]) {
#pragma unroll
  for (int qb = 0; qb < QB; ++qb)
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[qb][db][i] += xs[(4 * (DB * qb + db) + i) * 64];
}
template <int QB, int DB>
__device__ __forceinline__ void zero_acc(f32x4 (&acc)[QB][DB]) {
#pragma unroll
  for (int qb = 0; qb < QB; ++qb)
#pragma unroll
    for (int db = 0; db < DB; ++db) acc[qb][db] = f32x4{0.f, 0.f, 0.f, 0.f};
}

// s -> u = relu(s scale - tau) of the lane's four scores (rows first + i against position pos, in
// range below n): masked where `masked` says that the block straddles the diagonal or the end.
// KEYS: the rows are keys and pos the query (forward, dQ), else queries and pos the key.
template <bool CAUSAL, bool KEYS>
__device__ __forceinline__ void rectify(f32x4& s, float scale, float ntau, bool masked, int first,
                                        int pos, int N) {
#pragma unroll
  for (int i = 0; i < 4; ++i) s[i] = fmaxf(__builtin_fmaf(s[i], scale, ntau), 0.f);
  if (masked) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = first + i;
      if (row >= N || pos >= N || (CAUSAL && (KEYS ? row > pos : pos > row))) s[i] = 0.f;
    }
  }
}

// GEN: rows of any alignment, and the tie counts if asked for.
template <int D, bool CAUSAL, bool GEN>
__global__ __launch_bounds__(FwdCfg<D>::NT, GEN ? 2 : FwdCfg<D>::MINW) void f32_fwd_kernel(FwdParams p) {
  constexpr bool VEC = !GEN, COUNT = GEN;
  constexpr int QB = FwdCfg<D>::QB, NW = FwdCfg<D>::NW, NT = FwdCfg<D>::NT;
  constexpr int KS = D / 4, DB = D / 16;
  __shared__ __attribute__((aligned(16))) float Ks0[TB * D];
  __shared__ __attribute__((aligned(16))) float Vs0[TB * D];
  __shared__ __attribute__((aligned(16))) float Ks1[TB * D];
  __shared__ __attribute__((aligned(16))) float Vs1[TB * D];
  __shared__ float st_s[NW][QB][3][16];  // peak, tie count and mass of each wave's rows
  // each wave's activity bit per key tile (one 32-bit word per 32 tiles), for the tile mask
  __shared__ uint32_t act_s[NW][(kMaxTiles + 31) / 32];
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, g = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int N = p.N;
  int blk, bh;
  block_of((N + RB - 1) / RB, p.B * p.H, CAUSAL && D <= 64, true, blk, bh);
  const int b = bh / p.H, h = bh % p.H;
  // the wave's first 16-row group (it takes QB) and its 16-key block of every key tile
  const int rg = w >> 2, kp = w & 3;
  const int m0 = blk * RB, qw = m0 + 16 * rg, qlast = qw + 16 * QB - 1;
  if (lane < (kMaxTiles + 31) / 32) act_s[w][lane] = 0u;
  const float* Q = static_cast<const float*>(p.q) + b * p.qsb + h * p.qsh;
  const float* K = static_cast<const float*>(p.k) + b * p.ksb + h * p.ksh;
  const float* V = static_cast<const float*>(p.v) + b * p.vsb + h * p.vsh;
  const float ntau = -p.tau[0], scale = p.scale;
  const int kv_end = CAUSAL ? min(m0 + RB, N) : N;
  const int ntiles = (kv_end + TB - 1) / TB;
  const TileDma<D, VEC, NW> kdma(w, lane, p.ksn), vdma(w, lane, p.vsn);
  const auto load_tile = [&](int n, float* kt, float* vt) {
    kdma.load(K, p.ksn, n, N, kt, w, lane);
    vdma.load(V, p.vsn, n, N, vt, w, lane);
  };
  load_tile(0, Ks0, Vs0);
  score_t<D> qf[QB][KS];
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    const int row = qw + 16 * qb + r;
    load_row<D, VEC>(qf[qb], Q + (int64_t)row * p.qsn, row < N, g);
  }
  f32x4 acc[QB][DB];
  zero_acc(acc);
  float m[QB] = {}, mass[QB] = {};
  int cnt[QB] = {};
  // tile t, computed from kc/vc while tile t + 1 streams into kn/vn
  const auto step = [&](int t, const float* kc, const float* vc, float* kn, float* vn) {
    const int n0 = t * TB, kb = n0 + 16 * kp;  // the wave's keys
    wait_vmem();
    __syncthreads();
    if (t + 1 < ntiles) load_tile(n0 + TB, kn, vn);
    if (qw >= N || kb >= N || (CAUSAL && kb > qlast)) return;
    const bool tail = kb + 15 >= N;
    float x[4][DB];  // read ahead of the scores, whose chain hides their latency
#pragma unroll
    for (int i = 0; i < 4; ++i)
      ld_cols<D>(vc, 16 * kp + 4 * g + i, r, tail, kb + 4 * g + i < N, x[i]);
    f32x4 u[QB];
    dot64<D, QB>(kc, 16 * kp, r, g, qf, u);
    bool pos = false;
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
      rectify<CAUSAL, true>(u[qb], scale, ntau, tail || qlast >= N || (CAUSAL && kb + 15 > qw),
                            kb + 4 * g, qw + 16 * qb + r, N);
      const float mx = fmaxf(fmaxf(u[qb][0], u[qb][1]), fmaxf(u[qb][2], u[qb][3]));
      pos |= mx > 0.f;
      const float mm = fmaxf(m[qb], mx);
      if (COUNT) {
        cnt[qb] = m[qb] == mm ? cnt[qb] : 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) cnt[qb] += u[qb][i] == mm ? 1 : 0;
      }
      m[qb] = mm;
    }
    if (!__any(pos)) return;  // a silent block: nothing to add
    if (p.mask && lane == 0) act_s[w][t >> 5] |= 1u << (t & 31);  // nk64 <= kMaxTiles
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      // O^T[d][query] += V^T[d][key] P[key][query]: register i is k-slot g of MFMA i (key 4g + i)
      float pw[QB];
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) {
        pw[qb] = pow10f_(u[qb][i]);
        mass[qb] += pw[qb];
      }
      add_outer<D>(x[i], pw, acc);
    }
  };
  for (int t = 0; t < ntiles; t += 2) {
    step(t, Ks0, Vs0, Ks1, Vs1);
    if (t + 1 < ntiles) step(t + 1, Ks1, Vs1, Ks0, Vs0);
  }
  // the four lane groups of a query row hold disjoint keys: combine their statistics
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    float M = fmaxf(m[qb], __shfl_xor(m[qb], 16, 64));
    M = fmaxf(M, __shfl_xor(M, 32, 64));
    int c = (m[qb] == M) ? cnt[qb] : 0;
    c += __shfl_xor(c, 16, 64);
    c += __shfl_xor(c, 32, 64);
    float ms = mass[qb] + __shfl_xor(mass[qb], 16, 64);
    ms += __shfl_xor(ms, 32, 64);
    if (g == 0) {
      st_s[w][qb][0][r] = M;
      st_s[w][qb][1][r] = __int_as_float(c);
      st_s[w][qb][2][r] = ms;
    }
  }
  __syncthreads();  // every wave's tiles, statistics and activity bits are done
  if (p.mask) {  // the workgroup's 32-row group: all waves
    for (int t = tid; t < p.nk64; t += NT) {
      uint32_t a = 0u;
      if (t < ntiles)
#pragma unroll
        for (int v = 0; v < NW; ++v) a |= act_s[v][t >> 5];
      p.mask[((int64_t)bh * p.nq32 + blk) * p.nk64 + t] = (a >> (t & 31)) & 1u;
    }
  }
  // Waves kp = 1, 2, 3 of the row groups hand their sums to wave kp = 0 through the tiles' LDS.
  static_assert(RB / 16 * 4 * DB * 64 <= TB * D, "the row groups' sums fit one tile");
  const auto ex = [&](int k) { return k == 0 ? Ks0 : k == 1 ? Vs0 : Ks1; };
  const int xo = rg * 4 * DB * 64 + lane;
  if (kp > 0) put_acc(ex(kp - 1) + xo, acc);
  __syncthreads();
  if (kp > 0) return;
#pragma unroll
  for (int k = 0; k < 3; ++k) add_acc(ex(k) + xo, acc);
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    const int row = qw + 16 * qb + r;
    if (row >= N) continue;
    float M = 0.f, ms = 0.f;
    int c = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) M = fmaxf(M, st_s[w + k][qb][0][r]);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      c += st_s[w + k][qb][0][r] == M ? __float_as_int(st_s[w + k][qb][1][r]) : 0;
      ms += st_s[w + k][qb][2][r];
    }
    const float gate = M > 0.f ? (p.has_gamma ? M / (M + p.gamma) : 1.f) : 0.f;
    const float z = ms + 1e-12f;
    const float so = gate / z;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[qb][db][i] *= so;
    store_row<D, VEC>(static_cast<float*>(p.o) + b * p.osb + h * p.osh + (int64_t)row * p.osn,
                      acc[qb], g);
    if (g == 0) {
      const int64_t si = (int64_t)bh * N + row;
      p.M[si] = M;
      p.Z[si] = z;
      if (COUNT && p.Nmax) p.Nmax[si] = M > 0.f ? c : 0;
    }
  }
}

// Row constants of the backward, written by the dQ kernel for the dK/dV kernel: planes of N floats
// per (b, h): M, g/Z, 10 g/Z scale, D, and the dS share of a peak tie.
constexpr int NPL = 5;
__device__ __forceinline__ float* rc_plane(const BwdParams& p, int64_t bh, int k) {
  return p.rc + (bh * 8 + k) * (int64_t)p.N;
}

// dQ and the tau partials: query-parallel, the forward's tiling, in two sweeps over the keys.
// The first forms each row's D = sum_j (P_j / Z) dW_j (src/triton_pnfirtau.py:575-577 take it
// from the flash identity <dO, O>/g instead; in fp32 that difference of two separately rounded
// values loses the cancellation of dW - D on peaked rows, while this sum holds the very dW
// values the gradient subtracts it from, bitwise the same in every sweep and in the dK/dV
// kernel) and counts the peak ties; the second accumulates dQ, with G/Nmax for tied keys.  It
// goes back over the tiles from the last, which is in LDS already.
template <int D, bool CAUSAL, bool VEC>
__global__ __launch_bounds__(BwdCfg<D>::NT, VEC ? BwdCfg<D>::MINW : 2) void f32_bwd_dq_kernel(BwdParams p, bool has_gamma) {
  constexpr int QB = BwdCfg<D>::QB, NW = BwdCfg<D>::NW, NT = BwdCfg<D>::NT;
  constexpr int KS = D / 4, DB = D / 16;
  __shared__ __attribute__((aligned(16))) float Ks0[TB * D];
  __shared__ __attribute__((aligned(16))) float Vs0[TB * D];
  __shared__ __attribute__((aligned(16))) float Ks1[TB * D];
  __shared__ __attribute__((aligned(16))) float Vs1[TB * D];
  __shared__ double part_s[NW];
  __shared__ float pdw_s[NW][QB][16];  // each wave's row sums of P dW and tie counts, between sweeps
  __shared__ int nt_s[NW][QB][16];
  __shared__ uint8_t act_s[kMaxTiles];  // the tile mask's row of this workgroup
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, g = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int N = p.N, nb = (N + RB - 1) / RB;
  int blk, bh;
  block_of(nb, p.B * p.H, CAUSAL && D <= 64, true, blk, bh);
  const int b = bh / p.H, h = bh % p.H;
  const int rg = w >> 2, kp = w & 3;  // as in the forward
  const int m0 = blk * RB, qw = m0 + 16 * rg, qlast = qw + 16 * QB - 1;
  const float* Q = static_cast<const float*>(p.q) + b * p.qsb + h * p.qsh;
  const float* K = static_cast<const float*>(p.k) + b * p.ksb + h * p.ksh;
  const float* V = static_cast<const float*>(p.v) + b * p.vsb + h * p.vsh;
  const float* dO = static_cast<const float*>(p.dout) + b * p.dosb + h * p.dosh;
  const float ntau = -p.tau[0], scale = p.scale;
  const int kv_end = CAUSAL ? min(m0 + RB, N) : N;
  const int ntiles = (kv_end + TB - 1) / TB;
  const TileDma<D, VEC, NW> kdma(w, lane, p.ksn), vdma(w, lane, p.vsn);
  const auto load_tile = [&](int n, float* kt, float* vt) {
    kdma.load(K, p.ksn, n, N, kt, w, lane);
    vdma.load(V, p.vsn, n, N, vt, w, lane);
  };
  load_tile(0, Ks0, Vs0);
  const bool masked_tiles = p.mask && ntiles <= kMaxTiles;
  if (masked_tiles)
    for (int t = tid; t < ntiles; t += NT)
      act_s[t] = p.mask[((int64_t)bh * p.nq32 + blk) * p.nk64 + t];
  score_t<D> qf[QB][KS];
  float df[QB][KS];
  float rM[QB], Zr[QB], gate[QB], rcoef[QB];
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    const int row = qw + 16 * qb + r;
    const bool has = row < N;
    load_row<D, VEC>(qf[qb], Q + (int64_t)row * p.qsn, has, g);
    load_row<D, VEC>(df[qb], dO + (int64_t)row * p.dosn, has, g);
    const int64_t si = (int64_t)bh * N + (has ? row : 0);
    rM[qb] = has ? p.M[si] : 0.f;
    Zr[qb] = has ? p.Z[si] : 1.f;
    gate[qb] = rM[qb] > 0.f ? (has_gamma ? rM[qb] / (rM[qb] + p.gamma) : 1.f) : 0.f;
    rcoef[qb] = 10.f * gate[qb] / Zr[qb];  // of du, whose sum is the tau gradient
  }
  // the wave's block of tile t holds no key of its rows, or the tile is silent
  const auto skip = [&](int t) {
    const int kb = t * TB + 16 * kp;
    return qw >= N || kb >= N || (CAUSAL && kb > qlast) || (masked_tiles && act_s[t] == 0);
  };
  const auto scores = [&](int t, const float* kc, f32x4 (&u)[QB]) {
    const int kb = t * TB + 16 * kp;
    dot64<D, QB>(kc, 16 * kp, r, g, qf, u);
#pragma unroll
    for (int qb = 0; qb < QB; ++qb)
      rectify<CAUSAL, true>(u[qb], scale, ntau,
                            kb + 15 >= N || qlast >= N || (CAUSAL && kb + 15 > qw), kb + 4 * g,
                            qw + 16 * qb + r, N);
  };
  // First sweep: sum P dW and the peak-tie counts (the backward has no Nmax from the forward).
  float pdw[QB] = {};
  int nt[QB] = {};
  const auto sweep1 = [&](int t, const float* kc, const float* vc, float* kn, float* vn) {
    wait_vmem();
    __syncthreads();
    if (t + 1 < ntiles) load_tile((t + 1) * TB, kn, vn);
    if (skip(t)) return;
    f32x4 dw[QB], u[QB];
    dot32<D, QB>(vc, 16 * kp, r, g, df, dw);
    scores(t, kc, u);
#pragma unroll
    for (int qb = 0; qb < QB; ++qb)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        // where u = 0 the row may be masked, or repeat a row past N that is not finite: no term
        const bool on = u[qb][i] > 0.f;
        pdw[qb] = __builtin_fmaf(pow10f_(u[qb][i]), on ? dw[qb][i] : 0.f, pdw[qb]);
        nt[qb] += (u[qb][i] == rM[qb] && on) ? 1 : 0;
      }
  };
  for (int t = 0; t < ntiles; t += 2) {
    sweep1(t, Ks0, Vs0, Ks1, Vs1);
    if (t + 1 < ntiles) sweep1(t + 1, Ks1, Vs1, Ks0, Vs0);
  }
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    pdw[qb] += __shfl_xor(pdw[qb], 16, 64);
    pdw[qb] += __shfl_xor(pdw[qb], 32, 64);
    nt[qb] += __shfl_xor(nt[qb], 16, 64);
    nt[qb] += __shfl_xor(nt[qb], 32, 64);
    if (g == 0) {
      pdw_s[w][qb][r] = pdw[qb];
      nt_s[w][qb][r] = nt[qb];
    }
  }
  __syncthreads();
  float rD[QB], rG[QB];  // D, and the du share of a tied key
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    // the row group's four waves in order, the same sums in each of them
    float ps = 0.f;
    int c = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      ps += pdw_s[4 * rg + k][qb][r];
      c += nt_s[4 * rg + k][qb][r];
    }
    rD[qb] = rM[qb] > 0.f ? ps / Zr[qb] : 0.f;
    float rGu = 0.f;  // the whole row's peak-tie du
    if (has_gamma && rM[qb] > 0.f)
      rGu = rD[qb] * (p.gamma / ((rM[qb] + p.gamma) * (rM[qb] + p.gamma)));
    rG[qb] = c > 0 ? rGu / (float)c : 0.f;
    const int row = qw + 16 * qb + r;
    if (row < N && g == 0 && kp == 0) {  // read by the dK/dV kernel
      rc_plane(p, bh, 0)[row] = rM[qb];
      rc_plane(p, bh, 1)[row] = gate[qb] / Zr[qb];
      rc_plane(p, bh, 2)[row] = rcoef[qb] * scale;
      rc_plane(p, bh, 3)[row] = rD[qb];
      rc_plane(p, bh, 4)[row] = rG[qb] * scale;
    }
  }
  f32x4 acc[QB][DB];
  zero_acc(acc);
  double dsum = 0.0;  // the lane's sum of du; per-tile fp32 sums are added in fp64
  const auto sweep2 = [&](int t, const float* kc, const float* vc, float* kn, float* vn) {
    wait_vmem();
    __syncthreads();
    if (t > 0) load_tile((t - 1) * TB, kn, vn);
    if (skip(t)) return;
    const int kb = t * TB + 16 * kp;
    const bool tail = kb + 15 >= N;
    f32x4 dw[QB], u[QB];
    dot32<D, QB>(vc, 16 * kp, r, g, df, dw);
    scores(t, kc, u);
    float tsum = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float ds[QB], x[DB];
      ld_cols<D>(kc, 16 * kp + 4 * g + i, r, tail, kb + 4 * g + i < N, x);
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) {
        const float uv = u[qb][i], u2 = uv * uv, u4 = u2 * u2;
        float du = rcoef[qb] * (u4 * u4 * uv) * (dw[qb][i] - rD[qb]);
        if (uv == rM[qb]) du += rG[qb];
        du = uv > 0.f ? du : 0.f;
        tsum += du;
        ds[qb] = du * scale;
      }
      add_outer<D>(x, ds, acc);  // dQ^T[d][query] += K^T[d][key] dS^T[key][query]
    }
    dsum += (double)tsum;
  };
  for (int t = ntiles - 1; t >= 0; --t) {
    if (t & 1) sweep2(t, Ks1, Vs1, Ks0, Vs0);
    else sweep2(t, Ks0, Vs0, Ks1, Vs1);
  }
  dsum = wave_sum_d(dsum);
  if (lane == 0) part_s[w] = dsum;
  __syncthreads();  // also: every wave is done with the tiles, which take the waves' dQ sums
  if (tid == 0) {
    double ps = 0.0;
#pragma unroll
    for (int v = 0; v < NW; ++v) ps += part_s[v];
    p.partials[(int64_t)bh * nb + blk] = ps;
  }
  const auto ex = [&](int k) { return k == 0 ? Ks0 : k == 1 ? Vs0 : Ks1; };
  const int xo = rg * 4 * DB * 64 + lane;
  if (kp > 0) put_acc(ex(kp - 1) + xo, acc);
  __syncthreads();
  if (kp > 0) return;
#pragma unroll
  for (int k = 0; k < 3; ++k) add_acc(ex(k) + xo, acc);
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    const int row = qw + 16 * qb + r;
    if (row < N)
      store_row<D, VEC>(static_cast<float*>(p.dq) + b * p.dqsb + h * p.dqsh + (int64_t)row * p.dqsn,
                        acc[qb], g);
  }
}

// dtau = -(sum of the du partials), in fp64 and a fixed order, by one workgroup of NT threads.
template <int NT>
__device__ __forceinline__ void dtau_sum(const double* partials, int64_t n, float* dtau, int tid,
                                         double* red) {
  double acc = 0.0;
  for (int64_t i = tid; i < n; i += NT) acc += partials[i];
  acc = wave_sum_d(acc);
  if ((tid & 63) == 0) red[tid >> 6] = acc;
  __syncthreads();
  if (tid == 0) {
    double t = 0.0;
    for (int v = 0; v < NT / 64; ++v) t += red[v];
    dtau[0] = (float)(-t);
  }
}
__global__ __launch_bounds__(256) void f32_dtau_kernel(const double* partials, int64_t n,
                                                       float* dtau) {
  __shared__ double red[4];
  dtau_sum<256>(partials, n, dtau, threadIdx.x, red);
}

// dK and dV: key-parallel, 32 keys per workgroup, held as MFMA B operands; query tiles of 64 rows
// and their row constants stream through LDS, each wave taking one 16-row block of every tile.
// With sum_dtau its last workgroup also sums the dQ stage's tau partials (no launch of its own).
template <int D, bool CAUSAL, bool VEC>
__global__ __launch_bounds__(BwdCfg<D>::NT, VEC ? BwdCfg<D>::MINW : 2) void f32_bwd_dkdv_kernel(BwdParams p, bool sum_dtau) {
  constexpr int QB = BwdCfg<D>::QB, NW = BwdCfg<D>::NW, NT = BwdCfg<D>::NT;
  constexpr int KS = D / 4, DB = D / 16;
  __shared__ __attribute__((aligned(16))) float Qs0[TB * D];
  __shared__ __attribute__((aligned(16))) float dOs0[TB * D];
  __shared__ __attribute__((aligned(16))) float RC0[NPL * TB];
  __shared__ __attribute__((aligned(16))) float Qs1[TB * D];
  __shared__ __attribute__((aligned(16))) float dOs1[TB * D];
  __shared__ __attribute__((aligned(16))) float RC1[NPL * TB];
  __shared__ double red_s[NW];
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, g = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int N = p.N, nb = (N + RB - 1) / RB;
  int blk, bh;
  block_of(nb, p.B * p.H, CAUSAL && D <= 64, false, blk, bh);
  const int b = bh / p.H, h = bh % p.H;
  // the wave's first 16-key group (it takes QB) and its 16-query block of every query tile
  const int kg = w >> 2, qp = w & 3;
  const int k0 = blk * RB, kw = k0 + 16 * kg, klast = kw + 16 * QB - 1;
  const int kt = k0 / TB;  // the 64-key tile of the tile mask that holds these keys
  const float* Q = static_cast<const float*>(p.q) + b * p.qsb + h * p.qsh;
  const float* K = static_cast<const float*>(p.k) + b * p.ksb + h * p.ksh;
  const float* V = static_cast<const float*>(p.v) + b * p.vsb + h * p.vsh;
  const float* dO = static_cast<const float*>(p.dout) + b * p.dosb + h * p.dosh;
  const float ntau = -p.tau[0], scale = p.scale;
  const int nqt = (N + TB - 1) / TB;
  const int qt0 = CAUSAL ? kt : 0;
  // wave w stages row-constant plane w, and wave 0 also plane 4 where there are four waves
  const float* rcw = rc_plane(p, bh, w < NPL ? w : 0);
  const float* rc4 = rc_plane(p, bh, 4);
  const TileDma<D, VEC, NW> qdma(w, lane, p.qsn), odma(w, lane, p.dosn);
  const auto load_tile = [&](int m, float* qt, float* ot, float* rc) {
    qdma.load(Q, p.qsn, m, N, qt, w, lane);
    odma.load(dO, p.dosn, m, N, ot, w, lane);
    const int rr = min(m + lane, N - 1);
    if (w < NPL) lds_dma4(rcw + rr, rc + w * TB);
    if (NW == 4 && w == 0) lds_dma4(rc4 + rr, rc + 4 * TB);
  };
  load_tile(qt0 * TB, Qs0, dOs0, RC0);
  score_t<D> kf[QB][KS];
  float vf[QB][KS];
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    const int key = kw + 16 * qb + r;
    load_row<D, VEC>(kf[qb], K + (int64_t)key * p.ksn, key < N, g);
    load_row<D, VEC>(vf[qb], V + (int64_t)key * p.vsn, key < N, g);
  }
  f32x4 adk[QB][DB], adv[QB][DB];
  zero_acc(adk);
  zero_acc(adv);
  // The tile-mask byte of the wave's 32-query group, one tile ahead of its use.
  const uint8_t* mcol = p.mask ? p.mask + (int64_t)bh * p.nq32 * p.nk64 + kt : nullptr;
  const auto fetch_act = [&](int t) -> int {
    const int r32 = 2 * t + (qp >> 1);
    return mcol && r32 < p.nq32 ? mcol[(int64_t)r32 * p.nk64] : 1;
  };
  int act_next = fetch_act(qt0);
  const auto step = [&](int t, const float* qc, const float* oc, const float* rc, float* qn,
                        float* on, float* rn) {
    const int q0 = t * TB + 16 * qp;  // the wave's queries
    wait_vmem();
    __syncthreads();
    const int act = act_next;
    if (t + 1 < nqt) {
      load_tile((t + 1) * TB, qn, on, rn);
      act_next = fetch_act(t + 1);
    }
    if (kw >= N || q0 >= N || (CAUSAL && q0 + 15 < kw) || act == 0) return;
    const bool tail = q0 + 15 >= N;
    // S[query][key] = Q K^T (Q as A, fp64): bitwise the forward's S^T, transposed
    f32x4 dw[QB], u[QB];
    dot32<D, QB>(oc, 16 * qp, r, g, vf, dw);
    dot64<D, QB>(qc, 16 * qp, r, g, kf, u);
#pragma unroll
    for (int qb = 0; qb < QB; ++qb)
      rectify<CAUSAL, false>(u[qb], scale, ntau, tail || klast >= N || (CAUSAL && q0 < klast),
                             q0 + 4 * g, kw + 16 * qb + r, N);
    const auto plane = [&](int k) {
      return *reinterpret_cast<const f32x4*>(rc + k * TB + 16 * qp + 4 * g);
    };
    const f32x4 cM = plane(0), cw = plane(1), cs = plane(2), cD = plane(3), cT = plane(4);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float wv[QB], ds[QB], x[DB];
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) {
        const float uv = u[qb][i], u2 = uv * uv, u4 = u2 * u2, u8 = u4 * u4;
        wv[qb] = u8 * u2 * cw[i];
        float d = cs[i] * (u8 * uv) * (dw[qb][i] - cD[i]);
        if (uv == cM[i]) d += cT[i];
        ds[qb] = uv > 0.f ? d : 0.f;
      }
      // dV^T[d][key] += dO^T[d][query] W[query][key]; dK^T likewise with Q and dS
      const bool in = q0 + 4 * g + i < N;
      ld_cols<D>(oc, 16 * qp + 4 * g + i, r, tail, in, x);
      add_outer<D>(x, wv, adv);
      ld_cols<D>(qc, 16 * qp + 4 * g + i, r, tail, in, x);
      add_outer<D>(x, ds, adk);
    }
  };
  for (int t = qt0; t < nqt; t += 2) {
    step(t, Qs0, dOs0, RC0, Qs1, dOs1, RC1);
    if (t + 1 < nqt) step(t + 1, Qs1, dOs1, RC1, Qs0, dOs0, RC0);
  }
  // waves qp = 1, 2, 3 of the key groups hand their sums to wave qp = 0 through the tiles' LDS
  __syncthreads();
  static_assert(RB / 16 * 2 * 4 * DB * 64 <= TB * D, "the dK and dV sums fit one tile");
  const auto ex = [&](int k) { return k == 0 ? Qs0 : k == 1 ? dOs0 : Qs1; };
  const int xo = kg * 8 * DB * 64 + lane;
  if (qp > 0) {
    put_acc(ex(qp - 1) + xo, adk);
    put_acc(ex(qp - 1) + xo + QB * 4 * DB * 64, adv);
  }
  __syncthreads();
  if (qp == 0) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      add_acc(ex(k) + xo, adk);
      add_acc(ex(k) + xo + QB * 4 * DB * 64, adv);
    }
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
      const int key = kw + 16 * qb + r;
      if (key < N) {
        store_row<D, VEC>(static_cast<float*>(p.dk) + b * p.dksb + h * p.dksh +
                              (int64_t)key * p.dksn, adk[qb], g);
        store_row<D, VEC>(static_cast<float*>(p.dv) + b * p.dvsb + h * p.dvsh +
                              (int64_t)key * p.dvsn, adv[qb], g);
      }
    }
  }
  if (sum_dtau && blockIdx.x == gridDim.x - 1)
    dtau_sum<NT>(p.partials, (int64_t)p.B * p.H * nb, p.dtau, tid, red_s);
}

// Whether the rows of an operand are whole 16-byte chunks and 64 of them lie within 4 GB.
bool rows16(const void* ptr, int64_t sb, int64_t sh, int64_t sn) {
  return (reinterpret_cast<uintptr_t>(ptr) & 15u) == 0 && ((sb | sh | sn) & 3) == 0 && sn >= 0 &&
         sn < (1ll << 24);
}

template <int D>
int fwd_d(const FwdParams& fp, bool causal, hipStream_t st) {
  constexpr int NT = FwdCfg<D>::NT;
  const int64_t nwg = (int64_t)((fp.N + RB - 1) / RB) * fp.B * fp.H;
  if (nwg >= (1ll << 31)) {
    set_error("flash(f32): %lld workgroups exceed the grid", (long long)nwg);
    return PNFX_EINVAL;
  }
  const bool gen = fp.Nmax || !(rows16(fp.q, fp.qsb, fp.qsh, fp.qsn) &&
                                rows16(fp.k, fp.ksb, fp.ksh, fp.ksn) &&
                                rows16(fp.v, fp.vsb, fp.vsh, fp.vsn) &&
                                rows16(fp.o, fp.osb, fp.osh, fp.osn));
  const dim3 grid((unsigned)nwg), block(NT);
  if (causal) {
    if (gen) hipLaunchKernelGGL((f32_fwd_kernel<D, true, true>), grid, block, 0, st, fp);
    else hipLaunchKernelGGL((f32_fwd_kernel<D, true, false>), grid, block, 0, st, fp);
  } else {
    if (gen) hipLaunchKernelGGL((f32_fwd_kernel<D, false, true>), grid, block, 0, st, fp);
    else hipLaunchKernelGGL((f32_fwd_kernel<D, false, false>), grid, block, 0, st, fp);
  }
  return launch_status("pnfx_flash_fwd(f32)");
}

template <int D, bool VEC>
int bwd_dv(const BwdParams& bp, bool causal, bool has_gamma, int stages, hipStream_t st) {
  constexpr int NT = BwdCfg<D>::NT;
  const int64_t nb = (bp.N + RB - 1) / RB;
  if (nb * bp.B * bp.H >= (1ll << 31)) {
    set_error("flash(f32): %lld workgroups exceed the grid", (long long)(nb * bp.B * bp.H));
    return PNFX_EINVAL;
  }
  const dim3 grid((unsigned)(nb * bp.B * bp.H)), block(NT);
  const bool dkdv = stages & PNFX_BWD_DKDV;
  if (stages & PNFX_BWD_DQ) {
    if (causal)
      hipLaunchKernelGGL((f32_bwd_dq_kernel<D, true, VEC>), grid, block, 0, st, bp, has_gamma);
    else hipLaunchKernelGGL((f32_bwd_dq_kernel<D, false, VEC>), grid, block, 0, st, bp, has_gamma);
    if (!dkdv)  // otherwise the dK/dV kernel sums the partials
      hipLaunchKernelGGL(f32_dtau_kernel, dim3(1), dim3(256), 0, st, bp.partials,
                         bp.B * bp.H * nb, bp.dtau);
    const int rc = launch_status("pnfx_flash_bwd(f32 dq)");
    if (rc) return rc;
  }
  if (dkdv) {  // reads the row constants the dQ stage wrote
    const bool sum_dtau = stages & PNFX_BWD_DQ;
    if (causal)
      hipLaunchKernelGGL((f32_bwd_dkdv_kernel<D, true, VEC>), grid, block, 0, st, bp, sum_dtau);
    else hipLaunchKernelGGL((f32_bwd_dkdv_kernel<D, false, VEC>), grid, block, 0, st, bp, sum_dtau);
    const int rc = launch_status("pnfx_flash_bwd(f32 dkdv)");
    if (rc) return rc;
  }
  return PNFX_OK;
}

// The prepare stage has nothing to do: the dQ kernel forms the row constants it hands on.
template <int D>
int bwd_d(const BwdParams& bp, bool causal, bool has_gamma, int stages, hipStream_t st) {
  const bool vec = rows16(bp.q, bp.qsb, bp.qsh, bp.qsn) && rows16(bp.k, bp.ksb, bp.ksh, bp.ksn) &&
                   rows16(bp.v, bp.vsb, bp.vsh, bp.vsn) &&
                   rows16(bp.dout, bp.dosb, bp.dosh, bp.dosn) &&
                   rows16(bp.dq, bp.dqsb, bp.dqsh, bp.dqsn) &&
                   rows16(bp.dk, bp.dksb, bp.dksh, bp.dksn) &&
                   rows16(bp.dv, bp.dvsb, bp.dvsh, bp.dvsn);
  return vec ? bwd_dv<D, true>(bp, causal, has_gamma, stages, st)
             : bwd_dv<D, false>(bp, causal, has_gamma, stages, st);
}

}  // namespace

int flash_fwd_f32(const FwdParams& fp, int64_t D, bool causal, hipStream_t st) {
  switch (D) {
    case 16: return fwd_d<16>(fp, causal, st);
    case 32: return fwd_d<32>(fp, causal, st);
    case 64: return fwd_d<64>(fp, causal, st);
    case 128: return fwd_d<128>(fp, causal, st);
  }
  set_error("flash(f32): head dim %lld not in {16, 32, 64, 128}", (long long)D);
  return PNFX_EUNSUPPORTED;
}

int flash_bwd_f32(const BwdParams& bp, int64_t D, bool causal, bool has_gamma, int stages,
                  hipStream_t st) {
  switch (D) {
    case 16: return bwd_d<16>(bp, causal, has_gamma, stages, st);
    case 32: return bwd_d<32>(bp, causal, has_gamma, stages, st);
    case 64: return bwd_d<64>(bp, causal, has_gamma, stages, st);
    case 128: return bwd_d<128>(bp, causal, has_gamma, stages, st);
  }
  set_error("flash(f32): head dim %lld not in {16, 32, 64, 128}", (long long)D);
  return PNFX_EUNSUPPORTED;
}

}  // namespace pnfx
