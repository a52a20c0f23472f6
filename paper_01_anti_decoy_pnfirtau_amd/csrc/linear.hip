// Weight gradient of a bias-free linear layer: dW[M, N] = sum_k dY[k, m] X[k, n], with dY [K, M] and
// X [K, N] bf16 rows (the layer's output gradient and input), dW fp32 or bf16.
//
// The projections of an attention layer have small weights and many rows (M = 768, N = 256 over
// K = 16384 in a training step at B = 32, N = 512), so a kernel with one workgroup per output tile
// leaves most of the 256 CUs idle over a long serial reduction.  Here the rows are split over
// workgroups as well: each forms a 128 x 128 tile of its rows' products in fp32, and a second kernel
// sums the splits in a fixed order (no atomics: bitwise repeatable).
//
// MFMA mapping: both operands are contracted over rows, so both fragments come from row-major 64-row
// LDS tiles by transposing reads (tr_frag); the tiles go from global memory straight to LDS, two
// buffers deep.  A workgroup's four waves take a 64 x 64 quarter each.  X's fragment is the first
// operand, so a lane ends up with four consecutive columns of one row of dW and stores 16 bytes.
//
// Measured on MI355X (both kernels; the library's product and its cast in brackets): 768 x 256 over
// 16384 rows 29 us (93), of which summing the partial tiles takes 6; 256 x 256 17 (93); 768 x 256
// over 65536 rows 66 (240), 390 TFLOP/s.  Bound by the partial tiles' traffic at few rows and by the
// transposing LDS reads (one per two MFMAs and operand) at many; where a weight has tiles enough to
// fill the chip the library's larger tiles are faster (3072 x 1024 over 65536 rows 1272 against 492).
#include "tiles_bf16.h"

namespace pnfx {
namespace {

constexpr int kTile = 128;   // output tile
constexpr int kStep = 64;    // rows per step
constexpr int kMinSteps = 4; // steps that a split must have to cover its prologue and its partial tile
constexpr int kMaxSplits = 64;
// Workgroups aimed at: two for each of the 256 CUs (64 KB of LDS each).
constexpr int kTargetWgs = 512;

struct WgradArgs {
  const bf16* dy;
  const bf16* x;
  int64_t dy_rs, x_rs;
  float* part;  // [splits][M][N], or the result itself when splits == 1 and it is fp32
  int64_t K;
  int M, N, tiles_n, tiles, splits, chunk;  // chunk: steps per split
};

__global__ __launch_bounds__(256, 2) void linear_wgrad_kernel(WgradArgs a) {
  __shared__ __align__(16) bf16 sm[2][2][kStep * kTile];
  // The tiles of one split read the same rows: they run on one XCD (block id % 8), one after the
  // other, and share its L2.
  const int r = blockIdx.x >> 3;
  const int split = r / a.tiles * 8 + (blockIdx.x & 7), tile = r % a.tiles;
  if (split >= a.splits) return;
  const int m0 = tile / a.tiles_n * kTile, n0 = tile % a.tiles_n * kTile;
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, g = lane >> 4, r16 = lane & 15;
  const int K = (int)a.K;
  const int s0 = split * a.chunk, s1 = min(s0 + a.chunk, (K + kStep - 1) / kStep);
  // Columns past the matrix re-load its last chunk; their products are not stored.
  const TileDma<kTile, kTile> dma_y(w, lane, a.dy_rs, min(kTile, a.M - m0));
  const TileDma<kTile, kTile> dma_x(w, lane, a.x_rs, min(kTile, a.N - n0));
  const bf16 *dy = a.dy + m0, *x = a.x + n0;
  const auto load = [&](int s, int buf) {
    dma_y.load(dy, a.dy_rs, s * kStep, K, sm[buf][0], w);
    dma_x.load(x, a.x_rs, s * kStep, K, sm[buf][1], w);
  };
  const FragLane fl = tr_lane<kTile>(lane);
  const int wm = 4 * (w >> 1), wn = 4 * (w & 1);  // the wave's first 16-column block of dY and X
  f32x4 acc[4][4] = {};
  const auto products = [&](int buf, int hf, int rows) {
    bf16x8 fy[4], fx[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      fy[i] = tr_frag<kTile>(sm[buf][0], fl, hf, wm + i);
      fx[i] = tr_frag<kTile>(sm[buf][1], fl, hf, wn + i);
    }
    if (rows < kStep) {  // rows past K repeat the last one: zero in both operands
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int t = 0; t < 8; ++t)
          if (32 * hf + 8 * g + t >= rows) fy[i][t] = fx[i][t] = (bf16)0.f;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = mfma16x16x32(fx[j], fy[i], acc[i][j]);
  };
  load(s0, 0);
  wait_vmem();
  __syncthreads();
  for (int s = s0; s < s1; ++s) {
    const int buf = (s - s0) & 1;
    if (s + 1 < s1) load(s + 1, buf ^ 1);
    const int rows = min(K - s * kStep, kStep);
    products(buf, 0, rows);
    products(buf, 1, rows);
    wait_vmem();
    __syncthreads();
  }
  float* out = a.part + (int64_t)split * a.M * a.N;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int m = m0 + 16 * (wm + i) + r16, n = n0 + 16 * (wn + j) + 4 * g;
      if (m < a.M && n < a.N) *reinterpret_cast<f32x4*>(out + (int64_t)m * a.N + n) = acc[i][j];
    }
}

// Sum of the splits' partial results: 64 lanes of four columns, the splits dealt to the four waves
// (the loads of one output are a chain otherwise) and their sums added in wave order.
template <typename T>
__global__ __launch_bounds__(256) void linear_wgrad_sum_kernel(const float* part, int splits,
                                                               int64_t MN, T* out) {
  __shared__ f32x4 sums[3][64];
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t e = ((int64_t)blockIdx.x * 64 + lane) * 4;
  f32x4 acc = {};
  if (e < MN) {
#pragma unroll 4
    for (int s = w; s < splits; s += 4)
      acc += *reinterpret_cast<const f32x4*>(part + (int64_t)s * MN + e);
  }
  if (w) sums[w - 1][lane] = acc;
  __syncthreads();
  if (w || e >= MN) return;
#pragma unroll
  for (int i = 0; i < 3; ++i) acc += sums[i][lane];
#pragma unroll
  for (int i = 0; i < 4; ++i) out[e + i] = from_f32<T>(acc[i]);
}

// Splits of K rows over an [M, N] result.
int wgrad_chunk(int64_t M, int64_t N, int64_t K) {
  const int64_t tiles = ((M + kTile - 1) / kTile) * ((N + kTile - 1) / kTile);
  const int64_t steps = (K + kStep - 1) / kStep;
  int64_t splits = (kTargetWgs + tiles - 1) / tiles;
  splits = splits > kMaxSplits ? kMaxSplits : splits;
  splits = splits > steps / kMinSteps ? steps / kMinSteps : splits;
  splits = splits < 1 ? 1 : splits;
  return (int)((steps + splits - 1) / splits);
}

}  // namespace
}  // namespace pnfx

extern "C" int64_t pnfx_linear_wgrad_workspace_size(int64_t M, int64_t N, int64_t K, int dtype) {
  if (M < 1 || N < 1 || K < 1) return 0;
  const int64_t steps = (K + pnfx::kStep - 1) / pnfx::kStep, chunk = pnfx::wgrad_chunk(M, N, K);
  const int64_t splits = (steps + chunk - 1) / chunk;
  return splits == 1 && dtype == PNFX_F32 ? 0 : splits * M * N * 4;
}

extern "C" int pnfx_linear_wgrad(const void* dy, int64_t dy_rs, const void* x, int64_t x_rs,
                                 void* dw, int64_t M, int64_t N, int64_t K, int dtype,
                                 void* workspace, int64_t workspace_bytes, void* stream) {
  using namespace pnfx;
  PNFX_REQUIRE(dy && x && dw, "linear_wgrad: null pointer");
  PNFX_REQUIRE(dtype == PNFX_F32 || dtype == PNFX_BF16, "linear_wgrad: unsupported dtype %d", dtype);
  PNFX_REQUIRE(M >= 8 && N >= 8 && M % 8 == 0 && N % 8 == 0 && M <= 65536 && N <= 65536 && K >= 1 &&
                   K < (1ll << 30),
               "linear_wgrad: bad shape M=%lld N=%lld K=%lld", (long long)M, (long long)N,
               (long long)K);
  // 32-bit byte offsets within a 64-row tile
  PNFX_REQUIRE(dy_rs >= M && x_rs >= N && dy_rs % 8 == 0 && x_rs % 8 == 0 && dy_rs < (1 << 24) &&
                   x_rs < (1 << 24),
               "linear_wgrad: row strides %lld, %lld", (long long)dy_rs, (long long)x_rs);
  PNFX_REQUIRE(((reinterpret_cast<uintptr_t>(dy) | reinterpret_cast<uintptr_t>(x) |
                 reinterpret_cast<uintptr_t>(dw) | reinterpret_cast<uintptr_t>(workspace)) & 15) == 0,
               "linear_wgrad: operands must be 16-byte aligned");
  const int64_t need = pnfx_linear_wgrad_workspace_size(M, N, K, dtype);
  PNFX_REQUIRE(!need || (workspace && workspace_bytes >= need),
               "linear_wgrad: workspace needs %lld bytes", (long long)need);
  const int64_t steps = (K + kStep - 1) / kStep;
  WgradArgs a;
  a.dy = static_cast<const bf16*>(dy);
  a.x = static_cast<const bf16*>(x);
  a.dy_rs = dy_rs;
  a.x_rs = x_rs;
  a.part = static_cast<float*>(need ? workspace : dw);
  a.K = K;
  a.M = (int)M;
  a.N = (int)N;
  a.tiles_n = (int)((N + kTile - 1) / kTile);
  a.tiles = (int)((M + kTile - 1) / kTile) * a.tiles_n;
  a.chunk = wgrad_chunk(M, N, K);
  a.splits = (int)((steps + a.chunk - 1) / a.chunk);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const unsigned grid = (unsigned)(a.tiles * 8 * ((a.splits + 7) / 8));
  hipLaunchKernelGGL(linear_wgrad_kernel, dim3(grid), dim3(256), 0, st, a);
  if (need) {
    const unsigned nb = (unsigned)((M * N + 255) / 256);
    if (dtype == PNFX_F32)
      hipLaunchKernelGGL((linear_wgrad_sum_kernel<float>), dim3(nb), dim3(256), 0, st, a.part,
                         a.splits, M * N, static_cast<float*>(dw));
    else
      hipLaunchKernelGGL((linear_wgrad_sum_kernel<bf16>), dim3(nb), dim3(256), 0, st, a.part,
                         a.splits, M * N, static_cast<bf16*>(dw));
  }
  return launch_status("pnfx_linear_wgrad");
}
