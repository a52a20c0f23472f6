// Row-fused rectified power-norm score -> weight (the materialised-score path of pn_fir_tau).
//
// One wave64 per score row; any row length.  Forward makes two passes over the row:
// pass 1 accumulates the row peak and the power mass (lane-local, then a wave reduction),
// pass 2 counts peak ties and writes the weights from the register-held scores (re-reading
// only what did not fit).  Backward mirrors it: pass 1 forms <dW, w_hat>, pass 2 writes
// dScores and the row's tau partial.  A lane moves 16 bytes per access whatever the rows'
// alignment (rows that start at any element: unaligned vector accesses, and single elements
// for a last chunk that the row does not fill), but for short ragged bf16 rows (launch_rows).
//
// Bound: HBM for the bytes (the causal half of the inputs read, the whole output written), with
// the vector units close behind: about 19 operations per entry forward and 27 backward.  On the
// scores of [32, 4, 512, 512] bf16: forward 27.0 -> 26.2 us, backward 43.0 -> 32.6 us (per-entry 64-bit
// range tests and, in the backward, a division per entry before); [4, 8, 777, 777]: 23.8 -> 17.2 and
// 34.0 -> 23.3 us (single elements per lane, and every chunk that a register could hold computed
// whether or not the row reaches it, before).
//
// Semantics follow src/triton_pnfirtau.py:141-212 (forward) and :214-303 (backward):
// s = fma(raw, scale, -tau); u = relu(s) on valid columns (col <= t when causal,
// t = row % N); pw = u^p; Z = sum pw + 1e-12; gate = peak/(peak + gamma);
// w = pw * (gate / Z); silent rows (peak <= 0) short-circuit to zeros.
#include "pnfx_common.h"

namespace pnfx {
namespace {

struct RowsArgs {
  const void* raw;
  int64_t raw_rs;
  const void* dw;
  int64_t dw_rs;
  void* out;  // w (forward) or d_raw (backward)
  int64_t out_rs;
  float* M;
  float* Z;
  int32_t* Nmax;
  float* dtau_rows;
  int64_t R, N;
  const float* tau;
  float scale, p, gamma;
  int has_gamma, causal;
};

// Wave reductions by data-parallel-primitive moves within the register file (a butterfly through
// LDS waits for six LDS round trips): shifts by 1, 2, 4, 8 within rows of 16 lanes, then the
// rows' last lanes broadcast to the rows after them; lane 63 ends with the whole.  0 is neutral in
// all three (the maxima are of non-negative values).
template <int CTRL, int ROWS>
__device__ __forceinline__ int dpp_move(int x) {
  return __builtin_amdgcn_update_dpp(0, x, CTRL, ROWS, 0xf, false);
}
template <typename F>
__device__ __forceinline__ int dpp_reduce(int x, const F& f) {
  x = f(x, dpp_move<0x111, 0xf>(x));
  x = f(x, dpp_move<0x112, 0xf>(x));
  x = f(x, dpp_move<0x114, 0xf>(x));
  x = f(x, dpp_move<0x118, 0xf>(x));
  x = f(x, dpp_move<0x142, 0xa>(x));
  x = f(x, dpp_move<0x143, 0xc>(x));
  return __builtin_amdgcn_readlane(x, 63);
}
__device__ __forceinline__ float row_max(float v) {
  return __int_as_float(dpp_reduce(__float_as_int(v), [](int a, int b) { return max(a, b); }));
}
__device__ __forceinline__ float row_sum(float v) {
  return __int_as_float(dpp_reduce(__float_as_int(v), [](int a, int b) {
    return __float_as_int(__int_as_float(a) + __int_as_float(b));
  }));
}
__device__ __forceinline__ int row_sum_i(int v) {
  return dpp_reduce(v, [](int a, int b) { return a + b; });
}

// Query position of row r (32-bit where the sizes allow: a 64-bit remainder takes a long
// sequence).
__device__ __forceinline__ int64_t row_pos(int64_t r, int64_t N) {
  if (((r | N) >> 32) == 0) return (uint32_t)r % (uint32_t)N;
  return r % N;
}

// u^p of the general power, from u's logarithm
__device__ __forceinline__ float pow_log(float u, float lg, float p) {
  return u > 0.0f ? expf(lg * p) : 0.0f;
}
template <int PMODE>
__device__ __forceinline__ float pow_p(float u, float p) {
  if (PMODE == 10) {
    const float u2 = u * u;
    const float u4 = u2 * u2;
    return u4 * u4 * u2;
  } else if (PMODE == 2) {
    return u * u;
  } else {
    return pow_log(u, logf(u), p);
  }
}

// A chunk of V consecutive elements of a row, converted to fp32: 16 bytes, or one element.  ANY: rows
// of any alignment and length, else rows of whole 16-byte aligned chunks.
template <typename T, int V, bool ANY>
struct RowIO;
template <typename T>
struct RowIO<T, 1, true> {
  __device__ static __forceinline__ void load(const T* p, float (&x)[1]) { x[0] = to_f32(*p); }
  __device__ static __forceinline__ void store(T* p, const float (&x)[1]) { *p = from_f32<T>(x[0]); }
};
template <bool ANY>
struct RowIO<bf16, 8, ANY> {
  static constexpr int V = 8;
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
  struct __attribute__((packed, aligned(ANY ? 2 : 16))) Raw { u32x4 q; };
  struct __attribute__((packed, aligned(ANY ? 2 : 16))) Out { bf16x8 q; };
  __device__ static __forceinline__ void load(const bf16* p, float (&x)[V]) {
    const u32x4 w = reinterpret_cast<const Raw*>(p)->q;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      x[2 * j] = __uint_as_float(w[j] << 16);
      x[2 * j + 1] = __uint_as_float(w[j] & 0xffff0000u);
    }
  }
  __device__ static __forceinline__ void store(bf16* p, const float (&x)[V]) {
    bf16x8 v;
#pragma unroll
    for (int j = 0; j < V; ++j) v[j] = (bf16)x[j];
    reinterpret_cast<Out*>(p)->q = v;
  }
};
template <bool ANY>
struct RowIO<float, 4, ANY> {
  static constexpr int V = 4;
  struct __attribute__((packed, aligned(ANY ? 4 : 16))) Raw { f32x4 q; };
  __device__ static __forceinline__ void load(const float* p, float (&x)[V]) {
    const f32x4 q = reinterpret_cast<const Raw*>(p)->q;
#pragma unroll
    for (int j = 0; j < V; ++j) x[j] = q[j];
  }
  __device__ static __forceinline__ void store(float* p, const float (&x)[V]) {
    reinterpret_cast<Raw*>(p)->q = f32x4{x[0], x[1], x[2], x[3]};
  }
};
// The chunk of a row of N elements at c0 < N: zero past the row's end.
template <typename T, bool ANY, int V>
__device__ __forceinline__ void load_chunk(const T* row, int64_t c0, int64_t N, float (&x)[V]) {
  if (!ANY || c0 + V <= N) {
    RowIO<T, V, ANY>::load(row + c0, x);
  } else {
#pragma unroll
    for (int j = 0; j < V; ++j) x[j] = c0 + j < N ? to_f32(row[c0 + j]) : 0.f;
  }
}
template <typename T, bool ANY, int V>
__device__ __forceinline__ void store_chunk(T* row, int64_t c0, int64_t N, const float (&x)[V]) {
  if (!ANY || c0 + V <= N) {
    RowIO<T, V, ANY>::store(row + c0, x);
  } else {
#pragma unroll
    for (int j = 0; j < V; ++j)
      if (c0 + j < N) row[c0 + j] = from_f32<T>(x[j]);
  }
}
// u = relu(x scale - tau) of a chunk whose first nv entries (of any int) are valid, 0 elsewhere.
template <int V>
__device__ __forceinline__ void rectify(const float (&x)[V], float scale, float ntau, int nv,
                                        float (&u)[V]) {
#pragma unroll
  for (int j = 0; j < V; ++j) {
    const float s = fmaxf(__builtin_fmaf(x[j], scale, ntau), 0.0f);
    u[j] = j < nv ? s : 0.0f;
  }
}
__device__ __forceinline__ int valid_in_chunk(int64_t limit, int64_t c0) {
  const int64_t n = limit - c0;
  return n < 0 ? 0 : n > 16 ? 16 : (int)n;
}

// Chunks held in registers by the kernels of the longest rows (shorter rows have a kernel that holds
// all of theirs).
constexpr int kMaxChunks = 4;

// Lane l owns columns [l*V, l*V + V) of every 64*V-column chunk.  The first CH chunks of a
// row stay in registers between the two passes (u, and dW in the backward); columns beyond
// them are re-read in pass 2.  CH = 1 for rows of one chunk (512 bf16 / 256 fp32 entries),
// which keeps the register count low enough for 8 waves per SIMD -- the bytes in flight
// that a one-load-per-lane row needs to approach HBM bandwidth.  Chunks past the causal limit
// are not computed (a wave-uniform test).  p = 10 and 2 form a power again in pass 2; the general
// power, whose exponential and logarithm make most of the kernel, is kept in registers, in the
// backward its logarithm ([64, 1, 512, 512] bf16 at p = 3.5: forward 30.8 -> 21.5 us, backward 36.4 ->
// 33.4).
template <typename T, int PMODE, int V, bool ANY, int CH>
__global__ __launch_bounds__(256, V == 1 || CH <= 2 ? 8 : 4) void pn_rows_fwd_kernel(RowsArgs a) {
  constexpr int64_t SPAN = 64 * V;
  constexpr bool MORE = CH == kMaxChunks;  // rows longer than the registers
  const int64_t r = (int64_t)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (r >= a.R) return;
  const int64_t t = row_pos(r, a.N);
  const int64_t limit = a.causal ? t + 1 : a.N;
  const T* row = reinterpret_cast<const T*>(a.raw) + r * a.raw_rs;
  T* wrow = reinterpret_cast<T*>(a.out) + r * a.out_rs;
  const float ntau = -a.tau[0];
  const int64_t cl = (int64_t)lane * V;

  float u[CH][V], pw[PMODE ? 1 : CH][V];  // pw: the general power is costly, and taken once
  float peak = 0.0f, mass = 0.0f;
#pragma unroll
  for (int k = 0; k < CH; ++k) {
    if (k * SPAN >= limit) {
#pragma unroll
      for (int j = 0; j < V; ++j) u[k][j] = 0.0f;
      continue;
    }
    const int64_t c0 = k * SPAN + cl;
    float x[V] = {};
    if (c0 < limit) load_chunk<T, ANY>(row, c0, a.N, x);
    rectify(x, a.scale, ntau, valid_in_chunk(limit, c0), u[k]);
#pragma unroll
    for (int j = 0; j < V; ++j) {
      peak = fmaxf(peak, u[k][j]);
      const float pu = pow_p<PMODE>(u[k][j], a.p);
      if (!PMODE) pw[k][j] = pu;
      mass += pu;
    }
  }
  for (int64_t c0 = CH * SPAN + cl; MORE && c0 - cl < limit; c0 += SPAN) {
    if (c0 >= limit) continue;
    float x[V], uc[V];
    load_chunk<T, ANY>(row, c0, a.N, x);
    rectify(x, a.scale, ntau, valid_in_chunk(limit, c0), uc);
#pragma unroll
    for (int j = 0; j < V; ++j) {
      peak = fmaxf(peak, uc[j]);
      mass += pow_p<PMODE>(uc[j], a.p);
    }
  }
  peak = row_max(peak);
  mass = row_sum(mass);

  if (peak <= 0.0f) {
    const float zero[V] = {};
    for (int64_t c0 = cl; c0 < a.N; c0 += SPAN) store_chunk<T, ANY>(wrow, c0, a.N, zero);
    if (lane == 0) {
      a.M[r] = 0.0f;
      a.Z[r] = 1e-12f;
      a.Nmax[r] = 0;
    }
    return;
  }
  const float z = mass + 1e-12f;
  const float gate = a.has_gamma ? peak / (peak + a.gamma) : 1.0f;
  const float coef = gate / z;
  int cnt = 0;
#pragma unroll
  for (int k = 0; k < CH; ++k) {
    const int64_t c0 = k * SPAN + cl;
    if (k * SPAN >= a.N) break;
    float w[V] = {};
    if (k * SPAN < limit) {
#pragma unroll
      for (int j = 0; j < V; ++j) {
        w[j] = (PMODE ? pow_p<PMODE>(u[k][j], a.p) : pw[k][j]) * coef;
        cnt += (u[k][j] == peak) ? 1 : 0;
      }
    }
    if (c0 < a.N) store_chunk<T, ANY>(wrow, c0, a.N, w);
  }
  for (int64_t c0 = CH * SPAN + cl; MORE && c0 - cl < a.N; c0 += SPAN) {
    if (c0 >= a.N) continue;
    float w[V] = {};
    if (c0 < limit) {
      float x[V], uc[V];
      load_chunk<T, ANY>(row, c0, a.N, x);
      rectify(x, a.scale, ntau, valid_in_chunk(limit, c0), uc);
#pragma unroll
      for (int j = 0; j < V; ++j) {
        w[j] = pow_p<PMODE>(uc[j], a.p) * coef;
        cnt += (uc[j] == peak) ? 1 : 0;
      }
    }
    store_chunk<T, ANY>(wrow, c0, a.N, w);
  }
  cnt = row_sum_i(cnt);
  if (lane == 0) {
    a.M[r] = peak;
    a.Z[r] = z;
    a.Nmax[r] = cnt;
  }
}

template <int PMODE>  // u^(p - 1), p = 10 or 2
__device__ __forceinline__ float pow_pm1(float u) {
  if (PMODE == 10) {
    const float u2 = u * u;
    const float u4 = u2 * u2;
    return u4 * u4 * u;
  } else {
    return u;
  }
}

// The backward takes the scores in units of the power of two of the row's peak for p = 10 and 2
// (an exact scaling, folded into scale and tau): the powers are then at most 1, so that the sum
// <dW, u^p> can be divided by Z once instead of entry by entry without overflowing.  The unit is no
// smaller than 2^-16: Z holds 1e-12, which for p = 10 is 2^120 in that unit's powers, and in a
// smaller one would overflow.
template <typename T, int PMODE, int V, bool ANY, int CH>
__global__ __launch_bounds__(256, V == 1 ? 8 : CH == 1 ? (PMODE ? 8 : 7) : CH == 2 ? (PMODE ? 6 : 5) : PMODE ? 4 : 3) void pn_rows_bwd_kernel(RowsArgs a) {
  constexpr int64_t SPAN = 64 * V;
  constexpr bool MORE = CH == kMaxChunks;  // rows longer than the registers
  const int64_t r = (int64_t)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (r >= a.R) return;
  T* drow = reinterpret_cast<T*>(a.out) + r * a.out_rs;
  const int64_t cl = (int64_t)lane * V;
  const float peak = a.M[r];
  if (peak <= 0.0f) {
    const float zero[V] = {};
    for (int64_t c0 = cl; c0 < a.N; c0 += SPAN) store_chunk<T, ANY>(drow, c0, a.N, zero);
    if (lane == 0) a.dtau_rows[r] = 0.0f;
    return;
  }
  const int64_t t = row_pos(r, a.N);
  const int64_t limit = a.causal ? t + 1 : a.N;
  const T* row = reinterpret_cast<const T*>(a.raw) + r * a.raw_rs;
  const T* dyrow = reinterpret_cast<const T*>(a.dw) + r * a.dw_rs;
  const int e = PMODE ? min(max(__builtin_amdgcn_frexp_expf(peak), -16), 64) : 0;
  const float scale = __builtin_amdgcn_ldexpf(a.scale, -e);
  const float ntau = __builtin_amdgcn_ldexpf(-a.tau[0], -e);
  const float peak_e = __builtin_amdgcn_ldexpf(peak, -e);
  const float z = __builtin_amdgcn_ldexpf(a.Z[r], -PMODE * e);
  const float nmax = (float)a.Nmax[r];

  float u[CH][V], dy[CH][V], lg[PMODE ? 1 : CH][V];  // lg: u's logarithm, taken once
  float dot = 0.0f;
  const auto add_dot = [&](const float (&uc)[V], float (&lc)[V], const float (&g)[V]) {
#pragma unroll
    for (int j = 0; j < V; ++j) {
      if (!PMODE) lc[j] = logf(uc[j]);
      const float pw = PMODE ? pow_p<PMODE>(uc[j], a.p) : pow_log(uc[j], lc[j], a.p) / z;
      dot = __builtin_fmaf(g[j], pw, dot);
    }
  };
#pragma unroll
  for (int k = 0; k < CH; ++k) {
    if (k * SPAN >= limit) continue;
    const int64_t c0 = k * SPAN + cl;
    float x[V] = {}, g[V] = {};
    if (c0 < limit) {
      load_chunk<T, ANY>(row, c0, a.N, x);
      load_chunk<T, ANY>(dyrow, c0, a.N, g);
    }
    rectify(x, scale, ntau, valid_in_chunk(limit, c0), u[k]);
#pragma unroll
    for (int j = 0; j < V; ++j) dy[k][j] = g[j];
    add_dot(u[k], lg[PMODE ? 0 : k], g);
  }
  for (int64_t c0 = CH * SPAN + cl; MORE && c0 - cl < limit; c0 += SPAN) {
    if (c0 >= limit) continue;
    float x[V], g[V], uc[V], lc[V];
    load_chunk<T, ANY>(row, c0, a.N, x);
    load_chunk<T, ANY>(dyrow, c0, a.N, g);
    rectify(x, scale, ntau, valid_in_chunk(limit, c0), uc);
    add_dot(uc, lc, g);
  }
  dot = row_sum(dot);
  if (PMODE) dot /= z;
  // Rows whose sum does not tell: NaN may come from a chunk's dW past the causal limit (an infinity
  // there, times a power of 0), and where a power overflowed in the forward (inf / inf) this unit's
  // sum ends as 0.  The same sum over the valid entries alone.  (A test of each entry above instead
  // cost 17.2 -> 18.1 us at [64, 1, 512, 512] bf16.)
  if (dot != dot || (PMODE && z > __FLT_MAX__)) {
    dot = 0.0f;
    const auto add_valid = [&](int64_t c0, const float (&uc)[V], const float (&g)[V]) {
      const int nv = valid_in_chunk(limit, c0);
      float gv[V], lc[V];
#pragma unroll
      for (int j = 0; j < V; ++j) gv[j] = j < nv ? g[j] : 0.0f;
      add_dot(uc, lc, gv);
    };
#pragma unroll
    for (int k = 0; k < CH; ++k)
      if (k * SPAN < limit) add_valid(k * SPAN + cl, u[k], dy[k]);
    for (int64_t c0 = CH * SPAN + cl; MORE && c0 - cl < limit; c0 += SPAN) {
      if (c0 >= limit) continue;
      float x[V], g[V], uc[V];
      load_chunk<T, ANY>(row, c0, a.N, x);
      load_chunk<T, ANY>(dyrow, c0, a.N, g);
      rectify(x, scale, ntau, valid_in_chunk(limit, c0), uc);
      add_valid(c0, uc, g);
    }
    dot = row_sum(dot);
    if (PMODE) dot /= z;
    if (PMODE && pow_p<PMODE>(peak, a.p) > __FLT_MAX__) dot = __builtin_nanf("");
  }

  float gate = 1.0f, gterm = 0.0f;
  if (a.has_gamma) {
    gate = peak / (peak + a.gamma);
    const float dgate = a.gamma / ((peak + a.gamma) * (peak + a.gamma));
    gterm = dot * dgate / nmax;
  }
  // p gate u^(p-1) / Z: the unit's powers leave one factor 2^-e
  const float coef = __builtin_amdgcn_ldexpf(a.p * gate / z, -e);
  float acc = 0.0f;
  // du of a chunk, written over its dW; u == 0 covers both masked columns and the relu's dead side
  const auto du_chunk = [&](const float (&uc)[V], const float (&lc)[V], float (&g)[V]) {
#pragma unroll
    for (int j = 0; j < V; ++j) {
      const float pw = PMODE ? pow_pm1<PMODE>(uc[j]) : pow_log(uc[j], lc[j], a.p - 1.0f);
      const float du_norm = coef * pw * (g[j] - dot);
      const float du_gate = (a.has_gamma && uc[j] == peak_e) ? gterm : 0.0f;
      const float du = uc[j] > 0.0f ? du_norm + du_gate : 0.0f;
      acc += du;
      g[j] = du * a.scale;
    }
  };
#pragma unroll
  for (int k = 0; k < CH; ++k) {
    const int64_t c0 = k * SPAN + cl;
    if (k * SPAN >= a.N) break;
    float d[V] = {};
    if (k * SPAN < limit) {
#pragma unroll
      for (int j = 0; j < V; ++j) d[j] = dy[k][j];
      du_chunk(u[k], lg[PMODE ? 0 : k], d);
    }
    if (c0 < a.N) store_chunk<T, ANY>(drow, c0, a.N, d);
  }
  for (int64_t c0 = CH * SPAN + cl; MORE && c0 - cl < a.N; c0 += SPAN) {
    if (c0 >= a.N) continue;
    float d[V] = {};
    if (c0 < limit) {
      float x[V], uc[V], lc[V];
      load_chunk<T, ANY>(row, c0, a.N, x);
      load_chunk<T, ANY>(dyrow, c0, a.N, d);
      rectify(x, scale, ntau, valid_in_chunk(limit, c0), uc);
      if (!PMODE) {
#pragma unroll
        for (int j = 0; j < V; ++j) lc[j] = logf(uc[j]);
      }
      du_chunk(uc, lc, d);
    }
    store_chunk<T, ANY>(drow, c0, a.N, d);
  }
  acc = row_sum(acc);
  if (lane == 0) a.dtau_rows[r] = -acc;
}

// Sum of n floats in fp64 and a fixed order: each workgroup takes a contiguous part, four floats
// per lane and load, four loads in flight.  One workgroup writes the result itself (out32 or
// out64); more write their partial sums for a second launch.
constexpr int kSumPart = 1 << 17;  // floats per workgroup
template <typename S>
__global__ __launch_bounds__(1024) void sum_f64_kernel(const S* x, int64_t n, double* part,
                                                       float* out32, double* out64) {
  const int64_t first = (int64_t)blockIdx.x * kSumPart;
  const int64_t m = min(n - first, (int64_t)kSumPart);
  const S* p = x + first;
  double s[4] = {0.0, 0.0, 0.0, 0.0};
  int64_t i = 4 * threadIdx.x;
  typedef S vec __attribute__((ext_vector_type(4)));
  for (; i + 3 * 4096 + 3 < m; i += 4 * 4096) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const vec v = *reinterpret_cast<const vec*>(p + i + 4096 * k);
      s[k] += ((double)v[0] + (double)v[1]) + ((double)v[2] + (double)v[3]);
    }
  }
  for (; i < m; i += 4096)
    for (int64_t j = i; j < min(i + 4, m); ++j) s[0] += (double)p[j];
  __shared__ double red[16];
  const double w = wave_sum_d((s[0] + s[1]) + (s[2] + s[3]));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = w;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int k = 0; k < 16; ++k) t += red[k];
    if (part) part[blockIdx.x] = t;
    else if (out32) out32[0] = (float)t;
    else out64[0] = t;
  }
}

template <typename T, int V, bool ANY, int CH, bool BWD>
void launch_rows_v(const RowsArgs& a, int pm, dim3 grid, dim3 block, hipStream_t st) {
  if (BWD) {
    if (pm == 10) hipLaunchKernelGGL((pn_rows_bwd_kernel<T, 10, V, ANY, CH>), grid, block, 0, st, a);
    else if (pm == 2) hipLaunchKernelGGL((pn_rows_bwd_kernel<T, 2, V, ANY, CH>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((pn_rows_bwd_kernel<T, 0, V, ANY, CH>), grid, block, 0, st, a);
  } else {
    if (pm == 10) hipLaunchKernelGGL((pn_rows_fwd_kernel<T, 10, V, ANY, CH>), grid, block, 0, st, a);
    else if (pm == 2) hipLaunchKernelGGL((pn_rows_fwd_kernel<T, 2, V, ANY, CH>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((pn_rows_fwd_kernel<T, 0, V, ANY, CH>), grid, block, 0, st, a);
  }
}

// Rows of one or two chunks (64 lanes x 16 bytes) hold them in registers, longer ones up to four
// (fewer registers, more waves: two for four at N = 777 bf16 took the backward from 28 to 23.3 us).
// Short bf16 rows that are not whole aligned chunks go by single elements, 64 to a register: with
// eight to a lane few lanes compute, and the row's part of a chunk takes eight branches.  Forward /
// backward over 2^24 scores, by chunks -> by elements: N = 33 160 / 220 -> 89 / 137 us, N = 129
// 44.3 / 60.5 -> 35.1 / 52.5, N = 190 31.9 / 44.8 -> 26.6 / 38.9, N = 257 24.1 / 32.8 -> 25.8 / 37.5; with
// the general power, which is mostly computing, N = 300 34.5 / 57 -> 26.9 / 37.2, N = 511 22.5 /
// 36.4 -> 23.5 / 34.3.
template <typename T, bool BWD>
int launch_rows(const RowsArgs& a, hipStream_t st) {
  const dim3 grid((unsigned)((a.R + 3) / 4)), block(256);
  const int pm = a.p == 10.0f ? 10 : (a.p == 2.0f ? 2 : 0);
  constexpr int V = 16 / (int)sizeof(T);
  auto aligned = [](const void* ptr, int64_t rs) {
    return ((uintptr_t)ptr % 16 == 0) && rs % V == 0;
  };
  const bool vec = a.N % V == 0 && aligned(a.raw, a.raw_rs) && aligned(a.out, a.out_rs) &&
                   (!BWD || aligned(a.dw, a.dw_rs));
  const int64_t ch = (a.N + 64 * V - 1) / (64 * V);
  if constexpr (sizeof(T) == 2) {
    if (!vec && a.N <= (pm ? 256 : 384)) {
      if (a.N <= 64) launch_rows_v<T, 1, true, 1, BWD>(a, pm, grid, block, st);
      else if (a.N <= 128) launch_rows_v<T, 1, true, 2, BWD>(a, pm, grid, block, st);
      else launch_rows_v<T, 1, true, 6, BWD>(a, pm, grid, block, st);
      return launch_status(BWD ? "pnfx_pn_rows_bwd" : "pnfx_pn_rows_fwd");
    }
  }
  if (vec && ch <= 1) launch_rows_v<T, V, false, 1, BWD>(a, pm, grid, block, st);
  else if (vec && ch == 2) launch_rows_v<T, V, false, 2, BWD>(a, pm, grid, block, st);
  else if (vec) launch_rows_v<T, V, false, kMaxChunks, BWD>(a, pm, grid, block, st);
  else if (ch <= 1) launch_rows_v<T, V, true, 1, BWD>(a, pm, grid, block, st);
  else if (ch == 2) launch_rows_v<T, V, true, 2, BWD>(a, pm, grid, block, st);
  else launch_rows_v<T, V, true, kMaxChunks, BWD>(a, pm, grid, block, st);
  return launch_status(BWD ? "pnfx_pn_rows_bwd" : "pnfx_pn_rows_fwd");
}

template <bool BWD>
int rows_dispatch(const RowsArgs& a, int dtype, hipStream_t st) {
  if (a.R == 0 || a.N == 0) return PNFX_OK;
  if (dtype == PNFX_BF16) return launch_rows<bf16, BWD>(a, st);
  if (dtype == PNFX_F32) return launch_rows<float, BWD>(a, st);
  set_error("pn_rows: unsupported dtype %d", dtype);
  return PNFX_EUNSUPPORTED;
}

}  // namespace
}  // namespace pnfx

extern "C" int pnfx_pn_rows_fwd(const void* raw, int64_t raw_rs, void* w, int64_t w_rs, float* M,
                                float* Z, int32_t* Nmax, int64_t R, int64_t N, const float* tau,
                                float scale, float p, float gamma, int has_gamma, int causal,
                                int dtype, void* stream) {
  PNFX_REQUIRE(raw && w && M && Z && Nmax && tau, "pn_rows_fwd: null pointer");
  PNFX_REQUIRE(R >= 0 && N >= 0, "pn_rows_fwd: bad shape");
  pnfx::RowsArgs a{raw, raw_rs, nullptr, 0, w, w_rs, M, Z, Nmax, nullptr, R, N, tau, scale, p,
                   gamma, has_gamma, causal};
  return pnfx::rows_dispatch<false>(a, dtype, reinterpret_cast<hipStream_t>(stream));
}

extern "C" int pnfx_pn_rows_bwd(const void* dw, int64_t dw_rs, const void* raw, int64_t raw_rs,
                                const float* M, const float* Z, const int32_t* Nmax, void* draw,
                                int64_t draw_rs, float* dtau_rows, int64_t R, int64_t N,
                                const float* tau, float scale, float p, float gamma, int has_gamma,
                                int causal, int dtype, void* stream) {
  PNFX_REQUIRE(dw && raw && M && Z && Nmax && draw && dtau_rows && tau,
               "pn_rows_bwd: null pointer");
  PNFX_REQUIRE(R >= 0 && N >= 0, "pn_rows_bwd: bad shape");
  pnfx::RowsArgs a{raw, raw_rs, dw, dw_rs, draw, draw_rs, const_cast<float*>(M),
                   const_cast<float*>(Z), const_cast<int32_t*>(Nmax), dtau_rows, R, N, tau,
                   scale, p, gamma, has_gamma, causal};
  return pnfx::rows_dispatch<true>(a, dtype, reinterpret_cast<hipStream_t>(stream));
}

extern "C" int64_t pnfx_sum_f64_workspace_size(int64_t n) {
  return n <= pnfx::kSumPart ? 0 : (n + pnfx::kSumPart - 1) / pnfx::kSumPart * 8;
}

extern "C" int pnfx_sum_f64(const float* x, int64_t n, void* workspace, int64_t workspace_bytes,
                            float* out32, double* out64, void* stream) {
  PNFX_REQUIRE(x && n >= 1 && (out32 != nullptr) != (out64 != nullptr), "sum_f64: bad argument");
  PNFX_REQUIRE((reinterpret_cast<uintptr_t>(x) & 15u) == 0, "sum_f64: x must be 16-byte aligned");
  const int64_t need = pnfx_sum_f64_workspace_size(n);
  PNFX_REQUIRE(!need || (workspace && workspace_bytes >= need &&
                         (reinterpret_cast<uintptr_t>(workspace) & 31u) == 0),
               "sum_f64: workspace needs %lld bytes, 32-byte aligned", (long long)need);
  const int64_t nwg = (n + pnfx::kSumPart - 1) / pnfx::kSumPart;
  PNFX_REQUIRE(nwg <= pnfx::kSumPart, "sum_f64: %lld elements", (long long)n);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  double* part = need ? static_cast<double*>(workspace) : nullptr;
  hipLaunchKernelGGL((pnfx::sum_f64_kernel<float>), dim3((unsigned)nwg), dim3(1024), 0, st, x, n,
                     part, out32, out64);
  if (part)
    hipLaunchKernelGGL((pnfx::sum_f64_kernel<double>), dim3(1), dim3(1024), 0, st, part, nwg,
                       (double*)nullptr, out32, out64);
  return pnfx::launch_status("pnfx_sum_f64");
}
