// out[M, N] = x[M, K] . w[N, K]^T for M <= 16 (decode at small batch): a weight-streaming kernel.
//
// Call sites it serves: the four per-layer projections and the LM head at decode time -
// QKVParallelLinear / RowParallelLinear / MergedColumnParallelLinear.forward (nn/layers/linear.py:
// 696-760, 423-470, 1033-1155 -> F.linear) and LogitsProcessor._get_logits
// (nn/layers/logits_processor.py:340-376).  More rows, and 5 - 16 over large weights: gemm_dense.hip, then the library.
//
// At M <= 16 the product is a pure stream of the weight matrix (2 flop per weight byte per row): HBM-bound.  What decides the
// rate is how many bytes of each weight row one load covers and how many workgroups share the stream, so there are three forms:
//   1 row       a wave per weight row: a load covers 1 KB of the row, 4 of them in flight, the products on the vector unit (24
//               instructions a KB: a quarter of what the stream leaves room for), 2 waves a workgroup
//   2-4 rows    (few weight rows, or long ones) v_mfma_f32_4x4x4 (16 blocks): lane (b, i) loads 16 B of weight row i at chunk b,
//               so a load covers 256 B of 4 rows and its two halves are two products; the 16 blocks are 16 partial sums over K.
//               4 waves share K, 4 or 8 weight rows (columns of out) a workgroup
//   to 16 rows  v_mfma_f32_16x16x32: 64 B of 16 weight rows a load, x read in the same form (as many bytes out of L2 as weights:
//               what bounds it from 8 rows on), 8 waves share K
// Each form sums the partial results of its lanes and waves in a fixed order that M, K and the
// number of weight rows alone decide.
// us, cold weights under graph replay, N x K: 1 row / 4 rows / 8 rows; before (the third form for every M, the waves' k-steps
// interleaved) -> now (1 row of large weights: kRowOnce has the later figures; 5 - 16 rows of them go to sp_gemm_dense).  The second form ends at the 4 rows that its instruction holds: a second group of x rows for 5 to 8 was
// slower where there are many weight rows (8 rows: 20.1 against the third form's 17.3 at 16384 x 2048) and faster with few long ones (12.8
// against 14.6 at 2048 x 8192), which is left on the table.  Below 5 rows few_take_tiles has the line to the third form.
//   3072 x 2048     5.3 -> 4.6      5.9 -> 5.8      6.3 -> 6.1
//   2048 x 2048     5.0 -> 3.8      5.5 -> 5.3      5.7 -> 5.8
//   16384 x 2048   14.5 -> 12.3    15.9 -> 15.8    18.3 -> 18.2
//   2048 x 8192    13.3 -> 8.2     14.9 -> 12.0    16.4 -> 15.3
//   6144 x 4096    13.2 -> 9.9     15.4 -> 13.2    16.9 -> 16.4
//   28672 x 4096   43.7 -> 40.7    46.4 -> 42.9    52.7 -> 50.6
//   128256 x 2048  89.0 -> 83.1    98.5 -> 90.1   118.0 -> 113.2
// Tried and slower: x staged in LDS and a persistent loop over weight rows in any of 10 shapes (8 to 40 % slower: the copy and its
// barrier come before the first product, and the loop's tail is longer than a launch of many small workgroups), 16 products in
// flight, two weight rows a wave at one row.
//
// Epilogue fusion: with `epilogue` = 1 the weight is the merged gate|up matrix [2 I, K] of LlamaMLP
// (nn/models/llama/llama.py:62-66) and the output is SiluAndMul (nn/layers/activation.py:21-31) of the projection,
// [M, I]: a workgroup streams gate rows and the up rows of the same columns, and whoever finishes a gate column takes
// the up sum beside it and writes round(silu(round(gate))) * round(up), rounded - bit for bit the plain projection
// followed by sp_silu_and_mul, with the activation launch, its boundary and the [M, 2 I] round trip gone.  (The other
// way round - the activation in the PROLOGUE of the down projection, every workgroup recomputing the M x K activations
// it streams - measured 2 x SLOWER than the two launches: 76 vs 38 us at 1 row; the exponentials of every k-step are
// vector work the stream cannot hide.)
// `epilogue` = 2: out = max(product, 0)^2 on the fp32 sum, rounded once (the up projection of a squared-ReLU feed-forward).
// `epilogue` = 3: as 1 with the tanh form of GELU in SiLU's place, its product with the up sum rounded once (bit for bit the
// plain projection followed by sp_gelu_tanh_and_mul).
#include "sp_common.h"

namespace sp {

typedef float f32x4_g __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8_g __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_g __attribute__((ext_vector_type(8)));

template <typename Tag>
__device__ __forceinline__ f32x4_g mfma_g(const u32x4& a, const u32x4& b, const f32x4_g& c);
template <>
__device__ __forceinline__ f32x4_g mfma_g<bf16_tag>(const u32x4& a, const u32x4& b, const f32x4_g& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_g, a), __builtin_bit_cast(bf16x8_g, b),
                                                 c, 0, 0, 0);
}
template <>
__device__ __forceinline__ f32x4_g mfma_g<f16_tag>(const u32x4& a, const u32x4& b, const f32x4_g& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_g, a), __builtin_bit_cast(f16x8_g, b),
                                                c, 0, 0, 0);
}

struct SkinnyArgs {
  const char* x;
  const char* w;
  void* out;
  int M, N, K;
  int64_t x_stride, w_stride, out_stride;   // elements
};

// the value a finished sum is stored as (EPI 1 and 3 store glu_value instead)
template <int EPI>
__device__ __forceinline__ float plain_value(float s) {
  if constexpr (EPI == 2) {
    s = fmaxf(s, 0.f);
    s *= s;
  }
  return s;
}
// glu_mul_vec_kernel's arithmetic on the ROUNDED gate and up sums
template <typename Tag, int EPI>
__device__ __forceinline__ float glu_value(float gate, float up) {
  typedef Elem<Tag> E;
  const float act = EPI == 3 ? gelu_tanh_f32(E::round(gate)) : E::round(silu_ref(E::round(gate)));
  return mul_round<Tag>(act, E::round(up));
}

// ---- 1 row
constexpr int kRowWaves = 2, kRowLoads = 4;

// ONCE: weights past the L2 (launch_skinny_as has the line)
template <typename Tag, int EPI, bool ONCE>
__global__ __launch_bounds__(kRowWaves * 64) void gemm_row_kernel(SkinnyArgs a) {
  typedef Elem<Tag> E;
  constexpr bool GLU = EPI == 1 || EPI == 3;
  constexpr int R = GLU ? 2 : 1;                       // a gate row and its up row, or one row
  const int lane = threadIdx.x & 63, n = blockIdx.x * kRowWaves + (threadIdx.x >> 6);
  if (n >= a.N) return;                                // no barrier in this kernel
  const char* wp[R];
  float acc[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    wp[r] = a.w + ((int64_t)r * a.N + n) * a.w_stride * 2;
    acc[r] = 0.f;
  }
  const u32x4 zero = {0u, 0u, 0u, 0u};
  for (int k0 = 0; k0 < a.K; k0 += 512 * kRowLoads) {
    u32x4 wf[kRowLoads][R], xf[kRowLoads];
#pragma unroll
    for (int u = 0; u < kRowLoads; ++u) {
      const int k = k0 + u * 512 + lane * 8;           // K is a multiple of 8: a lane's 16 bytes are in the row or past it
      const bool in = k < a.K;
#pragma unroll
      for (int r = 0; r < R; ++r) wf[u][r] = !in ? zero : ONCE ? ld16_once(wp[r] + (int64_t)k * 2) : ld16(wp[r] + (int64_t)k * 2);
      xf[u] = in ? ld16(a.x + (int64_t)k * 2) : zero;
    }
    __builtin_amdgcn_sched_barrier(0);                 // all of them on their way before the first is waited for
#pragma unroll
    for (int u = 0; u < kRowLoads; ++u) {
      float xv[8];
      unpack16<Tag>(xf[u], xv);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        float wv[8];
        unpack16<Tag>(wf[u][r], wv);
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[r] = fmaf(wv[e], xv[e], acc[r]);
      }
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r) acc[r] = wave_sum(acc[r]);
  if (lane == 0) E::store(a.out, n, GLU ? glu_value<Tag, EPI>(acc[0], acc[R - 1]) : plain_value<EPI>(acc[0]));
}

// ---- 2-4 rows
typedef short s16x4_g __attribute__((ext_vector_type(4)));
typedef _Float16 f16x4_g __attribute__((ext_vector_type(4)));

// lane (b, i): a = weight row i, b = x row i, 8 elements of K; block b of the accumulator += rows . rows^T over those 8
template <typename Tag>
__device__ __forceinline__ f32x4_g mfma_quad(const u32x4& a, const u32x4& b, f32x4_g c) {
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const u32x2 ah = {a[2 * h], a[2 * h + 1]}, bh = {b[2 * h], b[2 * h + 1]};
    if constexpr (__is_same(Tag, bf16_tag))
      c = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(__builtin_bit_cast(s16x4_g, ah), __builtin_bit_cast(s16x4_g, bh), c, 0, 0, 0);
    else
      c = __builtin_amdgcn_mfma_f32_4x4x4f16(__builtin_bit_cast(f16x4_g, ah), __builtin_bit_cast(f16x4_g, bh), c, 0, 0, 0);
  }
  return c;
}

constexpr int kQuadWaves = 4, kQuadLoads = 4, kQuadRows = 4;

// G groups of 4 weight rows: two where there are enough of them to fill the card (x is read half as often) and for gate and up,
// else one and twice the length of K in flight.  The order of the sums is the same.
template <typename Tag, int G, int EPI, bool ONCE>
__global__ __launch_bounds__(kQuadWaves * 64) void gemm_quad_kernel(SkinnyArgs a) {
  typedef Elem<Tag> E;
  constexpr bool GLU = EPI == 1 || EPI == 3;
  static_assert(!GLU || G == 2, "gate rows and the up rows of the same columns");
  __shared__ float red[kQuadWaves][16 * G];            // [wave][group][weight row 4][x row 4]
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int b = lane >> 2, i = lane & 3;
  const int n0 = blockIdx.x * (GLU ? 4 : 4 * G);
  const char* wp[G];                                   // rows past N: row N - 1 again, computed and not stored
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const int n = GLU ? g * a.N + min(n0 + i, a.N - 1) : min(n0 + 4 * g + i, a.N - 1);
    wp[g] = a.w + ((int64_t)n * a.w_stride + 8 * b) * 2;
  }
  const bool mrow = i < a.M;
  const char* xp = a.x + ((int64_t)min(i, a.M - 1) * a.x_stride + 8 * b) * 2;
  f32x4_g acc[G];
#pragma unroll
  for (int g = 0; g < G; ++g) acc[g] = f32x4_g{0.f, 0.f, 0.f, 0.f};
  const u32x4 zero = {0u, 0u, 0u, 0u};
  constexpr int kSpan = 128 * kQuadLoads, kSpans = 2 / G;       // a wave's spans of K: wave, wave + 4, ...; kSpans at a time
  for (int k0 = wave * kSpan; k0 < a.K; k0 += kSpans * kQuadWaves * kSpan) {
    u32x4 wf[kSpans * kQuadLoads][G], xf[kSpans * kQuadLoads];
#pragma unroll
    for (int u = 0; u < kSpans * kQuadLoads; ++u) {
      const int k = k0 + (u / kQuadLoads) * kQuadWaves * kSpan + (u % kQuadLoads) * 128;
      const bool in = k + 8 * b < a.K;
#pragma unroll
      for (int g = 0; g < G; ++g) wf[u][g] = !in ? zero : ONCE ? ld16_once(wp[g] + (int64_t)k * 2) : ld16(wp[g] + (int64_t)k * 2);
      xf[u] = in && mrow ? ld16(xp + (int64_t)k * 2) : zero;
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < kSpans * kQuadLoads; ++u)
#pragma unroll
      for (int g = 0; g < G; ++g) acc[g] = mfma_quad<Tag>(wf[u][g], xf[u], acc[g]);
  }
  // lane (b, m): acc[g][r] = block b's part of out[m][row r of group g]
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float s = acc[g][r];
#pragma unroll
      for (int step = 4; step < 64; step *= 2) s += __shfl_xor(s, step);
      if (lane < 4) red[wave][(g * 4 + r) * 4 + lane] = s;
    }
  __syncthreads();
  if (threadIdx.x >= 16 * G) return;
  float s = 0.f;
#pragma unroll
  for (int w = 0; w < kQuadWaves; ++w) s += red[w][lane];
  const int m = lane & 3, r = (lane >> 2) & 3, g = lane >> 4;
  if constexpr (GLU) {
    const float up = __shfl_down(s, 16);
    if (g == 0 && m < a.M && n0 + r < a.N) E::store(a.out, (int64_t)m * a.out_stride + n0 + r, glu_value<Tag, EPI>(s, up));
  } else {
    const int n = n0 + 4 * g + r;
    if (m < a.M && n < a.N) E::store(a.out, (int64_t)m * a.out_stride + n, plain_value<EPI>(s));
  }
}

// ---- 5-16 rows
constexpr int kSkWaves = 8;

// The waves' k-steps: NEAR, a wave's loads in flight lie next to each other in K (4 of them: both halves of a 128-byte line are asked for
// by one wave), from K 2560 on; else they lie 8 steps apart and the workgroup's next to each other (8 of them), so that the waves
// share lines of x in the L1.  us at 5 / 16 rows, apart | NEAR: 4096 x 2048 6.2 / 7.5 | 7.0 / 7.9; 4608 x 1536 7.0 / 8.5 | 7.4 / 9.4;
// 1024 x 2560 5.8 / 7.0 | 5.5 / 6.9; 2048 x 3072 7.6 / 9.2 | 7.1 / 9.1; 16384 x 4096 29.2 / 39.6 | 28.7 / 38.7; 2048 x 8192 14.8 / 19.5 | 14.1 / 18.0.
// (NEAR with 8 in flight, and pairs of neighbours 8 pairs apart, are slower than one of the two everywhere.)
constexpr int kSkNearK = 2560;

// EPI 1 and 3: a.N = I output columns; the 16 W rows of a workgroup are gate rows n0 .. n0+7 (tile rows 0-7) and up rows
// I + n0 .. I + n0 + 7 (tile rows 8-15)
template <typename Tag, bool NEAR, int EPI>
__global__ __launch_bounds__(kSkWaves * 64) void gemm_skinny_kernel(SkinnyArgs a) {
  typedef Elem<Tag> E;
  constexpr int U = NEAR ? 4 : 8, STEP = NEAR ? 1 : kSkWaves;
  constexpr bool GLU = EPI == 1 || EPI == 3;
  __shared__ float red[kSkWaves][16 * 17];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int r16 = lane & 15, q = lane >> 4;            // operand row / k-quarter of the lane
  const int n0 = GLU ? blockIdx.x * 8 : blockIdx.x * 16;
  const bool mrow = r16 < a.M;
  int n = min(n0 + r16, a.N - 1);                      // clamp: columns past N are computed, never stored
  if constexpr (GLU) n = (r16 < 8 ? 0 : a.N) + min(n0 + (r16 & 7), a.N - 1);
  const char* wp = a.w + ((int64_t)n * a.w_stride + 8 * q) * 2;
  const char* xp = a.x + ((int64_t)min(r16, a.M - 1) * a.x_stride + 8 * q) * 2;
  const int ksteps = a.K / 32;
  f32x4_g acc = {0.f, 0.f, 0.f, 0.f};
  const u32x4 zero = {0u, 0u, 0u, 0u};
  // this wave's k-steps, U at a time, all loads of a group first
  for (int ks = wave * (NEAR ? U : 1); ks < ksteps; ks += U * kSkWaves) {
    u32x4 wf[U], xf[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t off = (int64_t)(ks + u * STEP) * 64;
      const bool in = ks + u * STEP < ksteps;
      wf[u] = in ? ld16(wp + off) : zero;
      xf[u] = in && mrow ? ld16(xp + off) : zero;
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < U; ++u) acc = mfma_g<Tag>(wf[u], xf[u], acc);
  }
  // acc[r] = partial of out[m = r16][n0 + 4q + r]; sum the waves in wave order
#pragma unroll
  for (int r = 0; r < 4; ++r) red[wave][(4 * q + r) * 17 + r16] = acc[r];
  __syncthreads();
  if (wave != 0) return;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int col = 4 * q + r;
    float s = 0.f;
#pragma unroll
    for (int w = 0; w < kSkWaves; ++w) s += red[w][col * 17 + r16];
    const int no = n0 + col;
    if constexpr (GLU) {
      // tile columns 0-7 are gate sums, 8-15 the up sums of the same output columns: the lanes of the gate half finish both
      // (same summation order as above)
      float su = 0.f;
#pragma unroll
      for (int w = 0; w < kSkWaves; ++w) su += red[w][((col & 7) + 8) * 17 + r16];
      if (mrow && q < 2 && no < a.N) E::store(a.out, (int64_t)r16 * a.out_stride + no, glu_value<Tag, EPI>(s, su));
    } else if (mrow && no < a.N) {
      E::store(a.out, (int64_t)r16 * a.out_stride + no, plain_value<EPI>(s));
    }
  }
}

// One group of 4 weight rows up to 2048 rows: 256 workgroups of two groups there (3 rows, K 4096, us: 1024 rows 4.6 one / 6.3 two,
// 2048 rows 6.3 / 6.9, 2560 rows 7.8 / 8.9, 8192 rows 16.0 / 14.6).
constexpr int kQuadOneGroup = 2048;
// Where 2-4 rows go to the tiles of 16 weight rows (us at 4 rows, groups of 4 / tiles): a short K, and more rows than one group takes while
// they are too few for two groups to fill the card (512 x 512 2.8 / 2.7; K 1536: 2560 4.9 / 4.9, 4096 5.6 / 5.2, 8192 8.2 / 7.2, 28672 19.2 /
// 19.5; K 2048: 3072 6.3 / 5.8, 4096 7.0 / 6.2, 4608 8.1 / 8.5, 16384 15.7 / 15.9; K 4096: 2048 7.4 / 8.3, 2560 9.7 / 8.8, 4096 10.3 / 10.1,
// 4608 12.7 / 14.7; K 8192: 3072 16.1 / 15.2; 2 rows there 14.2 / 14.6).
static bool few_take_tiles(int M, int64_t rows, int K) {
  if (K <= 512) return true;
  return rows > kQuadOneGroup && (K <= 1536 || (rows <= 4096 && (M > 2 || K <= 4096)));
}

// Weights past the L2, in elements: at 1 row from what the eight L2s hold together on (32 MB), at 2 - 4 rows, which read less of a row at
// a time, from half the last-level cache on.  us, kept / past it, 1 row, of weights out of HBM: 4096 x 4096 8.2 / 7.6, 2048 x 8192
// 8.3 / 7.7, 16384 x 2048 with the activation 13.6 / 12.3, 28672 x 4096 38.7 / 35.9, 128256 x 2048 86 / 78; out of the last-level cache (2
// weights in turn) 4096 x 4096 7.1 / 7.0, 16384 x 2048 11.2 / 11.1; below the line 3072 x 2048 4.2 / 4.2 and, out of the L2, 2.9 / 3.5.  2 rows:
// 28672 x 4096 41.1 / 38.6, 128256 x 2048 88 / 80; 16384 x 2048 14.3 / 14.0, but 12.5 / 13.6 out of the last-level cache.  (The tiles of 5 -
// 16 rows read half a line at a time: 28672 x 4096 47 / 54.)
constexpr int64_t kRowOnce = 1 << 24, kQuadOnce = 1 << 26;

template <typename Tag, int EPI>
static void launch_skinny_as(const SkinnyArgs& a, hipStream_t st) {
  constexpr bool GLU = EPI == 1 || EPI == 3;
  const int64_t elements = (GLU ? 2 : 1) * (int64_t)a.N * a.K;
  if (a.M == 1) {
    const dim3 grid((a.N + kRowWaves - 1) / kRowWaves), block(kRowWaves * 64);
    if (elements >= kRowOnce) gemm_row_kernel<Tag, EPI, true><<<grid, block, 0, st>>>(a);
    else gemm_row_kernel<Tag, EPI, false><<<grid, block, 0, st>>>(a);
  } else if (a.M <= kQuadRows && !few_take_tiles(a.M, GLU ? 2 * (int64_t)a.N : a.N, a.K)) {
    if (!GLU && a.N <= kQuadOneGroup) {
      if constexpr (!GLU) gemm_quad_kernel<Tag, 1, EPI, false><<<dim3((a.N + 3) / 4), dim3(kQuadWaves * 64), 0, st>>>(a);
    } else {
      constexpr int cols = GLU ? 4 : 8;
      const dim3 grid((a.N + cols - 1) / cols), block(kQuadWaves * 64);
      if (elements >= kQuadOnce) gemm_quad_kernel<Tag, 2, EPI, true><<<grid, block, 0, st>>>(a);
      else gemm_quad_kernel<Tag, 2, EPI, false><<<grid, block, 0, st>>>(a);
    }
  } else {
    constexpr int cols = GLU ? 8 : 16;
    const dim3 grid((a.N + cols - 1) / cols), block(kSkWaves * 64);
    if (a.K >= kSkNearK) gemm_skinny_kernel<Tag, true, EPI><<<grid, block, 0, st>>>(a);
    else gemm_skinny_kernel<Tag, false, EPI><<<grid, block, 0, st>>>(a);
  }
}

template <typename Tag>
static void launch_skinny(const SkinnyArgs& a, int epilogue, hipStream_t st) {
  if (epilogue == 1) launch_skinny_as<Tag, 1>(a, st);
  else if (epilogue == 2) launch_skinny_as<Tag, 2>(a, st);
  else if (epilogue == 3) launch_skinny_as<Tag, 3>(a, st);
  else launch_skinny_as<Tag, 0>(a, st);
}

}  // namespace sp

extern "C" int sp_gemm_skinny(void* out, const void* x, const void* w, int M, int N, int K, int64_t x_stride,
                              int64_t w_stride, int64_t out_stride, int epilogue, int dtype, void* stream) {
  SP_CHECK_ARG(M >= 0 && N >= 0 && K > 0 && epilogue >= 0 && epilogue <= 3);
  if (M == 0 || N == 0) return SP_OK;
  SP_CHECK_ARG(out && x && w);
  if (M > 16 || K % 32 != 0) return SP_ERR_UNSUPPORTED;
  if (dtype != SP_BF16 && dtype != SP_F16) return SP_ERR_UNSUPPORTED;
  SP_CHECK_ARG(x_stride % 8 == 0 && w_stride % 8 == 0 && x_stride >= K && w_stride >= K && out_stride >= N);
  SP_CHECK_ARG(((uintptr_t)x & 15) == 0 && ((uintptr_t)w & 15) == 0);
  sp::SkinnyArgs a{(const char*)x, (const char*)w, out, M, N, K, x_stride, w_stride, out_stride};
  if (dtype == SP_BF16) sp::launch_skinny<sp::bf16_tag>(a, epilogue, (hipStream_t)stream);
  else sp::launch_skinny<sp::f16_tag>(a, epilogue, (hipStream_t)stream);
  SP_LAUNCH_CHECK();
  return SP_OK;
}
