// Delta-rule recurrences with a decay per key channel (or per head), 16 tokens at a time on the matrix cores: fp32 products, or those of
// three bf16 parts of each operand (below: which, and why).
//
//   S = diag(w_t) S;   u_t = beta_t (v_t - S^T k_t);   S = S + k_t u_t^T;   o_t = S^T q_t        (k, q of the token, S [D, Dv])
//
// Over a chunk that starts from S_0, with G_t the product of the decays w_1 .. w_t per channel:
//   Kd_t = k_t G_t,  Qd_t = q_t G_t,  Ke_s = k_s (w_{s+1} ... w_16)                              (rows of D)
//   A_ts = beta_t sum_d k_td k_sd (w_{s+1} ... w_t)_d  (s < t),   P_ts = sum_d q_td k_sd (w_{s+1} ... w_t)_d  (s <= t)
//   U = (I + A)^{-1} diag(beta) (V - Kd S_0),   O = Qd S_0 + P U,   S_16 = diag(G_16) S_0 + Ke^T U
// so the serial chain is one step of matrix products per 16 tokens.  Every factor is a product of decays, never a quotient: with
// decays in [0, 1] nothing overflows however strong they are.
//
// What does not read the state - A, its inverse, P and the norms of q and k - is formed for all chunks at once
// (delta_chunk_prepare_kernel, a wave per chunk and head).  delta_chunk_scan_kernel then walks a request's chunks: a wave owns 16
// columns of S in the accumulator layout of v_mfma_f32_16x16x4_f32 (lane (r16, q): column r16, rows 16 i + 4 q + r), in which the
// register (i, r) IS the second operand of Kd S and Qd S for the channels 16 i + 4 q + r, and a product's four registers are the
// second operand of the next one over tokens: the waves of a head share operands through LDS and exchange nothing.  The read-outs
// go to fp32 rows that a last kernel norms over the head and gates.
//
// fp32 MFMAs: 64 multiply-adds per cycle and SIMD against 16 for fp32 vector code, whose sums over a column's lanes and LDS reads
// per token left the per-token kernels at a quarter of that.  16 heads of 128 x 128 with a decay per channel: 8 requests of 4096
// tokens together 682 -> 183 us (49 of them the preparation, 21 norm and gate), one request of 4096 tokens 4258 -> 725, 16 requests
// of 300 tokens 45 -> 33; since then the preparation sums eight values at a time over the lanes and takes 30 us in place of 49 - 53.  With one decay per head: 8 requests 364 -> 179, one request 2101 -> 672, 16 requests of 300 tokens 41 -> 33.
// Short portions are the per-token kernels': the callers' rules have the lines and both sides.
//
// A u that is not finite would reach the EARLIER tokens of its chunk too (zeros of (I + A)^{-1} and P times it): where a column has
// one, its read-outs are formed again without the rows from the first such token on, which become NaN, as does the column's state.
#pragma once
#include "seq_batch.h"

#include <type_traits>

namespace sp {

typedef float f32x4_d __attribute__((ext_vector_type(4)));
constexpr int kDC = 16;                               // tokens per chunk
// of a chunk and head, prepared: U's matrix (I + A)^{-1} diag(beta) and P (row major), 1 / |k|, D^(-1/2) / |q|, head decay
constexpr int kDcT = 0, kDcP = 256, kDcIk = 512, kDcIq = 528, kDcW = 544, kDcFloats = 560;

struct DeltaChunks {
  const void *q, *k, *v, *bpre;
  const float* decay;                                 // CHANNEL: [T, H * D]
  const float *pre, *dt_bias, *A_log;                 // per head: pre [T, >= 2 H] (step sizes, then decays)
  float *state, *work, *raw;                          // work [chunks, H, kDcFloats], raw [T, H * Dv]
  int64_t q_stride, k_stride, v_stride, b_stride, pre_stride, state_stride;
  int64_t T;
  int H, G, Dv, cols;                                 // cols: columns of a head per workgroup
};

__device__ __forceinline__ float softplus_dc(float z) { return fmaxf(z, 0.f) + log1pf(expf(-fabsf(z))); }

template <int N>
__device__ __forceinline__ float group_sum_dc(float v) {
  v = lanes_sum<(N < 16 ? N : 16)>(v);
  if constexpr (N >= 32) v += __shfl_xor(v, 16, 64);
  if constexpr (N >= 64) v += __shfl_xor(v, 32, 64);
  return v;
}

// chunks of the requests before `b` (one request per lane and round); all lanes get the sum
__device__ __forceinline__ int chunks_before(const SeqBatch& s, int b, int lane) {
  int n = 0;
  for (int i = lane; i < b; i += 64) n += (s.extend_seq_lens[i] + kDC - 1) / kDC;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) n += __shfl_xor(n, off, 64);
  return n;
}
// the request and first token (within it) of chunk `id`; false behind the last
__device__ __forceinline__ bool chunk_at(const SeqBatch& s, int id, int lane, int& b, int& t0) {
  for (int b0 = 0; b0 < s.B; b0 += 64) {
    const int i = b0 + lane;
    const int n = i < s.B ? (s.extend_seq_lens[i] + kDC - 1) / kDC : 0;
    int incl = n;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int o = __shfl_up(incl, off, 64);
      if (lane >= off) incl += o;
    }
    const uint64_t hit = __ballot(id < incl);
    if (hit) {
      const int l = __ffsll((unsigned long long)hit) - 1;
      b = __builtin_amdgcn_readfirstlane(b0 + l);
      t0 = __builtin_amdgcn_readfirstlane((id - __shfl(incl - n, l, 64)) * kDC);
      return true;
    }
    id -= __builtin_amdgcn_readfirstlane(__shfl(incl, 63, 64));
  }
  return false;
}

// One workgroup per (chunk, head), a wave per 32 channels.  A lane sums two columns s of A and P over 4 channels; the decays
// between s and t build up as t walks on, k, q and w of a token are broadcast reads of LDS that serve both columns.  (One wave for
// all channels left a CU with five waves, one LDS read in flight each: 50 us for 264 chunks of 16 heads.)
template <typename Tag, int D, bool CHANNEL>
__global__ void __launch_bounds__(D * 2) delta_chunk_prepare_kernel(DeltaChunks a, SeqBatch sb) {
  typedef Elem<Tag> E;
  constexpr int V = E::kVec, QP = D / V, ROW = D + 4, NW = D / 32, NT = 64 * NW;
  __shared__ __attribute__((aligned(16))) float sk[kDC][ROW], sq[kDC][ROW], sw[CHANNEL ? kDC : 1][ROW], sA[kDC][kDC + 4];
  __shared__ float sbeta[kDC], sdec[kDC];
  static_assert(NW * kDC * (kDC + 1) <= kDC * ROW, "the waves' sums take the place of the rows");
  float(*skk)[kDC][kDC + 1] = (float(*)[kDC][kDC + 1])&sk[0][0];
  float(*sqk)[kDC][kDC + 1] = (float(*)[kDC][kDC + 1])&sq[0][0];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, h = blockIdx.y;
  int b, c0;
  if (!chunk_at(sb, (int)blockIdx.x, lane, b, c0)) return;
  const int64_t row0 = (int64_t)sb.extend_start_loc[b] + c0;
  const int len = sb.extend_seq_lens[b] - c0, n = len < kDC ? len : kDC;
  float* work = a.work + ((int64_t)blockIdx.x * a.H + h) * kDcFloats;
  const int64_t qc = (int64_t)(h / (a.H / a.G)) * D;
  const float qscale = 1.f / sqrtf((float)D);
  // unit rows (zeros behind the request's end), QP lanes per row
  for (int e = tid; e < kDC * QP; e += NT) {
    const int t = e / QP, i = e % QP * V;
    float kf[V], qf[V], k2 = 0.f, q2 = 0.f;
    const u32x4 zero = {0u, 0u, 0u, 0u};
    unpack16<Tag>(t < n ? ld16((const char*)a.k + ((row0 + t) * a.k_stride + qc + i) * E::kBytes) : zero, kf);
    unpack16<Tag>(t < n ? ld16((const char*)a.q + ((row0 + t) * a.q_stride + qc + i) * E::kBytes) : zero, qf);
#pragma unroll
    for (int x = 0; x < V; ++x) {
      k2 += kf[x] * kf[x];
      q2 += qf[x] * qf[x];
    }
    const float ik = 1.f / sqrtf(group_sum_dc<QP>(k2) + 1e-6f), iq = qscale / sqrtf(group_sum_dc<QP>(q2) + 1e-6f);
#pragma unroll
    for (int x = 0; x < V; x += 4) {
      *(f32x4_d*)&sk[t][i + x] = f32x4_d{kf[x] * ik, kf[x + 1] * ik, kf[x + 2] * ik, kf[x + 3] * ik};
      *(f32x4_d*)&sq[t][i + x] = f32x4_d{qf[x] * iq, qf[x + 1] * iq, qf[x + 2] * iq, qf[x + 3] * iq};
    }
    if (e % QP == 0) {
      work[kDcIk + t] = ik;
      work[kDcIq + t] = iq;
    }
  }
  if constexpr (CHANNEL) {
    for (int e = tid * 4; e < kDC * D; e += 4 * NT) {
      const int t = e / D, i = e % D;
      *(f32x4_d*)&sw[t][i] = t < n ? *(const f32x4_d*)(a.decay + (row0 + t) * a.H * D + (int64_t)h * D + i) : f32x4_d{1.f, 1.f, 1.f, 1.f};
    }
  }
  if (tid < kDC) {
    float beta = 0.f, dec = 1.f;
    if (tid < n) {
      if constexpr (CHANNEL) {
        beta = over_one_plus_exp(1.f, E::load(a.bpre, (row0 + tid) * a.b_stride + h));
      } else {
        const float* pre = a.pre + (row0 + tid) * a.pre_stride;
        beta = over_one_plus_exp(1.f, pre[h]);
        dec = expf(-expf(a.A_log[h]) * softplus_dc(pre[a.H + h] + a.dt_bias[h]));
      }
    }
    sbeta[tid] = beta;
    sdec[tid] = dec;
    if constexpr (!CHANNEL) work[kDcW + tid] = dec;
  }
  __syncthreads();
  // lane (s0, part): columns s0 and s0 + 8 over 4 channels; only rows t >= 8 matter to the second
  const int s0 = lane & 7, part = lane >> 3, i = wave * 32 + part * 4;
  f32x4_d rat = *(const f32x4_d*)&sk[s0][i], rat8 = *(const f32x4_d*)&sk[s0 + 8][i];
  float kks[2][2], qks[2][2];                         // [half][column]: of token 8 half + part
#pragma unroll
  for (int half = 0; half < 2; ++half) {
    float kk[2][8], qk[2][8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int t = 8 * half + u;
      const f32x4_d kt = *(const f32x4_d*)&sk[t][i], qt = *(const f32x4_d*)&sq[t][i];
      if constexpr (CHANNEL) {
        const f32x4_d wt = *(const f32x4_d*)&sw[t][i];
#pragma unroll
        for (int x = 0; x < 4; ++x) rat[x] *= t >= 8 || t > s0 ? wt[x] : 1.f;
        if (t > 8) {
#pragma unroll
          for (int x = 0; x < 4; ++x) rat8[x] *= t > s0 + 8 ? wt[x] : 1.f;
        }
      }
      // (t < s: a number that nobody reads)
      kk[0][u] = (kt[0] * rat[0] + kt[1] * rat[1]) + (kt[2] * rat[2] + kt[3] * rat[3]);
      qk[0][u] = (qt[0] * rat[0] + qt[1] * rat[1]) + (qt[2] * rat[2] + qt[3] * rat[3]);
      kk[1][u] = (kt[0] * rat8[0] + kt[1] * rat8[1]) + (kt[2] * rat8[2] + kt[3] * rat8[3]);
      qk[1][u] = (qt[0] * rat8[0] + qt[1] * rat8[1]) + (qt[2] * rat8[2] + qt[3] * rat8[3]);
    }
#pragma unroll
    for (int z = 0; z < 2; ++z) {
      kks[half][z] = z <= half ? eight_sums(kk[z], lane) : 0.f;
      qks[half][z] = z <= half ? eight_sums(qk[z], lane) : 0.f;
    }
  }
  __syncthreads();                                    // every wave is done with the rows
#pragma unroll
  for (int half = 0; half < 2; ++half)
#pragma unroll
    for (int z = 0; z < 2; ++z) {
      skk[wave][8 * half + part][s0 + 8 * z] = kks[half][z];
      sqk[wave][8 * half + part][s0 + 8 * z] = qks[half][z];
    }
  __syncthreads();
  for (int e = tid; e < kDC * kDC; e += NT) {
    const int t = e / kDC, s = e % kDC;
    float kk = 0.f, qk = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      kk += skk[w][t][s];
      qk += sqk[w][t][s];
    }
    if constexpr (!CHANNEL) {                         // the decays between s and t as one factor
      float run = 1.f;
      for (int j = s + 1; j <= t; ++j) run *= sdec[j];
      kk *= run;
      qk *= run;
    }
    sA[t][s] = t > s ? sbeta[t] * kk : 0.f;
    work[kDcP + e] = t >= s ? qk : 0.f;
  }
  __syncthreads();
  if (wave > 0) return;
  // column s of (I + A)^{-1}: forward substitution
  const int s = lane & 15;
  float x[kDC];
#pragma unroll
  for (int t = 0; t < kDC; ++t) {
    float y = t == s ? 1.f : 0.f;
#pragma unroll
    for (int j = 0; j < t; ++j) y -= sA[t][j] * x[j];
    x[t] = y;
    if (lane < kDC) work[kDcT + t * kDC + s] = t >= s ? y * sbeta[s] : 0.f;      // (a step size that is not finite: zeros stay)
  }
}

__device__ __forceinline__ f32x4_d mfma_d(float a, float b, const f32x4_d& c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

typedef __bf16 bf16x8_d __attribute__((ext_vector_type(8)));
__device__ __forceinline__ f32x4_d mfma_parts(const u32x4& a, const u32x4& b, const f32x4_d& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_d, a), __builtin_bit_cast(bf16x8_d, b), c, 0, 0, 0);
}
// two fp32 values as three pairs of bf16 whose sums they are: the upper 16 bits (which cannot overflow), then what is left, rounded, then
// what is left of that (8 bits at the most: exact).  Not finite: the second part is NaN.
struct Parts {
  uint32_t p[3];
};
__device__ __forceinline__ Parts parts_of(float x, float y) {
  const auto pair = [](float a, float b) {
    bf16x2_t v;
    v[0] = (__bf16)a, v[1] = (__bf16)b;
    return __builtin_bit_cast(uint32_t, v);
  };
  const uint32_t xh = as_u32(x) & 0xffff0000u, yh = as_u32(y) & 0xffff0000u;
  x -= as_f32(xh), y -= as_f32(yh);
  const uint32_t mid = pair(x, y);
  return Parts{{__builtin_amdgcn_perm(yh, xh, 0x07060302u), mid, pair(x - as_f32(mid << 16), y - as_f32(mid & 0xffff0000u))}};
}

// One workgroup per (request, head, range of the head's columns): a wave per 16 columns runs the products of chunk c while
// kDcHelpers more waves form the operand rows of a chunk ahead and have those of the two chunks after it on their way into LDS; they
// meet at one barrier per chunk.  (The same waves doing both in turn left the matrix cores idle for two thirds of a chunk: 4.4 us.)
// With fp32 products (kParts false) a chunk is bound by the issue of vector and matrix instructions together: a fp32 matrix instruction keeps the
// vector unit for its 32 cycles, so its 104 (3380 of 5800 cycles) and every address, decay and conversion of both kinds of waves add up.  Hence
// rows by pointers that move on by a step, and masks in a request's last chunk alone.  Operands two chunks
// ahead, helpers ahead of the products in the issue, and stores behind the loads that are waited for gave nothing: the sum stays.
// bf16 products run beside vector work, so heads of 128 by ranges of 64 columns (kParts) take the products with S, and Ke^T U, as eight products of
// parts with 8 bits each: 96 instructions of 16 cycles in the place of 96 of 32, for 280 more of the vector unit.  The one left out, of both last
// parts, is at most 2^-32 of the whole.  (Without the two of a second and a last part as well, up to 2^-22 is left out where mantissas lie just below a
// cut, and a sum that one channel makes up is four times as far from 64 bits as fp32's; 25 us of the layers below.)  bf16 ends at 2^-133 where fp32
// ends at 2^-149: of states below 2^-109 the last part is cut there (300 tokens of values around 2^-120: 7e-5 of them, 1.3e-7 down to 2^-105).
// The helpers' chain is then about as long, so each takes a quarter of the tokens (K, Q and Ke as a wave each: 4900 cycles).
// us a chunk, one request of 4096 tokens, 16 heads of 128: decay per channel 2.44 -> 1.96, per head 2.2 -> 1.79 (the layers 855 -> 733 and 823 -> 717, 797 and
// 767 with fp32 products; of 8 requests 334 -> 316 and 333 -> 314, 323 and 320).  128 columns a workgroup, which many requests take, keep fp32: the parts do not fit 168
// registers (16 requests of 125 tokens 212 and 243 us), nor two workgroups a unit of heads of 64.
// S and the read-outs are otherwise no further from 64 bits than with fp32 products (S of those tokens 1.26e-7, 1.37e-7 with fp32).
constexpr int kDcHelpers = 4;

// COLS: columns of a workgroup at the most
template <typename Tag, int D, bool CHANNEL, int COLS>
struct DeltaScanLds {
  // heads of 128 by ranges of 64 columns: operands in three bf16 parts
  static constexpr bool kParts = D == 128 && COLS <= 64;
  static constexpr int kRow = D + 4;                                                     // floats per operand row
  static constexpr int kRaw = kDC * D * (2 * Elem<Tag>::kBytes + (CHANNEL ? 4 : 0));     // a chunk's k, q (and decay) rows
  // kParts: Kd and Qd three parts of 16 rows each, channels in the order that a lane takes them; Ke of a channel three parts of 16 tokens; G_end
  static constexpr int kPartRow = 2 * D + 16, kPart = kDC * kPartRow, kKe = 6 * kPart, kKeRow = 6 * kDC + 8, kG = kKe + D * kKeRow;
  static constexpr int kOps = kParts ? kG + 4 * D : (3 * kDC * kRow + D) * 4;            // Kd, Qd, Ke, G_end
  static constexpr int kOp = 3 * kRaw, kWork = kOp + 2 * kOps, kBytes = kWork + 4 * kDcFloats * 4;
  static constexpr int kWaves = (COLS / 16 + kDcHelpers) / 4 * (COLS <= 64 && kBytes <= 80 * 1024 ? 2 : 1);      // per SIMD
  static_assert(kBytes <= 160 * 1024, "LDS");
};

template <typename Tag, int D, bool CHANNEL, int COLS>
__global__ void __launch_bounds__(COLS * 4 + kDcHelpers * 64, (DeltaScanLds<Tag, D, CHANNEL, COLS>::kWaves)) delta_chunk_scan_kernel(DeltaChunks a, SeqBatch sb) {
  typedef Elem<Tag> E;
  typedef DeltaScanLds<Tag, D, CHANNEL, COLS> L;
  constexpr int DT = D / 16, ROW = L::kRow, kRowBytes = D * E::kBytes, HT = kDcHelpers * 64;
  extern __shared__ __attribute__((aligned(16))) char delta_lds[];
  const int tid = threadIdx.x, waves = a.cols / 16;    // the first `waves` waves own columns
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, r16 = lane & 15, q = lane >> 4;
  const int b = blockIdx.x, h = blockIdx.y;
  const int len = __builtin_amdgcn_readfirstlane(sb.extend_seq_lens[b]);
  if (len <= 0) return;
  const int64_t start = __builtin_amdgcn_readfirstlane(sb.extend_start_loc[b]);
  const int64_t qc = (int64_t)(h / (a.H / a.G)) * D;
  const int chunks = (len + kDC - 1) / kDC;
  if (wave >= waves) {
    const int ht = tid - 64 * waves, hw = wave - waves;
    const float* work = a.work + ((int64_t)chunks_before(sb, b, lane) * a.H + h) * kDcFloats;
    // a chunk's rows and prepared matrices, straight into LDS: 1 KiB per wave and load (rows past the end repeat the last one)
    constexpr int LK = kDC * kRowBytes / 1024, LW = CHANNEL ? kDC * D * 4 / 1024 : 0, LM = (kDcFloats * 4 + 1023) / 1024;
    const auto load = [&](const char* src, char* dst) {
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                       (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
    };
    constexpr int KU = (LK + kDcHelpers - 1) / kDcHelpers, WU = CHANNEL ? (LW + kDcHelpers - 1) / kDcHelpers : 1;
    const char *kp[KU], *qp[KU], *wp[WU], *mp = (const char*)work + hw * 1024 + lane * 16;
    const auto point = [&](int c, int last) {           // at chunk c, rows behind `last` as that one again
      const int64_t row0 = start + c * kDC;
#pragma unroll
      for (int i = 0; i < KU; ++i) {
        const int byte = (hw + i * kDcHelpers) * 1024 + lane * 16, t = byte / kRowBytes, x = byte % kRowBytes;
        const int64_t row = row0 + (t < last ? t : last);
        kp[i] = (const char*)a.k + (row * a.k_stride + qc) * E::kBytes + x;
        qp[i] = (const char*)a.q + (row * a.q_stride + qc) * E::kBytes + x;
      }
#pragma unroll
      for (int i = 0; CHANNEL && i < WU; ++i) {
        const int byte = (hw + i * kDcHelpers) * 1024 + lane * 16, t = byte / (D * 4), x = byte % (D * 4);
        const int64_t row = row0 + (t < last ? t : last);
        wp[i] = (const char*)(a.decay + row * a.H * D + (int64_t)h * D) + x;
      }
    };
    const int64_t kstep = kDC * a.k_stride * E::kBytes, qstep = kDC * a.q_stride * E::kBytes, wstep = (int64_t)kDC * a.H * D * 4,
                  mstep = (int64_t)a.H * kDcFloats * 4;
    static_assert(kDcFloats * 4 <= kDcHelpers * 1024, "one load of the matrices per helper");
    const auto fetch = [&](int c) {                    // (c = 0, 1, 2 ...)
      if (c >= chunks) return;
      char* raw = delta_lds + c % 3 * L::kRaw;
      if (c == chunks - 1) point(c, len - c * kDC - 1);
#pragma unroll
      for (int i = 0; i < KU; ++i) {
        const int u = hw + i * kDcHelpers;
        if (u < LK) {
          load(kp[i], raw + u * 1024);
          load(qp[i], raw + (LK + u) * 1024);
        }
        kp[i] += kstep, qp[i] += qstep;
      }
#pragma unroll
      for (int i = 0; CHANNEL && i < WU; ++i) {
        const int u = hw + i * kDcHelpers;
        if (u < LW) load(wp[i], raw + (2 * LK + u) * 1024);
        wp[i] += wstep;
      }
      if (hw * 1024 + lane * 16 < kDcFloats * 4) load(mp, delta_lds + L::kWork + (c & 3) * kDcFloats * 4 + hw * 1024);
      mp += mstep;
    };
    point(0, kDC);
    // operand rows of a chunk: a thread walks a channel forward (Kd, Qd, G_end) or backward (Ke); rows behind the end are zeros.  Rows
    // become unit rows here and not in the products, where their lengths would be fewer multiplications (12 of a wave for 48 of a
    // channel's two threads): a product with a row that is not of unit length can be past fp32 where the state is not, and zeros have a factor of 1000.
    const auto operands = [&](int c, auto whole) {
      const int n = len - c * kDC;
      const char* raw = delta_lds + c % 3 * L::kRaw;
      const float* wr = (const float*)(raw + 2 * kDC * kRowBytes);
      const float* m = (const float*)(delta_lds + L::kWork + (c & 3) * kDcFloats * 4);
      float* ops = (float*)(delta_lds + L::kOp + (c & 1) * L::kOps);
      for (int role = ht; role < 2 * D; role += HT) {
        const int d = role < D ? role : role - D;
        const bool fwd = role < D;                     // (D is a multiple of 64: whole waves)
        typename E::storage kr[kDC], qr[kDC];
        float w[kDC];
        f32x4_d ik[kDC / 4], iq[kDC / 4];
#pragma unroll
        for (int t = 0; t < kDC; ++t) {                // every read on its way before the first is used
          w[t] = CHANNEL ? wr[t * D + d] : m[kDcW + t];
          kr[t] = ((const typename E::storage*)raw)[t * D + d];
          qr[t] = ((const typename E::storage*)(raw + (fwd ? kDC * kRowBytes : 0)))[t * D + d];
        }
#pragma unroll
        for (int x = 0; x < kDC / 4; ++x) {
          ik[x] = *(const f32x4_d*)&m[kDcIk + 4 * x];
          iq[x] = *(const f32x4_d*)&m[kDcIq + 4 * x];
        }
        __builtin_amdgcn_sched_barrier(0);
        float k[kDC];
#pragma unroll
        for (int t = 0; t < kDC; ++t) {
          const bool on = whole || t < n;
          if (!on) w[t] = 1.f;
          k[t] = on ? E::load(&kr[t], 0) * ik[t / 4][t % 4] : 0.f;
        }
        float g = 1.f;
        if (fwd) {
#pragma unroll
          for (int t = 0; t < kDC; ++t) {
            g *= w[t];
            ops[t * ROW + d] = k[t] * g;
            ops[(kDC + t) * ROW + d] = whole || t < n ? E::load(&qr[t], 0) * iq[t / 4][t % 4] * g : 0.f;
          }
          ops[3 * kDC * ROW + d] = g;
        } else {
#pragma unroll
          for (int t = kDC - 1; t >= 0; --t) {
            ops[(2 * kDC + t) * ROW + d] = k[t] * g;
            g *= w[t];
          }
        }
      }
    };
    // kParts: a helper takes four tokens of every chunk, a thread two channels - the decays in front of them for Kd and Qd (and G_end), those
    // behind them for Ke
    struct __attribute__((aligned(2 * E::kBytes))) Two {
      typename E::storage x[2];
    };
    typedef float f32x2_d __attribute__((ext_vector_type(2)));
    const auto parts = [&](int c, auto whole) {
      const int n = len - c * kDC, d = 2 * lane, t0 = 4 * hw;
      const char* raw = delta_lds + c % 3 * L::kRaw;
      const float* wr = (const float*)(raw + 2 * kDC * kRowBytes);
      const float* m = (const float*)(delta_lds + L::kWork + (c & 3) * kDcFloats * 4);
      char* ops = delta_lds + L::kOp + (c & 1) * L::kOps;
      f32x2_d w[kDC];
      Two kr[4], qr[4];
#pragma unroll
      for (int t = 0; t < kDC; ++t) w[t] = CHANNEL ? *(const f32x2_d*)&wr[t * D + d] : f32x2_d{m[kDcW + t], m[kDcW + t]};
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        kr[x] = *(const Two*)(raw + (t0 + x) * kRowBytes + d * E::kBytes);
        qr[x] = *(const Two*)(raw + (kDC + t0 + x) * kRowBytes + d * E::kBytes);
      }
      const f32x4_d ik = *(const f32x4_d*)&m[kDcIk + t0], iq = *(const f32x4_d*)&m[kDcIq + t0];
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (!decltype(whole)::value) {
#pragma unroll
        for (int t = 0; t < kDC; ++t)
          if (t >= n) w[t] = f32x2_d{1.f, 1.f};
      }
      float y[3][4][2];                                // k, q, and k backward
#pragma unroll
      for (int x = 0; x < 4; ++x)
#pragma unroll
        for (int ch = 0; ch < 2; ++ch) {
          const bool on = whole || t0 + x < n;
          y[0][x][ch] = y[2][x][ch] = on ? E::load(kr[x].x, ch) * ik[x] : 0.f;
          y[1][x][ch] = on ? E::load(qr[x].x, ch) * iq[x] : 0.f;
        }
#pragma unroll
      for (int part = 0; part < kDcHelpers; ++part) {  // (hw is the wave's: one of four)
        if (hw != part) continue;
#pragma unroll
        for (int ch = 0; ch < 2; ++ch) {
          float g = 1.f, back = 1.f;
#pragma unroll
          for (int t = 0; t < 4 * part + 4; ++t) {
            g *= w[t][ch];
            if (t >= 4 * part) y[0][t - 4 * part][ch] *= g, y[1][t - 4 * part][ch] *= g;
          }
#pragma unroll
          for (int t = kDC - 1; t >= 4 * part; --t) {
            if (t < 4 * part + 4) y[2][t - 4 * part][ch] *= back;
            back *= w[t][ch];
          }
          if (part == kDcHelpers - 1) *(float*)(ops + L::kG + (d + ch) * 4) = g;
        }
      }
      // channels 4 q + r and 16 + 4 q + r of every 32 are a lane's eight
      char* rows = ops + t0 * L::kPartRow + (d / 32 * 32 + d % 16 / 4 * 8 + d % 32 / 16 * 4 + d % 4) * 2;
#pragma unroll
      for (int x = 0; x < 4; ++x)
#pragma unroll
        for (int which = 0; which < 2; ++which) {
          const Parts z = parts_of(y[which][x][0], y[which][x][1]);
#pragma unroll
          for (int i = 0; i < 3; ++i) *(uint32_t*)(rows + (3 * which + i) * L::kPart + x * L::kPartRow) = z.p[i];
        }
#pragma unroll
      for (int ch = 0; ch < 2; ++ch) {
        const Parts lo = parts_of(y[2][0][ch], y[2][1][ch]), hi = parts_of(y[2][2][ch], y[2][3][ch]);
#pragma unroll
        for (int i = 0; i < 3; ++i) *(u32x2*)(ops + L::kKe + (d + ch) * L::kKeRow + i * 2 * kDC + t0 * 2) = u32x2{lo.p[i], hi.p[i]};
      }
    };
    const auto form = [&](int c) {
      if (c >= chunks) return;
      const auto with = [&](auto whole) {
        if constexpr (L::kParts) parts(c, whole);
        else operands(c, whole);
      };
      if (len - c * kDC >= kDC) with(std::true_type());
      else with(std::false_type());
    };
    // loads of one fetch that every helper issues at the least: waiting for all but so many is waiting for the fetch before it
    constexpr int kLoads = 2 * (LK / kDcHelpers) + LW / kDcHelpers + LM / kDcHelpers;
    fetch(0);
    fetch(1);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    lds_barrier();
    fetch(2);
    form(0);
    lds_barrier();
    for (int c = 0; c < chunks; ++c) {
      fetch(c + 3);                                    // (over the rows of chunk c, whose operands are formed)
      form(c + 1);
      if (c + 3 < chunks) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kLoads) : "memory");
      else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      lds_barrier();                                   // the rows of chunk c + 2 have landed
    }
    return;
  }
  const bool held = sb.extend_prefix_lens[b] > 0;
  const int64_t slot = load_idx(sb.req_pool_indices, b, sb.idx64);
  const int col = blockIdx.z * a.cols + 16 * wave + r16;
  const bool live = __builtin_amdgcn_readfirstlane(col < a.Dv);      // (Dv is a multiple of 16: whole waves)
  float* st = a.state + slot * a.state_stride + (int64_t)h * D * a.Dv + (live ? col : 0);
  const int64_t vc = (int64_t)h * a.Dv + (live ? col : 0);
  f32x4_d S[DT];
#pragma unroll
  for (int i = 0; i < DT; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) S[i][r] = held && live ? st[(int64_t)(16 * i + 4 * q + r) * a.Dv] : 0.f;
  float v[4];
  typename E::storage vn[4];                           // the next chunk's values as they lie in memory
  const char* vp[4];
  char* op[4];
  const int64_t vstep = kDC * a.v_stride * E::kBytes, ostep = (int64_t)kDC * a.H * a.Dv * 4;
  const auto point_v = [&](int c, int last) {          // as the helpers'
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int t = 4 * q + r;
      vp[r] = (const char*)a.v + ((start + c * kDC + (t < last ? t : last)) * a.v_stride + vc) * E::kBytes;
    }
  };
  const auto fetch_v = [&](int c) {
    if (c == chunks - 1) point_v(c, len - c * kDC - 1);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      vn[r] = *(const typename E::storage*)vp[r];
      vp[r] += vstep;
    }
  };
#pragma unroll
  for (int r = 0; r < 4; ++r) op[r] = (char*)(a.raw + (start + 4 * q + r) * (int64_t)a.H * a.Dv + vc);
  point_v(0, kDC);
  fetch_v(0);
  lds_barrier();
  lds_barrier();
  for (int c = 0; c < chunks; ++c) {
    const int n = len - c * kDC;
    const float* m = (const float*)(delta_lds + L::kWork + (c & 3) * kDcFloats * 4);
    const float* ops = (const float*)(delta_lds + L::kOp + (c & 1) * L::kOps);
    f32x4_d kd = {0.f, 0.f, 0.f, 0.f}, o = {0.f, 0.f, 0.f, 0.f}, u = {0.f, 0.f, 0.f, 0.f}, tr, pr;
    float ke[L::kParts ? 1 : 4][DT];
    const auto values = [&] {
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = E::load(&vn[r], 0);
      if (n < kDC) {
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = 4 * q + r < n ? v[r] : 0.f;
      }
      if (c + 1 < chunks) fetch_v(c + 1);
    };
    if constexpr (L::kParts) {
      // Products of parts, the small ones first (those of two last parts are far below fp32's rounding).  The parts of
      // a block's state are formed between the products of the block before, whose operands are read a block ahead.
      constexpr int BLOCKS = D / 32;
      f32x4_d g[DT];
      const char* rows = (const char*)ops;
      u32x4 ak[2][3], aq[2][3], sp[2][3];
      u32x2 kp[DT][3];
      const auto read = [&](int x) {
#pragma unroll
        for (int p = 0; p < 3; ++p) {
          ak[x & 1][p] = ld16(rows + p * L::kPart + r16 * L::kPartRow + 64 * x + 16 * q);
          aq[x & 1][p] = ld16(rows + (3 + p) * L::kPart + r16 * L::kPartRow + 64 * x + 16 * q);
        }
#pragma unroll
        for (int i = 2 * x; i < 2 * x + 2; ++i) g[i] = *(const f32x4_d*)(rows + L::kG + (16 * i + 4 * q) * 4);
      };
      const auto split = [&](int x) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const Parts y = parts_of(S[2 * x + e / 2][2 * (e & 1)], S[2 * x + e / 2][2 * (e & 1) + 1]);
#pragma unroll
          for (int p = 0; p < 3; ++p) sp[x & 1][p][e] = y.p[p];
        }
      };
      constexpr int PA[8] = {2, 1, 2, 0, 1, 1, 0, 0}, PB[8] = {1, 2, 0, 2, 1, 0, 1, 0};
      read(0);
      split(0);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int x = 0; x < BLOCKS; ++x) {
        if (x + 1 < BLOCKS) read(x + 1);
#pragma unroll
        for (int i = 2 * x; i < 2 * x + 2; ++i)
#pragma unroll
          for (int p = 0; p < 3; ++p) kp[i][p] = *(const u32x2*)(rows + L::kKe + (16 * i + r16) * L::kKeRow + p * 2 * kDC + 8 * q);
#pragma unroll
        for (int y = 0; y < 8; ++y) {
          kd = mfma_parts(ak[x & 1][PA[y]], sp[x & 1][PB[y]], kd);
          o = mfma_parts(aq[x & 1][PA[y]], sp[x & 1][PB[y]], o);
        }
        if (x + 1 < BLOCKS) split(x + 1);
#pragma unroll
        for (int i = 2 * x; i < 2 * x + 2; ++i)
#pragma unroll
          for (int r = 0; r < 4; ++r) S[i][r] *= g[i][r];
#pragma unroll
        for (int y = 0; y < 16; ++y) {
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);      // a read of LDS, a product, four vector instructions
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      tr = *(const f32x4_d*)&m[kDcT + r16 * kDC + 4 * q], pr = *(const f32x4_d*)&m[kDcP + r16 * kDC + 4 * q];
      values();
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        v[r] -= kd[r];
        u = mfma_d(tr[r], v[r], u);
      }
      const Parts u0 = parts_of(u[0], u[1]), u1 = parts_of(u[2], u[3]);
      const u32x4 ub[4] = {u32x4{u0.p[2], u1.p[2], u0.p[1], u1.p[1]}, u32x4{u0.p[2], u1.p[2], u0.p[0], u1.p[0]},
                           u32x4{u0.p[1], u1.p[1], u0.p[1], u1.p[1]}, u32x4{u0.p[0], u1.p[0], u0.p[0], u1.p[0]}};
      // Ke's parts second and last, first and last, and first and second twice, against U's last and second, last and first, second twice, first twice
      constexpr int KA[4] = {1, 0, 0, 0}, KB[4] = {2, 2, 1, 1};
#pragma unroll
      for (int y = 0; y < 4; ++y)
#pragma unroll
        for (int i = 0; i < DT; ++i)
          S[i] = mfma_parts(u32x4{kp[i][KA[y]][0], kp[i][KA[y]][1], kp[i][KB[y]][0], kp[i][KB[y]][1]}, ub[y], S[i]);
    } else {
      // Every read of LDS goes out between two products: in one piece the four waves' reads hold their products up until LDS has taken them
      // (left to itself the compiler keeps registers free and waits for each read).
      f32x4_d ak[DT], aq[DT], g[DT];
      const auto read_k = [&](int i) { ak[i] = *(const f32x4_d*)&ops[r16 * ROW + 16 * i + 4 * q]; };
      read_k(0);
      read_k(1);
#pragma unroll
      for (int i = 0; i < DT; ++i) {
        if (i + 2 < DT) read_k(i + 2);
        aq[i] = *(const f32x4_d*)&ops[(kDC + r16) * ROW + 16 * i + 4 * q];
        if (i == DT - 1) tr = *(const f32x4_d*)&m[kDcT + r16 * kDC + 4 * q];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = 0; r < 4; ++r) kd = mfma_d(ak[i][r], S[i][r], kd);
        __builtin_amdgcn_sched_barrier(0);
      }
      values();
#pragma unroll
      for (int i = 0; i < DT; ++i) {
        g[i] = *(const f32x4_d*)&ops[3 * kDC * ROW + 16 * i + 4 * q];
        if (i == 0) pr = *(const f32x4_d*)&m[kDcP + r16 * kDC + 4 * q];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          __builtin_amdgcn_sched_barrier(0);
          ke[r][i] = ops[(2 * kDC + 4 * q + r) * ROW + 16 * i + r16];
          __builtin_amdgcn_sched_barrier(0);
          o = mfma_d(aq[i][r], S[i][r], o);
        }
        if (i == 1) {
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            v[r] -= kd[r];
            u = mfma_d(tr[r], v[r], u);
          }
        }
        if (i > 0) {
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int r = 0; r < 4; ++r) S[i - 1][r] *= g[i - 1][r];
        }
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) S[DT - 1][r] *= g[DT - 1][r];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < DT; ++i) S[i] = mfma_d(ke[0][i], u[0], S[i]);
    }
    int first = kDC;                                  // the column's first token whose u is not finite
    f32x4_d uf = u;
    const float probe = fmaf(u[0], 0.f, fmaf(u[1], 0.f, fmaf(u[2], 0.f, u[3] * 0.f)));
    const bool odd = __ballot(probe != probe) != 0;
    if (odd) {
      const auto finite = [](float x) { return fabsf(x) < INFINITY; };
#pragma unroll
      for (int r = 3; r >= 0; --r)
        if (!finite(v[r])) {
          v[r] = 0.f;
          first = 4 * q + r;
        }
      uf = f32x4_d{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int r = 0; r < 4; ++r) uf = mfma_d(tr[r], v[r], uf);
#pragma unroll
      for (int r = 3; r >= 0; --r)
        if (!finite(uf[r])) first = min(first, 4 * q + r);
      first = min(first, __shfl_xor(first, 16, 64));
      first = min(first, __shfl_xor(first, 32, 64));
#pragma unroll
      for (int r = 0; r < 4; ++r) uf[r] = 4 * q + r < first ? uf[r] : 0.f;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) o = mfma_d(pr[r], uf[r], o);
    if constexpr (!L::kParts) {
#pragma unroll
      for (int r = 1; r < 4; ++r)
#pragma unroll
        for (int i = 0; i < DT; ++i) S[i] = mfma_d(ke[r][i], u[r], S[i]);
    }
    if (odd) {
#pragma unroll
      for (int r = 0; r < 4; ++r) o[r] = 4 * q + r < first ? o[r] : as_f32(0x7fc00000u);
    }
    if (live) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if (n >= kDC || 4 * q + r < n) *(float*)op[r] = o[r];
        op[r] += ostep;
      }
    }
    lds_barrier();
  }
  if (live) {
#pragma unroll
    for (int i = 0; i < DT; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) st[(int64_t)(16 * i + 4 * q + r) * a.Dv] = S[i][r];
  }
}

// whether the chunk kernels take a step: several tokens per request, heads of 64 or 128 key channels and whole waves of value
// channels, rows that can be read 16 bytes at a time
inline bool delta_chunks_take(const DeltaChunks& a, int D, int dtype, const SeqBatch& s) {
  const int V = dtype == SP_F32 ? 4 : 8;
  return s.extend_seq_lens && (D == 64 || D == 128) && a.Dv % 16 == 0 && a.q_stride % V == 0 && a.k_stride % V == 0 &&
         (((uintptr_t)a.q | (uintptr_t)a.k | (uintptr_t)a.decay | (uintptr_t)a.work) & 15) == 0;
}

template <typename Tag, int D, bool CHANNEL, int COLS>
int launch_delta_scan(const DeltaChunks& a, const SeqBatch& s, hipStream_t st) {
  constexpr int lds = DeltaScanLds<Tag, D, CHANNEL, COLS>::kBytes;
  if (lds > 64 * 1024) {
    static PerDevice<int> raised;
    int ok = 0;
    raised.get(ok, [&](int) {
      return hipFuncSetAttribute((const void*)delta_chunk_scan_kernel<Tag, D, CHANNEL, COLS>, hipFuncAttributeMaxDynamicSharedMemorySize, lds) ==
             hipSuccess ? 1 : 0;
    });
    if (!ok) return SP_ERR_LAUNCH;
  }
  delta_chunk_scan_kernel<Tag, D, CHANNEL, COLS><<<dim3((unsigned)s.B, (unsigned)a.H, (unsigned)((a.Dv + a.cols - 1) / a.cols)),
                                                   a.cols * 4 + kDcHelpers * 64, lds, st>>>(a, s);
  SP_LAUNCH_CHECK();
  return SP_OK;
}

template <typename Tag, int D, bool CHANNEL>
int launch_delta_chunks(DeltaChunks a, const SeqBatch& s, hipStream_t st) {
  const int64_t chunks = a.T / kDC + s.B;              // at most: a request's last chunk may be partial
  if (chunks >= ((int64_t)1 << 31) || a.H > 65535) return SP_ERR_UNSUPPORTED;
  delta_chunk_prepare_kernel<Tag, D, CHANNEL><<<dim3((unsigned)chunks, (unsigned)a.H), D * 2, 0, st>>>(a, s);
  SP_LAUNCH_CHECK();
  // columns per workgroup: 128 while requests x heads fill the 256 CUs by themselves, fewer (the operand rows are then formed once
  // per range) until they do
  a.cols = 128;
  while (a.cols > 64 && (int64_t)s.B * a.H * ((a.Dv + a.cols - 1) / a.cols) < 256) a.cols /= 2;
  if (a.cols > a.Dv) a.cols = a.Dv;
  return a.cols <= 64 ? launch_delta_scan<Tag, D, CHANNEL, 64>(a, s, st) : launch_delta_scan<Tag, D, CHANNEL, 128>(a, s, st);
}

}  // namespace sp

// (weak: both delta rules' sources define it, a library may hold either or both)
extern "C" __attribute__((weak)) int64_t sp_delta_chunk_floats(int64_t num_tokens, int batch_size, int heads) {
  return (num_tokens / sp::kDC + batch_size) * heads * sp::kDcFloats;
}
