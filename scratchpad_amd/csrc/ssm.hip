// State-space mixer (Mamba-2 form) and the small pieces recurrent mixers share.
//   gate projections   out[t, n] = bias[n] + sum_i w[n, i] x[t, i]        few outputs (one per head), fp32 weights,
//                                                                         fp32 accumulation and fp32 OUTPUT: what enters
//                                                                         a recurrence's decay or gate is never rounded
//   causal convolution out[t, c] = silu(bias[c] + sum_j w[c, j] in[t - (taps-1) + j, c])   per channel; inputs before a
//                      step's first row come from the request's saved last taps-1 inputs (zeros before the sequence)
//   scan               dt = softplus(dt_raw + dt_bias);  S <- exp(-exp(A_log) dt) S + dt B x^T;  y = S^T C + D x
//                      per head, S [N, Dv] fp32 in the state pool; head h reads B, C of group h / (H / G)
//   gated group norm   out = (y silu(z)) / rms_part * w      the gate BEFORE the norm, `parts` equal parts per row
#include "chunk_scan.h"
#include "lds_ring.h"

namespace sp {
namespace {

__device__ __forceinline__ float softplus_f(float z) { return fmaxf(z, 0.f) + log1pf(expf(-fabsf(z))); }

// one workgroup per (token, 16 outputs): every wave forms 4 outputs at once; a lane takes 4 neighbouring inputs per step
// (16-byte weight loads where rows allow) and several steps are in flight, so the loop does not wait load by load
template <typename Tag, bool VEC>
__global__ void __launch_bounds__(256)
small_linear_f32_kernel(float* out, const void* x, int64_t x_stride, const float* w, const float* bias, int64_t T, int K, int N) {
  typedef Elem<Tag> E;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t t = blockIdx.x;
  const int n0 = (blockIdx.y * 4 + wave) * 4;
  if (n0 >= N) return;
  // rows past N repeat the last row (computed, never stored): no branch in the loop
  const float* w0 = w + (int64_t)n0 * K;
  const float* w1 = w + (int64_t)(n0 + 1 < N ? n0 + 1 : N - 1) * K;
  const float* w2 = w + (int64_t)(n0 + 2 < N ? n0 + 2 : N - 1) * K;
  const float* w3 = w + (int64_t)(n0 + 3 < N ? n0 + 3 : N - 1) * K;
  float d0 = 0.f, d1 = 0.f, d2 = 0.f, d3 = 0.f;
  if (VEC) {
#pragma unroll 4
    for (int i = 4 * lane; i < K; i += 256) {
      const u32x4 a0 = ld16(w0 + i), a1 = ld16(w1 + i), a2 = ld16(w2 + i), a3 = ld16(w3 + i);
      float xv[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) xv[e] = E::load(x, t * x_stride + i + e);
      d0 += as_f32(a0[0]) * xv[0] + as_f32(a0[1]) * xv[1] + as_f32(a0[2]) * xv[2] + as_f32(a0[3]) * xv[3];
      d1 += as_f32(a1[0]) * xv[0] + as_f32(a1[1]) * xv[1] + as_f32(a1[2]) * xv[2] + as_f32(a1[3]) * xv[3];
      d2 += as_f32(a2[0]) * xv[0] + as_f32(a2[1]) * xv[1] + as_f32(a2[2]) * xv[2] + as_f32(a2[3]) * xv[3];
      d3 += as_f32(a3[0]) * xv[0] + as_f32(a3[1]) * xv[1] + as_f32(a3[2]) * xv[2] + as_f32(a3[3]) * xv[3];
    }
  } else {
#pragma unroll 4
    for (int i = lane; i < K; i += 64) {
      const float xv = E::load(x, t * x_stride + i);
      d0 += w0[i] * xv;
      d1 += w1[i] * xv;
      d2 += w2[i] * xv;
      d3 += w3[i] * xv;
    }
  }
  d0 = wave_sum(d0), d1 = wave_sum(d1), d2 = wave_sum(d2), d3 = wave_sum(d3);
  if (lane == 0) {
    out[t * N + n0] = d0 + (bias ? bias[n0] : 0.f);
    if (n0 + 1 < N) out[t * N + n0 + 1] = d1 + (bias ? bias[n0 + 1] : 0.f);
    if (n0 + 2 < N) out[t * N + n0 + 2] = d2 + (bias ? bias[n0 + 2] : 0.f);
    if (n0 + 3 < N) out[t * N + n0 + 3] = d3 + (bias ? bias[n0 + 3] : 0.f);
  }
}

// The same for many rows of bf16 x, on the matrix cores with nothing rounded on the way: a weight is three bf16 parts whose sum is
// exact (split3), x is bf16 already, the sums are fp32.  A workgroup takes 16 MT tokens x 16 outputs; its W waves share K (a stretch each)
// and add up through LDS in wave order.  An infinity has no parts that are numbers: a sum that is not finite is formed again, element
// by element.
// What bounds it is the way of the operands to the lanes: a matrix instruction wants 16 rows in neighbouring lanes, and a load of that shape
// asks for 16 lines a quarter (65 rows of K 2048 took 9.7 us whatever was in flight).  So rows come by direct loads of 128 or 256 neighbouring
// bytes into LDS that is the wave's own - no barrier but the last - and the lanes take their operands from there; the next 64 of k load while
// those are split and multiplied (more stages in flight leave room for fewer workgroups: 4096 rows of 64 outputs 12.5 with two).
// us, K 2048, loads to registers -> this: 4096 rows of 64 outputs 15.6 -> 9.1, of 32 10.1 -> 6.7, 65 rows of 64 9.8 -> 5.5; K 1024, 4096 of 32
// 6.8 -> 5.1.  Layers of 4096 and 3001 tokens: Mamba-2 395 -> 388, mLSTM 207 -> 202.
constexpr int kLinOut = 16;
template <int MT, int W>
__global__ void __launch_bounds__(W * 64)
linear_f32_mfma_kernel(float* out, const char* x, int64_t x_stride, const float* w, const float* bias, int64_t T, int K, int N) {
  constexpr int TOK = 16 * MT, LX = 2 * MT, LW = 4, kX = TOK * 128, kStage = kX + kLinOut * 256, ROW = kLinOut + 4;
  static_assert(W / 2 * TOK * ROW * 4 <= W * kStage && W * kStage <= 160 * 1024, "LDS");
  extern __shared__ __attribute__((aligned(1024))) char lin_lds[];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, r16 = lane & 15, q = lane >> 4;
  const int64_t t0 = (int64_t)blockIdx.x * TOK;
  const int n0 = blockIdx.y * kLinOut;
  // rows past the last: that one again, never stored; 16-byte chunks permuted by the row's number
  uint32_t ox[LX], ow[LW];
  const int cx = (lane & 7) ^ (lane >> 3);
#pragma unroll
  for (int i = 0; i < LX; ++i) {
    const int64_t row = i * 8 + (lane >> 3), last = T - 1 - t0;
    ox[i] = (uint32_t)((row < last ? row : last) * x_stride * 2) + cx * 16;
  }
#pragma unroll
  for (int i = 0; i < LW; ++i) {
    const int row = i * 4 + q;
    ow[i] = (uint32_t)min(row, N - 1 - n0) * (uint32_t)K * 4 + ((lane & 15) ^ row) * 16;
  }
  const char *const xb = x + t0 * x_stride * 2, *const wb = (const char*)(w + (int64_t)n0 * K);
  char* const own = lin_lds + wave * kStage;
  const uint32_t own0 = lds_address(own);
  const int stages = (K + 63) / 64, first = stages * wave / W, last = stages * (wave + 1) / W;
  const auto load = [&](int s) {
    const bool half = s * 64 + 64 > K;                    // K ends in the middle: its second 32 are the first again, and not taken
#pragma unroll
    for (int i = 0; i < LX; ++i) ring_load<false>(half && cx >= 4 ? ox[i] - 64 : ox[i], xb + (int64_t)s * 128, own0 + i * 1024);
#pragma unroll
    for (int i = 0; i < LW; ++i)
      ring_load<false>(half && ((lane & 15) ^ (i * 4 + q)) >= 8 ? ow[i] - 128 : ow[i], wb + (int64_t)s * 256, own0 + kX + i * 1024);
  };
  f32x4_c acc[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) acc[i] = f32x4_c{0.f, 0.f, 0.f, 0.f};
  if (first < last) load(first);
  for (int s = first; s < last; ++s) {
    ring_wait<LX + LW, 0>(0);
    u32x4 xf[2][MT], wf[2][2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
#pragma unroll
      for (int h = 0; h < 2; ++h) wf[k][h] = ld16(own + kX + r16 * 256 + (((8 * k + 2 * q + h) ^ r16) * 16));
#pragma unroll
      for (int i = 0; i < MT; ++i) xf[k][i] = ld16(own + (16 * i + r16) * 128 + (((4 * k + q) ^ (r16 & 7)) * 16));
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // in registers: the stage is free
    if (s + 1 < last) load(s + 1);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      if (k && s * 64 + 64 > K) break;
      u32x4 b[3];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        uint32_t hi, mid, lo;
        split3(as_f32(wf[k][e / 2][2 * (e & 1)]), as_f32(wf[k][e / 2][2 * (e & 1) + 1]), hi, mid, lo);
        b[0][e] = hi, b[1][e] = mid, b[2][e] = lo;
      }
#pragma unroll
      for (int c = 2; c >= 0; --c)
#pragma unroll
        for (int i = 0; i < MT; ++i) acc[i] = mfma_c(xf[k][i], b[c], acc[i]);
    }
  }
  // lane (r16, q): tokens 16 i + 4 q + r, output r16; the upper half of the waves first, then the lower add their own
  __syncthreads();
  float* const part = (float*)lin_lds;
#pragma unroll
  for (int half = 1; half >= 0; --half) {
    if (wave / (W / 2) == half) {
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float* const to = part + (wave % (W / 2) * TOK + 16 * i + 4 * q + r) * ROW + r16;
          *to = half ? acc[i][r] : acc[i][r] + *to;
        }
    }
    __syncthreads();
  }
  for (int e = tid; e < TOK * kLinOut; e += W * 64) {
    const int t = e / kLinOut, n = e % kLinOut;
    if (t0 + t >= T || n0 + n >= N) continue;
    float v = 0.f;
#pragma unroll
    for (int u = 0; u < W / 2; ++u) v += part[(u * TOK + t) * ROW + n];
    if (!(fabsf(v) < INFINITY)) {
      v = 0.f;
      for (int k = 0; k < K; ++k) v += w[(int64_t)(n0 + n) * K + k] * Elem<bf16_tag>::load(x, (t0 + t) * x_stride + k);
    }
    out[(t0 + t) * N + n0 + n] = v + (bias ? bias[n0 + n] : 0.f);
  }
}

template <int MT, int W>
int launch_linear_f32(float* out, const char* x, int64_t x_stride, const float* w, const float* bias, int64_t T, int K, int N, hipStream_t st) {
  constexpr int lds = W * (MT * 2048 + kLinOut * 256);
  static PerDevice<int> raised;
  int ok = 0;
  raised.get(ok, [&](int) {
    return hipFuncSetAttribute((const void*)linear_f32_mfma_kernel<MT, W>, hipFuncAttributeMaxDynamicSharedMemorySize, lds) == hipSuccess ? 1 : 0;
  });
  if (!ok) return SP_ERR_LAUNCH;
  const dim3 tiles((unsigned)((T + 16 * MT - 1) / (16 * MT)), (unsigned)((N + kLinOut - 1) / kLinOut));
  linear_f32_mfma_kernel<MT, W><<<tiles, W * 64, lds, st>>>(out, x, x_stride, w, bias, T, K, N);
  SP_LAUNCH_CHECK();
  return SP_OK;
}

// state [slot][taps - 1][C]: entry k = the input at position (tokens held) - (taps - 1) + k
template <typename Tag>
__global__ void __launch_bounds__(kBlock)
conv_silu_kernel(void* out, int64_t out_stride, const void* in, int64_t in_stride, const float* w, const float* bias,
                 const float* state, int64_t state_stride, SeqBatch s, int C, int taps) {
  typedef Elem<Tag> E;
  const int64_t t = blockIdx.x;
  const int c = blockIdx.y * kBlock + threadIdx.x;
  if (c >= C) return;
  int b;
  int64_t start, prefix;
  seq_of_token(s, t, b, start, prefix);
  const float* st = state + load_idx(s.req_pool_indices, b, s.idx64) * state_stride;
  float acc = bias ? bias[c] : 0.f;
  for (int j = 0; j < taps; ++j) {
    const int64_t r = t - (taps - 1) + j;
    float val = 0.f;
    if (r >= start) {
      val = E::load(in, r * in_stride + c);
    } else {
      const int64_t back = start - r;                  // 1 .. taps - 1 rows before the step
      if (prefix - back >= 0) val = st[(int64_t)(taps - 1 - back) * C + c];
    }
    acc += w[(int64_t)c * taps + j] * val;
  }
  E::store(out, t * out_stride + c, over_one_plus_exp(acc, acc));
}

constexpr int kMaxTaps = 16;

// The same on 16-byte pieces of rows, at most 4 taps: a thread keeps one piece's latest inputs in registers while it walks RUN consecutive
// tokens of the step, so a row is read once, not once per tap, and a piece's taps once per run.  Bound by vector work (30 instructions of a
// channel and token, 18 of them the exponential and the quotient) and by bytes about equally: the next kConvAhead rows are on their way under the
// work on the ones before, which a load under a condition would wait for - runs inside one request, all but a few, have none.
// With the carried inputs' kernel, us, before (every row of 8 tokens loaded first) -> now: 4096 tokens x 6144 channels 44.9 -> 36.1, of 819 requests
// 89 -> 62, 16384 x 8192 179 -> 152, 500 x 2048 16.1 -> 11.6.
constexpr int kConvAhead = 4;
template <typename Tag, int TAPS, int RUN>
__global__ void __launch_bounds__(kBlock)
conv_silu_run_kernel(void* out, int64_t out_stride, const void* in, int64_t in_stride, const float* w, const float* bias,
                     const float* state, int64_t state_stride, SeqBatch s, int64_t T, int C) {
  typedef Elem<Tag> E;
  constexpr int V = E::kVec, A = kConvAhead, P = TAPS > 1 ? TAPS - 1 : 1;
  static_assert(RUN % A == 0, "run");
  const int piece = (blockIdx.y * kBlock + threadIdx.x) * V, c = min(piece, C - V);      // (past the end: the last piece again, not stored)
  const int64_t t0 = (int64_t)blockIdx.x * RUN;
  const int run = (int)(T - t0 < RUN ? T - t0 : RUN);
  const char* const from = (const char*)in + (int64_t)c * E::kBytes;
  u32x4 row[A], halo[P];
  int req[A];
#pragma unroll
  for (int u = 0; u < A; ++u) {
    const int64_t t = t0 + min(u, run - 1);
    row[u] = ld16(from + t * in_stride * E::kBytes);
    req[u] = s.token_req[t];
  }
#pragma unroll
  for (int j = 0; j < TAPS - 1; ++j) {
    const int64_t t = t0 - (TAPS - 1) + j;
    halo[j] = ld16(from + (t > 0 ? t : 0) * in_stride * E::kBytes);
  }
  float wt[TAPS][V], bs[V];
  const bool quads = TAPS == 4 && ((uintptr_t)w & 15) == 0;          // a channel's taps are one load
#pragma unroll
  for (int x = 0; x < V; ++x) {
    bs[x] = bias ? bias[c + x] : 0.f;
    if (quads) {
      const u32x4 w4 = ld16(w + (int64_t)(c + x) * 4);
#pragma unroll
      for (int j = 0; j < TAPS; ++j) wt[j][x] = as_f32(w4[j & 3]);
    } else {
#pragma unroll
      for (int j = 0; j < TAPS; ++j) wt[j][x] = w[(int64_t)(c + x) * TAPS + j];
    }
  }
  float past[P][V];                                                   // past[j]: the input TAPS - 1 - j rows back
#pragma unroll
  for (int j = 0; j < TAPS - 1; ++j) unpack16<Tag>(halo[j], past[j]);
  int b = __builtin_amdgcn_readfirstlane(req[0]);
  const bool same = b == s.token_req[t0 + run - 1];                    // all of the run one request's
  // request b's inputs before its token t: rows of the step stay, those before it are carried ones, or none
  const auto carry = [&](int64_t t) {
    const int64_t start = s.extend_start_loc[b], prefix = s.extend_prefix_lens[b];
    if (t - (TAPS - 1) >= start) return;
    const float* st = state + load_idx(s.req_pool_indices, b, s.idx64) * state_stride;
#pragma unroll
    for (int j = 0; j < TAPS - 1; ++j) {
      const int64_t back = start - (t - (TAPS - 1) + j);              // > 0: so many rows before the step
      if (back > 0) {
#pragma unroll
        for (int x = 0; x < V; ++x) past[j][x] = prefix - back >= 0 ? st[(TAPS - 1 - back) * C + c + x] : 0.f;
      }
    }
  };
  if (TAPS > 1) carry(t0);
  const auto walk = [&](auto several) {                                // several: requests may end inside the run
#pragma unroll 1
    for (int g = 0; g < run; g += A) {
      u32x4 next[A];
      int next_req[A];
#pragma unroll
      for (int u = 0; u < A; ++u) {
        const int64_t t = t0 + min(g + A + u, run - 1);
        next[u] = ld16(from + t * in_stride * E::kBytes);
        if constexpr (decltype(several)::value) next_req[u] = s.token_req[t];
      }
#pragma unroll
      for (int u = 0; u < A; ++u) {
        const int64_t t = t0 + g + u;
        if constexpr (TAPS > 1 && decltype(several)::value) {
          const int nb = __builtin_amdgcn_readfirstlane(req[u]);
          if (nb != b) b = nb, carry(t);
        }
        float here[V], o[V];
        unpack16<Tag>(row[u], here);
#pragma unroll
        for (int x = 0; x < V; ++x) {
          float acc = bs[x];
#pragma unroll
          for (int j = 0; j < TAPS - 1; ++j) acc += wt[j][x] * past[j][x];
          acc += wt[TAPS - 1][x] * here[x];
          o[x] = silu_ref(acc);
#pragma unroll
          for (int j = 0; j < TAPS - 2; ++j) past[j][x] = past[j + 1][x];
          past[P - 1][x] = here[x];
        }
        if (g + u < run && piece < C) st16((char*)out + (t * out_stride + c) * E::kBytes, pack16<Tag>(o));
      }
#pragma unroll
      for (int u = 0; u < A; ++u) {
        row[u] = next[u];
        if constexpr (decltype(several)::value) req[u] = next_req[u];
      }
    }
  };
  if (same) walk(std::false_type());                                   // (its loads stay on their way: no load is conditional)
  else walk(std::true_type());
}

// KEEP: taps - 1, or 0 for any number of them (whose values wait in memory, loaded one after the other: with the convolution, 400 requests of a
// token 30.4 us so, 27.0 with three in registers)
template <typename Tag, int KEEP>
__global__ void __launch_bounds__(kBlock)
conv_state_kernel(float* state, int64_t state_stride, const void* in, int64_t in_stride, SeqBatch s, int C, int taps) {
  typedef Elem<Tag> E;
  const int b = blockIdx.x;
  const int c = blockIdx.y * kBlock + threadIdx.x;
  if (c >= C) return;
  int64_t start, len, prefix;
  seq_span(s, b, start, len, prefix);
  if (len <= 0) return;
  float* st = state + load_idx(s.req_pool_indices, b, s.idx64) * state_stride;
  const int keep = KEEP ? KEEP : taps - 1;
  float fresh[KEEP ? KEEP : kMaxTaps];
#pragma unroll
  for (int k = 0; k < keep; ++k) {
    const int64_t p = prefix + len - keep + k;       // position of the new entry k
    float val = 0.f;
    if (p >= prefix) val = E::load(in, (start + (p - prefix)) * in_stride + c);
    else if (p >= 0) val = st[(p - prefix + keep) * C + c];
    fresh[k] = val;
  }
#pragma unroll
  for (int k = 0; k < keep; ++k) st[(int64_t)k * C + c] = fresh[k];
}

// a decode step's single row per request: output and the moved state in one launch (a thread owns a channel of a request)
template <typename Tag>
__global__ void __launch_bounds__(kBlock)
conv_silu_step_kernel(void* out, int64_t out_stride, const void* in, int64_t in_stride, const float* w, const float* bias,
                      float* state, int64_t state_stride, SeqBatch s, int C, int taps) {
  typedef Elem<Tag> E;
  const int b = blockIdx.x;
  const int c = blockIdx.y * kBlock + threadIdx.x;
  if (c >= C) return;
  int64_t start, len, prefix;
  seq_span(s, b, start, len, prefix);
  float* st = state + load_idx(s.req_pool_indices, b, s.idx64) * state_stride;
  const int keep = taps - 1;
  float acc = bias ? bias[c] : 0.f;
  for (int k = 0; k < keep; ++k) {
    const float val = prefix - (keep - k) >= 0 ? st[(int64_t)k * C + c] : 0.f;
    acc += w[(int64_t)c * taps + k] * val;
    if (k > 0) st[(int64_t)(k - 1) * C + c] = val;
  }
  const float cur = E::load(in, (int64_t)b * in_stride + c);
  acc += w[(int64_t)c * taps + keep] * cur;
  if (keep > 0) st[(int64_t)(keep - 1) * C + c] = cur;
  E::store(out, (int64_t)b * out_stride + c, over_one_plus_exp(acc, acc));
}

constexpr int kChunk = 16;      // tokens staged in LDS per pass
// lanes that share one column of S: each holds at most 64 of the column's N values (at 128 per lane the state alone
// fills the register file, one wave per SIMD remains and every LDS read of B and C waits in full)
constexpr int split_of(int NP) { return NP > 64 ? 4 : (NP > 32 ? 2 : 1); }

// one workgroup per (request, head); thread = (column col of S, part): part p of SP owns the rows [p NS, (p + 1) NS) of
// the column, the parts are neighbouring lanes and add their partial outputs by lane exchange.  LDS rows of B and C are
// padded by 4 floats per part so that the parts' simultaneous broadcast reads fall into different banks.
template <typename Tag, int NP>
__global__ void __launch_bounds__(256 * split_of(NP))
mamba2_scan_kernel(float* y, int64_t y_stride, const void* xbc, int64_t xbc_stride, const float* dt_raw, const float* dt_bias,
                   const float* A_log, const float* Dskip, float* state, int64_t state_stride, SeqBatch s, int H, int G, int N,
                   int Dv) {
  typedef Elem<Tag> E;
  constexpr int SP = split_of(NP), NS = NP / SP, ROW = NP + 4 * SP;
  __shared__ float sB[kChunk][ROW], sC[kChunk][ROW], sdt[kChunk], sdec[kChunk];
  extern __shared__ float sx[];                         // [kChunk][Dv]: no global load inside the token loop
  const int b = blockIdx.x, h = blockIdx.y, j = threadIdx.x;
  const int nthreads = blockDim.x;
  const int col = j / SP, part = j % SP;
  int64_t start, len, prefix;
  seq_span(s, b, start, len, prefix);
  if (len <= 0) return;
  const bool live = col < Dv;
  const int g = h / (H / G);
  const int64_t inner = (int64_t)H * Dv;
  const int64_t colx = (int64_t)h * Dv, colB = inner + (int64_t)g * N, colC = inner + (int64_t)G * N + (int64_t)g * N;
  float* st = state + load_idx(s.req_pool_indices, b, s.idx64) * state_stride + (int64_t)h * N * Dv;
  float S[NS];
#pragma unroll
  for (int ii = 0; ii < NS; ++ii) {
    const int i = part * NS + ii;
    S[ii] = (live && i < N && prefix > 0) ? st[(int64_t)i * Dv + col] : 0.f;
  }
  const float a = expf(A_log[h]), bias = dt_bias[h], skip = Dskip[h];
  const float* myB = &sB[0][part * (NS + 4)];
  const float* myC = &sC[0][part * (NS + 4)];
  for (int64_t c0 = 0; c0 < len; c0 += kChunk) {
    const int n = (int)(len - c0 < kChunk ? len - c0 : kChunk);
    __syncthreads();
    // staging: every load of the pass is issued before the first is used (rows past the pass's end repeat its last row)
#pragma unroll
    for (int tt = 0; tt < kChunk; ++tt) {
      const int64_t row = start + c0 + (tt < n ? tt : n - 1);
      for (int i = j; i < NP; i += nthreads) {
        const bool ok = i < N;
        const int at = i + 4 * (i / NS);
        sB[tt][at] = ok ? E::load(xbc, row * xbc_stride + colB + i) : 0.f;
        sC[tt][at] = ok ? E::load(xbc, row * xbc_stride + colC + i) : 0.f;
      }
      for (int c = j; c < Dv; c += nthreads) sx[tt * Dv + c] = E::load(xbc, row * xbc_stride + colx + c);
    }
    if (j < n) {
      const float dt = softplus_f(dt_raw[(start + c0 + j) * H + h] + bias);
      sdt[j] = dt;
      sdec[j] = expf(-a * dt);
    }
    __syncthreads();
    for (int tt = 0; tt < n; ++tt) {
      const int64_t row = start + c0 + tt;
      const float xj = live ? sx[tt * Dv + col] : 0.f;
      const float dec = sdec[tt], dx = sdt[tt] * xj;
      const float* Bt = myB + tt * ROW;
      const float* Ct = myC + tt * ROW;
      float o = 0.f;
#pragma unroll
      for (int ii = 0; ii < NS; ++ii) {
        S[ii] = dec * S[ii] + Bt[ii] * dx;
        o += S[ii] * Ct[ii];
      }
#pragma unroll
      for (int off = 1; off < SP; off <<= 1) o += __shfl_xor(o, off, 64);
      if (live && part == 0) y[row * y_stride + colx + col] = o + skip * xj;
    }
  }
  if (live) {
#pragma unroll
    for (int ii = 0; ii < NS; ++ii) {
      const int i = part * NS + ii;
      if (i < N) st[(int64_t)i * Dv + col] = S[ii];
    }
  }
}

// ---- steps of several tokens per request, bf16 rows: 64 tokens at a time (chunk_scan.h; q = C, k = B, v = x) -----------------
// With L the running sum of the log decays -exp(A_log) dt inside the chunk: token s weighs exp(L_t - L_s) dt_s at token t, the
// old state exp(L_t).  One workgroup of Dv / 16 waves per (request, head); B and C are read once per head of their group.
// The per-token form is a chain of LDS reads, sums and lane exchanges per token (1.2 us; 788 us at 8 requests of 4096 tokens
// together, 64 heads of 128 x 64); this one takes 87 us there and 351 us for one request of 4096 tokens (5.5 us per chunk).
// In segments (see chunk_scan.h): MODE.
template <int N, int NW, int MODE>
__global__ void __launch_bounds__(NW * 64, MODE == kSegmentSums ? 4 : 8 / NW)
mamba2_chunk_kernel(float* y, int64_t y_stride, const char* xbc, int64_t xbc_stride, const float* dt_raw, const float* dt_bias,
                    const float* A_log, const float* Dskip, float* state, int64_t state_stride, ScanSegments seg, SeqBatch s, int H, int G) {
  constexpr bool OUT = MODE != kSegmentSums;
  typedef ChunkScan<N, NW, OUT> C;
  constexpr int Dv = C::Dv;
  extern __shared__ __attribute__((aligned(16))) char chunk_lds[];
  C c(chunk_lds);
  const int h = blockIdx.y, g = h / (H / G);
  int b = blockIdx.x, t0 = 0;
  if constexpr (MODE != kWholeRequests)
    if (!segment_at(s, (int)blockIdx.x, seg.tokens, c.lane, b, t0)) return;
  int64_t start, len, prefix;
  seq_span(s, b, start, len, prefix);
  if (len <= 0) return;
  const bool split = MODE != kWholeRequests && len > seg.tokens, last = t0 + seg.tokens >= len;
  if (MODE == kSegmentSums && last) return;
  start = uniform64(start) + t0, len = uniform64(len) - t0;
  if (MODE != kWholeRequests && len > seg.tokens) len = seg.tokens;
  const bool held = OUT && (prefix > 0 || t0 > 0);
  float* st = state + uniform64(load_idx(s.req_pool_indices, b, s.idx64)) * state_stride + (int64_t)h * N * Dv;
  float* const part = MODE == kWholeRequests ? nullptr : seg.work + ((int64_t)blockIdx.x * H + h) * seg.stride;
  c.load_state(split ? part : st, held);
  const int64_t inner = (int64_t)H * Dv, row = xbc_stride * 2;
  const char* x0 = xbc + start * row + (int64_t)h * Dv * 2;
  const char* b0 = xbc + start * row + (inner + (int64_t)g * N) * 2;
  const char* c0p = xbc + start * row + (inner + (int64_t)(G + g) * N) * 2;
  const float a = expf(A_log[h]), bias = dt_bias[h], skip = Dskip[h];
  const auto load = [&](int64_t c0) {
    const int n = (int)(len - c0 < kCL ? len - c0 : kCL);
    c.load(c0p + c0 * row, row, b0 + c0 * row, row, x0 + c0 * row, row, n);
  };
  float raw = 0.f, decay = 1.f;
  const auto load_steps = [&](int64_t c0) {
    if (c.wave == NW - 1 && c0 + c.lane < len) raw = dt_raw[(start + c0 + c.lane) * H + h];
  };
  const auto steps = [&](int64_t c0) {                // by the last wave: its share of the tiles is the smallest
    if (c.wave != NW - 1) return;
    const bool live = c0 + c.lane < len;
    const float dt = live ? softplus_f(raw + bias) : 0.f, e = live ? -a * dt : 0.f;
    // (e^-128 is zero in fp32: a stronger decay is the same one, and the sums stay where their differences are exact)
    const double L = wave_scan_sum((double)(e < -128.f ? -128.f : e), c.lane), Lend = __shfl(L, 63, 64);
    ChunkScalars& sc = *c.scalars(c0 / kCL);
    if constexpr (OUT) {
      ChunkScalars::put(sc.lt, c.lane, L);
      ChunkScalars::put(sc.ls, c.lane, L);
      sc.cs[c.lane] = dt;
      sc.a0[c.lane] = expf((float)L);
    }
    sc.w[c.lane] = expf((float)(Lend - L)) * dt;
    const float a_end = expf((float)Lend);
    if (c.lane == 0) sc.a_end = a_end;
    decay *= a_end;
  };
  load(0);
  load_steps(0);
  steps(0);
  bool zero = !held;
  for (int64_t c0 = 0; c0 < len; c0 += kCL) {
    const int n = (int)(len - c0 < kCL ? len - c0 : kCL);
    c.sc = c.scalars(c0 / kCL);
    c.stage((int)(c0 / kCL));
    lds_barrier();
    if (c0 + kCL < len) {
      load_steps(c0 + kCL);                           // (first: they are waited for first, and loads arrive in order)
      load(c0 + kCL);
    }
    if constexpr (OUT) {
      c.scores();
      c.from_state(zero);
      zero = false;
      lds_barrier();
      c.template weigh<false>();
    }
    if (c0 + kCL < len) steps(c0 + kCL);
    if constexpr (OUT) lds_barrier();
    c.absorb((int)(c0 / kCL));
    if constexpr (OUT) {
      char* yc = (char*)(y + (start + c0) * y_stride + (int64_t)h * Dv);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int tt = 16 * i + 4 * c.q;
        const u32x2 xv = *(const u32x2*)(chunk_lds + C::kVT + c.column() * C::TROW + tt * 2);
        const float x[4] = {as_f32(xv[0] << 16), as_f32(xv[0] & 0xffff0000u), as_f32(xv[1] << 16), as_f32(xv[1] & 0xffff0000u)};
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (tt + r < n) *(float*)(yc + (uint32_t)((tt + r) * (uint32_t)y_stride + c.column()) * 4u) = c.o[i][r] + skip * x[r];
      }
    }
    lds_barrier();
  }
  if constexpr (MODE == kSegmentSums) {
    c.store_state(part);
    if (c.tid == (NW - 1) * 64) part[N * Dv + kSegDecay] = decay;
  } else if (MODE == kWholeRequests || last) {
    c.store_state(st);
  }
}

template <int N, int NW, int MODE>
int launch_mamba2_mode(float* y, int64_t y_stride, const void* xbc, int64_t xbc_stride, const float* dt_raw, const float* dt_bias,
                       const float* A_log, const float* Dskip, float* state, int64_t state_stride, const ScanSegments& seg, unsigned groups,
                       const SeqBatch& s, int H, int G, hipStream_t st) {
  constexpr int bytes = ChunkScan<N, NW, MODE != kSegmentSums>::kBytes;
  static PerDevice<int> raised;
  if (!chunk_lds_ready(raised, (const void*)mamba2_chunk_kernel<N, NW, MODE>, bytes)) return SP_ERR_LAUNCH;
  mamba2_chunk_kernel<N, NW, MODE><<<dim3(groups, (unsigned)H), NW * 64, bytes, st>>>(
      y, y_stride, (const char*)xbc, xbc_stride, dt_raw, dt_bias, A_log, Dskip, state, state_stride, seg, s, H, G);
  SP_LAUNCH_CHECK();
  return SP_OK;
}

// (seg.tokens 0: a request's chunks by one workgroup per head)
template <int N, int NW>
int launch_mamba2_chunks(float* y, int64_t y_stride, const void* xbc, int64_t xbc_stride, const float* dt_raw, const float* dt_bias,
                         const float* A_log, const float* Dskip, float* state, int64_t state_stride, const ScanSegments& seg, int64_t tokens,
                         const SeqBatch& s, int H, int G, hipStream_t st) {
#define SP_MODE(MODE, GROUPS)                                                                                                            \
  launch_mamba2_mode<N, NW, MODE>(y, y_stride, xbc, xbc_stride, dt_raw, dt_bias, A_log, Dskip, state, state_stride, seg, GROUPS, s, H, G, st)
  if (seg.tokens == 0) return SP_MODE(kWholeRequests, (unsigned)s.B);
  const unsigned groups = (unsigned)(tokens / seg.tokens + s.B);
  int rc = SP_MODE(kSegmentSums, groups);
  if (rc != SP_OK) return rc;
  segment_states_kernel<false><<<dim3((unsigned)s.B, (unsigned)H, N * NW * 16 / 1024), 256, 0, st>>>(
      seg, state, state_stride, nullptr, 0, nullptr, 0, s, H, N, NW * 16);
  SP_LAUNCH_CHECK();
  return SP_MODE(kSegmentOutputs, groups);
#undef SP_MODE
}

// The same with rows of 16-byte vectors: a wave per (token, part), the part's values in registers between the sum of squares and
// the store (VPL vectors of 8 per lane, parts of up to 512 VPL values).  One workgroup per token and a workgroup sum per part
// (two barriers each, eight parts) took 61 us for 4096 rows of 8 x 512; this takes 25.
template <typename Tag, int VPL>
__global__ void __launch_bounds__(kBlock)
gated_group_norm_vec_kernel(void* out, int64_t out_stride, const float* y, int64_t y_stride, const void* z, int64_t z_stride,
                            const float* w, int64_t T, int per, int parts, float eps) {
  typedef Elem<Tag> E;
  const int lane = threadIdx.x & 63;
  const int64_t id = (int64_t)blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6);
  if (id >= T * parts) return;
  const int64_t t = id / parts;
  const int c0 = (int)(id % parts) * per;
  u32x4 zr[VPL], ya[VPL], yb[VPL];
#pragma unroll
  for (int u = 0; u < VPL; ++u) {
    const int i = (u * 64 + lane) * 8;
    if (i < per) {
      zr[u] = ld16((const char*)z + (t * z_stride + c0 + i) * 2);
      ya[u] = ld16(y + t * y_stride + c0 + i);
      yb[u] = ld16(y + t * y_stride + c0 + i + 4);
    }
  }
  float v[VPL][8], ss = 0.f;
#pragma unroll
  for (int u = 0; u < VPL; ++u) {
    const int i = (u * 64 + lane) * 8;
    if (i >= per) continue;
    float zf[8];
    unpack16<Tag>(zr[u], zf);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      v[u][e] = as_f32(e < 4 ? ya[u][e] : yb[u][e - 4]) * silu_ref(zf[e]);
      ss += v[u][e] * v[u][e];
    }
  }
  const float inv = 1.f / sqrtf(wave_sum(ss) / (float)per + eps);
#pragma unroll
  for (int u = 0; u < VPL; ++u) {
    const int i = (u * 64 + lane) * 8;
    if (i >= per) continue;
    const u32x4 wa = ld16(w + c0 + i), wb = ld16(w + c0 + i + 4);
    float o[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = v[u][e] * inv * as_f32(e < 4 ? wa[e] : wb[e - 4]);
    st16((char*)out + (t * out_stride + c0 + i) * 2, pack16<Tag>(o));
  }
}

template <typename Tag>
__global__ void __launch_bounds__(kBlock)
gated_group_norm_kernel(void* out, int64_t out_stride, const float* y, int64_t y_stride, const void* z, int64_t z_stride,
                        const float* w, int n, int parts, float eps) {
  typedef Elem<Tag> E;
  __shared__ float red[kBlock / 64];
  const int64_t t = blockIdx.x;
  const int per = n / parts;
  for (int p = 0; p < parts; ++p) {
    float ss = 0.f;
    for (int i = threadIdx.x; i < per; i += blockDim.x) {
      const float zv = E::load(z, t * z_stride + p * per + i);
      const float v = y[t * y_stride + p * per + i] * over_one_plus_exp(zv, zv);
      ss += v * v;
    }
    ss = block_sum(ss, red);
    const float inv = 1.f / sqrtf(ss / (float)per + eps);
    for (int i = threadIdx.x; i < per; i += blockDim.x) {
      const int c = p * per + i;
      const float zv = E::load(z, t * z_stride + c);
      E::store(out, t * out_stride + c, y[t * y_stride + c] * over_one_plus_exp(zv, zv) * inv * w[c]);
    }
  }
}

}  // namespace
}  // namespace sp

using namespace sp;

extern "C" int sp_small_linear_f32(float* out, const void* x, int64_t x_stride, const float* weight, const float* bias,
                                   int64_t num_tokens, int k, int n, int dtype, void* stream) {
  SP_CHECK_ARG(num_tokens >= 0 && k > 0 && n > 0);
  if (num_tokens == 0) return SP_OK;
  SP_CHECK_ARG(out && x && weight && x_stride >= k);
  // the tiles' loads name a row by its distance from the tile's first in 32 bits, of x and of the weights
  const auto near = [&](int64_t rows) {
    const int64_t most = (int64_t)1 << 32;
    return k <= most / (4 * kLinOut) && x_stride <= most / (2 * rows);
  };
  if (num_tokens > 64 && dtype == SP_BF16 && k % 32 == 0 && x_stride % 8 == 0 && (((uintptr_t)x | (uintptr_t)weight) & 15) == 0 && near(32)) {
    // (up to 64 rows a workgroup per row has the shorter chain.)  Workgroups of 32 tokens, two of which fit a CU; of 64, one a CU, which
    // read the weights half as often, where their rounds are at least half full and not more than two (us, 32 / 64: 4096 rows of 32
    // outputs 6.7 / 8.4, of 64 10.3 / 9.1, of 128 15.9 / 14.9; 9000 of 32 16.9 / 18.8; 16384 of 64 43.3 / 48.4).  The order of the sums is the same.
    const int64_t nb = (n + kLinOut - 1) / kLinOut, wide = (num_tokens + 63) / 64 * nb;
    if (near(64) && (num_tokens + 31) / 32 * nb > 256 && wide <= 512 && (wide + 255) % 256 >= 127)
      return launch_linear_f32<4, 8>(out, (const char*)x, x_stride, weight, bias, num_tokens, k, n, (hipStream_t)stream);
    return launch_linear_f32<2, 8>(out, (const char*)x, x_stride, weight, bias, num_tokens, k, n, (hipStream_t)stream);
  }
  const dim3 grid((unsigned)num_tokens, (unsigned)((n + 15) / 16));
  if (k % 4 == 0 && ((uintptr_t)weight & 15) == 0)
    SP_DISPATCH_DTYPE(dtype, (small_linear_f32_kernel<Tag, true><<<grid, 256, 0, (hipStream_t)stream>>>(
                                 out, x, x_stride, weight, bias, num_tokens, k, n)));
  else
    SP_DISPATCH_DTYPE(dtype, (small_linear_f32_kernel<Tag, false><<<grid, 256, 0, (hipStream_t)stream>>>(
                                 out, x, x_stride, weight, bias, num_tokens, k, n)));
  SP_LAUNCH_CHECK();
  return SP_OK;
}

extern "C" int sp_causal_conv_silu(void* out, int64_t out_stride, const void* in, int64_t in_stride, const float* weight,
                                   const float* bias, float* state, int64_t state_stride, int64_t num_tokens, int channels,
                                   int taps, SP_SEQ_PARAMS, int dtype, void* stream) {
  SP_CHECK_ARG(num_tokens >= 0 && channels > 0 && taps >= 1 && taps <= kMaxTaps);
  if (num_tokens == 0) return SP_OK;
  SP_CHECK_ARG(out && in && weight && req_pool_indices && seq_lens);
  SP_CHECK_ARG(out_stride >= channels && in_stride >= channels);
  SP_CHECK_ARG(taps == 1 || (state && state_stride >= (int64_t)(taps - 1) * channels));      // one tap: nothing is carried
  SP_CHECK_ARG(!extend_seq_lens || (extend_prefix_lens && extend_start_loc && token_req));
  SP_CHECK_ARG(extend_seq_lens || num_tokens == batch_size);
  SEQ_BATCH(s);
  const unsigned cb = (unsigned)((channels + kBlock - 1) / kBlock);
  if (!extend_seq_lens) {
    SP_DISPATCH_DTYPE(dtype, (conv_silu_step_kernel<Tag><<<dim3((unsigned)batch_size, cb), kBlock, 0, (hipStream_t)stream>>>(
                                 out, out_stride, in, in_stride, weight, bias, state, state_stride, s, channels, taps)));
    SP_LAUNCH_CHECK();
    return SP_OK;
  }
  const int vecn = dtype == SP_F32 ? 4 : 8;
  if (taps <= 4 && num_tokens > 64 && channels % vecn == 0 && in_stride % vecn == 0 && out_stride % vecn == 0 &&
      (((uintptr_t)in | (uintptr_t)out) & 15) == 0) {
    // runs of 16 tokens where they leave two waves for every SIMD, else of 8 (500 tokens x 2048 channels: 63 workgroups)
    const unsigned pieces = (unsigned)((channels / vecn + kBlock - 1) / kBlock);
    const bool longer = (num_tokens + 15) / 16 * pieces * (kBlock / 64) >= 2048;
    const dim3 grid((unsigned)(longer ? (num_tokens + 15) / 16 : (num_tokens + 7) / 8), pieces);
#define SP_CONV(TAPS)                                                                                                  \
  SP_DISPATCH_DTYPE(dtype, ((longer ? conv_silu_run_kernel<Tag, TAPS, 16> : conv_silu_run_kernel<Tag, TAPS, 8>)<<<      \
                               grid, kBlock, 0, (hipStream_t)stream>>>(                                                \
                               out, out_stride, in, in_stride, weight, bias, state, state_stride, s, num_tokens, channels)))
    if (taps == 1) SP_CONV(1);
    else if (taps == 2) SP_CONV(2);
    else if (taps == 3) SP_CONV(3);
    else SP_CONV(4);
#undef SP_CONV
  } else {
    SP_DISPATCH_DTYPE(dtype, (conv_silu_kernel<Tag><<<dim3((unsigned)num_tokens, cb), kBlock, 0, (hipStream_t)stream>>>(
                                 out, out_stride, in, in_stride, weight, bias, state, state_stride, s, channels, taps)));
  }
  SP_LAUNCH_CHECK();
  if (taps > 1) {      // after every reader of the old state (stream order)
    SP_DISPATCH_DTYPE(dtype, ((taps == 4 ? conv_state_kernel<Tag, 3> : conv_state_kernel<Tag, 0>)<<<dim3((unsigned)batch_size, cb), kBlock, 0,
                                                                                                 (hipStream_t)stream>>>(
                                 state, state_stride, in, in_stride, s, channels, taps)));
    SP_LAUNCH_CHECK();
  }
  return SP_OK;
}

// Steps of short portions that the per-token form walks faster than a chunk of 64 mostly empty tokens costs: requests x heads that take
// the chunk form more than one round of workgroups (two per CU with Dv 64, one with 128), and few tokens per request on average.
// us, per token / in chunks, by tokens per request (N x Dv, W = requests x heads):
//   64 x 64     W 512: 1 14 / 12      W 640: 1 14 / 18, 8 18 / 19, 10 19 / 19     W 4096: 1 45 / 69, 10 66 / 71, 12 71 / 71
//   64 x 128    W 256: 1 13 / 11      W 1024: 1 28 / 37, 8 39 / 41, 10 43 / 42    W 4096: 1 84 / 134, 12 137 / 142, 16 154 / 145
//   128 x 64    W 512: 1 17 / 16      W 1024: 1 27 / 28, 4 30 / 28                W 4096: 1 91 / 97, 4 97 / 98    W 8192: 1 194 / 178
//   128 x 128   W 256: 1 16 / 15      W 1024: 1 49 / 55, 4 54 / 55, 6 58 / 55     W 4096: 1 197 / 191
static bool short_portions(int64_t tokens, int64_t B, int H, int N, int Dv) {
  const int64_t W = B * H;
  if (tokens < 0 || W <= (Dv == 64 ? 512 : 256)) return false;
  if (N == 64) return tokens <= (Dv == 128 && W >= 1536 ? 12 : 10) * B;
  return tokens <= (Dv == 128 ? 4 : 2) * B && W * Dv < (1 << 19);
}

template <typename Tag>
static int launch_mamba2(float* y, int64_t y_stride, const void* xbc, int64_t xbc_stride, const float* dt_raw,
                         const float* dt_bias, const float* A_log, const float* Dskip, float* state, int64_t state_stride,
                         const ScanSegments& seg, const SeqBatch& s, int H, int G, int N, int Dv, int64_t tokens,
                         hipStream_t st) {
  // a step of one token per request stays with the per-token form (one sweep over the state is all there is to do), and so do
  // the types and head sizes the matrix form is not built for, and short portions of many requests
  if (std::is_same<Tag, bf16_tag>::value && s.extend_seq_lens && (N == 64 || N == 128) && (Dv == 64 || Dv == 128) &&
      chunk_aligned(xbc, xbc_stride) && y_stride < ((int64_t)1 << 24) && (seg.tokens || !short_portions(tokens, s.B, H, N, Dv))) {
#define SP_CHUNKS(N_, NW_)                                                                                              \
  return launch_mamba2_chunks<N_, NW_>(y, y_stride, xbc, xbc_stride, dt_raw, dt_bias, A_log, Dskip, state, state_stride, seg, tokens, s, H, G, st)
    if (N == 128 && Dv == 128) SP_CHUNKS(128, 8);
    if (N == 128) SP_CHUNKS(128, 4);
    if (Dv == 128) SP_CHUNKS(64, 8);
    SP_CHUNKS(64, 4);
#undef SP_CHUNKS
  }
  if (seg.tokens) return SP_ERR_UNSUPPORTED;
  const dim3 grid((unsigned)s.B, (unsigned)H);
#define SP_SCAN(NP)                                                                                                    \
  mamba2_scan_kernel<Tag, NP><<<grid, (unsigned)((Dv * split_of(NP) + 63) / 64 * 64), (size_t)kChunk * Dv * sizeof(float), st>>>(y, y_stride, xbc, xbc_stride, dt_raw, dt_bias, A_log, Dskip, state, \
                                                        state_stride, s, H, G, N, Dv)
  if (N <= 16) SP_SCAN(16);
  else if (N <= 32) SP_SCAN(32);
  else if (N <= 64) SP_SCAN(64);
  else if (N <= 128) SP_SCAN(128);
  else if (N <= 256) SP_SCAN(256);
  else return SP_ERR_UNSUPPORTED;
#undef SP_SCAN
  SP_LAUNCH_CHECK();
  return SP_OK;
}

// (num_tokens: the step's rows, < 0 where the caller does not know; only the choice between the two forms depends on it)
static int mamba2_scan(float* y, int64_t y_stride, const void* xbc, int64_t xbc_stride, const float* dt_raw, const float* dt_bias,
                       const float* A_log, const float* Dskip, float* state, int64_t state_stride, const ScanSegments& seg,
                       int64_t num_tokens, int heads, int groups, int state_size, int vdim, SP_SEQ_PARAMS, int dtype, void* stream) {
  SP_CHECK_ARG(batch_size >= 0 && heads > 0 && groups > 0 && heads % groups == 0 && state_size > 0 && vdim > 0 && vdim <= 256);
  if (batch_size == 0) return SP_OK;
  SP_CHECK_ARG(y && xbc && dt_raw && dt_bias && A_log && Dskip && state && req_pool_indices && seq_lens);
  SP_CHECK_ARG(!extend_seq_lens || (extend_prefix_lens && extend_start_loc));
  const int64_t inner = (int64_t)heads * vdim;
  SP_CHECK_ARG(y_stride >= inner && xbc_stride >= inner + 2 * (int64_t)groups * state_size);
  SP_CHECK_ARG(state_stride >= (int64_t)heads * state_size * vdim);
  SEQ_BATCH(s);
  SP_DISPATCH_DTYPE(dtype, return (launch_mamba2<Tag>(y, y_stride, xbc, xbc_stride, dt_raw, dt_bias, A_log, Dskip, state,
                                                      state_stride, seg, s, heads, groups, state_size, vdim, num_tokens,
                                                      (hipStream_t)stream)));
}

extern "C" int sp_mamba2_scan_tokens(float* y, int64_t y_stride, const void* xbc, int64_t xbc_stride, const float* dt_raw,
                                     const float* dt_bias, const float* A_log, const float* Dskip, float* state,
                                     int64_t state_stride, int64_t num_tokens, int heads, int groups, int state_size, int vdim,
                                     SP_SEQ_PARAMS, int dtype, void* stream) {
  return mamba2_scan(y, y_stride, xbc, xbc_stride, dt_raw, dt_bias, A_log, Dskip, state, state_stride, ScanSegments{nullptr, 0, 0},
                     num_tokens, heads, groups, state_size, vdim, req_pool_indices, seq_lens, extend_seq_lens, extend_prefix_lens,
                     extend_start_loc, token_req, idx64, batch_size, dtype, stream);
}

// (weak: mlstm.hip and ssm.hip define it, a library may hold either or both)
extern "C" __attribute__((weak)) int64_t sp_scan_segment_floats(int64_t num_tokens, int batch_size, int heads, int dim, int vdim,
                                                                int segment_tokens) {
  return scan_segment_floats(num_tokens, batch_size, heads, dim, vdim, segment_tokens);
}

extern "C" int sp_mamba2_scan_segments(float* y, int64_t y_stride, const void* xbc, int64_t xbc_stride, const float* dt_raw,
                                       const float* dt_bias, const float* A_log, const float* Dskip, float* state, int64_t state_stride,
                                       float* work, int segment_tokens, int64_t num_tokens, int heads, int groups, int state_size,
                                       int vdim, SP_SEQ_PARAMS, int dtype, void* stream) {
  SP_CHECK_ARG(num_tokens >= 0 && segment_tokens > 0 && segment_tokens % kCL == 0 && work && ((uintptr_t)work & 15) == 0);
  return mamba2_scan(y, y_stride, xbc, xbc_stride, dt_raw, dt_bias, A_log, Dskip, state, state_stride,
                     ScanSegments{work, segment_floats(state_size, vdim, false), segment_tokens}, num_tokens, heads, groups, state_size,
                     vdim, req_pool_indices, seq_lens, extend_seq_lens, extend_prefix_lens, extend_start_loc, token_req, idx64, batch_size,
                     dtype, stream);
}

extern "C" int sp_mamba2_scan(float* y, int64_t y_stride, const void* xbc, int64_t xbc_stride, const float* dt_raw,
                              const float* dt_bias, const float* A_log, const float* Dskip, float* state,
                              int64_t state_stride, int heads, int groups, int state_size, int vdim, SP_SEQ_PARAMS,
                              int dtype, void* stream) {
  return sp_mamba2_scan_tokens(y, y_stride, xbc, xbc_stride, dt_raw, dt_bias, A_log, Dskip, state, state_stride, -1, heads, groups,
                               state_size, vdim, req_pool_indices, seq_lens, extend_seq_lens, extend_prefix_lens, extend_start_loc,
                               token_req, idx64, batch_size, dtype, stream);
}

extern "C" int sp_gated_group_norm(void* out, int64_t out_stride, const float* y, int64_t y_stride, const void* z,
                                   int64_t z_stride, const float* weight, int64_t num_tokens, int n, int parts, float eps,
                                   int dtype, void* stream) {
  SP_CHECK_ARG(num_tokens >= 0 && n > 0 && parts > 0 && n % parts == 0);
  if (num_tokens == 0) return SP_OK;
  SP_CHECK_ARG(out && y && z && weight && out_stride >= n && y_stride >= n && z_stride >= n);
  const int per = n / parts;
  const int64_t waves = (num_tokens * parts + kBlock / 64 - 1) / (kBlock / 64);
  if (dtype != SP_F32 && per % 8 == 0 && per <= 2048 && waves < ((int64_t)1 << 31) && out_stride % 8 == 0 && y_stride % 4 == 0 &&
      z_stride % 8 == 0 && (((uintptr_t)out | (uintptr_t)y | (uintptr_t)z | (uintptr_t)weight) & 15) == 0) {
#define SP_GGN(T_, VPL)                                                                                              \
  gated_group_norm_vec_kernel<T_, VPL><<<dim3((unsigned)waves), kBlock, 0, (hipStream_t)stream>>>(                    \
      out, out_stride, y, y_stride, z, z_stride, weight, num_tokens, per, parts, eps)
#define SP_GGN2(T_)                 \
  do {                              \
    if (per <= 512) SP_GGN(T_, 1);  \
    else if (per <= 1024) SP_GGN(T_, 2); \
    else SP_GGN(T_, 4);             \
  } while (0)
    if (dtype == SP_BF16) SP_GGN2(bf16_tag);
    else SP_GGN2(f16_tag);
#undef SP_GGN2
#undef SP_GGN
    SP_LAUNCH_CHECK();
    return SP_OK;
  }
  SP_DISPATCH_DTYPE(dtype, (gated_group_norm_kernel<Tag><<<dim3((unsigned)num_tokens), kBlock, 0, (hipStream_t)stream>>>(
                               out, out_stride, y, y_stride, z, z_stride, weight, n, parts, eps)));
  SP_LAUNCH_CHECK();
  return SP_OK;
}
