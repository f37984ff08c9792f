// Generalized delta rule: a per-head matrix state with a per-channel decay and a per-channel removal along the unit key.
// Per head, with r, k, v of a token, decay w and removal rate a per key channel, all of the recurrence in fp32:
//   u  = k / sqrt(|k|^2 + 1e-6)
//   S' = diag(w) S - (a * u) (u^T S) + k v^T            (both first terms read the state the previous token left)
//   o  = S'^T r
//   out = o / rms_head(o) * norm_w * sigmoid(g)
// The gates come from sp_delta_gates:
//   w = exp(-rate * sigmoid(W2 tanh(p) + w0))            (p = the low-rank projection's output)
//   a = sigmoid(apre + a_bias)
//
// One workgroup per (request, head): a column of S (one value channel) lives in the registers of 2, 4 or 8 neighbouring
// lanes; the request's tokens of this step are walked in order from the state the previous step left in the pool (zeros
// at a sequence's first token), staged through LDS in passes.  A token costs ONE sweep over the column: the update, the
// numerator and - on the state just completed - the next token's u^T S, then two independent sums over the column's lanes
// (register moves); no workgroup barrier.  The order of its sums depends on the head only.  Prompts
// take it, but for longer portions with heads of 64, which go 16 tokens at a time (delta_prepare_kernel and the walk of chunk16.h); a decode step (one token
// per request, heads of 64 or 128, rank up to 512) takes delta_step_kernel, which forms the gates too and adds a head's sums in
// another order.
#include "chunk16.h"

namespace sp {
namespace {

// w2t: [rank, channels] fp32 (the up-projection transposed: neighbouring threads read neighbouring channels).  A workgroup
// takes TPB tokens x 256 channels, a thread one channel: every weight it loads serves all TPB tokens (TPB = 8 for prompts'
// portions), and a step of few tokens (TPB = 1) still spreads over channels / 256 workgroups per token.
template <typename Tag, int TPB>
__global__ void __launch_bounds__(kBlock)
delta_gates_kernel(float* decay, float* remove, const void* p, int64_t p_stride, const float* w2t, const float* w0,
                   const void* apre, int64_t a_stride, const float* a_bias, int64_t T, int channels, int rank, float rate) {
  typedef Elem<Tag> E;
  extern __shared__ float tp[];                          // [TPB][rank]
  const int64_t t0 = (int64_t)blockIdx.x * TPB;
  const int c = blockIdx.y * kBlock + threadIdx.x;
  for (int e = threadIdx.x; e < TPB * rank; e += kBlock) {
    const int tt = e / rank, r = e % rank;
    tp[e] = t0 + tt < T ? tanhf(E::load(p, (t0 + tt) * p_stride + r)) : 0.f;
  }
  __syncthreads();
  if (c >= channels) return;
  float acc[TPB];
#pragma unroll
  for (int tt = 0; tt < TPB; ++tt) acc[tt] = 0.f;
  int r = 0;
  for (; r + 4 <= rank; r += 4) {                        // four weights in flight
    const float w_0 = w2t[(int64_t)r * channels + c], w_1 = w2t[(int64_t)(r + 1) * channels + c];
    const float w_2 = w2t[(int64_t)(r + 2) * channels + c], w_3 = w2t[(int64_t)(r + 3) * channels + c];
#pragma unroll
    for (int tt = 0; tt < TPB; ++tt) {
      const float* q = tp + tt * rank + r;
      acc[tt] += w_0 * q[0];
      acc[tt] += w_1 * q[1];
      acc[tt] += w_2 * q[2];
      acc[tt] += w_3 * q[3];
    }
  }
  for (; r < rank; ++r) {
    const float w = w2t[(int64_t)r * channels + c];
#pragma unroll
    for (int tt = 0; tt < TPB; ++tt) acc[tt] += w * tp[tt * rank + r];
  }
  const float bias = w0[c], ab = a_bias[c];
#pragma unroll
  for (int tt = 0; tt < TPB; ++tt) {
    const int64_t t = t0 + tt;
    if (t < T) {
      decay[t * channels + c] = expf(-over_one_plus_exp(rate, acc[tt] + bias));
      remove[t * channels + c] = over_one_plus_exp(1.f, E::load(apre, t * a_stride + c) + ab);
    }
  }
}

constexpr int delta_chunk(int KP) { return KP > 64 ? 8 : 16; }                      // tokens staged in LDS per pass
// lanes that share one column of S: 8 state values per lane where the workgroup's 1024 threads allow it (measured at heads of
// 64: 2 lanes 1.07 ms, 4 lanes 0.58 ms, 8 lanes 0.38 ms, 16 lanes 0.49 ms per 4096 tokens with two sweeps per token and
// lane exchanges through LDS; 8 lanes 0.29 ms, 16 lanes 0.32 ms with one sweep and register moves - more waves per SIMD
// hide the waits of the per-token chain until the sums over the lanes take over)
constexpr int delta_split(int KP) { return KP > 128 ? 4 : (KP > 32 ? 8 : (KP > 16 ? 4 : 2)); }

// wave_sum's additions by shuffles.  The recurrence's columns fill the registers, and the lane swaps' copies pushed 36 bytes of them a lane
// into scratch at heads of 128 (64 requests of 4 tokens, 16 heads: 64.7 -> 69.0 us; 16 single tokens 16.3 -> 17.4).
__device__ __forceinline__ float wave_sum_shuffled(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// thread = (column col of S, part): part p of SP owns the rows [p DS, (p + 1) DS) of the column.  LDS rows are padded by
// 4 floats per part so that the parts' simultaneous broadcast reads fall into different banks.
// A pass's operands come from global memory into registers in ONE burst (every load issued before the first is used), and
// the burst of pass n + 1 is issued right before the token loop of pass n, so it flies while the recurrence runs; the loop
// itself touches LDS and registers only.
template <typename Tag, int KP>
__global__ void __launch_bounds__(KP * delta_split(KP) < 64 ? 64 : KP * delta_split(KP))
delta_recurrence_kernel(void* out, int64_t out_stride, const void* r, int64_t r_stride, const void* k, int64_t k_stride,
                        const void* v, int64_t v_stride, const void* g, int64_t g_stride, const float* decay,
                        const float* remove, const float* norm_w, float* state, int64_t state_stride, SeqBatch s, int H,
                        int K, float eps) {
  typedef Elem<Tag> E;
  constexpr int kChunk = delta_chunk(KP), SP = delta_split(KP), DS = KP / SP, ROW = KP + 4 * SP;
  constexpr int NT = KP * SP < 64 ? 64 : KP * SP;       // threads of the workgroup (the launch uses exactly these)
  constexpr int TSTEP = NT / KP, PER = kChunk / TSTEP;  // staging: thread j takes channel j % KP of tokens j / KP + u TSTEP
  constexpr int PERG = kChunk / SP;                     // epilogue: thread (col, part) takes tokens part + u SP
  // (rows and parts start at multiples of 16 bytes: the token loop reads them four floats at a time)
  __shared__ __attribute__((aligned(16))) float sr[kChunk][ROW], sk[kChunk][ROW], sw[kChunk][ROW], su[kChunk + 1][ROW], sau[kChunk][ROW];
  __shared__ float sv[kChunk][KP], so[kChunk][KP], sinv[kChunk];
  const int b = blockIdx.x, h = blockIdx.y, j = threadIdx.x;
  const int wave = j >> 6, lane = j & 63, waves = NT >> 6;
  const int col = j / SP, part = j % SP;
  int64_t start, len, prefix;
  seq_span(s, b, start, len, prefix);
  if (len <= 0) return;
  const bool live = col < K;
  float* st = state + load_idx(s.req_pool_indices, b, s.idx64) * state_stride + (int64_t)h * K * K;
  const bool held = prefix > 0;
  const int64_t hc = (int64_t)h * K, HK = (int64_t)H * K;
  const int mine = part * (DS + 4);
  const int si = j % KP, st0 = j / KP;                  // this thread's staged channel and first staged token
  const bool sok = si < K;
  const int sat = si + 4 * (si / DS);
  float fr[PER], fk[PER], fw[PER], fa[PER], fv[PER], fg[PERG];
  // the operands of the pass that starts at c0 (rows past the pass's end repeat its last row; they are never used)
  auto fetch = [&](int64_t c0) {
    const int n = (int)(len - c0 < kChunk ? len - c0 : kChunk);
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int tt = st0 + u * TSTEP;
      const int64_t row = start + c0 + (tt < n ? tt : n - 1);
      fr[u] = sok ? E::load(r, row * r_stride + hc + si) : 0.f;
      fk[u] = sok ? E::load(k, row * k_stride + hc + si) : 0.f;
      fv[u] = sok ? E::load(v, row * v_stride + hc + si) : 0.f;
      fw[u] = sok ? decay[row * HK + hc + si] : 0.f;
      fa[u] = sok ? remove[row * HK + hc + si] : 0.f;
    }
#pragma unroll
    for (int u = 0; u < PERG; ++u) {
      const int tt = part + u * SP;
      fg[u] = live ? E::load(g, (start + c0 + (tt < n ? tt : n - 1)) * g_stride + hc + col) : 0.f;
    }
  };
  fetch(0);
  float S[DS];
#pragma unroll
  for (int ii = 0; ii < DS; ++ii) {
    const int i = part * DS + ii;
    S[ii] = (live && i < K && held) ? st[(int64_t)i * K + col] : 0.f;
  }
  const float nw = live ? norm_w[hc + col] : 0.f;
  for (int64_t c0 = 0; c0 < len; c0 += kChunk) {
    const int n = (int)(len - c0 < kChunk ? len - c0 : kChunk);
    __syncthreads();                                     // the previous pass's epilogue is done with so and sinv
    float gate[PERG];
#pragma unroll
    for (int u = 0; u < PERG; ++u) gate[u] = fg[u];
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int tt = st0 + u * TSTEP;
      sr[tt][sat] = fr[u];
      sk[tt][sat] = fk[u];
      sw[tt][sat] = fw[u];
      sau[tt][sat] = fa[u];
      sv[tt][si] = fv[u];
    }
    __syncthreads();
    // the unit key of every token of the pass: a wave per token
    for (int tt = wave; tt < n; tt += waves) {
      float ss = 0.f;
      for (int i = lane; i < K; i += 64) {
        const float x = sk[tt][i + 4 * (i / DS)];
        ss += x * x;
      }
      ss = wave_sum_shuffled(ss);
      const float inv = 1.f / sqrtf(ss + 1e-6f);
      for (int i = lane; i < KP; i += 64) {
        const int at = i + 4 * (i / DS);
        const float uu = sk[tt][at] * inv;
        su[tt][at] = uu;
        sau[tt][at] *= uu;
      }
    }
    __syncthreads();
    if (c0 + kChunk < len) fetch(c0 + kChunk);           // in flight while the recurrence runs
    // u^T S of the pass's first token; every later token's is formed in the sweep that completes the state it reads
    // (four partial sums per sum: the chain of dependent additions is a quarter as long; DS is a multiple of 4)
    float proj;
    {
      const float4* pu = reinterpret_cast<const float4*>(&su[0][mine]);
      float pj[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ii = 0; ii < DS; ii += 4) {
        const float4 u4 = pu[ii / 4];
        pj[0] += u4.x * S[ii];
        pj[1] += u4.y * S[ii + 1];
        pj[2] += u4.z * S[ii + 2];
        pj[3] += u4.w * S[ii + 3];
      }
      proj = lanes_sum<SP>((pj[0] + pj[1]) + (pj[2] + pj[3]));
    }
    for (int tt = 0; tt < n; ++tt) {
      const float4* pau = reinterpret_cast<const float4*>(&sau[tt][mine]);
      const float4* pw = reinterpret_cast<const float4*>(&sw[tt][mine]);
      const float4* pk = reinterpret_cast<const float4*>(&sk[tt][mine]);
      const float4* pr = reinterpret_cast<const float4*>(&sr[tt][mine]);
      const float4* pun = reinterpret_cast<const float4*>(&su[tt + 1][mine]);      // the next token's unit key (row n: unused)
      const float vj = live ? sv[tt][col] : 0.f;
      float nm[4] = {0.f, 0.f, 0.f, 0.f}, pj[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ii = 0; ii < DS; ii += 4) {
        const float4 w4 = pw[ii / 4], a4 = pau[ii / 4], k4 = pk[ii / 4], r4 = pr[ii / 4], u4 = pun[ii / 4];
        S[ii] = w4.x * S[ii] - a4.x * proj + k4.x * vj;
        S[ii + 1] = w4.y * S[ii + 1] - a4.y * proj + k4.y * vj;
        S[ii + 2] = w4.z * S[ii + 2] - a4.z * proj + k4.z * vj;
        S[ii + 3] = w4.w * S[ii + 3] - a4.w * proj + k4.w * vj;
        nm[0] += S[ii] * r4.x;
        nm[1] += S[ii + 1] * r4.y;
        nm[2] += S[ii + 2] * r4.z;
        nm[3] += S[ii + 3] * r4.w;
        pj[0] += S[ii] * u4.x;
        pj[1] += S[ii + 1] * u4.y;
        pj[2] += S[ii + 2] * u4.z;
        pj[3] += S[ii + 3] * u4.w;
      }
      const float num = lanes_sum<SP>((nm[0] + nm[1]) + (nm[2] + nm[3]));
      proj = lanes_sum<SP>((pj[0] + pj[1]) + (pj[2] + pj[3]));
      if (live && part == 0) so[tt][col] = num;
    }
    __syncthreads();
    // per-head RMS of o, output weight and gate
    for (int tt = wave; tt < n; tt += waves) {
      float ss = 0.f;
      for (int i = lane; i < K; i += 64) ss += so[tt][i] * so[tt][i];
      ss = wave_sum_shuffled(ss);
      if (lane == 0) sinv[tt] = 1.f / sqrtf(ss / (float)K + eps);
    }
    __syncthreads();
    if (live) {
#pragma unroll
      for (int u = 0; u < PERG; ++u) {
        const int tt = part + u * SP;
        if (tt < n)
          E::store(out, (start + c0 + tt) * out_stride + hc + col, over_one_plus_exp(so[tt][col] * sinv[tt] * nw, gate[u]));
      }
    }
  }
  if (live) {
#pragma unroll
    for (int ii = 0; ii < DS; ++ii) {
      const int i = part * DS + ii;
      if (i < K) st[(int64_t)i * K + col] = S[ii];
    }
  }
}

// A decode step - one token per request - with its gates formed where they are used: one launch in place of two, and decay and
// removal never in memory.  Thread (part, col): a wave reads whole rows of S, a part of NT / K owns every part-th block of K / parts
// rows of its column; sums over the parts, and over the slices of the gates' rank, go through LDS.  A step of 16 requests of 16
// heads of 64 (4 MB of states: 1 us) is bound by its launches: this one takes 6.7 us of the GPU, the mixer's step 58.5 -> 49 us.
constexpr int kStepRank = 512;
template <typename Tag, int K, int PARTS>
__global__ void __launch_bounds__(K * PARTS)
delta_step_kernel(void* out, int64_t out_stride, const void* r, int64_t r_stride, const void* k, int64_t k_stride,
                  const void* v, int64_t v_stride, const void* g, int64_t g_stride, const void* p, int64_t p_stride,
                  const void* apre, int64_t a_stride, const float* w2t, const float* w0, const float* a_bias, int rank, float rate,
                  const float* norm_w, float* state, int64_t state_stride, SeqBatch s, int H, float eps) {
  typedef Elem<Tag> E;
  constexpr int NT = K * PARTS, DS = K / PARTS;
  __shared__ float tp[kStepRank], part_sum[PARTS][K], sw[K], sau[K], su[K], sk[K], sr[K], red[NT / 64];
  const int b = blockIdx.x, h = blockIdx.y, j = threadIdx.x, col = j % K, part = j / K;
  int64_t start, len, prefix;
  seq_span(s, b, start, len, prefix);
  const bool held = prefix > 0;
  const int64_t hc = (int64_t)h * K, channels = (int64_t)H * K;
  float* st = state + load_idx(s.req_pool_indices, b, s.idx64) * state_stride + hc * K;
  float S[DS];
#pragma unroll
  for (int ii = 0; ii < DS; ++ii) S[ii] = held ? st[(int64_t)(part * DS + ii) * K + col] : 0.f;
  const float kf = E::load(k, b * k_stride + hc + col), rf = E::load(r, b * r_stride + hc + col);
  const float vf = E::load(v, b * v_stride + hc + col), gf = E::load(g, b * g_stride + hc + col);
  const float af = E::load(apre, b * a_stride + hc + col) + a_bias[hc + col], nw = norm_w[hc + col], bias = w0[hc + col];
  for (int x = j; x < rank; x += NT) tp[x] = tanhf(E::load(p, b * p_stride + x));
  const float k2 = block_sum(part == 0 ? kf * kf : 0.f, red);      // (its barriers also publish tp)
  float acc = 0.f;
#pragma unroll 8
  for (int x = part; x < rank; x += PARTS) acc += w2t[x * channels + hc + col] * tp[x];
  part_sum[part][col] = acc;
  __syncthreads();
  const auto over_parts = [&]() {
    float t = 0.f;
#pragma unroll
    for (int q = 0; q < PARTS; ++q) t += part_sum[q][col];
    return t;
  };
  if (part == 0) {
    const float u = kf / sqrtf(k2 + 1e-6f);
    sw[col] = expf(-over_one_plus_exp(rate, over_parts() + bias));
    su[col] = u;
    sau[col] = over_one_plus_exp(u, af);
    sk[col] = kf;
    sr[col] = rf;
  }
  __syncthreads();
  float proj = 0.f;
#pragma unroll
  for (int ii = 0; ii < DS; ++ii) proj += su[part * DS + ii] * S[ii];
  part_sum[part][col] = proj;
  __syncthreads();
  proj = over_parts();
  __syncthreads();
  float num = 0.f;
#pragma unroll
  for (int ii = 0; ii < DS; ++ii) {
    const int i = part * DS + ii;
    S[ii] = sw[i] * S[ii] - sau[i] * proj + sk[i] * vf;
    st[(int64_t)i * K + col] = S[ii];
    num += S[ii] * sr[i];
  }
  part_sum[part][col] = num;
  __syncthreads();
  const float o = over_parts();
  const float ss = block_sum(part == 0 ? o * o : 0.f, red);
  if (part == 0) E::store(out, b * out_stride + hc + col, over_one_plus_exp(o / sqrtf(ss / (float)K + eps) * nw, gf));
}

template <typename Tag>
static int launch_delta(void* out, int64_t out_stride, const void* r, int64_t r_stride, const void* k, int64_t k_stride,
                        const void* v, int64_t v_stride, const void* g, int64_t g_stride, const float* decay,
                        const float* remove, const float* norm_w, float* state, int64_t state_stride, const SeqBatch& s,
                        int H, int K, float eps, hipStream_t st) {
  const dim3 grid((unsigned)s.B, (unsigned)H);
#define SP_DELTA(KP)                                                                                                    \
  delta_recurrence_kernel<Tag, KP><<<grid, (unsigned)(KP * delta_split(KP) < 64 ? 64 : KP * delta_split(KP)), 0, st>>>(  \
      out, out_stride, r, r_stride, k, k_stride, v, v_stride, g, g_stride, decay, remove, norm_w, state, state_stride, s, H, K, \
      eps)
  if (K <= 16) SP_DELTA(16);
  else if (K <= 32) SP_DELTA(32);
  else if (K <= 64) SP_DELTA(64);
  else if (K <= 128) SP_DELTA(128);
  else if (K <= 256) SP_DELTA(256);
  else return SP_ERR_UNSUPPORTED;
#undef SP_DELTA
  SP_LAUNCH_CHECK();
  return SP_OK;
}

// ---- steps of several tokens per request, 16 tokens at a time on the matrix cores (chunk16.h: u the unit key, b = remove * u) ----------
// The per-token form above is a chain of a sweep over the column and two sums over its lanes per token.  32 heads of 64 (width 2048), us per
// layer: one request of 4096 tokens 2309 -> 1010 (the walk 625: 2.4 per chunk; prepare 80, gates 57), 4 requests of 4096 tokens together
// 835 -> 531, 16 of them 558 -> 497.  Heads of 128 stay with the per-token form (their operands and state crowd the registers).
template <typename Tag, int D>
__global__ void __launch_bounds__(256)
delta_prepare_kernel(float* work, const char* r, int64_t r_stride, const char* k, int64_t k_stride, const float* decay, const float* remove,
                     SeqBatch s, int H) {
  typedef Elem<Tag> E;
  constexpr int V = E::kVec, QP = D / V;
  const int h = blockIdx.y;
  int b, t0;
  if (!segment_at(s, (int)blockIdx.x, kC16, threadIdx.x & 63, b, t0)) return;
  const int64_t row0 = (int64_t)s.extend_start_loc[b] + t0;
  const int n = s.extend_seq_lens[b] - t0;
  chunk16_prepare<D, true>(work + ((int64_t)blockIdx.x * H + h) * Chunk16<D, true>::kFloats,
                           [&](auto& sr, auto& sk, auto& sw, auto& su, auto& sb) {
    for (int e = threadIdx.x; e < kC16 * QP; e += 256) {               // (whole groups of QP lanes)
      const int t = e / QP, i = e % QP * V, c = h * D + i;
      float rf[V], kf[V], k2 = 0.f;
      const u32x4 zero = {0u, 0u, 0u, 0u};
      unpack16<Tag>(t < n ? ld16(r + ((row0 + t) * r_stride + c) * E::kBytes) : zero, rf);
      unpack16<Tag>(t < n ? ld16(k + ((row0 + t) * k_stride + c) * E::kBytes) : zero, kf);
#pragma unroll
      for (int x = 0; x < V; ++x) k2 += kf[x] * kf[x];
      k2 = lanes_sum<(QP < 16 ? QP : 16)>(k2);
      if constexpr (QP == 32) k2 += __shfl_xor(k2, 16, 64);
      const float inv = 1.f / sqrtf(k2 + 1e-6f);
#pragma unroll
      for (int x = 0; x < V; x += 4) {
        const int64_t at = (row0 + t) * H * D + c + x;
        const f32x4_c w = t < n ? *(const f32x4_c*)(decay + at) : f32x4_c{1.f, 1.f, 1.f, 1.f};
        const f32x4_c a = t < n ? *(const f32x4_c*)(remove + at) : f32x4_c{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int z = 0; z < 4; ++z) {
          const float u = kf[x + z] * inv;
          sr[t][i + x + z] = rf[x + z];
          sk[t][i + x + z] = kf[x + z];
          sw[t][i + x + z] = w[z];
          su[t][i + x + z] = u;
          sb[t][i + x + z] = a[z] * u;
        }
      }
    }
  });
}

template <typename Tag>
static int launch_delta_chunks16(Tag, const Walk16& w, float* work, const void* r, int64_t r_stride, const void* k, int64_t k_stride,
                                 const float* decay, const float* remove, int64_t num_tokens, const SeqBatch& step, hipStream_t st) {
  return each_window16(work, num_tokens, w.H, Chunk16<64, true>::kFloats, step, st, [&](const SeqBatch& s, int64_t units, int64_t tokens) -> int {
    delta_prepare_kernel<Tag, 64><<<dim3((unsigned)units, (unsigned)w.H), 256, 0, st>>>(
        work, (const char*)r, r_stride, (const char*)k, k_stride, decay, remove, s, w.H);
    SP_LAUNCH_CHECK();
    return launch_walk16<Tag, 64, 4, true>(w, tokens, s, st);
  });
}

}  // namespace
}  // namespace sp

using namespace sp;

extern "C" int sp_delta_gates(float* decay, float* remove, const void* p, int64_t p_stride, const float* w2t, const float* w0,
                              const void* apre, int64_t a_stride, const float* a_bias, int64_t num_tokens, int channels,
                              int rank, float rate, int dtype, void* stream) {
  SP_CHECK_ARG(num_tokens >= 0 && channels > 0 && rank > 0 && rank <= 8192);
  if (num_tokens == 0) return SP_OK;
  SP_CHECK_ARG(decay && remove && p && w2t && w0 && apre && a_bias && p_stride >= rank && a_stride >= channels);
  const unsigned cb = (unsigned)((channels + kBlock - 1) / kBlock);
  if (num_tokens >= 64 && rank <= 1024) {
    SP_DISPATCH_DTYPE(dtype, (delta_gates_kernel<Tag, 8><<<dim3((unsigned)((num_tokens + 7) / 8), cb), kBlock,
                                                            8 * rank * sizeof(float), (hipStream_t)stream>>>(
                                 decay, remove, p, p_stride, w2t, w0, apre, a_stride, a_bias, num_tokens, channels, rank, rate)));
  } else {
    SP_DISPATCH_DTYPE(dtype, (delta_gates_kernel<Tag, 1><<<dim3((unsigned)num_tokens, cb), kBlock, rank * sizeof(float),
                                                            (hipStream_t)stream>>>(
                                 decay, remove, p, p_stride, w2t, w0, apre, a_stride, a_bias, num_tokens, channels, rank, rate)));
  }
  SP_LAUNCH_CHECK();
  return SP_OK;
}

extern "C" int sp_delta_recurrence(void* out, int64_t out_stride, const void* r, int64_t r_stride, const void* k,
                                   int64_t k_stride, const void* v, int64_t v_stride, const void* g, int64_t g_stride,
                                   const float* decay, const float* remove, const float* norm_w, float* state,
                                   int64_t state_stride, int heads, int head_dim, float eps, SP_SEQ_PARAMS, int dtype,
                                   void* stream) {
  SP_CHECK_ARG(batch_size >= 0 && heads > 0 && head_dim > 0);
  if (batch_size == 0) return SP_OK;
  SP_CHECK_ARG(out && r && k && v && g && decay && remove && norm_w && state && req_pool_indices && seq_lens);
  SP_CHECK_ARG(!extend_seq_lens || (extend_prefix_lens && extend_start_loc));
  SP_CHECK_ARG(state_stride >= (int64_t)heads * head_dim * head_dim);
  const int64_t n = (int64_t)heads * head_dim;
  SP_CHECK_ARG(r_stride >= n && k_stride >= n && v_stride >= n && g_stride >= n && out_stride >= n);
  SEQ_BATCH(s);
  SP_DISPATCH_DTYPE(dtype, return (launch_delta<Tag>(out, out_stride, r, r_stride, k, k_stride, v, v_stride, g, g_stride, decay,
                                                     remove, norm_w, state, state_stride, s, heads, head_dim, eps,
                                                     (hipStream_t)stream)));
}

extern "C" int64_t sp_delta_recurrence_chunk_floats(int64_t num_tokens, int batch_size, int heads, int head_dim) {
  return head_dim == 64 && heads > 0 ? chunk16_work_floats(num_tokens, batch_size, heads, Chunk16<64, true>::kFloats) : 0;
}

extern "C" int sp_delta_recurrence_chunks(void* out, int64_t out_stride, const void* r, int64_t r_stride, const void* k, int64_t k_stride,
                                          const void* v, int64_t v_stride, const void* g, int64_t g_stride, const float* decay,
                                          const float* remove, const float* norm_w, float* state, int64_t state_stride, float* work,
                                          int64_t num_tokens, int heads, int head_dim, float eps, SP_SEQ_PARAMS, int dtype, void* stream) {
  SP_CHECK_ARG(batch_size >= 0 && num_tokens >= 0 && heads > 0 && head_dim > 0);
  if (batch_size == 0 || num_tokens == 0) return SP_OK;
  SP_CHECK_ARG(out && r && k && v && g && decay && remove && norm_w && state && work && req_pool_indices && seq_lens);
  SP_CHECK_ARG(!extend_seq_lens || (extend_prefix_lens && extend_start_loc));
  SP_CHECK_ARG(state_stride >= (int64_t)heads * head_dim * head_dim);
  const int64_t n = (int64_t)heads * head_dim;
  SP_CHECK_ARG(r_stride >= n && k_stride >= n && v_stride >= n && g_stride >= n && out_stride >= n);
  SEQ_BATCH(s);
  if (!extend_seq_lens || head_dim != 64 || heads > 65535 || !rows_aligned(r, r_stride, dtype) ||
      !rows_aligned(k, k_stride, dtype) || !rows_aligned(v, v_stride, dtype) || !rows_aligned(g, g_stride, dtype) ||
      (((uintptr_t)decay | (uintptr_t)remove | (uintptr_t)work) & 15) ||
      chunk16_units(num_tokens, batch_size) >> 31)
    return SP_ERR_UNSUPPORTED;
  const Walk16 w{out, v, g, norm_w, work, state, out_stride, v_stride, g_stride, state_stride, ScanSegments{nullptr, 0, 0}, heads, eps,
                 rows_aligned(out, out_stride, dtype)};
  SP_DISPATCH_DTYPE(dtype, return (launch_delta_chunks16(Tag(), w, work, r, r_stride, k, k_stride, decay, remove, num_tokens, s,
                                                         (hipStream_t)stream)));
}

extern "C" int sp_delta_step(void* out, int64_t out_stride, const void* r, int64_t r_stride, const void* k, int64_t k_stride,
                             const void* v, int64_t v_stride, const void* g, int64_t g_stride, const void* p, int64_t p_stride,
                             const void* apre, int64_t a_stride, const float* w2t, const float* w0, const float* a_bias, int rank,
                             float rate, const float* norm_w, float* state, int64_t state_stride, int heads, int head_dim,
                             float eps, SP_SEQ_PARAMS, int dtype, void* stream) {
  SP_CHECK_ARG(batch_size >= 0 && heads > 0 && head_dim > 0 && rank > 0);
  if (batch_size == 0) return SP_OK;
  SP_CHECK_ARG(out && r && k && v && g && p && apre && w2t && w0 && a_bias && norm_w && state && req_pool_indices && seq_lens);
  SP_CHECK_ARG(!extend_seq_lens && state_stride >= (int64_t)heads * head_dim * head_dim && p_stride >= rank);
  const int64_t n = (int64_t)heads * head_dim;
  SP_CHECK_ARG(r_stride >= n && k_stride >= n && v_stride >= n && g_stride >= n && out_stride >= n && a_stride >= n);
  if ((head_dim != 64 && head_dim != 128) || rank > kStepRank || heads > 65535) return SP_ERR_UNSUPPORTED;
  SEQ_BATCH(s);
  const dim3 grid((unsigned)batch_size, (unsigned)heads);
#define SP_STEP(K, PARTS)                                                                                                    \
  SP_DISPATCH_DTYPE(dtype, (delta_step_kernel<Tag, K, PARTS><<<grid, K * PARTS, 0, (hipStream_t)stream>>>(                   \
                               out, out_stride, r, r_stride, k, k_stride, v, v_stride, g, g_stride, p, p_stride, apre, a_stride, \
                               w2t, w0, a_bias, rank, rate, norm_w, state, state_stride, s, heads, eps)))
  if (head_dim == 64) SP_STEP(64, 8);
  else SP_STEP(128, 8);
#undef SP_STEP
  SP_LAUNCH_CHECK();
  return SP_OK;
}
