// Channel-gated delta rule: a per-head matrix state S [D, Dv] whose rows (key channels) each have a decay of their own,
// corrected along the unit key.  Per value head h (its query/key head is h / (H / G)), all of the recurrence in fp32:
//   qn = q / sqrt(|q|^2 + 1e-6) * D^(-1/2)       kn = k / sqrt(|k|^2 + 1e-6)        beta = sigmoid(bpre)
//   S  = diag(w) S                                (w: the token's decay per key channel)
//   u  = beta (v - S^T kn)                        (what the state does not yet return for this key)
//   S  = S + kn u^T                               o = S^T qn       (the read-out sees the token's own write)
//   out = o / rms_head(o) * norm_w * gate         (norm_w [Dv] shared by the heads, gate fp32 per value channel)
// Decay and gate come from sp_lowrank_gate, an fp32 product with a low-rank projection's output p [T, rank]:
//   z = W2 p + bias;   decay = exp(-exp(A_log[head]) softplus(z))   or   gate = sigmoid(z).
//
// One workgroup per (request, value head): a column of S (one value channel) lives in the registers of SP neighbouring
// lanes; the request's tokens of this step are walked in order from the state the previous step left in the pool (zeros at
// a sequence's first token), staged through LDS in passes.  A token costs ONE sweep over the column: the update, the
// read-out and - on the state just completed - the next token's (w * kn)^T S, then two independent sums over the column's
// lanes (register moves); no workgroup barrier inside a pass.  The order of its sums depends on the head's sizes only.
//
// Decode steps and short portions take that path, longer ones (by the mean tokens per request, the head's sizes and their number; of
// the sizes that chunk_delta.h takes) the 16-token chunks of sp_gated_delta_chunks, whose sums associate by a token's place in its
// portion: a request's roundings depend on how its prompt was cut and, through the mean, on the lengths of the others in the step.
#include "chunk_delta.h"
#include "chunk_scan.h"

namespace sp {
namespace {

// log(1 + e), e in [0, 1], as 2 atanh(e / (2 + e)) = s (1 + z / 3 + z^2 / 5 + ...), s = 2 e / (2 + e) <= 2/3, z = s^2 / 4: the terms
// past z^7 are 2e-9 of it.  s takes the hardware's reciprocal and then what its division leaves (and the rounding of 2 + e); what s
// itself rounds away (`rest`) is added last, 0.6 ulp in all.  The library's log1p is as exact in four times the instructions: 36.7
// against 22.0 us for the decays of 4096 tokens x 2048 channels.
__device__ __forceinline__ float log1p_unit(float e) {
#pragma clang fp contract(off)                         // (s - q is what the sum rounded away, not what q did)
  const float d = 2.f + e, low = e - (d - 2.f), r = __builtin_amdgcn_rcpf(d), q = (e + e) * r;
  const float left = fmaf(-low, q, fmaf(-d, q, e + e)) * r, s = q + left, rest = left - (s - q), z = 0.25f * s * s;
  float p = fmaf(1.f / 15.f, z, 1.f / 13.f);
  p = fmaf(p, z, 1.f / 11.f);
  p = fmaf(p, z, 1.f / 9.f);
  p = fmaf(p, z, 1.f / 7.f);
  p = fmaf(p, z, 1.f / 5.f);
  p = fmaf(p, z, 1.f / 3.f);
  return s + fmaf(s * z, p, rest);
}
__device__ __forceinline__ float softplus_gd(float z) { return fmaxf(z, 0.f) + log1p_unit(expf(-fabsf(z))); }

// w2t: [rank, channels] fp32 (the up-projection transposed: neighbouring threads read neighbouring channels).  A workgroup
// takes TPB tokens x 256 channels, a thread one channel: every weight it loads serves all TPB tokens.
// ACT 0: exp(-exp(A_log[c / per_head]) softplus(z));  ACT 1: sigmoid(z)
// (one function for both forms below: a portion of a prompt may take either.  A decay near 1 repeats over a prompt: log(1 + e^z) in
// place of log1p has lost e^z's low bits there, all of them from z = -17 down)
template <int ACT>
__device__ __forceinline__ float gate_value(float z, float rate) {
  return ACT == 0 ? expf(-rate * softplus_gd(z)) : over_one_plus_exp(1.f, z);
}

template <typename Tag, int TPB, int ACT>
__global__ void __launch_bounds__(kBlock)
lowrank_gate_kernel(float* out, const void* p, int64_t p_stride, const float* w2t, const float* bias, const float* A_log,
                    int64_t T, int channels, int rank, int per_head) {
  typedef Elem<Tag> E;
  extern __shared__ float tp[];                          // [TPB][rank]
  const int64_t t0 = (int64_t)blockIdx.x * TPB;
  const int c = blockIdx.y * kBlock + threadIdx.x;
  for (int e = threadIdx.x; e < TPB * rank; e += kBlock) {
    const int tt = e / rank, r = e % rank;
    tp[e] = t0 + tt < T ? E::load(p, (t0 + tt) * p_stride + r) : 0.f;
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
  const float b = bias ? bias[c] : 0.f;
  const float rate = ACT == 0 ? expf(A_log[c / per_head]) : 0.f;
#pragma unroll
  for (int tt = 0; tt < TPB; ++tt) {
    const int64_t t = t0 + tt;
    if (t < T) out[t * channels + c] = gate_value<ACT>(acc[tt] + b, rate);
  }
}

// The same for steps of many tokens, bf16 rows and ranks that are multiples of 32, up to 128: the product on the matrix cores.  A
// wave keeps 16 channels of w2t as three bf16 parts each (an exact split, chunk_scan.h) and walks `run` tokens, 16 at a time:
// p's rows are the other operand as they lie, a lane ends with 4 neighbouring channels of a token.  One channel per thread was bound
// by its LDS reads (one per 4 multiply-adds): 51 us for 4096 tokens x 2048 channels of rank 64, 22 here (16 for a sigmoid).
// Where that leaves the chip idle a wave walks fewer: 128 tokens each were a chain of 8 products, exponentials and stores whatever the
// step's size, longer than the form above in small ones (decays, rank 64: 128 tokens x 2048 channels 7.7 above, 10.3 with 128, 4.2 now; 512 x
// 1024 8.0, 10.4, 4.8).
constexpr int kGateTokens = 128, kGateGroups = 512;      // tokens per wave at the most; workgroups that fill the chip

template <int RANK, int ACT>
__global__ void __launch_bounds__(kBlock)
lowrank_gate_mfma_kernel(float* out, const char* p, int64_t p_stride, const float* w2t, const float* bias, const float* A_log,
                         int64_t T, int channels, int per_head, int run) {
  const int lane = threadIdx.x & 63, r16 = lane & 15, q = lane >> 4;
  const int c0 = (blockIdx.y * (kBlock / 64) + (threadIdx.x >> 6)) * 16;
  if (c0 >= channels) return;                          // (channels is a multiple of 16)
  u32x4 w[RANK / 32][3];
#pragma unroll
  for (int kk = 0; kk < RANK / 32; ++kk) {
    float f[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) f[e] = w2t[(int64_t)(32 * kk + 8 * q + e) * channels + c0 + r16];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      uint32_t hi, mid, lo;
      split3(f[2 * e], f[2 * e + 1], hi, mid, lo);
      w[kk][0][e] = hi, w[kk][1][e] = mid, w[kk][2][e] = lo;
    }
  }
  float b[4], rate[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    b[r] = bias ? bias[c0 + 4 * q + r] : 0.f;
    rate[r] = ACT == 0 ? expf(A_log[(c0 + 4 * q + r) / per_head]) : 0.f;
  }
  const int64_t t1 = (int64_t)(blockIdx.x + 1) * run < T ? (int64_t)(blockIdx.x + 1) * run : T;
  for (int64_t t0 = (int64_t)blockIdx.x * run; t0 < t1; t0 += 16) {
    const int64_t t = t0 + r16 < t1 ? t0 + r16 : t1 - 1;
    f32x4_c z = {b[0], b[1], b[2], b[3]};
#pragma unroll
    for (int kk = 0; kk < RANK / 32; ++kk) {
      const u32x4 x = ld16(p + (t * p_stride + 32 * kk + 8 * q) * 2);
#pragma unroll
      for (int part = 2; part >= 0; --part) z = mfma_c(w[kk][part], x, z);
    }
    if (t0 + r16 < t1) {
      f32x4_c o;
#pragma unroll
      for (int r = 0; r < 4; ++r) {                    // an infinity's parts are not numbers: such a sum is formed again as it is
        if (fabsf(z[r]) < INFINITY) continue;
        const int c = c0 + 4 * q + r;
        float sum = b[r];
        for (int x = 0; x < RANK; ++x) sum += w2t[(int64_t)x * channels + c] * Elem<bf16_tag>::load(p, t * p_stride + x);
        z[r] = sum;
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) o[r] = gate_value<ACT>(z[r], rate[r]);
      *(f32x4_c*)(out + t * channels + c0 + 4 * q) = o;
    }
  }
}

constexpr int gd_chunk(int KP) { return KP > 64 ? 8 : 16; }       // tokens staged in LDS per pass
constexpr int kGdMaxV = 256;                                      // value channels per head

// thread = (column col of S, part): part p of SP owns the rows [p DS, (p + 1) DS) of the column (DS = KP / SP, KP = the
// key width rounded up).  LDS rows are padded by 4 floats per part so that the parts' simultaneous broadcast reads fall
// into different banks.  The workgroup has ceil(Dv SP / 64) waves.
template <typename Tag, int KP, int SP>
__global__ void __launch_bounds__(1024)
gated_delta_scan_kernel(void* out, int64_t out_stride, const void* q, int64_t q_stride, const void* k, int64_t k_stride,
                        const void* v, int64_t v_stride, const void* bpre, int64_t b_stride, const float* decay,
                        const float* gate, const float* norm_w, float* state, int64_t state_stride, SeqBatch s, int H, int G,
                        int K, int Dv, float eps) {
  typedef Elem<Tag> E;
  constexpr int kChunk = gd_chunk(KP), DS = KP / SP, ROW = KP + 4 * SP;
  static_assert(DS % 4 == 0, "a part's rows are read four at a time");
  __shared__ __attribute__((aligned(16))) float sq[kChunk][ROW], sk[kChunk][ROW], sw[kChunk][ROW], sgk[kChunk + 1][ROW];
  __shared__ float sv[kChunk][kGdMaxV], so[kChunk][kGdMaxV], sbeta[kChunk], sinv[kChunk];
  const int b = blockIdx.x, h = blockIdx.y, j = threadIdx.x, NT = blockDim.x;
  const int wave = j >> 6, lane = j & 63, waves = NT >> 6;
  const int col = j / SP, part = j % SP;
  int64_t start, len, prefix;
  seq_span(s, b, start, len, prefix);
  if (len <= 0) return;
  const bool live = col < Dv;
  const int g = h / (H / G);
  float* st = state + load_idx(s.req_pool_indices, b, s.idx64) * state_stride + (int64_t)h * K * Dv;
  const bool held = prefix > 0;
  const int64_t qc = (int64_t)g * K, wc = (int64_t)h * K, vc = (int64_t)h * Dv, HK = (int64_t)H * K, HV = (int64_t)H * Dv;
  const int mine = part * (DS + 4);
  const float qscale = 1.f / sqrtf((float)K);
  float S[DS];
#pragma unroll
  for (int ii = 0; ii < DS; ++ii) {
    const int i = part * DS + ii;
    S[ii] = (live && i < K && held) ? st[(int64_t)i * Dv + col] : 0.f;
  }
  const float nw = live ? norm_w[col] : 0.f;
  for (int64_t c0 = 0; c0 < len; c0 += kChunk) {
    const int n = (int)(len - c0 < kChunk ? len - c0 : kChunk);
    __syncthreads();                                     // the previous pass's epilogue is done with so and sinv
    for (int e = j; e < n * KP; e += NT) {
      const int tt = e / KP, i = e % KP;
      const int at = i + 4 * (i / DS);
      const int64_t row = start + c0 + tt;
      const bool ok = i < K;
      sq[tt][at] = ok ? E::load(q, row * q_stride + qc + i) : 0.f;
      sk[tt][at] = ok ? E::load(k, row * k_stride + qc + i) : 0.f;
      sw[tt][at] = ok ? decay[row * HK + wc + i] : 0.f;
    }
    for (int e = j; e < n * Dv; e += NT) {
      const int tt = e / Dv, i = e % Dv;
      sv[tt][i] = E::load(v, (start + c0 + tt) * v_stride + vc + i);
    }
    if (j < n) sbeta[j] = over_one_plus_exp(1.f, E::load(bpre, (start + c0 + j) * b_stride + h));
    __syncthreads();
    // unit query and key of every token of the pass, and the decayed key: a wave per token
    for (int tt = wave; tt < n; tt += waves) {
      float sk2 = 0.f, sq2 = 0.f;
      for (int i = lane; i < K; i += 64) {
        const int at = i + 4 * (i / DS);
        sk2 += sk[tt][at] * sk[tt][at];
        sq2 += sq[tt][at] * sq[tt][at];
      }
      sk2 = wave_sum(sk2);
      sq2 = wave_sum(sq2);
      const float ik = 1.f / sqrtf(sk2 + 1e-6f), iq = qscale / sqrtf(sq2 + 1e-6f);
      for (int i = lane; i < KP; i += 64) {
        const int at = i + 4 * (i / DS);
        const float kn = sk[tt][at] * ik;
        sk[tt][at] = kn;
        sq[tt][at] *= iq;
        sgk[tt][at] = kn * sw[tt][at];
      }
    }
    __syncthreads();
    // (w * kn)^T S of the pass's first token; every later token's is formed in the sweep that completes the state it reads
    float proj;
    {
      const float4* pu = reinterpret_cast<const float4*>(&sgk[0][mine]);
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
      const float4* pw = reinterpret_cast<const float4*>(&sw[tt][mine]);
      const float4* pk = reinterpret_cast<const float4*>(&sk[tt][mine]);
      const float4* pq = reinterpret_cast<const float4*>(&sq[tt][mine]);
      const float4* pun = reinterpret_cast<const float4*>(&sgk[tt + 1][mine]);     // the next token's (row n: unused)
      const float u = live ? sbeta[tt] * (sv[tt][col] - proj) : 0.f;
      float nm[4] = {0.f, 0.f, 0.f, 0.f}, pj[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ii = 0; ii < DS; ii += 4) {
        const float4 w4 = pw[ii / 4], k4 = pk[ii / 4], q4 = pq[ii / 4], u4 = pun[ii / 4];
        S[ii] = w4.x * S[ii] + k4.x * u;
        S[ii + 1] = w4.y * S[ii + 1] + k4.y * u;
        S[ii + 2] = w4.z * S[ii + 2] + k4.z * u;
        S[ii + 3] = w4.w * S[ii + 3] + k4.w * u;
        nm[0] += S[ii] * q4.x;
        nm[1] += S[ii + 1] * q4.y;
        nm[2] += S[ii + 2] * q4.z;
        nm[3] += S[ii + 3] * q4.w;
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
    // per-head RMS of o, then the output weight and gate
    for (int tt = wave; tt < n; tt += waves) {
      float ss = 0.f;
      for (int i = lane; i < Dv; i += 64) ss += so[tt][i] * so[tt][i];
      ss = wave_sum(ss);
      if (lane == 0) sinv[tt] = 1.f / sqrtf(ss / (float)Dv + eps);
    }
    __syncthreads();
    for (int e = j; e < n * Dv; e += NT) {
      const int tt = e / Dv, i = e % Dv;
      const int64_t row = start + c0 + tt;
      E::store(out, row * out_stride + vc + i, so[tt][i] * sinv[tt] * norm_w[i] * gate[row * HV + vc + i]);
    }
  }
  (void)nw;
  if (live) {
#pragma unroll
    for (int ii = 0; ii < DS; ++ii) {
      const int i = part * DS + ii;
      if (i < K) st[(int64_t)i * Dv + col] = S[ii];
    }
  }
}

// out[t, h] = raw[t, h] / rms * norm_w * gate[t, h]: a wave per (token, head)
template <typename Tag>
__global__ void __launch_bounds__(kBlock)
gated_norm_kernel(void* out, int64_t out_stride, const float* raw, const float* gate, const float* norm_w, int H, int Dv, float eps,
                  int64_t jobs) {
  typedef Elem<Tag> E;
  const int lane = threadIdx.x & 63;
  const int64_t job = (int64_t)blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6);
  if (job >= jobs) return;
  const int64_t t = job / H, h = job % H;
  float f[kGdMaxV / 64], ss = 0.f;
#pragma unroll
  for (int u = 0; u < kGdMaxV / 64; ++u) {
    const int i = lane + 64 * u;
    f[u] = i < Dv ? raw[job * Dv + i] : 0.f;
    ss += f[u] * f[u];
  }
  const float inv = 1.f / sqrtf(wave_sum(ss) / (float)Dv + eps);
#pragma unroll
  for (int u = 0; u < kGdMaxV / 64; ++u) {
    const int i = lane + 64 * u;
    if (i < Dv) E::store(out, t * out_stride + h * Dv + i, f[u] * inv * norm_w[i] * gate[job * Dv + i]);
  }
}

// The same with the gate sigmoid(p w2t) formed on the spot (bf16 rows, RANK 32 or 64, heads of 16 TILES values): a workgroup keeps its head's
// columns of w2t in LDS as three bf16 parts each, in the order the matrix instructions take them, and a wave takes 16 tokens - a lane ends with 4
// neighbouring channels of every tile of its token, the head's sum of squares is over the four lanes of a token.  Memory bounds it: read-outs
// in, results out.  The gates as a launch of their own are written and read once more in fp32: 4096 tokens of 16 heads of 128, rank 64, 16.2 us
// for the gates and 19.5 for the norm; together 20.6.
constexpr int kGateNormWaves = 8;
template <int RANK, int TILES>
__global__ void __launch_bounds__(kGateNormWaves * 64)
gated_norm_lowrank_kernel(char* out, int64_t out_stride, const float* raw, const char* p, int64_t p_stride, const float* w2t,
                          const float* norm_w, int64_t T, int H, float eps) {
  constexpr int Dv = TILES * 16, KS = RANK / 32, FRAGS = KS * TILES * 64;
  __shared__ u32x4 parts[3][FRAGS];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, r16 = lane & 15, q = lane >> 4, h = blockIdx.y;
  const int64_t channels = (int64_t)H * Dv, t = ((int64_t)blockIdx.x * kGateNormWaves + wave) * 16 + r16, tt = t < T ? t : T - 1;
  // this wave's rows are on their way while the weights are split
  f32x4_c o[TILES];
  u32x4 x[KS];
#pragma unroll
  for (int kk = 0; kk < KS; ++kk) x[kk] = ld16(p + (tt * p_stride + 32 * kk + 8 * q) * 2);
#pragma unroll
  for (int i = 0; i < TILES; ++i) o[i] = *(const f32x4_c*)(raw + (tt * H + h) * Dv + 16 * i + 4 * q);
  for (int f = tid; f < FRAGS; f += kGateNormWaves * 64) {
    const int l = f & 63, i = (f >> 6) % TILES, kk = (f >> 6) / TILES;
    const float* from = w2t + (int64_t)(32 * kk + 8 * (l >> 4)) * channels + h * Dv + 16 * i + (l & 15);
    float w[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) w[e] = from[e * channels];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      uint32_t hi, mid, lo;
      split3(w[2 * e], w[2 * e + 1], hi, mid, lo);
      parts[0][f][e] = hi, parts[1][f][e] = mid, parts[2][f][e] = lo;
    }
  }
  __syncthreads();
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < TILES; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) ss += o[i][r] * o[i][r];
  ss += __shfl_xor(ss, 16, 64);
  ss += __shfl_xor(ss, 32, 64);
  const float inv = 1.f / sqrtf(ss / (float)Dv + eps);
#pragma unroll
  for (int i = 0; i < TILES; ++i) {
    f32x4_c z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < KS; ++kk)
#pragma unroll
      for (int part = 2; part >= 0; --part) z = mfma_c(parts[part][(kk * TILES + i) * 64 + lane], x[kk], z);
    const f32x4_c nw = *(const f32x4_c*)(norm_w + 16 * i + 4 * q);
    float y[8] = {};
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (!(fabsf(z[r]) < INFINITY)) {                 // an infinity's parts are not numbers: such a sum is formed again as it is
        float sum = 0.f;
        for (int k = 0; k < RANK; ++k)
          sum += w2t[k * channels + h * Dv + 16 * i + 4 * q + r] * Elem<bf16_tag>::load(p, tt * p_stride + k);
        z[r] = sum;
      }
      y[r] = o[i][r] * inv * nw[r] * gate_value<1>(z[r], 0.f);
    }
    const u32x4 two = pack16<bf16_tag>(y);
    if (t < T) *(u32x2*)(out + (t * out_stride + h * Dv + 16 * i + 4 * q) * 2) = u32x2{two[0], two[1]};
  }
}

template <typename Tag>
static int launch_gated_delta(void* out, int64_t out_stride, const void* q, int64_t q_stride, const void* k, int64_t k_stride,
                              const void* v, int64_t v_stride, const void* bpre, int64_t b_stride, const float* decay,
                              const float* gate, const float* norm_w, float* state, int64_t state_stride, const SeqBatch& s,
                              int H, int G, int K, int Dv, float eps, hipStream_t st) {
  const dim3 grid((unsigned)s.B, (unsigned)H);
#define SP_GD(KP, SPL)                                                                                                   \
  gated_delta_scan_kernel<Tag, KP, SPL><<<grid, (unsigned)((Dv * SPL + 63) / 64 * 64), 0, st>>>(                          \
      out, out_stride, q, q_stride, k, k_stride, v, v_stride, bpre, b_stride, decay, gate, norm_w, state, state_stride, s, H, \
      G, K, Dv, eps)
  // lanes per column: 8 state values per lane where the workgroup's 1024 threads allow it
  const bool wide = Dv > 128;                            // 8 lanes per column would need more than 1024 threads
  if (K <= 16) SP_GD(16, 2);
  else if (K <= 32) SP_GD(32, 4);
  else if (K <= 64) { if (wide) SP_GD(64, 4); else SP_GD(64, 8); }
  else if (K <= 128) { if (wide) SP_GD(128, 4); else SP_GD(128, 8); }
  else if (K <= 256) SP_GD(256, 4);
  else return SP_ERR_UNSUPPORTED;
#undef SP_GD
  SP_LAUNCH_CHECK();
  return SP_OK;
}

}  // namespace
}  // namespace sp

using namespace sp;

extern "C" int sp_lowrank_gate(float* out, const void* p, int64_t p_stride, const float* w2t, const float* bias,
                               const float* A_log, int64_t num_tokens, int channels, int rank, int per_head, int act,
                               int dtype, void* stream) {
  SP_CHECK_ARG(num_tokens >= 0 && channels > 0 && rank > 0 && rank <= 8192 && (act == 0 || act == 1));
  if (num_tokens == 0) return SP_OK;
  SP_CHECK_ARG(out && p && w2t && p_stride >= rank);
  SP_CHECK_ARG(act != 0 || (A_log && per_head > 0 && channels % per_head == 0));
  const unsigned cb = (unsigned)((channels + kBlock - 1) / kBlock);
  if (per_head <= 0) per_head = 1;
  if (dtype == SP_BF16 && num_tokens >= 64 && (rank == 32 || rank == 64 || rank == 96 || rank == 128) && channels % 16 == 0 &&
      p_stride % 8 == 0 && (((uintptr_t)p | (uintptr_t)out) & 15) == 0) {
    const int64_t groups = (channels + kBlock / 4 - 1) / (kBlock / 4);
    int run = kGateTokens;
    while (run > 16 && (num_tokens + run - 1) / run * groups < kGateGroups) run /= 2;
    const dim3 grid((unsigned)((num_tokens + run - 1) / run), (unsigned)groups);
#define SP_LM(R, ACT)                                                                                                    \
  lowrank_gate_mfma_kernel<R, ACT><<<grid, kBlock, 0, (hipStream_t)stream>>>(out, (const char*)p, p_stride, w2t, bias, A_log, \
                                                                              num_tokens, channels, per_head, run)
#define SP_LM2(R)              \
  do {                         \
    if (act == 0) SP_LM(R, 0); \
    else SP_LM(R, 1);          \
  } while (0)
    if (rank == 32) SP_LM2(32);
    else if (rank == 64) SP_LM2(64);
    else if (rank == 96) SP_LM2(96);
    else SP_LM2(128);
#undef SP_LM2
#undef SP_LM
    SP_LAUNCH_CHECK();
    return SP_OK;
  }
#define SP_LG(TPB, ACT)                                                                                                  \
  SP_DISPATCH_DTYPE(dtype, (lowrank_gate_kernel<Tag, TPB, ACT><<<dim3((unsigned)((num_tokens + TPB - 1) / TPB), cb), kBlock, \
                                                                  TPB * rank * sizeof(float), (hipStream_t)stream>>>(     \
                               out, p, p_stride, w2t, bias, A_log, num_tokens, channels, rank, per_head)))
  if (num_tokens >= 64 && rank <= 1024) {
    if (act == 0) SP_LG(8, 0);
    else SP_LG(8, 1);
  } else {
    if (act == 0) SP_LG(1, 0);
    else SP_LG(1, 1);
  }
#undef SP_LG
  SP_LAUNCH_CHECK();
  return SP_OK;
}

extern "C" int sp_gated_delta_scan(void* out, int64_t out_stride, const void* q, int64_t q_stride, const void* k,
                                   int64_t k_stride, const void* v, int64_t v_stride, const void* bpre, int64_t b_stride,
                                   const float* decay, const float* gate, const float* norm_w, float* state,
                                   int64_t state_stride, int heads, int kv_heads, int dim, int vdim, float eps,
                                   SP_SEQ_PARAMS, int dtype, void* stream) {
  SP_CHECK_ARG(batch_size >= 0 && heads > 0 && kv_heads > 0 && heads % kv_heads == 0 && dim > 0 && vdim > 0);
  if (batch_size == 0) return SP_OK;
  SP_CHECK_ARG(out && q && k && v && bpre && decay && gate && norm_w && state && req_pool_indices && seq_lens);
  SP_CHECK_ARG(!extend_seq_lens || (extend_prefix_lens && extend_start_loc));
  SP_CHECK_ARG(state_stride >= (int64_t)heads * dim * vdim);
  SP_CHECK_ARG(q_stride >= (int64_t)kv_heads * dim && k_stride >= (int64_t)kv_heads * dim && b_stride >= heads);
  SP_CHECK_ARG(v_stride >= (int64_t)heads * vdim && out_stride >= (int64_t)heads * vdim);
  if (vdim > kGdMaxV) return SP_ERR_UNSUPPORTED;
  SEQ_BATCH(s);
  SP_DISPATCH_DTYPE(dtype, return (launch_gated_delta<Tag>(out, out_stride, q, q_stride, k, k_stride, v, v_stride, bpre, b_stride,
                                                           decay, gate, norm_w, state, state_stride, s, heads, kv_heads, dim,
                                                           vdim, eps, (hipStream_t)stream)));
}

// (gate: the gates themselves; else p [T, rank] and w2t [rank, heads * vdim])
static int gated_delta_chunks(void* out, int64_t out_stride, const void* q, int64_t q_stride, const void* k, int64_t k_stride, const void* v,
                              int64_t v_stride, const void* bpre, int64_t b_stride, const float* decay, const float* gate, const void* p,
                              int64_t p_stride, const float* w2t, int rank, const float* norm_w, float* state, int64_t state_stride,
                              float* work, float* raw, int64_t num_tokens, int heads, int kv_heads, int dim, int vdim, float eps,
                              SP_SEQ_PARAMS, int dtype, void* stream) {
  SP_CHECK_ARG(batch_size >= 0 && num_tokens >= 0 && heads > 0 && kv_heads > 0 && heads % kv_heads == 0 && dim > 0 && vdim > 0);
  if (batch_size == 0 || num_tokens == 0) return SP_OK;
  SP_CHECK_ARG(out && q && k && v && bpre && decay && (gate || (p && w2t && p_stride >= rank)) && norm_w && state && work && raw &&
               req_pool_indices && seq_lens);
  SP_CHECK_ARG(!extend_seq_lens || (extend_prefix_lens && extend_start_loc));
  SP_CHECK_ARG(state_stride >= (int64_t)heads * dim * vdim);
  SP_CHECK_ARG(q_stride >= (int64_t)kv_heads * dim && k_stride >= (int64_t)kv_heads * dim && b_stride >= heads);
  SP_CHECK_ARG(v_stride >= (int64_t)heads * vdim && out_stride >= (int64_t)heads * vdim);
  if (vdim > kGdMaxV) return SP_ERR_UNSUPPORTED;
  SEQ_BATCH(s);
  const DeltaChunks a{q, k, v, bpre, decay, nullptr, nullptr, nullptr, state, work, raw, q_stride, k_stride, v_stride, b_stride, 0,
                      state_stride, num_tokens, heads, kv_heads, vdim, vdim};
  if (!delta_chunks_take(a, dim, dtype, s)) return SP_ERR_UNSUPPORTED;
  if (!gate && (dtype != SP_BF16 || (rank != 32 && rank != 64) || (vdim != 64 && vdim != 128) || p_stride % 8 != 0 || out_stride % 4 != 0 ||
                ((((uintptr_t)p | (uintptr_t)raw | (uintptr_t)norm_w) & 15) | ((uintptr_t)out & 7)) || heads > 65535))
    return SP_ERR_UNSUPPORTED;
  hipStream_t st = (hipStream_t)stream;
  int rc = SP_OK;
  SP_DISPATCH_DTYPE(dtype, rc = (dim == 64 ? launch_delta_chunks<Tag, 64, true>(a, s, st) : launch_delta_chunks<Tag, 128, true>(a, s, st)));
  if (rc != SP_OK) return rc;
  if (!gate) {
    const dim3 grid((unsigned)((num_tokens + 16 * kGateNormWaves - 1) / (16 * kGateNormWaves)), (unsigned)heads);
#define SP_GN(R, TILES)                                                                                                         \
  gated_norm_lowrank_kernel<R, TILES><<<grid, kGateNormWaves * 64, 0, st>>>((char*)out, out_stride, raw, (const char*)p, p_stride, \
                                                                            w2t, norm_w, num_tokens, heads, eps)
    if (rank == 64 && vdim == 128) SP_GN(64, 8);
    else if (rank == 64) SP_GN(64, 4);
    else if (vdim == 128) SP_GN(32, 8);
    else SP_GN(32, 4);
#undef SP_GN
    SP_LAUNCH_CHECK();
    return SP_OK;
  }
  const int64_t jobs = num_tokens * heads;
  SP_DISPATCH_DTYPE(dtype, (gated_norm_kernel<Tag><<<dim3((unsigned)((jobs + kBlock / 64 - 1) / (kBlock / 64))), kBlock, 0, st>>>(
                               out, out_stride, raw, gate, norm_w, heads, vdim, eps, jobs)));
  SP_LAUNCH_CHECK();
  return SP_OK;
}

extern "C" int sp_gated_delta_chunks(void* out, int64_t out_stride, const void* q, int64_t q_stride, const void* k,
                                     int64_t k_stride, const void* v, int64_t v_stride, const void* bpre, int64_t b_stride,
                                     const float* decay, const float* gate, const float* norm_w, float* state, int64_t state_stride, float* work, float* raw,
                                     int64_t num_tokens, int heads, int kv_heads, int dim, int vdim, float eps, SP_SEQ_PARAMS, int dtype,
                                     void* stream) {
  SP_CHECK_ARG(gate || batch_size == 0 || num_tokens == 0);
  return gated_delta_chunks(out, out_stride, q, q_stride, k, k_stride, v, v_stride, bpre, b_stride, decay, gate, nullptr, 0, nullptr, 0, norm_w, state,
                            state_stride, work, raw, num_tokens, heads, kv_heads, dim, vdim, eps, req_pool_indices, seq_lens,
                            extend_seq_lens, extend_prefix_lens, extend_start_loc, token_req, idx64, batch_size, dtype, stream);
}

extern "C" int sp_gated_delta_chunks_lowrank(void* out, int64_t out_stride, const void* q, int64_t q_stride, const void* k,
                                             int64_t k_stride, const void* v, int64_t v_stride, const void* bpre, int64_t b_stride,
                                             const float* decay, const void* p, int64_t p_stride, const float* w2t, int rank,
                                             const float* norm_w, float* state, int64_t state_stride, float* work, float* raw,
                                             int64_t num_tokens, int heads, int kv_heads, int dim, int vdim, float eps, SP_SEQ_PARAMS, int dtype,
                                             void* stream) {
  SP_CHECK_ARG(rank > 0);
  return gated_delta_chunks(out, out_stride, q, q_stride, k, k_stride, v, v_stride, bpre, b_stride, decay, nullptr, p, p_stride, w2t, rank, norm_w, state,
                            state_stride, work, raw, num_tokens, heads, kv_heads, dim, vdim, eps, req_pool_indices, seq_lens,
                            extend_seq_lens, extend_prefix_lens, extend_start_loc, token_req, idx64, batch_size, dtype, stream);
}
