// Matrix-memory recurrence with exponential gating kept stable by a running maximum (the mLSTM cell of xLSTM).
// Per head, with log gates i and f of a token and state (S [D, Dv], n [D], m), all fp32:
//   i = cap tanh(ipre / cap)                 f = logsigmoid(cap tanh(fpre / cap))         (ipre, fpre: fp32 projections)
//   m' = max(f + m, i)
//   S' = exp(f + m - m') S + exp(i - m') k v^T          n' = exp(f + m - m') n + exp(i - m') k
//   o  = S'^T q / (max(|n' . q|, exp(-m')) + 1e-6)      q = (projection) * D^(-1/2)
//   out = o / rms_head(o) * w * sigmoid(g)
// S, n and m start at ZERO for a sequence (m too: not minus infinity).  One workgroup per (request, head): a column of S
// lives in the registers of 1, 2 or 4 neighbouring lanes and n is one more column, so a token costs no workgroup barrier
// and no sum over a wave; tokens are staged through LDS in passes and the per-head norm and gate run as the pass's epilogue.
#include "chunk_scan.h"

namespace sp {
namespace {

// tokens staged in LDS per pass (fewer for the widest heads: static + dynamic LDS stay under 64 KB)
constexpr int chunk_of(int DP) { return DP > 128 ? 8 : 16; }
// lanes that share one column of S: each holds 16 - 64 of the column's D values, so the state never crowds the register
// file (at 128 values per lane the compiler is at its 256-register limit with one wave per SIMD) and a head gives the
// chip more waves - the recurrence is a chain of waits per token, and idle SIMDs are what a prompt leaves most of
constexpr int split_of(int DP) { return DP > 64 ? 4 : (DP > 32 ? 2 : 1); }

__device__ __forceinline__ float logsigmoid_f(float z) { return fminf(z, 0.f) - log1pf(expf(-fabsf(z))); }

// thread = (column col of S, part): part p of SP owns the rows [p DS, (p + 1) DS) of the column; the parts of a column
// are neighbouring lanes and add their partial numerators by lane exchange.  LDS rows of q and k are padded by 4 floats
// per part so that the parts' simultaneous broadcast reads fall into different banks.
// The normaliser n is column Dv of the same recurrence (its "value" is 1): its lanes form n . q like any numerator, and
// the division by max(|n . q|, exp(-m)) + 1e-6 waits for the pass's epilogue - no sum over a wave inside the token loop.
template <typename Tag, int DP>
__global__ void __launch_bounds__(split_of(DP) == 1 ? 320 : (split_of(DP) == 2 ? 576 : 1024))
mlstm_scan_kernel(void* out, int64_t out_stride, const void* q, int64_t q_stride, const void* k, int64_t k_stride,
                  const void* v, int64_t v_stride, const void* g, int64_t g_stride, const float* ipre, const float* fpre,
                  int64_t gate_stride, const float* norm_w, float* S_state, int64_t S_stride, float* n_state, int64_t n_stride,
                  float* m_state, int64_t m_stride, SeqBatch s, int H, int D, int Dv, float cap, float eps) {
  typedef Elem<Tag> E;
  constexpr int kChunk = chunk_of(DP), SP = split_of(DP), DS = DP / SP, ROW = DP + 4 * SP;
  __shared__ float sq[kChunk][ROW], sk[kChunk][ROW], si[kChunk], sf[kChunk], sinv[kChunk], sden[kChunk], sm[kChunk];
  extern __shared__ float so[];                         // [kChunk][Dv + 1] numerators (column Dv: n . q), then [kChunk][Dv] values
  float* sv = so + (size_t)kChunk * (Dv + 1);           // (no global load inside the token loop)
  const int b = blockIdx.x, h = blockIdx.y, j = threadIdx.x;
  const int nthreads = blockDim.x, wave = j >> 6, lane = j & 63, waves = nthreads >> 6;
  const int col = j / SP, part = j % SP;
  int64_t start, len, prefix;
  seq_span(s, b, start, len, prefix);
  if (len <= 0) return;
  const bool live = col <= Dv, isn = col == Dv;         // column Dv is the normaliser
  const int64_t slot = load_idx(s.req_pool_indices, b, s.idx64);
  float* Sst = S_state + slot * S_stride + (int64_t)h * D * Dv;
  float* nst = n_state + slot * n_stride + (int64_t)h * D;
  float* mst = m_state + slot * m_stride + h;
  const bool held = prefix > 0;
  float S[DS];
#pragma unroll
  for (int ii = 0; ii < DS; ++ii) {
    const int i = part * DS + ii;
    S[ii] = (live && i < D && held) ? (isn ? nst[i] : Sst[(int64_t)i * Dv + col]) : 0.f;
  }
  float m = held ? mst[0] : 0.f;
  const float qscale = 1.f / sqrtf((float)D);
  const int64_t colk = (int64_t)h * D, colv = (int64_t)h * Dv;
  const float* myq = &sq[0][part * (DS + 4)];
  const float* myk = &sk[0][part * (DS + 4)];
  for (int64_t c0 = 0; c0 < len; c0 += kChunk) {
    const int n = (int)(len - c0 < kChunk ? len - c0 : kChunk);
    __syncthreads();
    // staging: every load of the pass is issued before the first is used (rows past the pass's end repeat its last row)
#pragma unroll
    for (int tt = 0; tt < kChunk; ++tt) {
      const int64_t row = start + c0 + (tt < n ? tt : n - 1);
      for (int i = j; i < DP; i += nthreads) {
        const bool ok = i < D;
        const int at = i + 4 * (i / DS);
        sq[tt][at] = ok ? E::load(q, row * q_stride + colk + i) * qscale : 0.f;
        sk[tt][at] = ok ? E::load(k, row * k_stride + colk + i) : 0.f;
      }
      for (int c = j; c < Dv; c += nthreads) sv[tt * Dv + c] = E::load(v, row * v_stride + colv + c);
    }
    if (j < n) {
      const int64_t row = start + c0 + j;
      si[j] = cap * tanhf(ipre[row * gate_stride + h] / cap);
      sf[j] = logsigmoid_f(cap * tanhf(fpre[row * gate_stride + h] / cap));
    }
    __syncthreads();
    for (int tt = 0; tt < n; ++tt) {
      const float ig = si[tt], fg = sf[tt];
      const float m_new = fmaxf(fg + m, ig);
      const float keep = expf(fg + m - m_new), take = expf(ig - m_new);
      m = m_new;
      const float tv = take * (isn ? 1.f : (live ? sv[tt * Dv + col] : 0.f));
      const float* kq = myk + tt * ROW;
      const float* qq = myq + tt * ROW;
      float num = 0.f;
#pragma unroll
      for (int ii = 0; ii < DS; ++ii) {
        S[ii] = keep * S[ii] + kq[ii] * tv;
        num += S[ii] * qq[ii];
      }
#pragma unroll
      for (int off = 1; off < SP; off <<= 1) num += __shfl_xor(num, off, 64);
      if (live && part == 0) so[tt * (Dv + 1) + col] = num;
      if (j == 0) sm[tt] = m_new;
    }
    __syncthreads();
    // the division, then the per-head RMS of every token of the pass (a wave per token, LDS only), then every column of
    // all tokens at once
    for (int tt = wave; tt < n; tt += waves) {
      const float den = 1.f / (fmaxf(fabsf(so[tt * (Dv + 1) + Dv]), expf(-sm[tt])) + 1e-6f);
      float ss = 0.f;
      for (int i = lane; i < Dv; i += 64) {
        const float o = so[tt * (Dv + 1) + i] * den;
        ss += o * o;
      }
      ss = wave_sum(ss);
      if (lane == 0) {
        sden[tt] = den;
        sinv[tt] = 1.f / sqrtf(ss / (float)Dv + eps);
      }
    }
    __syncthreads();
    if (col < Dv) {                                     // part p takes the tokens p, p + SP, ...
      const float nw = norm_w[colv + col];
      constexpr int PER = kChunk / SP;
      float gv[PER];
#pragma unroll
      for (int u = 0; u < PER; ++u) {
        const int tt = part + u * SP;
        gv[u] = E::load(g, (start + c0 + (tt < n ? tt : n - 1)) * g_stride + colv + col);
      }
#pragma unroll
      for (int u = 0; u < PER; ++u) {
        const int tt = part + u * SP;
        if (tt < n)
          E::store(out, (start + c0 + tt) * out_stride + colv + col,
                   over_one_plus_exp(so[tt * (Dv + 1) + col] * sden[tt] * sinv[tt] * nw, gv[u]));
      }
    }
  }
  if (live) {
#pragma unroll
    for (int ii = 0; ii < DS; ++ii) {
      const int i = part * DS + ii;
      if (i < D) {
        if (isn) nst[i] = S[ii];
        else Sst[(int64_t)i * Dv + col] = S[ii];
      }
    }
  }
  if (j == 0) mst[0] = m;
}

// ---- steps of several tokens per request, bf16 rows: 64 tokens at a time (chunk_scan.h) -------------------------------------
// With F the running sum of the log forget gates inside the chunk, b_s = i_s - F_s and G_t = max(m_0, max_{s <= t} b_s), the
// running maximum is m_t = F_t + G_t and the weight of token s at t is exp(b_s - G_t) <= 1, that of the old state
// exp(m_0 - G_t).  The normaliser n . q is a row sum of the weighted tiles plus n_0 . q.
// One workgroup of Dv / 16 waves per (request, head).  The per-token form is a chain of one token's exponentials, sums and
// lane exchanges (1.6 us per token: 1546 us at 3001 tokens of 5 requests, 16 heads of 128 x 128); this one takes 140 us there
// and 568 us for one request of 4096 tokens, 8.9 us per chunk: about 1500 vector instructions per wave at two waves per SIMD
// (the splits, the weights' exponentials, the epilogue) against 126 MFMAs and 0.5 MB of LDS reads.
template <int D, int NW, bool OUT = true>
struct MlstmLds {
  typedef ChunkScan<D, NW, OUT> C;
  static constexpr int kN = (C::kBytes + 15) / 16 * 16, kNq = kN + D * 4, kFloor = kNq + kCL * 4, kRed = kFloor + 2 * kCL * 4;
  static constexpr int kGates = (kRed + NW * kCL * 4 + 7) / 8 * 8;             // double [NW][3][kCL]: F, b and its running maximum of NW chunks
  static constexpr int kBytes = kGates + NW * 3 * kCL * 8;
};

// (heads of 64 x 64: registers for the two workgroups per CU that LDS has room for)
// In segments (see chunk_scan.h): MODE.
template <int D, int NW, int MODE>
__global__ void __launch_bounds__(NW * 64, MODE == kSegmentSums ? 4 : D == 64 ? 8 / NW : 1)
mlstm_chunk_kernel(void* out, int64_t out_stride, const char* q, int64_t q_stride, const char* k, int64_t k_stride, const char* v,
                   int64_t v_stride, const void* g, int64_t g_stride, const float* ipre, const float* fpre,
                   int64_t gate_stride, const float* norm_w, float* S_state, int64_t S_stride, float* n_state, int64_t n_stride,
                   float* m_state, int64_t m_stride, ScanSegments seg, SeqBatch s, int H, float cap, float eps) {
  constexpr bool OUT = MODE != kSegmentSums;
  typedef Elem<bf16_tag> E;
  typedef ChunkScan<D, NW, OUT> C;
  typedef MlstmLds<D, NW, OUT> L;
  constexpr int Dv = C::Dv, NT = C::NT;
  extern __shared__ __attribute__((aligned(16))) char chunk_lds[];
  C c(chunk_lds);
  const int h = blockIdx.y;
  int b = blockIdx.x, t0 = 0;
  if constexpr (MODE != kWholeRequests)
    if (!segment_at(s, (int)blockIdx.x, seg.tokens, c.lane, b, t0)) return;
  int64_t start, len, prefix;
  seq_span(s, b, start, len, prefix);
  if (len <= 0) return;
  const bool split = MODE != kWholeRequests && len > seg.tokens, final = t0 + seg.tokens >= len;
  if (MODE == kSegmentSums && final) return;
  float* sn = (float*)(chunk_lds + L::kN);
  float* snq = (float*)(chunk_lds + L::kNq);
  float* sfloor = (float*)(chunk_lds + L::kFloor);
  float* red = (float*)(chunk_lds + L::kRed);
  double* sgate = (double*)(chunk_lds + L::kGates);
  const bool held = OUT && (prefix > 0 || t0 > 0);
  start = uniform64(start) + t0, len = uniform64(len) - t0;
  if (MODE != kWholeRequests && len > seg.tokens) len = seg.tokens;
  const int64_t slot = uniform64(load_idx(s.req_pool_indices, b, s.idx64));
  float* Sst = S_state + slot * S_stride + (int64_t)h * D * Dv;
  float* nst = n_state + slot * n_stride + (int64_t)h * D;
  float* mst = m_state + slot * m_stride + h;
  float* const part = MODE == kWholeRequests ? nullptr : seg.work + ((int64_t)blockIdx.x * H + h) * seg.stride;
  c.load_state(split ? part : Sst, held);
  if (c.tid < D) sn[c.tid] = held ? (split ? part + D * Dv : nst)[c.tid] : 0.f;
  // (kept by the wave that forms the scalars; a segment's sums know no earlier token)
  float m = MODE == kSegmentSums ? -INFINITY : split ? part[D * Dv + D + kSegStart] : held ? mst[0] : 0.f;
  double passed = 0.;                                 // kSegmentSums: the sum of the log forget gates
  const float qscale = 1.f / sqrtf((float)D);
  q += (start * q_stride + (int64_t)h * D) * 2;
  k += (start * k_stride + (int64_t)h * D) * 2;
  v += (start * v_stride + (int64_t)h * Dv) * 2;
  const char* gb = (const char*)g + (start * g_stride + (int64_t)h * Dv) * 2;
  char* ob = (char*)out + (start * out_stride + (int64_t)h * Dv) * 2;
  const int col = c.column();
  float nw = norm_w[(int64_t)h * Dv + col];
  asm volatile("" : "+v"(nw), "+v"(m));               // (as the state: waited for here)
  const auto load = [&](int64_t c0) {
    const int n = (int)(len - c0 < kCL ? len - c0 : kCL);
    c.load(q + c0 * q_stride * 2, q_stride * 2, k + c0 * k_stride * 2, k_stride * 2, v + c0 * v_stride * 2, v_stride * 2, n);
  };
  // F, b and the running maximum of b do not depend on m: the NW waves form those of NW chunks at a time (two scans and five
  // transcendentals of latency), and a chunk's scalars are a few exponentials more once the chunk before it has fixed m
  const auto scan_gates = [&](int64_t c0) {
    const int64_t t = c0 + c.tid;
    double* to = sgate + c.wave * 3 * kCL + c.lane;
    const bool live = t < len;
    const float gi = live ? ipre[(start + t) * gate_stride + h] : 0.f, gf = live ? fpre[(start + t) * gate_stride + h] : 0.f;
    const double F = wave_scan_sum(live ? (double)logsigmoid_f(cap * tanhf(gf / cap)) : 0., c.lane);
    const double bs = live ? (double)(cap * tanhf(gi / cap)) - F : -INFINITY;
    to[0] = F;
    to[kCL] = bs;
    to[2 * kCL] = wave_scan_max(bs, c.lane);
  };
  const auto gates = [&](int64_t c0) {                // by the last wave: its share of the tiles is the smallest
    if (c.wave != NW - 1) return;
    const double* from = sgate + c0 / kCL % NW * 3 * kCL + c.lane;
    const double F = from[0], bs = from[kCL], G = fmax((double)m, from[2 * kCL]);
    const double Gend = __shfl(G, 63, 64), Fend = __shfl(F, 63, 64);
    ChunkScalars& sc = *c.scalars(c0 / kCL);
    if constexpr (OUT) {
      ChunkScalars::put(sc.lt, c.lane, Gend - G);
      ChunkScalars::put(sc.ls, c.lane, Gend - bs);
      sc.cs[c.lane] = qscale;
      sc.a0[c.lane] = expf((float)(m - G)) * qscale;
      sfloor[(c0 / kCL & 1) * kCL + c.lane] = expf((float)-(F + G));
    }
    sc.w[c.lane] = expf((float)(bs - Gend));
    passed += Fend;
    if (c.lane == 0) sc.a_end = expf((float)(m - Gend));
    m = (float)(Fend + Gend);
  };
  load(0);
  bool zero = !held;
  for (int64_t c0 = 0; c0 < len; c0 += kCL) {
    const int n = (int)(len - c0 < kCL ? len - c0 : kCL);
    c.sc = c.scalars(c0 / kCL);
    if (c0 / kCL % NW == 0) {
      scan_gates(c0);
      lds_barrier();
      gates(c0);
    }
    c.stage((int)(c0 / kCL));
    lds_barrier();
    if (c0 + kCL < len) load(c0 + kCL);
    uint16_t gv[4][4];
    if constexpr (OUT) {
      c.scores();
      c.from_state(zero);
      zero = false;
      {      // n_0 . q of a token: the lanes of a token share its D channels
        constexpr int PER = NT / kCL, DP = D / PER;
        const int t = c.tid / PER, part = c.tid % PER;
        float d = 0.f;
#pragma unroll
        for (int i = 0; i < DP; i += 8) {
          float f[8];
          unpack16<bf16_tag>(ld16(chunk_lds + C::kQ + t * C::QROW + (part * DP + i) * 2), f);
#pragma unroll
          for (int e = 0; e < 8; ++e) d += sn[part * DP + i + e] * f[e];
        }
        d = lanes_sum<PER>(d);
        if (part == 0) snq[t] = d;
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int t = 16 * i + 4 * c.q + r;
          gv[i][r] = *(const uint16_t*)(gb + c0 * g_stride * 2 + (uint32_t)((t < n ? t : n - 1) * (uint32_t)g_stride + col) * 2u);
        }
      lds_barrier();
      c.template weigh<true>();
    }
    if (c0 + kCL < len && (c0 / kCL + 1) % NW != 0) gates(c0 + kCL);
    {      // the normaliser's update: the lanes of a channel share the chunk's tokens
      constexpr int PER = NT / D, TP = kCL / PER;
      const int d = c.tid / PER, part = c.tid % PER;
      const ChunkScalars& sc = *c.sc;
      float x = 0.f;
#pragma unroll
      for (int i = 0; i < TP; i += 8) {
        float f[8];
        unpack16<bf16_tag>(ld16(chunk_lds + C::kKT + d * C::TROW + (part * TP + i) * 2), f);
#pragma unroll
        for (int e = 0; e < 8; ++e) x += sc.w[part * TP + i + e] * f[e];
      }
      x = lanes_sum<PER>(x);
      if (part == 0) sn[d] = sc.a_end * sn[d] + x;
    }
    if constexpr (OUT) lds_barrier();
    c.absorb((int)(c0 / kCL));
    if constexpr (!OUT) {
      lds_barrier();
      continue;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float ss = lanes_sum<16>(c.o[i][r] * c.o[i][r]);
        if (c.r16 == 0) red[c.wave * kCL + 16 * i + 4 * c.q + r] = ss;
      }
    lds_barrier();
    // lane t of every wave: the division by the normaliser and the RMS of the divided row as one factor
    float nq = snq[c.lane] * c.sc->a0[c.lane], ss = 0.f;
    for (int j = 0; j <= c.q; ++j) nq += c.sums()[j * kCL + c.lane];
#pragma unroll
    for (int w = 0; w < NW; ++w) ss += red[w * kCL + c.lane];
    const float den = 1.f / (fmaxf(fabsf(nq), sfloor[(c0 / kCL & 1) * kCL + c.lane]) + 1e-6f);
    const float factor = den / sqrtf(den * den * ss / (float)Dv + eps);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int t = 16 * i + 4 * c.q + r;
        const float gate = bf16_bits_to_f32(gv[i][r]), f = __shfl(factor, t, 64);
        if (t < n)
          E::store(ob + c0 * out_stride * 2 + (uint32_t)(t * (uint32_t)out_stride + col) * 2u, 0,
                   over_one_plus_exp(c.o[i][r] * f * nw, gate));
      }
  }
  if constexpr (MODE == kSegmentSums) {
    c.store_state(part);
    if (c.tid < D) part[D * Dv + c.tid] = sn[c.tid];
    if (c.tid == (NW - 1) * 64) {
      *(double*)(part + D * Dv + D + kSegDecay) = passed;
      part[D * Dv + D + kSegMax] = m;
    }
  } else if (MODE == kWholeRequests || final) {
    c.store_state(Sst);
    if (c.tid < D) nst[c.tid] = sn[c.tid];
    if (c.tid == (NW - 1) * 64) mst[0] = m;
  }
}

#define SP_MLSTM_SCAN_PARAMS                                                                                                             \
  void *out, int64_t out_stride, const void *q, int64_t q_stride, const void *k, int64_t k_stride, const void *v, int64_t v_stride,       \
      const void *g, int64_t g_stride, const float *ipre, const float *fpre, int64_t gate_stride, const float *norm_w, float *S_state,    \
      int64_t S_stride, float *n_state, int64_t n_stride, float *m_state, int64_t m_stride, const ScanSegments &seg, const SeqBatch &s,   \
      int H, float cap, float eps, hipStream_t st
#define SP_MLSTM_SCAN_ARGS                                                                                                                \
  out, out_stride, q, q_stride, k, k_stride, v, v_stride, g, g_stride, ipre, fpre, gate_stride, norm_w, S_state, S_stride, n_state,       \
      n_stride, m_state, m_stride, seg, s, H, cap, eps, st

template <int D, int NW, int MODE>
static int launch_mlstm_mode(unsigned groups, SP_MLSTM_SCAN_PARAMS) {
  constexpr int bytes = MlstmLds<D, NW, MODE != kSegmentSums>::kBytes;
  static PerDevice<int> raised;
  if (!chunk_lds_ready(raised, (const void*)mlstm_chunk_kernel<D, NW, MODE>, bytes)) return SP_ERR_LAUNCH;
  mlstm_chunk_kernel<D, NW, MODE><<<dim3(groups, (unsigned)H), NW * 64, bytes, st>>>(
      out, out_stride, (const char*)q, q_stride, (const char*)k, k_stride, (const char*)v, v_stride, g, g_stride, ipre, fpre, gate_stride,
      norm_w, S_state, S_stride, n_state, n_stride, m_state, m_stride, seg, s, H, cap, eps);
  SP_LAUNCH_CHECK();
  return SP_OK;
}

// (seg.tokens 0: a request's chunks by one workgroup per head)
template <int D, int NW>
static int launch_mlstm_chunks(int64_t tokens, SP_MLSTM_SCAN_PARAMS) {
  if (seg.tokens == 0) return launch_mlstm_mode<D, NW, kWholeRequests>((unsigned)s.B, SP_MLSTM_SCAN_ARGS);
  const unsigned groups = (unsigned)(tokens / seg.tokens + s.B);
  const int rc = launch_mlstm_mode<D, NW, kSegmentSums>(groups, SP_MLSTM_SCAN_ARGS);
  if (rc != SP_OK) return rc;
  segment_states_kernel<true><<<dim3((unsigned)s.B, (unsigned)H, D * NW * 16 / 1024 + 1), 256, 0, st>>>(
      seg, S_state, S_stride, n_state, n_stride, m_state, m_stride, s, H, D, NW * 16);
  SP_LAUNCH_CHECK();
  return launch_mlstm_mode<D, NW, kSegmentOutputs>(groups, SP_MLSTM_SCAN_ARGS);
}

// Steps of short portions that the per-token form walks faster than a chunk of 64 mostly empty tokens costs: requests x heads of few
// values that take the chunk form more than one round of workgroups, few tokens per request on average.  us, per token / in chunks, by
// tokens per request (D x Dv, W = requests x heads):
//   64 x 64     W 512: 1 18 / 15    W 640: 1 19 / 24, 6 24 / 25, 8 26 / 25    W 2048: 1 46 / 51, 2 49 / 51, 4 58 / 52
//   128 x 64    W 256: 1 23 / 16    W 512: 1 27 / 30, 2 28 / 30, 4 30 / 30    W 640: 1 44 / 42
//   64 x 128    W 320: 1 29 / 24    W 4096: 1 203 / 176      128 x 128   W 320: 1 46 / 31    W 4096: 1 487 / 239
static bool short_portions(int64_t tokens, int64_t B, int H, int D, int Dv) {
  const int64_t W = B * H;
  if (tokens < 0 || Dv != 64) return false;
  if (D == 64) return W > 512 && tokens <= (W <= 1024 ? 6 : 2) * B;
  return W > 256 && W <= 512 && tokens <= 2 * B;
}

template <typename Tag>
static int launch_mlstm(int D, int Dv, int64_t tokens, SP_MLSTM_SCAN_PARAMS) {
  // a step of one token per request stays with the per-token form (one sweep over the state is all there is to do), and so do
  // the types and head sizes the matrix form is not built for, and short portions of many requests
  if (std::is_same<Tag, bf16_tag>::value && s.extend_seq_lens && (D == 64 || D == 128) && (Dv == 64 || Dv == 128) &&
      chunk_aligned(q, q_stride) && chunk_aligned(k, k_stride) && chunk_aligned(v, v_stride) &&
      g_stride < ((int64_t)1 << 24) && out_stride < ((int64_t)1 << 24) && (seg.tokens || !short_portions(tokens, s.B, H, D, Dv))) {
    if (D == 128 && Dv == 128) return launch_mlstm_chunks<128, 8>(tokens, SP_MLSTM_SCAN_ARGS);
    if (D == 128) return launch_mlstm_chunks<128, 4>(tokens, SP_MLSTM_SCAN_ARGS);
    if (Dv == 128) return launch_mlstm_chunks<64, 8>(tokens, SP_MLSTM_SCAN_ARGS);
    return launch_mlstm_chunks<64, 4>(tokens, SP_MLSTM_SCAN_ARGS);
  }
  if (seg.tokens) return SP_ERR_UNSUPPORTED;
  const dim3 grid((unsigned)s.B, (unsigned)H);
  if ((Dv + 1) * (D > 64 ? 4 : (D > 32 ? 2 : 1)) > 1024) return SP_ERR_UNSUPPORTED;      // vdim 256 with dim > 64
#define SP_MLSTM(DP)                                                                                                    \
  mlstm_scan_kernel<Tag, DP><<<grid, (unsigned)(((Dv + 1) * split_of(DP) + 63) / 64 * 64),                              \
                               (size_t)chunk_of(DP) * (2 * Dv + 1) * sizeof(float), st>>>(                              \
      out, out_stride, q, q_stride, k, k_stride, v, v_stride, g, g_stride, ipre, fpre, gate_stride, norm_w, S_state, S_stride, n_state,  \
      n_stride, m_state, m_stride, s, H, D, Dv, cap, eps)
  if (D <= 16) SP_MLSTM(16);
  else if (D <= 32) SP_MLSTM(32);
  else if (D <= 64) SP_MLSTM(64);
  else if (D <= 128) SP_MLSTM(128);
  else if (D <= 256) SP_MLSTM(256);
  else return SP_ERR_UNSUPPORTED;
#undef SP_MLSTM
  SP_LAUNCH_CHECK();
  return SP_OK;
}
#undef SP_MLSTM_SCAN_PARAMS
#undef SP_MLSTM_SCAN_ARGS

}  // namespace
}  // namespace sp

using namespace sp;

// (gate_stride: values between the gates of a token and the next one's, so that both may be halves of one product's rows; num_tokens:
// the step's rows, < 0 where the caller does not know; only the choice between the two forms depends on it)
static int mlstm_scan(void* out, int64_t out_stride, const void* q, int64_t q_stride, const void* k, int64_t k_stride, const void* v,
                      int64_t v_stride, const void* g, int64_t g_stride, const float* ipre, const float* fpre, int64_t gate_stride,
                      const float* norm_w, float* S_state, int64_t S_stride, float* n_state, int64_t n_stride, float* m_state,
                      int64_t m_stride, const ScanSegments& seg, int64_t num_tokens, int heads, int dim, int vdim, float cap, float eps,
                      SP_SEQ_PARAMS, int dtype, void* stream) {
  SP_CHECK_ARG(batch_size >= 0 && heads > 0 && dim > 0 && vdim > 0 && vdim <= 256 && cap > 0.f);
  if (batch_size == 0) return SP_OK;
  SP_CHECK_ARG(out && q && k && v && g && ipre && fpre && norm_w && S_state && n_state && m_state && req_pool_indices && seq_lens);
  SP_CHECK_ARG(!extend_seq_lens || (extend_prefix_lens && extend_start_loc));
  const int64_t nk = (int64_t)heads * dim, nv = (int64_t)heads * vdim;
  SP_CHECK_ARG(q_stride >= nk && k_stride >= nk && v_stride >= nv && g_stride >= nv && out_stride >= nv);
  SP_CHECK_ARG(S_stride >= nk * vdim && n_stride >= nk && m_stride >= heads && gate_stride >= heads);
  SEQ_BATCH(s);
  SP_DISPATCH_DTYPE(dtype, return (launch_mlstm<Tag>(dim, vdim, num_tokens, out, out_stride, q, q_stride, k, k_stride, v, v_stride, g,
                                                     g_stride, ipre, fpre, gate_stride, norm_w, S_state, S_stride, n_state, n_stride,
                                                     m_state, m_stride, seg, s, heads, cap, eps, (hipStream_t)stream)));
}

extern "C" int sp_mlstm_scan_tokens(void* out, int64_t out_stride, const void* q, int64_t q_stride, const void* k, int64_t k_stride, const void* v,
                                    int64_t v_stride, const void* g, int64_t g_stride, const float* ipre, const float* fpre, int64_t gate_stride,
                                    const float* norm_w, float* S_state, int64_t S_stride, float* n_state, int64_t n_stride, float* m_state,
                                    int64_t m_stride, int64_t num_tokens, int heads, int dim, int vdim, float cap, float eps, SP_SEQ_PARAMS,
                                    int dtype, void* stream) {
  return mlstm_scan(out, out_stride, q, q_stride, k, k_stride, v, v_stride, g, g_stride, ipre, fpre, gate_stride, norm_w, S_state, S_stride,
                    n_state, n_stride, m_state, m_stride, ScanSegments{nullptr, 0, 0}, num_tokens, heads, dim, vdim, cap, eps,
                    req_pool_indices, seq_lens, extend_seq_lens, extend_prefix_lens, extend_start_loc, token_req, idx64, batch_size, dtype,
                    stream);
}

// (weak: mlstm.hip and ssm.hip define it, a library may hold either or both)
extern "C" __attribute__((weak)) int64_t sp_scan_segment_floats(int64_t num_tokens, int batch_size, int heads, int dim, int vdim,
                                                                int segment_tokens) {
  return scan_segment_floats(num_tokens, batch_size, heads, dim, vdim, segment_tokens);
}

extern "C" int sp_mlstm_scan_segments(void* out, int64_t out_stride, const void* q, int64_t q_stride, const void* k, int64_t k_stride, const void* v,
                                      int64_t v_stride, const void* g, int64_t g_stride, const float* ipre, const float* fpre, int64_t gate_stride,
                                      const float* norm_w, float* S_state, int64_t S_stride, float* n_state, int64_t n_stride, float* m_state,
                                      int64_t m_stride, float* work, int segment_tokens, int64_t num_tokens, int heads, int dim, int vdim,
                                      float cap, float eps, SP_SEQ_PARAMS, int dtype, void* stream) {
  SP_CHECK_ARG(num_tokens >= 0 && segment_tokens > 0 && segment_tokens % kCL == 0 && work && ((uintptr_t)work & 15) == 0);
  return mlstm_scan(out, out_stride, q, q_stride, k, k_stride, v, v_stride, g, g_stride, ipre, fpre, gate_stride, norm_w, S_state, S_stride,
                    n_state, n_stride, m_state, m_stride, ScanSegments{work, segment_floats(dim, vdim, true), segment_tokens}, num_tokens,
                    heads, dim, vdim, cap, eps, req_pool_indices, seq_lens, extend_seq_lens, extend_prefix_lens, extend_start_loc, token_req,
                    idx64, batch_size, dtype, stream);
}

extern "C" int sp_mlstm_scan_gates(void* out, int64_t out_stride, const void* q, int64_t q_stride, const void* k, int64_t k_stride,
                                   const void* v, int64_t v_stride, const void* g, int64_t g_stride, const float* ipre,
                                   const float* fpre, int64_t gate_stride, const float* norm_w, float* S_state, int64_t S_stride,
                                   float* n_state, int64_t n_stride, float* m_state, int64_t m_stride, int heads, int dim,
                                   int vdim, float cap, float eps, SP_SEQ_PARAMS, int dtype, void* stream) {
  return sp_mlstm_scan_tokens(out, out_stride, q, q_stride, k, k_stride, v, v_stride, g, g_stride, ipre, fpre, gate_stride, norm_w,
                              S_state, S_stride, n_state, n_stride, m_state, m_stride, -1, heads, dim, vdim, cap, eps, req_pool_indices,
                              seq_lens, extend_seq_lens, extend_prefix_lens, extend_start_loc, token_req, idx64, batch_size, dtype, stream);
}

extern "C" int sp_mlstm_scan(void* out, int64_t out_stride, const void* q, int64_t q_stride, const void* k, int64_t k_stride,
                             const void* v, int64_t v_stride, const void* g, int64_t g_stride, const float* ipre,
                             const float* fpre, const float* norm_w, float* S_state, int64_t S_stride, float* n_state,
                             int64_t n_stride, float* m_state, int64_t m_stride, int heads, int dim, int vdim, float cap,
                             float eps, SP_SEQ_PARAMS, int dtype, void* stream) {
  return sp_mlstm_scan_gates(out, out_stride, q, q_stride, k, k_stride, v, v_stride, g, g_stride, ipre, fpre, heads, norm_w, S_state,
                             S_stride, n_state, n_stride, m_state, m_stride, heads, dim, vdim, cap, eps, req_pool_indices, seq_lens,
                             extend_seq_lens, extend_prefix_lens, extend_start_loc, token_req, idx64, batch_size, dtype, stream);
}
