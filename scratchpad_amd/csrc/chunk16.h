// Linear recurrences with a decay per key channel, 16 tokens at a time, fp32 on the matrix cores, their operands formed beforehand.
//
//   FORGET:  S_t = diag(w_t) S_{t-1} + k_t v_t^T                                            o_t = S_t^T r_t        (S [D, Dv])
//   DELTA:   S_t = diag(w_t) S_{t-1} - b_t (u_t^T S_{t-1}) + k_t v_t^T                       o_t = S_t^T r_t        (b = a * u)
//
// Over a chunk that starts from S_0, with w_{i..j} the product of the decays of tokens i .. j per channel:
//   Rd_t = r_t w_{1..t},   Ke_s = k_s w_{s+1..16},   P_ts = r_t . (k_s w_{s+1..t})  (s <= t),   G = w_{1..16}
//   FORGET:  O = Rd S_0 + P V,            S_16 = diag(G) S_0 + Ke^T V
//   DELTA:   Ud_t = u_t w_{1..t-1},  Be_s = b_s w_{s+1..16},  L_ts = u_t . (b_s w_{s+1..t-1}),  M_ts = u_t . (k_s w_{s+1..t-1})  (s < t),
//            Q_ts = r_t . (b_s w_{s+1..t})  (s <= t):   Y = (I + L)^{-1} (Ud S_0 + M V)     (y_t = u_t^T S_{t-1})
//            O = Rd S_0 + P V - Q Y,       S_16 = diag(G) S_0 + Ke^T V - Be^T Y
// Every factor is a product of decays, never a quotient: with decays in [0, 1] nothing overflows however strong they are.
//
// chunk16_prepare_kernel forms all of this but the products with S_0, V and Y for all chunks at once (one workgroup per chunk and
// head) and lays it out as the walk reads it from LDS.  chunk16_walk_kernel walks a request's chunks: a wave owns 16 columns of S in the
// accumulator layout of v_mfma_f32_16x16x4_f32 (lane (r16, q): column r16, rows 16 i + 4 q + r), in which register (i, r) IS the second
// operand of Rd S for the channels 16 i + 4 q + r, and the registers of v and Y are the second operands of the products over tokens.
// Operands and rows come into LDS by direct loads, two chunks ahead; one barrier per chunk.  Read-outs go
// through LDS to the waves that norm, gate and store them, a chunk behind.
//
// A FORGET request's tokens may be cut into segments that run side by side (chunk_scan.h: the state is linear in the one a segment
// starts from, here with a decay per row).
//
// A value that is not finite would reach the EARLIER tokens of its chunk (zeros of P and M times it): where a column has one, it is
// taken out, the column's read-outs from that token on become NaN, and so does the column of the state.
#pragma once
#include "chunk_scan.h"

#include <algorithm>

namespace sp {

constexpr int kC16 = 16;

// floats of a chunk and head: KeT [D][16], G [D], Rd [16][D], P [16][16]; DELTA: BeT (negative) [D][16], Ud [16][D], T = (I + L)^{-1},
// M and Q (negative), [16][16] each.  Pieces of 4 floats are permuted so that the 16 lanes of an LDS read phase meet no bank twice: in
// rows of 16 by place16, in rows of D by XOR with the row's number.
template <int D, bool DELTA>
struct Chunk16 {
  static constexpr int kKe = 0, kG = 16 * D, kSums = kG + D;               // what a segment's sums need comes first
  static constexpr int kRd = kSums, kP = kRd + 16 * D, kBe = kP + 256, kUd = kBe + 16 * D, kT = kUd + 16 * D, kM = kT + 256, kQ = kM + 256;
  static constexpr int kUsed = DELTA ? kQ + 256 : kBe;
  static constexpr int kFloats = (kUsed + 255) / 256 * 256;                // whole direct loads of 1 KiB
};
// the walk's LDS: three chunks' operands, rows of v (and of the gate), then two chunks' read-outs in fp32 (rows of Dv + 4: the four rows that
// a wave writes at a time lie in different banks)
template <typename Tag, int D, int NW, bool DELTA, int MODE>
struct Walk16Lds {
  static constexpr int kOps = (MODE != kSegmentSums ? Chunk16<D, DELTA>::kFloats : (Chunk16<D, DELTA>::kSums + 255) / 256 * 256) * 4;
  static constexpr int kRows = kC16 * NW * 16 * Elem<Tag>::kBytes, kBuf = kOps + (DELTA ? 2 : 1) * kRows, kRow = NW * 16 + 4;
  static constexpr int kOut = 3 * kBuf, kBytes = kOut + (MODE != kSegmentSums ? 2 * kC16 * kRow * 4 : 0);
};
// where piece q of row `row` lies, in rows of four pieces
__device__ __forceinline__ int place16(int row, int q) { return ((q & 1) * 2 + (q >> 1)) ^ ((row >> 3) & 1); }

__device__ __forceinline__ f32x4_c mfma_4(float a, float b, const f32x4_c& c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// Workgroup (chunk, head).  `fill` puts the chunk's rows of r, k, w (DELTA: u and b too) into LDS in fp32, rows past the request's end
// as zeros with decay 1.  Vector work bounds it: a lane sums two columns s of the 16 x 16 matrices over D / 32 channels, the decays
// between s and t building up as t walks on.
template <int D, bool DELTA, typename Fill>
__device__ __forceinline__ void chunk16_prepare(float* work, const Fill& fill) {
  typedef Chunk16<D, DELTA> C;
  constexpr int ROW = D + 4, CH = D / 32, NM = DELTA ? 4 : 1;             // matrices: P; L, M, Q
  __shared__ __attribute__((aligned(16))) float sr[kC16][ROW], sk[kC16][ROW], sw[kC16][ROW];
  __shared__ __attribute__((aligned(16))) float su[DELTA ? kC16 : 1][ROW], sb[DELTA ? kC16 : 1][ROW];
  __shared__ float part[4][NM][kC16][kC16 + 1];
  __shared__ float sL[DELTA ? kC16 : 1][kC16 + 1];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  fill(sr, sk, sw, su, sb);
  __syncthreads();
  const int s0 = lane & 7, c0 = wave * (D / 4) + (lane >> 3) * CH;
  typedef float vec __attribute__((ext_vector_type(CH)));
  vec rk[2], rb[2];
#pragma unroll
  for (int z = 0; z < 2; ++z) {
    rk[z] = *(const vec*)&sk[s0 + 8 * z][c0];
    if constexpr (DELTA) rb[z] = *(const vec*)&sb[s0 + 8 * z][c0];
  }
#pragma unroll
  for (int half = 0; half < 2; ++half) {
    float sums[NM][2][8];                             // of tokens t = 8 half + u and columns s0 + 8 z
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int t = 8 * half + u;
      const vec rt = *(const vec*)&sr[t][c0], wt = *(const vec*)&sw[t][c0];
      vec ut;
      if constexpr (DELTA) ut = *(const vec*)&su[t][c0];
#pragma unroll
      for (int z = 0; z <= half; ++z) {               // (tokens below 8 are before every second column)
        float sum[4] = {0.f, 0.f, 0.f, 0.f};
        if constexpr (DELTA) {
#pragma unroll
          for (int x = 0; x < CH; ++x) {
            sum[1] += ut[x] * rb[z][x];
            sum[2] += ut[x] * rk[z][x];
          }
        }
#pragma unroll
        for (int x = 0; x < CH; ++x) {
          rk[z][x] *= t > s0 + 8 * z ? wt[x] : 1.f;
          sum[0] += rt[x] * rk[z][x];
          if constexpr (DELTA) {
            rb[z][x] *= t > s0 + 8 * z ? wt[x] : 1.f;
            sum[3] += rt[x] * rb[z][x];
          }
        }
#pragma unroll
        for (int m = 0; m < NM; ++m) sums[m][z][u] = sum[m];
      }
    }
#pragma unroll
    for (int m = 0; m < NM; ++m)
#pragma unroll
      for (int z = 0; z <= half; ++z) part[wave][m][8 * half + (lane >> 3)][s0 + 8 * z] = eight_sums(sums[m][z], lane);
  }
  // Rd, Ud, G by one half of the threads, Ke and Be by the other: a channel's tokens forward or backward
  for (int e = tid; e < 2 * D; e += 256) {
    const int d = e < D ? e : e - D;
    float g = 1.f;
    if (e < D) {
#pragma unroll
      for (int t = 0; t < kC16; ++t) {
        const int at = t * D + (((d >> 2) ^ t) << 2) + (d & 3);
        if constexpr (DELTA) work[C::kUd + at] = su[t][d] * g;
        g *= sw[t][d];
        work[C::kRd + at] = sr[t][d] * g;
      }
      work[C::kG + d] = g;
    } else {
#pragma unroll
      for (int p4 = 3; p4 >= 0; --p4) {
        f32x4_c ke, be;
#pragma unroll
        for (int x = 3; x >= 0; --x) {
          const int t = 4 * p4 + x;
          ke[x] = sk[t][d] * g;
          if constexpr (DELTA) be[x] = -(sb[t][d] * g);
          g *= sw[t][d];
        }
        *(f32x4_c*)(work + C::kKe + d * 16 + place16(d, p4) * 4) = ke;
        if constexpr (DELTA) *(f32x4_c*)(work + C::kBe + d * 16 + place16(d, p4) * 4) = be;
      }
    }
  }
  __syncthreads();
  const int t = tid >> 4, s = tid & 15, at = t * 16 + place16(t, s >> 2) * 4 + (s & 3);
  float sum[NM];
#pragma unroll
  for (int m = 0; m < NM; ++m) sum[m] = (part[0][m][t][s] + part[1][m][t][s]) + (part[2][m][t][s] + part[3][m][t][s]);
  work[C::kP + at] = t >= s ? sum[0] : 0.f;
  if constexpr (DELTA) {
    work[C::kM + at] = t > s ? sum[2] : 0.f;
    work[C::kQ + at] = t >= s ? -sum[3] : 0.f;
    sL[t][s] = t > s ? sum[1] : 0.f;
    __syncthreads();
    if (tid < kC16) {                                 // column tid of (I + L)^{-1}: forward substitution
      float x[kC16];
#pragma unroll
      for (int i = 0; i < kC16; ++i) {
        float y = i == tid ? 1.f : 0.f;
#pragma unroll
        for (int j = 0; j < i; ++j) y -= sL[i][j] * x[j];
        x[i] = i >= tid ? y : 0.f;
        work[C::kT + i * 16 + place16(i, tid >> 2) * 4 + (tid & 3)] = x[i];
      }
    }
  }
}

// 16 bytes per lane from `from` to lds + 16 lane.  (The builtin of the same makes every later read of LDS wait for it; the walk waits
// once a chunk.  m0 is named, so that no value another instruction needs in it is carried past; the compiler calls that reserved.)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void load_to_lds(const void* from, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(from), "s"(lds) : "memory", "m0");
}
#pragma clang diagnostic pop

// chunks of the requests before `b`, by all lanes of a wave
__device__ __forceinline__ int chunks16_before(const SeqBatch& s, int b, int lane) {
  int n = 0;
  for (int i = lane; i < b; i += 64) n += segments_of(max(s.extend_seq_lens[i], 0), kC16);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) n += __shfl_xor(n, off, 64);
  return __builtin_amdgcn_readfirstlane(n);
}

struct Walk16 {
  void* out;
  const void *v, *gate;                               // gate: DELTA
  const float *norm_w, *work;                         // norm_w [Dv] (DELTA: [H * Dv])
  float* state;
  int64_t out_stride, v_stride, gate_stride, state_stride;
  ScanSegments seg;
  int H;
  float eps;
  int vec_out;                                        // rows of `out` take 16-byte stores (fp32: two of them per 8 values)
};

// Workgroup (request or segment, head): NW waves own 16 columns each, NW / 2 more fetch the operands of the chunk after the next and finish
// the one before - the head's norm, the gate, the stores.  What bounds it is the chain of a wave's matrix instructions of 32 cycles, 2 D / 4 + 4
// per chunk (DELTA: 4 D / 4 + 16): with waves that also finished their own columns a chunk
// of a single request (DELTA, heads of 64) took 3.2 us, now 2.4.
template <typename Tag, int D, int NW, bool DELTA, int MODE>
__global__ void __launch_bounds__(NW * 96) chunk16_walk_kernel(Walk16 a, SeqBatch sb) {
  typedef Elem<Tag> E;
  typedef Chunk16<D, DELTA> C;
  typedef Walk16Lds<Tag, D, NW, DELTA, MODE> L;
  constexpr bool OUT = MODE != kSegmentSums;
  constexpr int Dv = NW * 16, DT = D / 16, NH = NW / 2, OPS = L::kOps / 1024, ROWS = L::kRows / 1024;
  extern __shared__ __attribute__((aligned(16))) char walk_lds[];
  const int tid = threadIdx.x, lane = tid & 63, r16 = lane & 15, q = lane >> 4, h = blockIdx.y;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int b = blockIdx.x, t0 = 0;
  if constexpr (MODE != kWholeRequests)
    if (!segment_at(sb, (int)blockIdx.x, a.seg.tokens, lane, b, t0)) return;
  int len = __builtin_amdgcn_readfirstlane(sb.extend_seq_lens[b]);
  if (len <= 0) return;
  const bool split = MODE != kWholeRequests && len > a.seg.tokens, last = MODE == kWholeRequests || t0 + a.seg.tokens >= len;
  if (MODE == kSegmentSums && last) return;
  const bool held = OUT && (sb.extend_prefix_lens[b] > 0 || t0 > 0);
  const int64_t start = __builtin_amdgcn_readfirstlane(sb.extend_start_loc[b]) + t0;
  const int whole = len;
  len -= t0;
  if (MODE != kWholeRequests && whole > a.seg.tokens && len > a.seg.tokens) len = a.seg.tokens;
  const int chunks = (len + kC16 - 1) / kC16;
  float* const outs = (float*)(walk_lds + L::kOut);
  if (wave >= NW) {
    const int hw = wave - NW;
    // (their vector instructions go in front of the other waves' products, which keep the vector unit for 32 cycles each: general delta rule, one
    // request of 4096 tokens, the layer 967 -> 945 us; HGRN2, 16 requests of 125 tokens, 118 -> 115)
    __builtin_amdgcn_s_setprio(3);
    const float* work = a.work + (int64_t)(chunks16_before(sb, b, lane) + t0 / kC16) * a.H * C::kFloats + (int64_t)h * C::kFloats;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)walk_lds;
    // a chunk's operands and rows (past the request's end: its last one again), 1 KiB per load, shared out over the helpers; the gates of a
    // helper's tokens are its own loads (it reads them when the others may be on to the next chunk)
    constexpr int LEAST = (OPS + ROWS) / NH + (DELTA ? ROWS / NH : 0);      // loads of a chunk by any helper, at the least
    const auto row_piece = [&](const void* rows, int64_t stride, int c, int piece) {
      const int at = piece * 1024 + lane * 16, t = at / (Dv * E::kBytes);
      const int64_t row = start + c * kC16 + min(t, len - c * kC16 - 1);
      return (const char*)rows + (row * stride + (int64_t)h * Dv) * E::kBytes + at % (Dv * E::kBytes);
    };
    const auto fetch = [&](int c) {
      const uint32_t to = lds0 + c % 3 * L::kBuf;
      for (int u = hw; u < OPS + ROWS; u += NH) {
        const char* from = (const char*)(work + (int64_t)c * a.H * C::kFloats) + u * 1024 + lane * 16;
        if (u >= OPS) from = row_piece(a.v, a.v_stride, c, u - OPS);
        load_to_lds(from, to + u * 1024);
      }
      if constexpr (DELTA) {
#pragma unroll
        for (int u = 0; u < ROWS / NH; ++u) {
          const int piece = hw * (ROWS / NH) + u;
          load_to_lds(row_piece(a.gate, a.gate_stride, c, piece), to + (OPS + ROWS + piece) * 1024);
        }
      }
    };
    // lane: 8 values of a token
    constexpr int PER = Dv / 8;
    const int t = hw * (kC16 / NH) + lane / PER, at = lane % PER * 8;
    float nw[8];
#pragma unroll
    for (int x = 0; x < 8; ++x) nw[x] = OUT ? a.norm_w[(DELTA ? (int64_t)h * Dv : 0) + at + x] : 0.f;
    const auto finish = [&](int c) {
      const float* o = outs + ((c & 1) * kC16 + t) * L::kRow + at;
      const f32x4_c o0 = *(const f32x4_c*)o, o1 = *(const f32x4_c*)(o + 4);
      float f[8] = {o0[0], o0[1], o0[2], o0[3], o1[0], o1[1], o1[2], o1[3]}, ss = 0.f;
#pragma unroll
      for (int x = 0; x < 8; ++x) ss += f[x] * f[x];
      const float inv = 1.f / sqrtf(lanes_sum<PER>(ss) / (float)Dv + a.eps);
#pragma unroll
      for (int x = 0; x < 8; ++x) f[x] = f[x] * inv * nw[x];
      if constexpr (DELTA) {
        float g[8];
        const char* rows = walk_lds + c % 3 * L::kBuf + L::kOps + L::kRows + (t * Dv + at) * E::kBytes;
#pragma unroll
        for (int x = 0; x < 8; x += E::kVec) unpack16<Tag>(ld16(rows + x * E::kBytes), g + x);
#pragma unroll
        for (int x = 0; x < 8; ++x) f[x] = over_one_plus_exp(f[x], g[x]);
      }
      if (t >= len - c * kC16) return;
      char* to = (char*)a.out + ((start + c * kC16 + t) * a.out_stride + (int64_t)h * Dv + at) * E::kBytes;
      if (a.vec_out) {
#pragma unroll
        for (int x = 0; x < 8; x += E::kVec) st16(to + x * E::kBytes, pack16<Tag>(f + x));
      } else {
#pragma unroll
        for (int x = 0; x < 8; ++x) E::store(to, x, f[x]);
      }
    };
    fetch(0);
    if (chunks > 1) fetch(1);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    lds_barrier();
    for (int c = 0; c < chunks; ++c) {
      if (OUT && c > 0) finish(c - 1);                 // (the gates of chunk c - 1 lie where chunk c + 2 goes)
      if (c + 2 < chunks) {
        if constexpr (DELTA) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        fetch(c + 2);
      }
      // waiting for all but the last LEAST loads is waiting for the chunk before
      if (c + 2 < chunks) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LEAST) : "memory");
      else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      lds_barrier();
    }
    if constexpr (OUT) finish(chunks - 1);
    return;
  }
  const int col = 16 * wave + r16;
  float* st = a.state + load_idx(sb.req_pool_indices, b, sb.idx64) * a.state_stride + (int64_t)h * D * Dv;
  float* const part = MODE == kWholeRequests ? nullptr : a.seg.work + ((int64_t)blockIdx.x * a.H + h) * a.seg.stride;
  const float* from = split ? part : st;
  f32x4_c S[DT], decay[MODE == kSegmentSums ? DT : 1];
#pragma unroll
  for (int i = 0; i < DT; ++i) {
    if constexpr (MODE == kSegmentSums) decay[i] = f32x4_c{1.f, 1.f, 1.f, 1.f};
#pragma unroll
    for (int r = 0; r < 4; ++r) S[i][r] = held ? from[(int64_t)(16 * i + 4 * q + r) * Dv + col] : 0.f;
  }
  lds_barrier();
  for (int c = 0; c < chunks; ++c) {
    const int n = len - c * kC16;
    const float* m = (const float*)(walk_lds + c % 3 * L::kBuf);
    const auto row16 = [&](int at) { return *(const f32x4_c*)(m + at + r16 * 16 + place16(r16, q) * 4); };
    const auto row_d = [&](int at, int i) { return *(const f32x4_c*)(m + at + r16 * D + (((4 * i + q) ^ r16) << 2)); };
    f32x4_c rd[OUT ? DT : 1], ud[DELTA ? DT : 1], g[DT], ke[DT], be[DELTA ? DT : 1], mr, pr, tr, qr;
    float v[4];
    // the operands of the next products are read while the matrix cores are on the ones before (left to itself the compiler keeps
    // registers free and waits for each read)
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = E::load((const char*)m + L::kOps, (4 * q + r) * Dv + col);
    if constexpr (DELTA) mr = row16(C::kM);
    if constexpr (OUT) {
#pragma unroll
      for (int i = 0; i < DT; ++i) {
        rd[i] = row_d(C::kRd, i);
        if constexpr (DELTA) ud[i] = row_d(C::kUd, i);
      }
    }
    const auto read_update = [&] {
#pragma unroll
      for (int i = 0; i < DT; ++i) {
        g[i] = *(const f32x4_c*)(m + C::kG + 16 * i + 4 * q);
        ke[i] = *(const f32x4_c*)(m + C::kKe + (16 * i + r16) * 16 + place16(r16, q) * 4);
        if constexpr (DELTA) be[i] = *(const f32x4_c*)(m + C::kBe + (16 * i + r16) * 16 + place16(r16, q) * 4);
      }
    };
    if constexpr (!OUT) read_update();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = 4 * q + r < n ? v[r] : 0.f;
    int first = kC16;                                 // the column's first token that is not finite
    bool any = false;
    f32x4_c y = {0.f, 0.f, 0.f, 0.f};
    if constexpr (OUT) {
      const auto finite = [](float x) { return fabsf(x) < INFINITY; };
      const auto odd = [](const auto& x) {            // (in any lane)
        const float probe = fmaf(x[0], 0.f, fmaf(x[1], 0.f, fmaf(x[2], 0.f, x[3] * 0.f)));
        return __ballot(probe != probe) != 0;
      };
      const auto share_first = [&] {                  // over the lanes of the column
        first = min(first, __shfl_xor(first, 16, 64));
        first = min(first, __shfl_xor(first, 32, 64));
      };
      if (odd(v)) {
        any = true;
#pragma unroll
        for (int r = 3; r >= 0; --r)
          if (!finite(v[r])) v[r] = 0.f, first = 4 * q + r;
        share_first();
      }
      f32x4_c o = {0.f, 0.f, 0.f, 0.f}, x = {0.f, 0.f, 0.f, 0.f};
      if constexpr (DELTA) {
#pragma unroll
        for (int r = 0; r < 4; ++r) x = mfma_4(mr[r], v[r], x);
      }
      const auto read_state = [&](int i0, int i1) {
#pragma unroll
        for (int i = i0; i < i1; ++i)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            if constexpr (DELTA) x = mfma_4(ud[i][r], S[i][r], x);
            o = mfma_4(rd[i][r], S[i][r], o);
          }
      };
      read_state(0, DT / 2);
      __builtin_amdgcn_sched_barrier(0);
      pr = row16(C::kP);
      if constexpr (DELTA) tr = row16(C::kT), qr = row16(C::kQ);
      read_update();
      __builtin_amdgcn_sched_barrier(0);
      read_state(DT / 2, DT);
      if constexpr (DELTA) {
        if (odd(x)) {
          any = true;
#pragma unroll
          for (int r = 3; r >= 0; --r)
            if (!finite(x[r])) x[r] = 0.f, first = min(first, 4 * q + r);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          y = mfma_4(tr[r], x[r], y);
          o = mfma_4(pr[r], v[r], o);
        }
        if (any || odd(y)) {
          any = true;
#pragma unroll
          for (int r = 3; r >= 0; --r)
            if (!finite(y[r])) first = min(first, 4 * q + r);
          share_first();
#pragma unroll
          for (int r = 0; r < 4; ++r) y[r] = 4 * q + r < first ? y[r] : 0.f;
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) o = mfma_4(qr[r], y[r], o);
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) o = mfma_4(pr[r], v[r], o);
      }
#pragma unroll
      for (int i = 0; i < DT; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) S[i][r] *= g[i][r];
      if (any) {
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] = 4 * q + r < first ? o[r] : as_f32(0x7fc00000u);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int i = 0; i < DT; ++i) S[i] = mfma_4(ke[i][r], v[r], S[i]);
      if constexpr (DELTA) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int i = 0; i < DT; ++i) S[i] = mfma_4(be[i][r], y[r], S[i]);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) outs[((c & 1) * kC16 + 4 * q + r) * L::kRow + col] = o[r];
      if (any) {
#pragma unroll
        for (int i = 0; i < DT; ++i)
#pragma unroll
          for (int r = 0; r < 4; ++r) S[i][r] = first < kC16 ? as_f32(0x7fc00000u) : S[i][r];
      }
    } else {
#pragma unroll
      for (int i = 0; i < DT; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          S[i][r] *= g[i][r];
          decay[i][r] *= g[i][r];
        }
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int i = 0; i < DT; ++i) S[i] = mfma_4(ke[i][r], v[r], S[i]);
    }
    lds_barrier();
  }
  float* to = MODE == kSegmentSums ? part : st;
  if (MODE == kSegmentSums || last) {
#pragma unroll
    for (int i = 0; i < DT; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) to[(int64_t)(16 * i + 4 * q + r) * Dv + col] = S[i][r];
  }
  if constexpr (MODE == kSegmentSums) {
    if (wave == 0 && r16 == 0) {
#pragma unroll
      for (int i = 0; i < DT; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) part[D * Dv + 16 * i + 4 * q + r] = decay[i][r];
    }
  }
}

// Workgroup (request, head, 1024 values of S): segment_states_kernel with a decay per row
template <int D, int Dv>
__global__ void __launch_bounds__(256) segment_rows_kernel(ScanSegments g, const float* state, int64_t state_stride, SeqBatch s, int H) {
  const int b = blockIdx.x, h = blockIdx.y, lane = threadIdx.x & 63;
  const int segments = segments_of(s.extend_seq_lens[b], g.tokens);
  if (segments <= 1) return;
  int before = 0;
  for (int i = lane; i < b; i += 64) before += segments_of(max(s.extend_seq_lens[i], 0), g.tokens);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) before += __shfl_xor(before, off, 64);
  const int e = (blockIdx.z * 256 + threadIdx.x) * 4;
  float* const first = g.work + ((int64_t)before * H + h) * g.stride;
  const int64_t step = H * g.stride;
  f32x4_c S = {0.f, 0.f, 0.f, 0.f};
  if (s.extend_prefix_lens[b] > 0) {
    const float* from = state + load_idx(s.req_pool_indices, b, s.idx64) * state_stride + (int64_t)h * D * Dv + e;
    S = f32x4_c{from[0], from[1], from[2], from[3]};
  }
  constexpr int AHEAD = 8;
  for (int i0 = 0; i0 < segments; i0 += AHEAD) {
    f32x4_c sum[AHEAD];
    float decay[AHEAD];
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
      const float* at = first + min(i0 + u, segments - 2) * step;      // (the last segment has no sums)
      sum[u] = *(const f32x4_c*)(at + e);
      decay[u] = at[D * Dv + e / Dv];
    }
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
      if (i0 + u >= segments) break;
      *(f32x4_c*)(first + (i0 + u) * step + e) = S;
#pragma unroll
      for (int r = 0; r < 4; ++r) S[r] = decay[u] * S[r] + sum[u][r];
    }
  }
}

template <typename Tag, int D, int NW, bool DELTA, int MODE>
int launch_walk16_mode(const Walk16& a, unsigned groups, const SeqBatch& s, hipStream_t st) {
  constexpr int bytes = Walk16Lds<Tag, D, NW, DELTA, MODE>::kBytes;
  static PerDevice<int> raised;
  if (!chunk_lds_ready(raised, (const void*)chunk16_walk_kernel<Tag, D, NW, DELTA, MODE>, bytes)) return SP_ERR_LAUNCH;
  chunk16_walk_kernel<Tag, D, NW, DELTA, MODE><<<dim3(groups, (unsigned)a.H), NW * 96, bytes, st>>>(a, s);
  SP_LAUNCH_CHECK();
  return SP_OK;
}
template <typename Tag, int D, int NW, bool DELTA>
int launch_walk16(const Walk16& a, int64_t tokens, const SeqBatch& s, hipStream_t st) {
  if (a.seg.tokens == 0) return launch_walk16_mode<Tag, D, NW, DELTA, kWholeRequests>(a, (unsigned)s.B, s, st);
  if constexpr (!DELTA) {
    const unsigned groups = (unsigned)(tokens / a.seg.tokens + s.B);
    const int rc = launch_walk16_mode<Tag, D, NW, DELTA, kSegmentSums>(a, groups, s, st);
    if (rc != SP_OK) return rc;
    segment_rows_kernel<D, NW * 16><<<dim3((unsigned)s.B, (unsigned)a.H, D * NW * 16 / 1024), 256, 0, st>>>(a.seg, a.state, a.state_stride, s, a.H);
    SP_LAUNCH_CHECK();
    return launch_walk16_mode<Tag, D, NW, DELTA, kSegmentOutputs>(a, groups, s, st);
  }
  return SP_ERR_UNSUPPORTED;
}

// 16-byte loads of rows of `type` at `p`
inline bool rows_aligned(const void* p, int64_t stride, int dtype) {
  return ((uintptr_t)p & 15) == 0 && stride % (dtype == SP_F32 ? 4 : 8) == 0;
}

inline int64_t chunk16_units(int64_t tokens, int B) { return tokens / kC16 + B; }      // at most: a request's last chunk may be partial

// ---- windows: a step's chunks in passes over one bounded workspace ----------------------------------------------------------------
// A chunk's prepared operands take 18 - 21 KB per head, so a step takes the chunks that 192 MiB hold at a time (general delta rule, 32 heads
// of 64: 4672 tokens; HGRN2, 8 heads of 128: 21840), and a request's state goes from pass to pass through the pool.  A window
// is a range of the chunks in the order (chunk within its request, request): all requests advance side by side in every pass.  To the
// kernels it is a step of its own - lengths, prefixes and first rows of the requests' pieces (each 16 tokens a chunk but a request's last,
// so the chunks and their bits are the same).  us, whole step at once -> in passes (scratch in MB): general delta rule 1 x 16384 2851 -> 2875 (736
// -> 256 with the rows out), 16 x 1024 663 -> 738, 16 x 2048 1289 -> 1459 (1482 -> 319), 1 x 65536 11419 -> 11423 (2944 -> 447); HGRN2 1 x 65536
// 973 -> 1062, 16 x 2048 524 -> 568.
constexpr int64_t kChunk16Work = (int64_t)192 << 20;

inline int64_t chunk16_window(int H, int floats) { return std::max<int64_t>(1, kChunk16Work / ((int64_t)H * floats * (int64_t)sizeof(float))); }
inline int64_t chunk16_work_floats(int64_t tokens, int B, int H, int floats) {
  const int64_t units = chunk16_units(tokens, B), per = chunk16_window(H, floats);
  return std::min(units, per) * H * floats + (units > per ? (units + per - 1) / per * 3 * B : 0);
}

__device__ __forceinline__ int block_count(int v, int* red) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  return (red[0] + red[1]) + (red[2] + red[3]);
}
// the rounds (a chunk of every request that has one) among the first `rank` chunks, and how many chunks of the round after: by a block of 256
__device__ __forceinline__ void rounds_of(const SeqBatch& s, int rank, int longest, int* red, int& rounds, int& rest) {
  const auto chunks = [&](int c) {
    int n = 0;
    for (int b = threadIdx.x; b < s.B; b += 256) n += min(segments_of(max(s.extend_seq_lens[b], 0), kC16), c);
    return block_count(n, red);
  };
  int lo = 0, hi = longest;                            // the most rounds with at most `rank` chunks
  while (lo < hi) {
    const int mid = lo + (hi - lo + 1) / 2;
    if (chunks(mid) <= rank) lo = mid;
    else hi = mid - 1;
  }
  rounds = lo;
  rest = rank - chunks(lo);
}
// Workgroup: window blockIdx.x.  tables: [window][length, prefix, first row][request]
static __global__ void __launch_bounds__(256) chunk16_windows_kernel(int32_t* tables, SeqBatch s, int per) {
  __shared__ int red[4];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  int longest = 0;
  for (int b = threadIdx.x; b < s.B; b += 256) longest = max(longest, segments_of(max(s.extend_seq_lens[b], 0), kC16));
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) longest = max(longest, __shfl_xor(longest, off, 64));
  if (lane == 0) red[wave] = longest;
  __syncthreads();
  longest = max(max(red[0], red[1]), max(red[2], red[3]));
  int rounds[2], rest[2];
  for (int i = 0; i < 2; ++i) rounds_of(s, (int)(blockIdx.x + i) * per, longest, red, rounds[i], rest[i]);
  int before[2] = {0, 0};                              // requests below this tile of 256 with a chunk in the round that a bound cuts
  int32_t* table = tables + (int64_t)blockIdx.x * 3 * s.B;
  for (int b0 = 0; b0 < s.B; b0 += 256) {
    const int b = b0 + threadIdx.x, len = b < s.B ? max(s.extend_seq_lens[b], 0) : 0, n = segments_of(len, kC16);
    int at[2];
    for (int i = 0; i < 2; ++i) {
      const uint64_t has = __ballot(n > rounds[i]);
      __syncthreads();
      if (lane == 0) red[wave] = __popcll(has);
      __syncthreads();
      int below = before[i] + __popcll(has & ((1ull << lane) - 1));
      for (int w = 0; w < wave; ++w) below += red[w];
      at[i] = min(n, rounds[i]) + (n > rounds[i] && below < rest[i] ? 1 : 0);
      before[i] += (red[0] + red[1]) + (red[2] + red[3]);
    }
    if (b < s.B) {
      table[b] = min(len, at[1] * kC16) - min(len, at[0] * kC16);
      table[s.B + b] = s.extend_prefix_lens[b] + at[0] * kC16;
      table[2 * s.B + b] = s.extend_start_loc[b] + at[0] * kC16;
    }
  }
}

// launch(the step or a window of it, its chunks and tokens at the most) for every window of the step
template <typename Launch>
int each_window16(float* work, int64_t tokens, int H, int floats, const SeqBatch& s, hipStream_t st, const Launch& launch) {
  const int64_t units = chunk16_units(tokens, s.B), per = chunk16_window(H, floats);
  if (units <= per) return launch(s, units, tokens);
  const int windows = (int)((units + per - 1) / per);
  int32_t* table = (int32_t*)(work + per * H * floats);
  chunk16_windows_kernel<<<dim3((unsigned)windows), 256, 0, st>>>(table, s, (int)per);
  SP_LAUNCH_CHECK();
  for (int w = 0; w < windows; ++w, table += 3 * s.B) {
    SeqBatch piece = s;
    piece.extend_seq_lens = table, piece.extend_prefix_lens = table + s.B, piece.extend_start_loc = table + 2 * s.B;
    const int rc = launch(piece, per, per * kC16);
    if (rc != SP_OK) return rc;
  }
  return SP_OK;
}

}  // namespace sp
