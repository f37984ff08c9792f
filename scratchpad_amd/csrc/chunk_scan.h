// Linear recurrences with one decay per head, a chunk of 64 tokens at a time on the matrix cores (bf16 rows, fp32 state).
//
//   S_t = e_t S_{t-1} + c_t k_t v_t^T,   o_t = S_t^T q_t            (S [D, Dv] fp32; e, c scalars of token and head)
//
// is, over a chunk that starts from S_0 and with A_ts = weight of token s's contribution at token t <= s' ... in closed form:
//   o_t = a0_t S_0^T q_t + sum_{s <= t} A_ts (q_t . k_s) v_s,        S_end = a_end S_0 + sum_s w_s k_s v_s^T
// so the serial chain is one step per 64 tokens instead of one per token, and every sum is a matrix product.  The user of this
// header forms A, a0, w and a_end (their logarithms are sums of the tokens' log decays) and owns the state's load and store.
//
// Precision: q, k and v are the 16-bit rows themselves, so q . k has exact products in fp32 sums.  Whatever is fp32 in the
// serial form - the state, the weighted products A (q . k), the weighted values w v - enters the matrix cores as THREE bf16
// parts (8 + 8 + 8 bits by truncation: the split is exact), one MFMA each into the same fp32 accumulator.
//
// Work split: wave w owns the columns [16 w, 16 w + 16) of S and of o for all D and all tokens, S in the accumulator layout of
// v_mfma_f32_16x16x32 (lane (r16, q): column r16, rows 4 q + r of a tile).  Row m of tile i stands for
// d = 32 (i / 2) + 8 (m / 4) + 4 (i % 2) + m % 4, so the 8 values a lane holds in tiles 2 kk, 2 kk + 1 are the neighbouring
// d = 32 kk + 8 q + 0 .. 7: split in place they ARE the operand of S^T q, the state never passes through LDS.  The 10 lower
// 16 x 16 tiles of q k^T (and two of zeros) are dealt to the waves and exchanged through LDS.  Two products sum over tokens
// and take their operands transposed: k and v are also staged as [channel][token], two tokens packed per 4-byte write.
//
// Values that are not finite: a product with the tokens' values would carry one to the EARLIER tokens of its chunk (zero weights
// times it), so such values are taken out of a chunk that has any (stage, clear), and in their column the outputs from their token on
// and the state become NaN (spoil).  What is not finite in q, k, the weights or the state meets only its own tokens and later ones.
#pragma once
#include "seq_batch.h"

#include <type_traits>

namespace sp {

typedef float f32x4_c __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8_c __attribute__((ext_vector_type(8)));
__device__ __forceinline__ f32x4_c mfma_c(const u32x4& a, const u32x4& b, const f32x4_c& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_c, a), __builtin_bit_cast(bf16x8_c, b), c, 0, 0, 0);
}

// two fp32 as three packed bf16 pairs whose sum is exact: the upper 16 bits, then those of what is left, twice
__device__ __forceinline__ void split3(float x, float y, uint32_t& hi, uint32_t& mid, uint32_t& lo) {
  hi = __builtin_amdgcn_perm(as_u32(y), as_u32(x), 0x07060302u);
  x -= as_f32(as_u32(x) & 0xffff0000u);
  y -= as_f32(as_u32(y) & 0xffff0000u);
  mid = __builtin_amdgcn_perm(as_u32(y), as_u32(x), 0x07060302u);
  x -= as_f32(as_u32(x) & 0xffff0000u);
  y -= as_f32(as_u32(y) & 0xffff0000u);
  lo = __builtin_amdgcn_perm(as_u32(y), as_u32(x), 0x07060302u);
}

constexpr int kCL = 64;      // tokens per chunk

// inclusive scans over a wave, in 64 bits: a chunk's log decays are summed and then subtracted from each other, and an exponent
// that is wrong by the sum's fp32 rounding would be a weight wrong by as much (6e-5 where the sums reach -1000).  For the same
// reason the sums go to the weights as two fp32 parts, subtracted part by part: an exponent is then off by an ulp of itself.
__device__ __forceinline__ double wave_scan_sum(double v, int lane) {
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const double o = __shfl_up(v, off, 64);
    if (lane >= off) v += o;
  }
  return v;
}
__device__ __forceinline__ double wave_scan_max(double v, int lane) {
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const double o = __shfl_up(v, off, 64);
    if (lane >= off) v = fmax(v, o);
  }
  return v;
}

// what the products need of a chunk's tokens, in LDS: weight of s at t = exp(lt[t] - ls[s]) * cs[s] (s <= t), lt and ls each the
// sum of two parts, see above
struct ChunkScalars {
  float lt[2][kCL], ls[2][kCL], cs[kCL], a0[kCL], w[kCL];
  float a_end, pad[3];

  static __device__ __forceinline__ void put(float (*to)[kCL], int i, double v) {
    const float hi = (float)v;
    to[0][i] = hi;
    to[1][i] = fabsf(hi) == INFINITY ? 0.f : (float)(v - (double)hi);
  }
};

// rows that can be read 16 bytes at a time, a chunk's worth of them within 32-bit offsets
inline bool chunk_aligned(const void* p, int64_t stride) {
  return stride % 8 == 0 && stride < ((int64_t)1 << 24) && ((uintptr_t)p & 15) == 0;
}
// a value that is the same in all lanes, moved to scalar registers (addresses then cost a 32-bit offset per lane)
__device__ __forceinline__ int64_t uniform64(int64_t v) {
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return (int64_t)(((uint64_t)hi << 32) | lo);
}

// (OUT false: the state's part only, for the sums of a request's segments - no q, no rows of k, no outputs)
template <int D, int NW, bool OUT = true>
struct ChunkScan {
  static constexpr int Dv = NW * 16, NT = NW * 64, QROW = D * 2 + 16, TROW = kCL * 2 + 16;
  static constexpr int kQ = 0, kKT = kQ + (OUT ? kCL * QROW : 0), kVT = kKT + D * TROW, kP = kVT + Dv * TROW;
  static constexpr int kK = kP;                                  // the rows of k are gone when the weighted tiles arrive
  static constexpr int kPBytes = !OUT ? 0 : 3 * kCL * TROW > kCL * QROW ? 3 * kCL * TROW : kCL * QROW;
  static constexpr int kSum = kP + kPBytes;                      // float [4][kCL]: sums of the weighted tiles over s
  static constexpr int kScalars = kSum + (OUT ? 4 * kCL * 4 : 0);
  static constexpr int kOdd = kScalars + 2 * (int)sizeof(ChunkScalars);      // int: the last chunk's number + 1 with such values
  static constexpr int kFirst = kOdd + 16;                                   // int [Dv]: a column's first token of it
  static constexpr int kBytes = kFirst + Dv * 4;
  static constexpr int QN = kCL * (D / 8), KN = kCL / 2 * (D / 8), VN = kCL / 2 * (Dv / 8);
  static constexpr int QU = (QN + NT - 1) / NT, KU = (KN + NT - 1) / NT, VU = (VN + NT - 1) / NT;
  static constexpr int TILES = 12 / NW + (12 % NW != 0), DT = D / 16;

  u32x4 rq[QU], rk[KU][2], rv[VU][2];       // the next chunk's rows
  f32x4_c S[DT], o[4], p[TILES];
  char* lds;
  const ChunkScalars* sc;
  int tid, wave, lane, r16, q;

  __device__ __forceinline__ ChunkScan(char* l) : lds(l) {
    tid = threadIdx.x;
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    lane = tid & 63;
    r16 = lane & 15;
    q = lane >> 4;
  }
  // the scalars of a chunk are formed while the one before it is worked on: two sets, the running chunk's in `sc`
  __device__ __forceinline__ ChunkScalars* scalars(int64_t chunk) const { return (ChunkScalars*)(lds + kScalars) + (chunk & 1); }
  __device__ __forceinline__ float* sums() const { return (float*)(lds + kSum); }
  __device__ __forceinline__ int* odd() const { return (int*)(lds + kOdd); }
  // the d of register (i, r) and the column of this lane's part of the state
  __device__ __forceinline__ int row_of(int i, int r) const { return 32 * (i / 2) + 8 * q + 4 * (i & 1) + r; }
  __device__ __forceinline__ int column() const { return 16 * wave + r16; }

  static __device__ __forceinline__ u32x4 row16(const char* base, uint32_t stride, int t, int n, int at) {
    return t < n ? ld16(base + (uint32_t)(t * stride + at)) : u32x4{0u, 0u, 0u, 0u};
  }
  // rows of the chunk (bases at its first token, strides in bytes), zeros from token n on
  __device__ __forceinline__ void load(const char* qb, uint32_t qs, const char* kb, uint32_t ks, const char* vb, uint32_t vs, int n) {
#pragma unroll
    for (int u = 0; u < QU; ++u) {
      const int x = tid + u * NT;
      if (OUT && x < QN) rq[u] = row16(qb, qs, x / (D / 8), n, x % (D / 8) * 16);
    }
#pragma unroll
    for (int u = 0; u < KU; ++u) {
      const int x = tid + u * NT, t = x % (kCL / 2) * 2, c = x / (kCL / 2) * 16;
      if (x < KN) {
        rk[u][0] = row16(kb, ks, t, n, c);
        rk[u][1] = row16(kb, ks, t + 1, n, c);
      }
    }
#pragma unroll
    for (int u = 0; u < VU; ++u) {
      const int x = tid + u * NT, t = x % (kCL / 2) * 2, c = x / (kCL / 2) * 16;
      if (x < VN) {
        rv[u][0] = row16(vb, vs, t, n, c);
        rv[u][1] = row16(vb, vs, t + 1, n, c);
      }
    }
  }
  __device__ __forceinline__ void put_transposed(char* dst, const u32x4& a, const u32x4& b) const {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      *(uint32_t*)(dst + 2 * e * TROW) = __builtin_amdgcn_perm(b[e], a[e], 0x05040100u);          // the two low halves
      *(uint32_t*)(dst + (2 * e + 1) * TROW) = __builtin_amdgcn_perm(b[e], a[e], 0x07060302u);    // the two high halves
    }
  }
  __device__ __forceinline__ void stage(int chunk) const {
#pragma unroll
    for (int u = 0; u < QU; ++u) {
      const int x = tid + u * NT;
      if (OUT && x < QN) st16(lds + kQ + x / (D / 8) * QROW + x % (D / 8) * 16, rq[u]);
    }
#pragma unroll
    for (int u = 0; u < KU; ++u) {
      const int x = tid + u * NT, t = x % (kCL / 2) * 2, c = x / (kCL / 2);
      if (x < KN) {
        if constexpr (OUT) {
          st16(lds + kK + t * QROW + c * 16, rk[u][0]);
          st16(lds + kK + (t + 1) * QROW + c * 16, rk[u][1]);
        }
        put_transposed(lds + kKT + c * 8 * TROW + t * 2, rk[u][0], rk[u][1]);
      }
    }
#pragma unroll
    for (int u = 0; u < VU; ++u) {
      const int x = tid + u * NT, t = x % (kCL / 2) * 2, c = x / (kCL / 2);
      if (x < VN) {
        if constexpr (OUT) {
          uint32_t ones = 0u;                          // (an exponent of ones carries into the sign)
#pragma unroll
          for (int e = 0; e < 8; ++e) ones |= (rv[u][e & 1][e / 2] & 0x7f807f80u) + 0x00800080u;
          if (ones & 0x80008000u) *odd() = chunk + 1;
        }
        put_transposed(lds + kVT + c * 8 * TROW + t * 2, rv[u][0], rv[u][1]);
      }
    }
  }
  static __device__ __forceinline__ void tile_of(int id, int& i, int& j) {      // ids 0 .. 9 lower tiles, 10 and 11 zeros
    i = id < 1 ? 0 : (id < 3 ? 1 : (id < 6 ? 2 : 3));
    j = id - i * (i + 1) / 2;
    if (id == 10) i = 0, j = 1;
    if (id == 11) i = 2, j = 3;
  }
  // this wave's tiles of k q^T: lane (r16, q) gets s = 16 j + 4 q + r of t = 16 i + r16
  __device__ __forceinline__ void scores() {
    int i[TILES], j[TILES];
#pragma unroll
    for (int u = 0; u < TILES; ++u) {
      p[u] = f32x4_c{0.f, 0.f, 0.f, 0.f};
      tile_of(min(wave + u * NW, 9), i[u], j[u]);                // (ids past 9: computed, never used)
    }
#pragma unroll
    for (int kk = 0; kk < D / 32; ++kk)
#pragma unroll
      for (int u = 0; u < TILES; ++u)
        p[u] = mfma_c(ld16(lds + kK + (16 * j[u] + r16) * QROW + kk * 64 + 16 * q),
                      ld16(lds + kQ + (16 * i[u] + r16) * QROW + kk * 64 + 16 * q), p[u]);
  }
  // o = a0 S_0^T q
  __device__ __forceinline__ void from_state(bool zero_state) {
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = f32x4_c{0.f, 0.f, 0.f, 0.f};
    if (zero_state) return;
#pragma unroll
    for (int kk = 0; kk < D / 32; ++kk) {
      u32x4 a[4], b[3];
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = ld16(lds + kQ + (16 * i + r16) * QROW + kk * 64 + 16 * q);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        uint32_t hi, mid, lo;
        split3(S[2 * kk + e / 2][2 * (e & 1)], S[2 * kk + e / 2][2 * (e & 1) + 1], hi, mid, lo);
        b[0][e] = hi, b[1][e] = mid, b[2][e] = lo;
      }
#pragma unroll
      for (int x = 2; x >= 0; --x)
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = mfma_c(a[i], b[x], o[i]);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const f32x4_c a0 = *(const f32x4_c*)(sc->a0 + 16 * i + 4 * q);
#pragma unroll
      for (int r = 0; r < 4; ++r) o[i][r] *= a0[r];
    }
  }
  // the weighted tiles into LDS, and (SUMS) their sums over s
  template <bool SUMS>
  __device__ __forceinline__ void weigh() {
#pragma unroll
    for (int u = 0; u < TILES; ++u) {
      const int id = wave + u * NW;
      if (id >= 12) break;
      int i, j;
      tile_of(id, i, j);
      const int t = 16 * i + r16, s0 = 16 * j + 4 * q;
      const float lt = sc->lt[0][t], lt2 = sc->lt[1][t];
      const f32x4_c ls = *(const f32x4_c*)(sc->ls[0] + s0), ls2 = *(const f32x4_c*)(sc->ls[1] + s0), cs = *(const f32x4_c*)(sc->cs + s0);
      float v[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = s0 + r <= t ? p[u][r] * (expf((lt - ls[r]) + (lt2 - ls2[r])) * cs[r]) : 0.f;
      if constexpr (SUMS) {
        float sum = (v[0] + v[1]) + (v[2] + v[3]);
        sum += __shfl_xor(sum, 16, 64);
        sum += __shfl_xor(sum, 32, 64);
        if (q == 0) sums()[j * kCL + t] = sum;
      }
      uint32_t part[3][2];
#pragma unroll
      for (int e = 0; e < 2; ++e) split3(v[2 * e], v[2 * e + 1], part[0][e], part[1][e], part[2][e]);
#pragma unroll
      for (int x = 0; x < 3; ++x)
        *(u32x2*)(lds + kP + (x * kCL + t) * TROW + s0 * 2) = u32x2{part[x][0], part[x][1]};
    }
  }
  // the values of this wave's columns without those that are not finite (lane (r16, q): 16 tokens of a column), and the first of them
  __device__ __forceinline__ void clear() const {
    uint16_t* v = (uint16_t*)(lds + kVT + column() * TROW) + 16 * q;
    int first = kCL;
    for (int t = 15; t >= 0; --t)
      if ((v[t] & 0x7f80) == 0x7f80) {
        v[t] = 0;
        first = 16 * q + t;
      }
    first = min(first, __shfl_xor(first, 16, 64));
    first = min(first, __shfl_xor(first, 32, 64));
    ((int*)(lds + kFirst))[column()] = first;
  }
  __device__ __forceinline__ void spoil() {
    const int first = ((const int*)(lds + kFirst))[column()];
    const float nan = as_f32(0x7fc00000u);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) o[i][r] = 16 * i + 4 * q + r >= first ? nan : o[i][r];
#pragma unroll
    for (int i = 0; i < DT; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) S[i][r] = first < kCL ? nan : S[i][r];
  }
  // o += (weighted tiles) v;  S = a_end S + k^T (w v)
  __device__ __forceinline__ void absorb(int chunk) {
    // (OUT false: a value that is not finite leaves its column of the state so by itself)
    const bool any = OUT && __builtin_amdgcn_readfirstlane(*odd()) == chunk + 1;
    if (any) clear();
    const float a_end = sc->a_end;
#pragma unroll
    for (int i = 0; i < DT; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) S[i][r] *= a_end;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const u32x4 v = ld16(lds + kVT + column() * TROW + ks * 64 + 16 * q);
      if constexpr (OUT)
#pragma unroll
        for (int x = 2; x >= 0; --x)
#pragma unroll
          for (int i = 2 * ks; i < 4; ++i)
            o[i] = mfma_c(ld16(lds + kP + (x * kCL + 16 * i + r16) * TROW + ks * 64 + 16 * q), v, o[i]);
      float f[8];
      unpack16<bf16_tag>(v, f);
      const f32x4_c w0 = *(const f32x4_c*)(sc->w + ks * 32 + 8 * q), w1 = *(const f32x4_c*)(sc->w + ks * 32 + 8 * q + 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) f[e] *= w0[e], f[4 + e] *= w1[e];
      u32x4 b[3];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        uint32_t hi, mid, lo;
        split3(f[2 * e], f[2 * e + 1], hi, mid, lo);
        b[0][e] = hi, b[1][e] = mid, b[2][e] = lo;
      }
#pragma unroll
      for (int i0 = 0; i0 < DT; i0 += 4) {
        u32x4 a[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
          a[i] = ld16(lds + kKT + (32 * ((i0 + i) / 2) + 8 * (r16 / 4) + 4 * (i & 1) + r16 % 4) * TROW + ks * 64 + 16 * q);
#pragma unroll
        for (int x = 2; x >= 0; --x)
#pragma unroll
          for (int i = 0; i < 4; ++i) S[i0 + i] = mfma_c(a[i], b[x], S[i0 + i]);
      }
    }
    if (any) spoil();
  }
  __device__ __forceinline__ void load_state(const float* st, bool held) {      // (st is not read unless held)
#pragma unroll
    for (int i = 0; i < DT; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) S[i][r] = held ? st[(int64_t)row_of(i, r) * Dv + column()] : 0.f;
    // here before the loop over chunks: a wait for them inside it would be one for the next chunk's loads, every time
#pragma unroll
    for (int i = 0; i < DT; ++i) asm volatile("" : "+v"(S[i]));
    if (tid == 0) *odd() = 0;
    lds_barrier();                                   // (before a first chunk's)
  }
  __device__ __forceinline__ void store_state(float* st) const {
#pragma unroll
    for (int i = 0; i < DT; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) st[(int64_t)row_of(i, r) * Dv + column()] = S[i][r];
  }
};

// ---- segments: a request's chunks as several workgroups -----------------------------------------------------------------------
// One workgroup per (request, head) walks the request's chunks in turn; few requests leave most of the chip idle and the longest one
// sets the time.  The state is linear in the one a segment starts from, so segments of `tokens` tokens (a multiple of kCL) run side by
// side in three launches: every segment but a request's last walks its own tokens from an empty state (kSegmentSums; no outputs, about
// a third of the work), segment_states_kernel chains these sums into the state that each segment starts from, and every segment
// walks its tokens once more from there (kSegmentOutputs); a request's last one leaves the new state in the pool.  3001
// tokens of 5 requests, 16 heads of 128 x 128 (mLSTM), segments of 256: 146 us -> 19 (sums) + 8 (states) + 54 (outputs); the rule for the
// segments' length (_native.py) has both sides' times of whole layers.
enum { kWholeRequests = 0, kSegmentSums = 1, kSegmentOutputs = 2 };

// of a segment and head, in the workspace: S [D * Dv], n [D] (mLSTM), then kSegScalars floats: the decay of what the segment started
// from (mLSTM: as the sum of the log forget gates, a double, and the largest exponent of its own sums; the one that it starts from)
constexpr int kSegScalars = 8, kSegDecay = 0, kSegMax = 2, kSegStart = 3;

inline int64_t segment_floats(int D, int Dv, bool normaliser) { return (int64_t)D * Dv + (normaliser ? D : 0) + kSegScalars; }

// floats of a step's segments (with mLSTM's normaliser, for either recurrence); no segments: none
inline int64_t scan_segment_floats(int64_t num_tokens, int batch_size, int heads, int dim, int vdim, int segment_tokens) {
  return segment_tokens > 0 ? (num_tokens / segment_tokens + batch_size) * heads * segment_floats(dim, vdim, true) : 0;
}

struct ScanSegments {
  float* work;
  int64_t stride;            // floats per segment and head
  int tokens;
};

__device__ __forceinline__ int segments_of(int len, int tokens) { return (len + tokens - 1) / tokens; }
// the request, first token (within it) and length of segment `id` of the step; false behind the last (all lanes of a wave ask)
__device__ __forceinline__ bool segment_at(const SeqBatch& s, int id, int tokens, int lane, int& b, int& t0) {
  for (int b0 = 0; b0 < s.B; b0 += 64) {
    const int i = b0 + lane;
    const int n = i < s.B ? segments_of(max(s.extend_seq_lens[i], 0), tokens) : 0;
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
      t0 = __builtin_amdgcn_readfirstlane((id - __shfl(incl - n, l, 64)) * tokens);
      return true;
    }
    id -= __builtin_amdgcn_readfirstlane(__shfl(incl, 63, 64));
  }
  return false;
}

// Workgroup (request, head, 1024 values of S): the sums of the request's segments become the states they start from.  Memory: a read
// and a write of all segments' states.  MAXED (mLSTM): sums are relative to exp(their largest exponent), n is chained too.
template <bool MAXED>
__global__ void __launch_bounds__(256)
segment_states_kernel(ScanSegments g, const float* S_state, int64_t S_stride, const float* n_state, int64_t n_stride, const float* m_state,
                      int64_t m_stride, SeqBatch s, int H, int D, int Dv) {
  const int b = blockIdx.x, h = blockIdx.y, lane = threadIdx.x & 63;
  const int segments = segments_of(s.extend_seq_lens[b], g.tokens);
  if (segments <= 1) return;
  int before = 0;
  for (int i = lane; i < b; i += 64) before += segments_of(max(s.extend_seq_lens[i], 0), g.tokens);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) before += __shfl_xor(before, off, 64);
  const bool held = s.extend_prefix_lens[b] > 0;
  const int64_t slot = load_idx(s.req_pool_indices, b, s.idx64);
  const int states = D * Dv, scalars = states + (MAXED ? D : 0), e = (blockIdx.z * 256 + threadIdx.x) * 4;
  float* const first = g.work + ((int64_t)before * H + h) * g.stride;
  const int64_t step = H * g.stride;
  const bool live = e < scalars;                       // (n's values follow those of S)
  f32x4_c S = {0.f, 0.f, 0.f, 0.f};
  if (held && live) {
    const float* from = e < states ? S_state + slot * S_stride + (int64_t)h * states + e : n_state + slot * n_stride + (int64_t)h * D + e - states;
    S = f32x4_c{from[0], from[1], from[2], from[3]};
  }
  float m = MAXED && held ? m_state[slot * m_stride + h] : 0.f;
  constexpr int AHEAD = 8;
  for (int i0 = 0; i0 < segments; i0 += AHEAD) {
    f32x4_c sum[AHEAD];
    double F[AHEAD];
    float top[AHEAD];
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
      const float* at = first + min(i0 + u, segments - 2) * step;      // (the last segment has no sums)
      sum[u] = live ? *(const f32x4_c*)(at + e) : f32x4_c{0.f, 0.f, 0.f, 0.f};
      if constexpr (MAXED) {
        F[u] = *(const double*)(at + scalars + kSegDecay);
        top[u] = at[scalars + kSegMax];
      } else {
        top[u] = at[scalars + kSegDecay];
      }
    }
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
      if (i0 + u >= segments) break;
      float* at = first + (i0 + u) * step;
      if (live) *(f32x4_c*)(at + e) = S;
      if (MAXED && e == 0) at[scalars + kSegStart] = m;
      if constexpr (MAXED) {
        const double old = F[u] + (double)m, now = fmax(old, (double)top[u]);
        const float keep = expf((float)(old - now)), take = expf((float)((double)top[u] - now));
#pragma unroll
        for (int r = 0; r < 4; ++r) S[r] = keep * S[r] + take * sum[u][r];
        m = F[u] != F[u] ? (float)F[u] : (float)now;
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) S[r] = top[u] * S[r] + sum[u][r];
      }
    }
  }
}

// raise a kernel's dynamic-LDS limit to `bytes`, once per device of the process (`raised`: a static of the launching function)
inline bool chunk_lds_ready(PerDevice<int>& raised, const void* kernel, int bytes) {
  int ok = 0;
  raised.get(ok, [&](int) { return hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) == hipSuccess ? 1 : 0; });
  return ok != 0;
}

}  // namespace sp
