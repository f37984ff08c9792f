// Grouped-query attention over a sliding window plus pooled blocks, on a token-level key/value pool.
//
// A query at position p sees the tokens j with 0 <= p - j < size and, for every block of P consecutive positions that
// lies wholly before the window (block b = positions bP .. bP + P - 1, seen once bP + P - 1 <= p - size), ONE key and
// value: the means of the block's cached keys and values.  Tokens and blocks share one softmax.  Tokens that left the
// window while their block is still incomplete behind it are not seen.  size <= 0 means no window (plain causal),
// P <= 0 no pooling.  With `keep_first` = n > 0 (and no pooling) the tokens j < n stay visible to every later query: they are
// numbered like blocks of one token whose mean is the token itself, of which only the first n exist.
//
// Cache: per token a key row [G, D] (rotated) and a value row [G, Dv] (each head divided by its root mean square); the
// pooled key/value of block b lives in a second pair of buffers at the slot of the block's LAST token, written by the
// step that brings this token, so the pooled rows need no allocator of their own and are freed with the token.
//
// Rotation: "rotate half" - coordinate i < dims/2 pairs with i + dims/2 - or, with `adjacent`, coordinate 2i with 2i + 1;
// angle = position * freq[i] in fp32, cos and sin times mag; coordinates from dims on pass.  Optional fp32 biases join q, k
// and v before the rotation; the per-head norm of the values can be switched off.  Scores, softmax and the weighted sum are
// fp32.  With `sinks` (one fp32 number per query head) the softmax's denominator holds one more term exp(sink): a key that
// is seen by every query, is not scaled and has no value.
//
// Further forms of the same layer (each a parameter): q and k divided per head by their root mean square after the
// rotation, or before it and then times a learned weight per coordinate (shared by the heads); values that are the keys as
// projected, before norm and rotation; q times a number per head and times 1 + coef ln(floor((position + 1) / every) + 1); values blended with the
// values an earlier layer cached for the same token, v <- (1 - lambda) v + lambda v_first; scores capped as
// cap tanh(score / cap); and, instead of the softmax, every visible key weighted by sigmoid(score + bias[head]) without
// normalisation.  The result can be multiplied element by element with sigmoid(gate) on its way out.
#include "seq_batch.h"

namespace sp {
namespace {

// a pair (u, w) turned by an angle, rounded to Tag's type.  The fused operations are written out: the compiler fuses one product or the
// other, and rounds to 16 bits inside or behind the sum, as a loop's unrolling suggests to it - a token's row must not depend on the
// kernel that stores it.
template <typename Tag>
__device__ __forceinline__ void turn_pair(float u, float w, float cosine, float sine, float& first, float& second) {
  first = fma_round<Tag>(u, cosine, -(w * sine));
  second = fma_round<Tag>(u, sine, w * cosine);
}

// q rotated in place; k rotated and v (normed per head unless norm_v is 0) into the pool rows loc[t]
template <typename Tag>
__global__ void __launch_bounds__(kBlock)
qkv_rotary_store_kernel(void* q, int64_t q_stride, const void* k, int64_t k_stride, const void* v, int64_t v_stride,
                        void* kpool, int64_t kp_stride, void* vpool, int64_t vp_stride, const int64_t* positions,
                        const int64_t* loc, const float* freq, float mag, const float* qb, const float* kb, const float* vb,
                        int H, int G, int D, int Dv, int dims, int adjacent, int norm_v, float eps) {
  typedef Elem<Tag> E;
  const int64_t t = blockIdx.x;
  const float pos = (float)positions[t];
  const int half = dims / 2;
  const int64_t slot = loc[t];
  const int second = adjacent ? 1 : half, step = adjacent ? 2 : 1;      // a pair is (i * step, i * step + second)
  for (int e = threadIdx.x; e < H * half; e += blockDim.x) {
    const int h = e / half, i = e % half;
    const float a = pos * freq[i];
    const float c = cosf(a) * mag, sn = sinf(a) * mag;
    const int col = h * D + i * step;
    const int64_t at = t * q_stride + col;
    const float u = E::load(q, at) + (qb ? qb[col] : 0.f), w = E::load(q, at + second) + (qb ? qb[col + second] : 0.f);
    float x, y;
    turn_pair<Tag>(u, w, c, sn, x, y);
    E::store(q, at, x);
    E::store(q, at + second, y);
  }
  for (int e = threadIdx.x; e < G * half; e += blockDim.x) {
    const int g = e / half, i = e % half;
    const float a = pos * freq[i];
    const float c = cosf(a) * mag, sn = sinf(a) * mag;
    const int col = g * D + i * step;
    const int64_t at = t * k_stride + col, to = slot * kp_stride + col;
    const float u = E::load(k, at) + (kb ? kb[col] : 0.f), w = E::load(k, at + second) + (kb ? kb[col + second] : 0.f);
    float x, y;
    turn_pair<Tag>(u, w, c, sn, x, y);
    E::store(kpool, to, x);
    E::store(kpool, to + second, y);
  }
  const int rest = D - dims;
  if (qb)
    for (int e = threadIdx.x; e < H * rest; e += blockDim.x) {
      const int col = (e / rest) * D + dims + e % rest;
      E::store(q, t * q_stride + col, E::load(q, t * q_stride + col) + qb[col]);
    }
  for (int e = threadIdx.x; e < G * rest; e += blockDim.x) {
    const int col = (e / rest) * D + dims + e % rest;
    E::store(kpool, slot * kp_stride + col, E::load(k, t * k_stride + col) + (kb ? kb[col] : 0.f));
  }
  if (!norm_v) {
    for (int e = threadIdx.x; e < G * Dv; e += blockDim.x)
      E::store(vpool, slot * vp_stride + e, E::load(v, t * v_stride + e) + (vb ? vb[e] : 0.f));
    return;
  }
  // value heads: one wave each
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, waves = blockDim.x >> 6;
  for (int g = wave; g < G; g += waves) {
    const int64_t at = t * v_stride + (int64_t)g * Dv, to = slot * vp_stride + (int64_t)g * Dv;
    float ss = 0.f;
    for (int i = lane; i < Dv; i += 64) {
      const float x = E::load(v, at + i) + (vb ? vb[g * Dv + i] : 0.f);
      ss += x * x;
    }
    ss = wave_sum(ss);
    const float inv = 1.f / sqrtf(ss / (float)Dv + eps);
    for (int i = lane; i < Dv; i += 64) E::store(vpool, to + i, mul_round<Tag>(E::load(v, at + i) + (vb ? vb[g * Dv + i] : 0.f), inv));
  }
}

// The same for steps of more than 64 tokens (prompts, and decode steps of so many requests) in 16-byte pieces, a wave per token: its
// angles' cosines and sines are formed once, a lane each, and wait in LDS; a lane then takes V neighbouring pairs of a head, or V of its
// values (halves, no biases, values normed; VL lanes share a value head).  The kernel above forms the two functions pair by pair of every
// head and takes a value per lane and load.  16 + 4 heads of 128 with 64 rotated, it / this one in us: 65 tokens 4.4 / 4.1, 256: 4.5 / 4.1,
// 1024: 6.0 / 4.5, 4096: 15.0 / 7.6 (a workgroup per token with these pieces: 13.4).  The same bits.
template <typename Tag, int VL>
__global__ void __launch_bounds__(kBlock)
qkv_rotary_wave_kernel(char* q, int64_t q_stride, const char* k, int64_t k_stride, const char* v, int64_t v_stride, char* kpool,
                       int64_t kp_stride, char* vpool, int64_t vp_stride, const int64_t* positions, const int64_t* loc, const float* freq,
                       float mag, int64_t T, int H, int G, int D, int dims, float eps) {
  typedef Elem<Tag> E;
  constexpr int V = E::kVec, Dv = VL * V;
  __shared__ __attribute__((aligned(16))) float angles[kBlock / 64][2][64];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, half = dims / 2;
  const int64_t t = (int64_t)blockIdx.x * (kBlock / 64) + wave;
  if (t >= T) return;
  const float pos = (float)positions[t];
  const int64_t slot = loc[t];
  float *const cosine = angles[wave][0], *const sine = angles[wave][1];
  if (lane < half) {
    const float a = pos * freq[lane];
    cosine[lane] = cosf(a) * mag;
    sine[lane] = sinf(a) * mag;
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  const int per = half / V, pieces = (H + G) * per;
#pragma unroll 2
  for (int e = lane; e < pieces; e += 64) {
    const int head = e / per, i = e % per * V;
    const bool isq = head < H;
    const int col = (isq ? head : head - H) * D + i;
    char* const at = q + (t * q_stride + col) * E::kBytes;
    const char* const from = isq ? at : k + (t * k_stride + col) * E::kBytes;
    char* const to = isq ? at : kpool + (slot * kp_stride + col) * E::kBytes;
    float u[V], w[V], a[V], b[V];
    unpack16<Tag>(ld16(from), u);
    unpack16<Tag>(ld16(from + half * E::kBytes), w);
#pragma unroll
    for (int x = 0; x < V; ++x) turn_pair<Tag>(u[x], w[x], cosine[i + x], sine[i + x], a[x], b[x]);
    st16(to, pack16<Tag>(a));
    st16(to + half * E::kBytes, pack16<Tag>(b));
  }
  const int rest = (D - dims) / V;
  for (int e = lane; e < G * rest; e += 64) {
    const int col = e / rest * D + dims + e % rest * V;
    st16(kpool + (slot * kp_stride + col) * E::kBytes, ld16(k + (t * k_stride + col) * E::kBytes));
  }
  for (int e = lane; e < (G * VL + 63) / 64 * 64; e += 64) {          // (whole waves: the sum is over lanes)
    const bool in = e < G * VL;
    float x[V], sq[V];
    unpack16<Tag>(ld16(v + (t * v_stride + (in ? e : 0) * V) * E::kBytes), x);
    // the squares in the order of the kernel above (a value per lane, wave_sum): values 64 apart, then 32, 16 ... 1 - here over the
    // lanes of a head first, then over a lane's own values - so that a row's bits do not depend on how many tokens a step has
#pragma unroll
    for (int c = 0; c < V; ++c) {
      sq[c] = x[c] * x[c];
      asm("" : "+v"(sq[c]));                          // (rounded here, not inside a fused multiply-add)
      if constexpr (VL == 16) {
        sq[c] += dpp_f32<0x128>(sq[c]);               // row_ror 8: lane ^ 8
        sq[c] += dpp_f32<0x124>(sq[c]);               // row_ror 4: lane ^ 4, since lanes 8 apart hold the same by now
      } else {
        sq[c] += __shfl_xor(sq[c], 4, 64);
      }
      sq[c] += dpp_f32<0x4E>(sq[c]);                  // lane ^ 2
      sq[c] += dpp_f32<0xB1>(sq[c]);                  // lane ^ 1
    }
#pragma unroll
    for (int off = V / 2; off > 0; off /= 2)
#pragma unroll
      for (int c = 0; c < off; ++c) sq[c] += sq[c + off];
    const float inv = 1.f / sqrtf(sq[0] / (float)Dv + eps);
#pragma unroll
    for (int c = 0; c < V; ++c) x[c] = mul_round<Tag>(x[c], inv);
    if (in) st16(vpool + (slot * vp_stride + e * V) * E::kBytes, pack16<Tag>(x));
  }
}

// The same store with a wave per head: q and k can be divided by their root mean square over the head AFTER the rotation
// (qk_norm 1) or BEFORE it, times a weight per coordinate (qk_norm 2), q scaled per head and by position, v blended with the
// row another layer's pool holds for the same slot.  v null: the values are the keys as projected (bias included, neither
// normed nor rotated), written by the wave that makes the key.  A lane holds the coordinates lane, lane + 64, ... of its head (dim, vdim <= 64 * kStorePerLane).
// The token's angles are the same for all its heads: their cosines and sines (times mag) wait in LDS.
constexpr int kStorePerLane = 4;
template <typename Tag>
__device__ __forceinline__ void rotated_head(float* val, const void* src, int64_t at, const float* bias, int col0, int D,
                                             int dims, int adjacent, const float* cosine, const float* sine, int lane) {
  typedef Elem<Tag> E;
  const int half = dims / 2;
#pragma unroll
  for (int u = 0; u < kStorePerLane; ++u) {
    const int i = lane + 64 * u;
    float out = 0.f;
    if (i < D) {
      const float x = E::load(src, at + i) + (bias ? bias[col0 + i] : 0.f);
      out = x;
      if (i < dims) {
        int pi, fi;
        bool first;
        if (adjacent) {
          first = (i & 1) == 0;
          pi = first ? i + 1 : i - 1;
          fi = i >> 1;
        } else {
          first = i < half;
          pi = first ? i + half : i - half;
          fi = first ? i : i - half;
        }
        const float y = E::load(src, at + pi) + (bias ? bias[col0 + pi] : 0.f);
        const float c = cosine[fi], sn = sine[fi];
        out = first ? x * c - y * sn : x * c + y * sn;
      }
    }
    val[u] = out;
  }
}

// the head before the rotation divided by its root mean square and times weight[i], then rotated; raw: the head as projected
template <typename Tag>
__device__ __forceinline__ void normed_rotated_head(float* val, float* raw, const void* src, int64_t at, const float* bias,
                                                    int col0, int D, int dims, int adjacent, const float* cosine,
                                                    const float* sine, const float* weight, float eps, int lane) {
  typedef Elem<Tag> E;
  const int half = dims / 2;
  float ss = 0.f;
#pragma unroll
  for (int u = 0; u < kStorePerLane; ++u) {
    const int i = lane + 64 * u;
    raw[u] = i < D ? E::load(src, at + i) + (bias ? bias[col0 + i] : 0.f) : 0.f;
    ss += raw[u] * raw[u];
  }
  const float inv = 1.f / sqrtf(wave_sum(ss) / (float)D + eps);
#pragma unroll
  for (int u = 0; u < kStorePerLane; ++u) {
    const int i = lane + 64 * u;
    float out = 0.f;
    if (i < D) {
      const float x = raw[u] * inv * (weight ? weight[i] : 1.f);
      out = x;
      if (i < dims) {
        const bool first = adjacent ? (i & 1) == 0 : i < half;
        const int pi = adjacent ? (first ? i + 1 : i - 1) : (first ? i + half : i - half);
        const int fi = adjacent ? i >> 1 : (first ? i : i - half);
        const float y = (E::load(src, at + pi) + (bias ? bias[col0 + pi] : 0.f)) * inv * (weight ? weight[pi] : 1.f);
        const float c = cosine[fi], sn = sine[fi];
        out = first ? x * c - y * sn : x * c + y * sn;
      }
    }
    val[u] = out;
  }
}

template <typename Tag>
__global__ void __launch_bounds__(1024)
qkv_norm_store_kernel(void* q, int64_t q_stride, const void* k, int64_t k_stride, const void* v, int64_t v_stride,
                      void* kpool, int64_t kp_stride, void* vpool, int64_t vp_stride, const int64_t* positions,
                      const int64_t* loc, const float* freq, float mag, const float* qb, const float* kb, const float* vb,
                      int H, int G, int D, int Dv, int dims, int adjacent, int norm_v, float eps, int qk_norm,
                      const float* q_norm_w, const float* k_norm_w, const float* q_head_scale, float q_temp_coef, int q_temp_every, const void* v_first,
                      int64_t vf_stride, const float* v_mix) {
  typedef Elem<Tag> E;
  const int64_t t = blockIdx.x;
  const int64_t ipos = positions[t];
  const float pos = (float)ipos;
  const int64_t slot = loc[t];
  __shared__ float cosine[32 * kStorePerLane], sine[32 * kStorePerLane];      // dims <= D <= 64 * kStorePerLane
  for (int i = threadIdx.x; i < dims / 2; i += blockDim.x) {
    const float ang = pos * freq[i];
    cosine[i] = cosf(ang) * mag;
    sine[i] = sinf(ang) * mag;
  }
  __syncthreads();
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, waves = blockDim.x >> 6;
  float qmul = 1.f;
  if (q_temp_every > 0) qmul = 1.f + q_temp_coef * logf((float)((ipos + 1) / q_temp_every) + 1.f);
  for (int job = wave; job < H + (v ? 2 * G : G); job += waves) {
    float val[kStorePerLane], raw[kStorePerLane];
    if (job < H + G) {
      const bool isq = job < H;
      const int h = isq ? job : job - H;
      const void* src = isq ? q : k;
      const int64_t at = t * (isq ? q_stride : k_stride) + (int64_t)h * D;
      if (qk_norm == 2) {
        normed_rotated_head<Tag>(val, raw, src, at, isq ? qb : kb, h * D, D, dims, adjacent, cosine, sine,
                                 isq ? q_norm_w : k_norm_w, eps, lane);
        if (!isq && !v) {
#pragma unroll
          for (int u = 0; u < kStorePerLane; ++u) {
            const int i = lane + 64 * u;
            if (i < D) E::store(vpool, slot * vp_stride + (int64_t)h * D + i, raw[u]);
          }
        }
      } else {
        rotated_head<Tag>(val, src, at, isq ? qb : kb, h * D, D, dims, adjacent, cosine, sine, lane);
        if (!isq && !v) {
#pragma unroll
          for (int u = 0; u < kStorePerLane; ++u) {
            const int i = lane + 64 * u;
            if (i < D) E::store(vpool, slot * vp_stride + (int64_t)h * D + i, E::load(k, at + i) + (kb ? kb[h * D + i] : 0.f));
          }
        }
      }
      float mul = 1.f;
      if (qk_norm == 1) {
        float ss = 0.f;
#pragma unroll
        for (int u = 0; u < kStorePerLane; ++u) ss += val[u] * val[u];       // (coordinates past D are zeros)
        ss = wave_sum(ss);
        mul = 1.f / sqrtf(ss / (float)D + eps);
      }
      if (isq) mul *= qmul * (q_head_scale ? q_head_scale[h] : 1.f);
      void* dst = isq ? q : kpool;
      const int64_t to = isq ? at : slot * kp_stride + (int64_t)h * D;
#pragma unroll
      for (int u = 0; u < kStorePerLane; ++u) {
        const int i = lane + 64 * u;
        if (i < D) E::store(dst, to + i, val[u] * mul);
      }
    } else {
      const int g = job - H - G;
      const int64_t at = t * v_stride + (int64_t)g * Dv, to = slot * vp_stride + (int64_t)g * Dv;
      float ss = 0.f;
#pragma unroll
      for (int u = 0; u < kStorePerLane; ++u) {
        const int i = lane + 64 * u;
        val[u] = i < Dv ? E::load(v, at + i) + (vb ? vb[g * Dv + i] : 0.f) : 0.f;
        ss += val[u] * val[u];
      }
      float mul = 1.f;
      if (norm_v) mul = 1.f / sqrtf(wave_sum(ss) / (float)Dv + eps);
      const float lam = v_first ? v_mix[0] : 0.f;
#pragma unroll
      for (int u = 0; u < kStorePerLane; ++u) {
        const int i = lane + 64 * u;
        if (i < Dv) {
          float x = val[u] * mul;
          if (v_first) x = (1.f - lam) * x + lam * E::load(v_first, slot * vf_stride + (int64_t)g * Dv + i);
          E::store(vpool, to + i, x);
        }
      }
    }
  }
}

// a token that completes a block (position + 1 divisible by P) writes the block's mean key and value at its own slot.
// A workgroup looks at `rows` rows of the step (a lane each) and takes the completing ones in turn; a thread owns V
// neighbouring channels (16 bytes of a row where rows and buffers allow it) and adds the block's rows in order, kPoolAhead of
// them in flight.  One workgroup per row with a scalar channel per thread and a dependent table read per key took 86 us for
// 4096 tokens in blocks of 64 x 1024 channels; this takes 9.  One row per workgroup up to kPoolSingles rows: a decode step's requests
// may all complete a block at once, and 16 blocks in turn took longer than one scalar one (64 requests, blocks of 64 x 1024 channels: 35 us
// scalar, 100 by sixteens, 8 one by one; 1000 rows of a prompt 8.2 by sixteens, 9.5 one by one).
constexpr int kPoolRows = 16, kPoolSingles = 256, kPoolAhead = 16;

// Where 16-byte pieces would leave threads of the workgroup without channels, a thread takes half or a quarter of one and keeps as many
// bytes on their way (AHEAD rows of V channels); the block's rows of the table come in one load, a lane each.  The rows are added in their
// order whatever the piece: a block's bits depend on its rows alone.  4096 tokens in blocks of 64 x 1024 channels: 10.4 us with
// 16-byte pieces and a dependent table read per row, in half pieces 7.7; x 512 channels 7.8, in quarters 5.4.  (Shares of the rows
// side by side, added up at the end, take 6.6 and 4.2, but give other bits.)
template <typename Tag, int V>
__device__ __forceinline__ u32x4 load_piece(const char* row, int at) {
  const char* p = row + (uint32_t)(at * Elem<Tag>::kBytes);
  if constexpr (V * Elem<Tag>::kBytes == 16) return ld16(p);
  else if constexpr (V * Elem<Tag>::kBytes == 8) { const u32x2 h = *(const u32x2*)p; return u32x4{h[0], h[1], 0u, 0u}; }
  else if constexpr (V * Elem<Tag>::kBytes == 4) return u32x4{*(const uint32_t*)p, 0u, 0u, 0u};
  else return u32x4{*(const uint16_t*)p, 0u, 0u, 0u};
}
template <typename Tag, int V, int AHEAD>
__global__ void __launch_bounds__(kBlock)
pool_blocks_kernel(void* kpooled, void* vpooled, const void* kpool, const void* vpool, int64_t kp_stride, int64_t vp_stride,
                   const int32_t* req_to_token, int64_t table_stride, SeqBatch s, int64_t T, int rows, int kw, int vw, int P) {
  typedef Elem<Tag> E;
  const int64_t t0 = (int64_t)blockIdx.x * rows;
  const int lane = threadIdx.x & 63;
  int64_t pos = -1;
  int b = 0;
  if (lane < rows && t0 + lane < T) {
    int64_t start, prefix;
    seq_of_token(s, t0 + lane, b, start, prefix);
    pos = prefix + (t0 + lane - start);
  }
  uint64_t hits = __ballot(pos >= 0 && (pos + 1) % P == 0);          // (the same in every wave of the workgroup)
  const float inv = 1.f / (float)P;
  for (; hits; hits &= hits - 1) {
    const int l = __ffsll((unsigned long long)hits) - 1;
    const int64_t p = __shfl(pos, l, 64);
    const int32_t* table = req_to_token + load_idx(s.req_pool_indices, __shfl(b, l, 64), s.idx64) * table_stride;
    const int64_t first = p - P + 1, dst = table[p];
    // a wave's pieces are of one buffer (the keys' share is filled up to whole waves): the rows' addresses are scalar
    const int keys = (kw / V + 63) / 64 * 64, pieces = keys + (vw / V + 63) / 64 * 64;
    for (int e0 = blockIdx.y * kBlock + (threadIdx.x & ~63); e0 < pieces; e0 += gridDim.y * kBlock) {
      const bool isk = __builtin_amdgcn_readfirstlane(e0) < keys;
      const int64_t stride = isk ? kp_stride : vp_stride;
      const int c = (e0 - (isk ? 0 : keys) + lane) * V;
      const bool live = c < (isk ? kw : vw);
      const int col = live ? c : 0;
      const char* src = (const char*)(isk ? kpool : vpool);
      float acc[8];
#pragma unroll
      for (int x = 0; x < 8; ++x) acc[x] = 0.f;
      for (int j64 = 0; j64 < P; j64 += 64) {
        const int64_t row = table[first + min(j64 + lane, P - 1)] * stride * E::kBytes;
        const int row_lo = (int)row, row_hi = (int)(row >> 32);
        for (int j0 = j64; j0 < min(j64 + 64, P); j0 += AHEAD) {
          const int n = min(AHEAD, P - j0);
          u32x4 raw[AHEAD];
#pragma unroll
          for (int j = 0; j < AHEAD; ++j) {
            const int at = j0 - j64 + j;               // (past the block: its last row again)
            const int64_t off = ((int64_t)__builtin_amdgcn_readlane(row_hi, at) << 32) | (uint32_t)__builtin_amdgcn_readlane(row_lo, at);
            raw[j] = load_piece<Tag, V>(src + off, col);
          }
#pragma unroll
          for (int j = 0; j < AHEAD; ++j)
            if (j < n) {
              float f[8];
              unpack16<Tag>(raw[j], f);
#pragma unroll
              for (int x = 0; x < V; ++x) acc[x] += f[x];
            }
        }
      }
      if (!live) continue;
#pragma unroll
      for (int x = 0; x < V; ++x) acc[x] *= inv;
      char* out = (char*)(isk ? kpooled : vpooled) + (dst * stride + col) * E::kBytes;
      const u32x4 w = pack16<Tag>(acc);
      if constexpr (V * E::kBytes == 16) st16(out, w);
      else if constexpr (V * E::kBytes == 8) *(u32x2*)out = u32x2{w[0], w[1]};
      else if constexpr (V * E::kBytes == 4) *(uint32_t*)out = w[0];
      else *(uint16_t*)out = (uint16_t)w[0];
    }
  }
}

template <typename Tag>
static int launch_pool_blocks(void* kpooled, void* vpooled, const void* kpool, const void* vpool, int64_t kp_stride,
                              int64_t vp_stride, const int32_t* req_to_token, int64_t table_stride, const SeqBatch& s, int64_t T,
                              int kw, int vw, int P, hipStream_t st) {
  constexpr int V = Elem<Tag>::kVec;
  const int rows = T <= kPoolSingles ? 1 : kPoolRows;
  const unsigned groups = (unsigned)((T + rows - 1) / rows);
  const bool vec = kw % V == 0 && vw % V == 0 && kp_stride % V == 0 && vp_stride % V == 0 &&
                   (((uintptr_t)kpooled | (uintptr_t)vpooled | (uintptr_t)kpool | (uintptr_t)vpool) & 15) == 0;
  const auto pieces = [&](int per) { return (kw / per + 63) / 64 * 64 + (vw / per + 63) / 64 * 64; };
#define SP_POOL(VEC, AHEAD)                                                                                                             \
  pool_blocks_kernel<Tag, VEC, AHEAD><<<dim3(groups, (unsigned)((pieces(VEC) + kBlock - 1) / kBlock)), kBlock, 0, st>>>(                \
      kpooled, vpooled, kpool, vpool, kp_stride, vp_stride, req_to_token, table_stride, s, T, rows, kw, vw, P)
  // (rows past the block are loaded for nothing: as many on their way as it has)
  if (vec && P >= 4 * kPoolAhead && pieces(V / 4) <= kBlock) SP_POOL(V / 4, 4 * kPoolAhead);
  else if (vec && P >= 2 * kPoolAhead && pieces(V / 2) <= kBlock) SP_POOL(V / 2, 2 * kPoolAhead);
  else if (vec) SP_POOL(V, kPoolAhead);
  else SP_POOL(1, kPoolAhead);
#undef SP_POOL
  SP_LAUNCH_CHECK();
  return SP_OK;
}

constexpr int kMaxPerLane = 4;       // value width Dv <= 64 * kMaxPerLane
constexpr int kRows = 8;             // value rows a wave has in flight

template <typename Tag, bool VEC>
__device__ __forceinline__ float dot_row(const float* sq, const void* base, int64_t at, int D) {
  typedef Elem<Tag> E;
  float d = 0.f;
  if (VEC) {
    constexpr int V = E::kVec;
#pragma unroll 4
    for (int i = 0; i < D; i += V) {
      float f[V];
      unpack16<Tag>(ld16((const char*)base + (at + i) * E::kBytes), f);
#pragma unroll
      for (int e = 0; e < V; ++e) d += sq[i + e] * f[e];
    }
  } else {
    for (int i = 0; i < D; ++i) d += sq[i] * E::load(base, at + i);
  }
  return d;
}

// One workgroup of NW waves per (token, query head) - 4 for the rows of prompts, 16 for single decoded tokens, where the
// rows are few and each is long.  The query's keys are numbered blocks first, then the window's tokens, in tiles of 64;
// wave w takes tiles w, w + NW, ...: lane = key for the scores, lane = value channel for the
// weighted sum; the waves' partial (maximum, sum, weighted values) meet in LDS.
// The order of every sum depends on the query's position only, never on the batch or on how the prompt was cut.
template <typename Tag, bool VEC, bool SIG>
__global__ void __launch_bounds__(1024)
window_attention_kernel(void* out, int64_t out_stride, const void* q, int64_t q_stride, const void* kpool, const void* vpool,
                        const void* kpooled, const void* vpooled, int64_t kp_stride, int64_t vp_stride,
                        const int32_t* req_to_token, int64_t table_stride, SeqBatch s, int H, int G, int D, int Dv,
                        int64_t size, int P, int64_t lead, float scale, const float* sinks, float softcap,
                        const float* head_bias, const void* gate, int64_t gate_stride) {
  typedef Elem<Tag> E;
  extern __shared__ float smem[];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, NW = blockDim.x >> 6;
  const int64_t t = blockIdx.x;
  const int h = blockIdx.y;
  float* sq = smem;                              // [D] the scaled query
  float* sw = smem + D + wave * 64;              // this wave's 64 weights
  float* sacc = smem + D + 64 * NW;              // [NW][Dv]
  float* sml = sacc + NW * Dv;                   // [NW] maxima, [NW] sums
  int b;
  int64_t start, prefix;
  seq_of_token(s, t, b, start, prefix);
  const int64_t pos = prefix + (t - start);
  const int64_t w0 = (size > 0 && pos - size + 1 > 0) ? pos - size + 1 : 0;      // first token of the window
  int64_t nb = (size > 0 && P > 0) ? w0 / P : 0;                                  // blocks wholly before it
  if (nb > lead) nb = lead;                                                       // (no more of them exist)
  const int64_t total = nb + (pos - w0 + 1);
  const int g = h / (H / G);
  const int32_t* table = req_to_token + load_idx(s.req_pool_indices, b, s.idx64) * table_stride;
  for (int i = threadIdx.x; i < D; i += blockDim.x) sq[i] = E::load(q, t * q_stride + (int64_t)h * D + i) * scale;
  __syncthreads();
  float m = -INFINITY, l = 0.f;
  const float hbias = (SIG && head_bias) ? head_bias[h] : 0.f;
  float acc[kMaxPerLane];
#pragma unroll
  for (int i = 0; i < kMaxPerLane; ++i) acc[i] = 0.f;
  const int64_t vcol = (int64_t)g * Dv;
  for (int64_t k0 = (int64_t)wave * 64; k0 < total; k0 += 64 * NW) {
    const int n = (int)(total - k0 < 64 ? total - k0 : 64);
    float sc = -INFINITY;
    int32_t slot = 0;
    if (lane < n) {
      const int64_t kk = k0 + lane;
      const bool blk = kk < nb;
      slot = blk ? table[kk * P + P - 1] : table[w0 + (kk - nb)];
      sc = dot_row<Tag, VEC>(sq, blk ? kpooled : kpool, (int64_t)slot * kp_stride + (int64_t)g * D, D);
      if (softcap > 0.f) sc = softcap * tanhf(sc / softcap);
    }
    if constexpr (SIG) {                                // every visible key on its own: no maximum, no denominator
      sw[lane] = lane < n ? over_one_plus_exp(1.f, sc + hbias) : 0.f;
      __builtin_amdgcn_wave_barrier();
    } else {
      float tm = sc;
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) tm = fmaxf(tm, __shfl_xor(tm, off, 64));
      const float m_new = fmaxf(m, tm);
      const float corr = expf(m - m_new);                 // first tile: exp(-inf) = 0
      const float p = lane < n ? expf(sc - m_new) : 0.f;
      l = l * corr + wave_sum(p);
      m = m_new;
      sw[lane] = p;
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int i = 0; i < kMaxPerLane; ++i) acc[i] *= corr;
    }
    // eight keys' rows in flight; the rows are what the lanes looked up for the scores.  Behind the last key its row comes again
    // with a weight of zero
    for (int j = 0; j < n; j += kRows) {
      int64_t at[kRows];
      const void* src[kRows];
      float wt[kRows];
#pragma unroll
      for (int u = 0; u < kRows; ++u) {
        const int ju = j + u < n ? j + u : n - 1;
        at[u] = (int64_t)__builtin_amdgcn_readlane(slot, ju) * vp_stride + vcol;
        src[u] = k0 + ju < nb ? vpooled : vpool;
        wt[u] = j + u < n ? sw[j + u] : 0.f;
      }
#pragma unroll
      for (int i = 0; i < kMaxPerLane; ++i) {
        const int c = lane + 64 * i;
        if (c < Dv) {
          float v[kRows];
#pragma unroll
          for (int u = 0; u < kRows; ++u) v[u] = E::load(src[u], at[u] + c);
#pragma unroll
          for (int u = 0; u < kRows; ++u) acc[i] += wt[u] * v[u];
        }
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
#pragma unroll
  for (int i = 0; i < kMaxPerLane; ++i) {
    const int c = lane + 64 * i;
    if (c < Dv) sacc[wave * Dv + c] = acc[i];
  }
  if (lane == 0) {
    sml[wave] = m;
    sml[NW + wave] = l;
  }
  __syncthreads();
  if constexpr (SIG) {
    for (int c = threadIdx.x; c < Dv; c += blockDim.x) {
      float num = 0.f;
      for (int w = 0; w < NW; ++w) num += sacc[w * Dv + c];
      if (gate) num = over_one_plus_exp(num, E::load(gate, t * gate_stride + (int64_t)h * Dv + c));
      E::store(out, t * out_stride + (int64_t)h * Dv + c, num);
    }
    return;
  }
  float M = sml[0];                                                         // wave 0 always holds a key: M is finite
  for (int w = 1; w < NW; ++w) M = fmaxf(M, sml[w]);
  float den = 0.f;
  if (sinks) {                                                              // one more term of the denominator
    M = fmaxf(M, sinks[h]);
    den = expf(sinks[h] - M);
  }
  for (int w = 0; w < NW; ++w) den += sml[NW + w] * expf(sml[w] - M);       // a wave without keys: exp(-inf) = 0
  const float inv = 1.f / den;
  for (int c = threadIdx.x; c < Dv; c += blockDim.x) {
    float num = 0.f;
    for (int w = 0; w < NW; ++w) num += sacc[w * Dv + c] * expf(sml[w] - M);
    num *= inv;
    if (gate) num = over_one_plus_exp(num, E::load(gate, t * gate_stride + (int64_t)h * Dv + c));
    E::store(out, t * out_stride + (int64_t)h * Dv + c, num);
  }
}


// ---- the same attention on the matrix cores, for portions of prompts in 16-bit types ------------------------------------
// One workgroup per (16 consecutive tokens of one request's portion, key/value head); wave w works for the group's query
// head w (w + 4, ... in further passes).  Keys of the 16 queries' UNION (blocks up to the last query's, tokens from the
// first query's window start to the last query) go by in tiles of 64; who sees what is a mask per (key, query).
//   S^T = K Q^T   v_mfma_f32_16x16x32: first operand = 16 key rows from LDS (a fragment taken straight from the pool would
//                 touch 16 lines per 16 lanes), second = the query fragment held in registers; a lane receives S^T[key 4q + r][query r16]: four keys of ONE query,
//                 so the softmax of a query is a reduction over r, the tile's four key groups and the lanes q = 0..3.
//   O^T = V^T P^T first operand = V^T by transposing reads of the value rows in LDS, second =
//                 P^T - exactly the registers the lane already holds: the key order inside a step of 32 is (4q .. 4q + 3 of
//                 the first 16 keys, then of the second 16) for both operands, so P needs no exchange between lanes.
// Scores, softmax and O are fp32; P enters the second product as a 16-bit value plus its 16-bit remainder (two products).
// The vector unit bounds it: a tile's 48 products take 768 cycles, its LDS reads 1024 per workgroup, and masks in 64-bit positions,
// the library's exponential and a rescaling of O per tile took 3500 per wave.  So masks are formed only where a tile is not wholly
// visible, in the list's own 32-bit positions; a weight is one fma and one hardware exp2 (a score's product and difference are
// rounded once; a layer's error against 64 bits is the one with the library's exponential, 4.72e-3); O is rescaled when a maximum
// moved; and a query's denominator stays spread over its lanes until the end.  4 requests of 4096 tokens together, 16 heads of 128 on
// 4, window 512 and blocks of 64: 95 -> 62 us.  Keys (two buffers) and values go to LDS by direct loads: held in registers on the way,
// with the next tile's on top, they left two workgroups per CU; three fit now, 62 -> 57.
typedef float f32x4_w __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8_w __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_w __attribute__((ext_vector_type(8)));
template <typename Tag>
__device__ __forceinline__ f32x4_w mfma_w(const u32x4& a, const u32x4& b, const f32x4_w& c);
template <>
__device__ __forceinline__ f32x4_w mfma_w<bf16_tag>(const u32x4& a, const u32x4& b, const f32x4_w& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_w, a), __builtin_bit_cast(bf16x8_w, b), c, 0, 0, 0);
}
template <>
__device__ __forceinline__ f32x4_w mfma_w<f16_tag>(const u32x4& a, const u32x4& b, const f32x4_w& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_w, a), __builtin_bit_cast(f16x8_w, b), c, 0, 0, 0);
}

typedef short s16x4_w __attribute__((ext_vector_type(4)));

// by what a row's 16-byte chunks are turned in LDS: rows of 256 bytes begin in one bank, of 128 bytes in two, and a transposing
// read takes pairs of chunks from four rows
template <int RB>
__device__ __forceinline__ int row_turn(int row) {
  return RB == 256 ? 2 * (row & 7) : 2 * ((row >> 1) & 3);
}

template <typename Tag, int DS, int DT, bool SIG>      // DS = dim / 32, DT = vdim / 16
__global__ void __launch_bounds__(256, 3)
window_attention_mfma_kernel(void* out, int64_t out_stride, const void* q, int64_t q_stride, const void* kpool,
                             const void* vpool, const void* kpooled, const void* vpooled, int64_t kp_stride, int64_t vp_stride,
                             const int32_t* req_to_token, int64_t table_stride, SeqBatch s, int H, int G, int64_t size, int P,
                             int64_t lead, float scale, const float* sinks, float softcap, const float* head_bias, const void* gate,
                             int64_t gate_stride) {
  constexpr int D = 32 * DS, Dv = 16 * DT;
  constexpr int KB = 2 * D, VB = 2 * Dv;                 // bytes of an LDS row
  constexpr int KL = KB / 64, VL = VB / 64;              // direct loads of 1 KB per wave for a tile of 64 keys
  extern __shared__ __attribute__((aligned(16))) char wlds[];      // two tiles of keys, one of values
  char *keys = wlds, *keys_next = wlds + 64 * KB, *const sval = wlds + 128 * KB;
  __shared__ int32_t sslot[2][64];                       // pool rows of a tile's keys
  // which request and which of its 16-row tiles
  int tile = blockIdx.x, b = 0;
  for (; b < s.B; ++b) {
    const int tiles = (s.extend_seq_lens[b] + 15) / 16;
    if (tile < tiles) break;
    tile -= tiles;
  }
  if (b >= s.B) return;
  const int g = blockIdx.y, R = H / G;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, r16 = lane & 15, qd = lane >> 4;
  const int64_t start = s.extend_start_loc[b], len = s.extend_seq_lens[b], prefix = s.extend_prefix_lens[b];
  const int rows = (int)(len - 16 * tile < 16 ? len - 16 * tile : 16);
  const int64_t t0 = start + 16 * tile, pos0 = prefix + 16 * tile, pos_last = pos0 + rows - 1;
  const int32_t* table = req_to_token + load_idx(s.req_pool_indices, b, s.idx64) * table_stride;
  const bool pooled = size > 0 && P > 0;
  const int64_t w0U = (size > 0 && pos0 - size + 1 > 0) ? pos0 - size + 1 : 0;
  const int64_t w0L = (size > 0 && pos_last - size + 1 > 0) ? pos_last - size + 1 : 0;
  int64_t nbU = pooled ? w0L / P : 0;
  if (nbU > lead) nbU = lead;
  const int64_t totalU = nbU + (pos_last - w0U + 1);
  // this lane's query (column r16 of every S^T tile) sees the entries [0, blocks) and [first, last] of that list
  const bool qvalid = r16 < rows;
  const int64_t pos_q = pos0 + r16;
  const int64_t w0_q = (size > 0 && pos_q - size + 1 > 0) ? pos_q - size + 1 : 0;
  int64_t nb_q = pooled ? w0_q / P : 0;
  if (nb_q > lead) nb_q = lead;
  const int blocks = qvalid ? (int)nb_q : 0, last = qvalid ? (int)(nbU + (pos_q - w0U)) : -1;
  const int first = qvalid ? (int)(nbU + (w0_q - w0U)) : 0;
  // [open0, open1]: entries that every query of the tile sees (the last one's window begins, the first one's position ends it)
  const int open0 = (int)(nbU + (w0L - w0U)), open1 = (int)(nbU + (pos0 - w0U));
  // scores in units that make a weight one exp2: the product itself times `unit`, or what the cap makes of it
  const bool plain = softcap <= 0.f && scale > 0.f;
  const float unit = (plain ? scale : 1.f) * 1.4426950408889634f;
  for (int h0 = 0; h0 < R; h0 += 4) {
    const int hq = g * R + h0 + wave;
    const bool work = h0 + wave < R;
    const float hbias = (SIG && head_bias && work) ? head_bias[hq] : 0.f;
    u32x4 qf[DS];
#pragma unroll
    for (int st = 0; st < DS; ++st)
      qf[st] = (work && qvalid) ? ld16((const char*)q + ((t0 + r16) * q_stride + (int64_t)hq * D + 32 * st + 8 * qd) * 2)
                                : u32x4{0u, 0u, 0u, 0u};
    f32x4_w oacc[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) oacc[dt] = f32x4_w{0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.f;
    // keys behind the last one repeat it, unseen by every query
    auto entry = [&](int64_t k0, int key) { return k0 + key < totalU ? k0 + key : totalU - 1; };
    auto slot_of = [&](int64_t k0) {                     // (threads 0 .. 63 use it)
      const int64_t kk = entry(k0, threadIdx.x & 63);
      return kk < nbU ? table[kk * P + P - 1] : table[w0U + (kk - nbU)];
    };
    // a tile's rows straight into LDS, 1 KB per wave and load; a row's 16-byte chunks lie permuted by its number (the source address
    // is: a direct load writes lane after lane), so that neither operand's reads meet a bank twice
    // (its pool rows come out of LDS before any load is under way: a read of LDS behind one would wait for it)
    auto rows_of = [&](auto row_bytes, int par, int32_t* slots) {
      constexpr int RB = decltype(row_bytes)::value, CH = RB / 16, ROWS = 64 / CH;
#pragma unroll
      for (int u = 0; u < RB / 64; ++u) slots[u] = sslot[par][(wave * (RB / 64) + u) * ROWS + lane / CH];
    };
    auto fetch = [&](char* lds, const void* pool, const void* pooled_rows, int64_t stride, auto row_bytes, int64_t k0,
                     const int32_t* slots) {
      constexpr int RB = decltype(row_bytes)::value, CH = RB / 16, ROWS = 64 / CH;
#pragma unroll
      for (int u = 0; u < RB / 64; ++u) {
        const int piece = wave * (RB / 64) + u, key = piece * ROWS + lane / CH;
        const char* src = (const char*)(entry(k0, key) < nbU ? pooled_rows : pool) +
                          ((int64_t)slots[u] * stride + (int64_t)g * (RB / 2)) * 2 + ((lane % CH) ^ row_turn<RB>(key)) * 16;
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                         (__attribute__((address_space(3))) void*)(lds + piece * 1024), 16, 0, 0);
      }
    };
    const std::integral_constant<int, KB> key_bytes;
    const std::integral_constant<int, VB> value_bytes;
    lds_barrier();                                       // (a further pass of heads: the last tile's readers are done)
    if (threadIdx.x < 64) {
      sslot[0][threadIdx.x] = slot_of(0);
      sslot[1][threadIdx.x] = slot_of(64);
    }
    lds_barrier();
    int32_t kslots[KL], vslots[VL];
    rows_of(key_bytes, 0, kslots);
#pragma unroll
    for (int st = 0; st < DS; ++st) asm volatile("" : "+v"(qf[st]));      // (the queries are here: no wait for them in the loop)
    fetch(keys, kpool, kpooled, kp_stride, key_bytes, 0, kslots);
    for (int64_t k0 = 0; k0 < totalU; k0 += 64) {
      const int par = (int)(k0 >> 6) & 1;
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      lds_barrier();                                     // the tile's keys have landed; everyone is done with the values before
      rows_of(value_bytes, par, vslots);
      rows_of(key_bytes, par ^ 1, kslots);
      fetch(sval, vpool, vpooled, vp_stride, value_bytes, k0, vslots);
      __builtin_amdgcn_sched_barrier(0);                 // in this order: the wait below counts
      const bool more = k0 + 64 < totalU;
      if (more) fetch(keys_next, kpool, kpooled, kp_stride, key_bytes, k0 + 64, kslots);
      __builtin_amdgcn_sched_barrier(0);
      const int32_t slot = slot_of(k0 + 128);
      u32x4 pb[2], pr[2];
      if (work) {
        f32x4_w sacc[4];
#pragma unroll
        for (int sb = 0; sb < 4; ++sb) {
          sacc[sb] = f32x4_w{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int st = 0; st < DS; ++st)
            sacc[sb] = mfma_w<Tag>(ld16(keys + (16 * sb + r16) * KB + ((4 * st + qd) ^ row_turn<KB>(r16)) * 16), qf[st], sacc[sb]);
        }
        if (!plain) {
#pragma unroll
          for (int sb = 0; sb < 4; ++sb) {
            if (k0 + 16 * sb >= totalU) continue;         // (nobody sees these; 16 tanh a lane are 0.5 us of a short prompt's 8)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const float v = sacc[sb][r] * scale;
              sacc[sb][r] = softcap > 0.f ? softcap * tanhf(v / softcap) : v;
            }
          }
        }
        if (k0 < open0 || k0 + 63 > open1) {              // (most tiles of a long window lie inside)
          const int e0 = (int)k0 + 4 * qd;
#pragma unroll
          for (int sb = 0; sb < 4; ++sb)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const int kk = e0 + 16 * sb + r;
              sacc[sb][r] = kk < blocks || (kk >= first && kk <= last) ? sacc[sb][r] : -INFINITY;
            }
        }
        float pf[2][8];
        if constexpr (SIG) {                              // sigmoid(score + bias) per visible key, nothing to rescale
#pragma unroll
          for (int sb = 0; sb < 4; ++sb)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const float v = plain ? sacc[sb][r] * scale : sacc[sb][r];
              pf[sb >> 1][4 * (sb & 1) + r] = v == -INFINITY ? 0.f : over_one_plus_exp(1.f, v + hbias);
            }
        } else {
          float mx = fmaxf(fmaxf(sacc[0][0], sacc[0][1]), fmaxf(sacc[0][2], sacc[0][3]));
#pragma unroll
          for (int sb = 1; sb < 4; ++sb) mx = fmaxf(fmaxf(mx, fmaxf(sacc[sb][0], sacc[sb][1])), fmaxf(sacc[sb][2], sacc[sb][3]));
          const auto half = __builtin_amdgcn_permlane16_swap(as_u32(mx), as_u32(mx), false, false);
          mx = fmaxf(as_f32(half[0]), as_f32(half[1]));
          const auto whole = __builtin_amdgcn_permlane32_swap(as_u32(mx), as_u32(mx), false, false);
          mx = fmaxf(as_f32(whole[0]), as_f32(whole[1]));
          const float m_new = fmaxf(m, mx * unit);
          const float m_safe = m_new == -INFINITY ? 0.f : m_new;      // nothing seen yet: every weight is exp2(-inf) = 0
          if (__ballot(m_new != m)) {                     // (rare after the first tiles)
            const float corr = __builtin_amdgcn_exp2f(m - m_safe);
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
#pragma unroll
              for (int r = 0; r < 4; ++r) oacc[dt][r] *= corr;
            l *= corr;
            m = m_new;
          }
#pragma unroll
          for (int sb = 0; sb < 4; ++sb)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const float p = __builtin_amdgcn_exp2f(fmaf(sacc[sb][r], unit, -m_safe));
              l += p;                                     // this lane's keys; the lanes of a query are added up at the end
              pf[sb >> 1][4 * (sb & 1) + r] = p;
            }
        }
        // the weights enter the product as a 16-bit value plus a 16-bit remainder: they are never rounded to 8 bits of
        // mantissa (the second product costs an eighth of the step's matrix work again)
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) {
          pb[hh] = pack16<Tag>(pf[hh]);
          float rest[8], back[8];
          unpack16<Tag>(pb[hh], back);
#pragma unroll
          for (int e = 0; e < 8; ++e) rest[e] = pf[hh][e] - back[e];
          pr[hh] = pack16<Tag>(rest);
        }
      }
      // the values were asked for before the next tile's keys: at most those (KL of them per wave) may still be under way
      if (more) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(KL) : "memory");
      else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      lds_barrier();
      if (work) {
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) {
          // lane i of a 16-lane group addresses row 4 qd + (i >> 2), elements 4 (i & 3) .. + 3, and receives column i
          const int row = 32 * hh + 4 * qd + (r16 >> 2), turn = row_turn<VB>(row);      // (16 rows on: the same turn)
          const char* vr = sval + row * VB + 8 * (r16 & 1);
#pragma unroll
          for (int dt = 0; dt < DT; ++dt) {
            const char* vp = vr + ((2 * dt + ((r16 & 3) >> 1)) ^ turn) * 16;
            const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                                           (__attribute__((address_space(3))) s16x4_w*)vp));
            const u32x2 hi = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                                           (__attribute__((address_space(3))) s16x4_w*)(vp + 16 * VB)));
            const u32x4 a = {lo[0], lo[1], hi[0], hi[1]};
            oacc[dt] = mfma_w<Tag>(a, pb[hh], oacc[dt]);
            oacc[dt] = mfma_w<Tag>(a, pr[hh], oacc[dt]);
          }
        }
      }
      if (threadIdx.x < 64) sslot[par][threadIdx.x] = slot;      // (waits for all loads: at the tile's end)
      char* const t = keys;
      keys = keys_next, keys_next = t;
    }
    if constexpr (!SIG) {                              // (outside the branch: every lane of a wave takes part)
      l += __shfl_xor(l, 16, 64);
      l += __shfl_xor(l, 32, 64);
    }
    if (work && qvalid) {
      float inv = 1.f;
      if constexpr (!SIG) {
        inv = 1.f / l;
        if (sinks) {                                   // (a valid query has seen itself: m is finite)
          const float sk = sinks[hq] * 1.4426950408889634f, m2 = fmaxf(m, sk), keep = __builtin_amdgcn_exp2f(m - m2);
          inv = keep / (l * keep + __builtin_amdgcn_exp2f(sk - m2));
        }
      }
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        float f[8] = {oacc[dt][0] * inv, oacc[dt][1] * inv, oacc[dt][2] * inv, oacc[dt][3] * inv, 0.f, 0.f, 0.f, 0.f};
        if (gate) {
          float gf[8];
          const u32x2 g2 = *(const u32x2*)((const char*)gate + ((t0 + r16) * gate_stride + (int64_t)hq * Dv + 16 * dt + 4 * qd) * 2);
          unpack16<Tag>(u32x4{g2[0], g2[1], 0u, 0u}, gf);
#pragma unroll
          for (int e = 0; e < 4; ++e) f[e] = over_one_plus_exp(f[e], gf[e]);
        }
        const u32x4 pk = pack16<Tag>(f);
        *(u32x2*)((char*)out + ((t0 + r16) * out_stride + (int64_t)hq * Dv + 16 * dt + 4 * qd) * 2) = u32x2{pk[0], pk[1]};
      }
    }
  }
}

}  // namespace
}  // namespace sp

using namespace sp;

extern "C" int sp_qkv_rotary_store(void* q, int64_t q_stride, const void* k, int64_t k_stride, const void* v,
                                   int64_t v_stride, void* kpool, int64_t kp_stride, void* vpool, int64_t vp_stride,
                                   const int64_t* positions, const int64_t* loc, const float* freq, float mag,
                                   const float* q_bias, const float* k_bias, const float* v_bias, int64_t num_tokens,
                                   int heads, int kv_heads, int dim, int vdim, int rot_dims, int adjacent, int norm_values,
                                   float eps, int qk_norm, const float* q_norm_weight, const float* k_norm_weight,
                                   const float* q_head_scale, float q_temp_coef, int q_temp_every, const void* v_first,
                                   int64_t vf_stride, const float* v_mix, int dtype, void* stream) {
  SP_CHECK_ARG(num_tokens >= 0 && heads > 0 && kv_heads > 0 && dim > 0 && vdim > 0);
  SP_CHECK_ARG(rot_dims >= 0 && rot_dims % 2 == 0 && rot_dims <= dim);
  SP_CHECK_ARG(qk_norm >= 0 && qk_norm <= 2 && (qk_norm == 2 || (!q_norm_weight && !k_norm_weight)));
  if (num_tokens == 0) return SP_OK;
  SP_CHECK_ARG(q && k && kpool && vpool && positions && loc && (freq || rot_dims == 0));
  SP_CHECK_ARG(q_stride >= (int64_t)heads * dim && k_stride >= (int64_t)kv_heads * dim);
  SP_CHECK_ARG(v ? v_stride >= (int64_t)kv_heads * vdim : (dim == vdim && !v_bias && !norm_values && !v_first));
  SP_CHECK_ARG(kp_stride >= (int64_t)kv_heads * dim && vp_stride >= (int64_t)kv_heads * vdim);
  SP_CHECK_ARG(q_temp_every >= 0 && (!v_first || (v_mix && vf_stride >= (int64_t)kv_heads * vdim)));
  if (qk_norm || q_head_scale || q_temp_every > 0 || v_first || !v) {      // the wave-per-head form
    if (dim > 64 * kStorePerLane || vdim > 64 * kStorePerLane) return SP_ERR_UNSUPPORTED;
    // four waves take a prompt token's heads in turn; the few tokens of a decode step get a wave per head (16 at most)
    const int jobs = heads + (v ? 2 : 1) * kv_heads;
    const int threads = num_tokens > 256 ? kBlock : 64 * (jobs < 4 ? 4 : (jobs > 16 ? 16 : jobs));
    SP_DISPATCH_DTYPE(dtype, (qkv_norm_store_kernel<Tag><<<dim3((unsigned)num_tokens), threads, 0, (hipStream_t)stream>>>(
                                 q, q_stride, k, k_stride, v, v_stride, kpool, kp_stride, vpool, vp_stride, positions, loc,
                                 freq, mag, q_bias, k_bias, v_bias, heads, kv_heads, dim, vdim, rot_dims, adjacent,
                                 norm_values, eps, qk_norm, q_norm_weight, k_norm_weight, q_head_scale, q_temp_coef,
                                 q_temp_every, v_first, vf_stride, v_mix)));
    SP_LAUNCH_CHECK();
    return SP_OK;
  }
  // (the line of 64 tokens is not a crossing: at 1 - 64 tokens of 16 + 4 heads of 128 the wave takes 3.4 - 4.1 us, the workgroup 4.0 - 4.3)
  const int per = dtype == SP_F32 ? 4 : 8, half = rot_dims / 2;
  if (num_tokens > 64 && !adjacent && !q_bias && !k_bias && !v_bias && norm_values && v && half <= 64 && half % per == 0 && dim % per == 0 &&
      (vdim == 8 * per || vdim == 16 * per) && q_stride % per == 0 && k_stride % per == 0 && v_stride % per == 0 && kp_stride % per == 0 &&
      vp_stride % per == 0 && (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)kpool | (uintptr_t)vpool) & 15) == 0) {
    const dim3 grid((unsigned)((num_tokens + kBlock / 64 - 1) / (kBlock / 64)));
#define SP_STORE(VL)                                                                                                               \
  SP_DISPATCH_DTYPE(dtype, (qkv_rotary_wave_kernel<Tag, VL><<<grid, kBlock, 0, (hipStream_t)stream>>>(                             \
                               (char*)q, q_stride, (const char*)k, k_stride, (const char*)v, v_stride, (char*)kpool, kp_stride,    \
                               (char*)vpool, vp_stride, positions, loc, freq, mag, num_tokens, heads, kv_heads, dim, rot_dims, eps)))
    if (vdim == 8 * per) SP_STORE(8);
    else SP_STORE(16);
#undef SP_STORE
    SP_LAUNCH_CHECK();
    return SP_OK;
  }
  SP_DISPATCH_DTYPE(dtype, (qkv_rotary_store_kernel<Tag><<<dim3((unsigned)num_tokens), kBlock, 0, (hipStream_t)stream>>>(
                               q, q_stride, k, k_stride, v, v_stride, kpool, kp_stride, vpool, vp_stride, positions, loc,
                               freq, mag, q_bias, k_bias, v_bias, heads, kv_heads, dim, vdim, rot_dims, adjacent, norm_values,
                               eps)));
  SP_LAUNCH_CHECK();
  return SP_OK;
}

extern "C" int sp_pool_blocks(void* kpooled, void* vpooled, const void* kpool, const void* vpool, int64_t kp_stride,
                              int64_t vp_stride, const int32_t* req_to_token, int64_t table_stride, int64_t num_tokens,
                              int key_width, int value_width, int block, SP_SEQ_PARAMS, int dtype, void* stream) {
  SP_CHECK_ARG(num_tokens >= 0 && key_width > 0 && value_width > 0 && block > 0);
  if (num_tokens == 0) return SP_OK;
  SP_CHECK_ARG(kpooled && vpooled && kpool && vpool && req_to_token && req_pool_indices && seq_lens);
  SP_CHECK_ARG(kp_stride >= key_width && vp_stride >= value_width);
  SP_CHECK_ARG(!extend_seq_lens || (extend_prefix_lens && extend_start_loc && token_req));
  SP_CHECK_ARG(extend_seq_lens || num_tokens == batch_size);
  SEQ_BATCH(s);
  SP_DISPATCH_DTYPE(dtype, return (launch_pool_blocks<Tag>(kpooled, vpooled, kpool, vpool, kp_stride, vp_stride, req_to_token,
                                                           table_stride, s, num_tokens, key_width, value_width, block,
                                                           (hipStream_t)stream)));
}

extern "C" int sp_window_attention(void* out, int64_t out_stride, const void* q, int64_t q_stride, const void* kpool,
                                   const void* vpool, const void* kpooled, const void* vpooled, int64_t kp_stride,
                                   int64_t vp_stride, const int32_t* req_to_token, int64_t table_stride,
                                   int64_t num_tokens, int heads, int kv_heads, int dim, int vdim, int64_t window, int block,
                                   int keep_first, float scale, const float* sinks, float softcap, int sigmoid_weights,
                                   const float* head_bias, const void* gate, int64_t gate_stride, int matrix, SP_SEQ_PARAMS,
                                   int dtype, void* stream) {
  SP_CHECK_ARG(num_tokens >= 0 && heads > 0 && kv_heads > 0 && heads % kv_heads == 0 && dim > 0 && vdim > 0);
  if (num_tokens == 0) return SP_OK;
  SP_CHECK_ARG(out && q && kpool && vpool && req_to_token && req_pool_indices && seq_lens);
  SP_CHECK_ARG((kpooled && vpooled) || block <= 0 || window <= 0);
  SP_CHECK_ARG(keep_first >= 0 && (keep_first == 0 || block <= 0));
  int64_t lead = INT64_MAX;                      // how many blocks exist at most
  if (keep_first > 0) {                          // the kept tokens: blocks of one token, read from the token rows
    block = 1;
    lead = keep_first;
    kpooled = kpool;
    vpooled = vpool;
  }
  SP_CHECK_ARG(!extend_seq_lens || (extend_prefix_lens && extend_start_loc && token_req));
  SP_CHECK_ARG(extend_seq_lens || num_tokens == batch_size);
  SP_CHECK_ARG(q_stride >= (int64_t)heads * dim && out_stride >= (int64_t)heads * vdim);
  SP_CHECK_ARG(kp_stride >= (int64_t)kv_heads * dim && vp_stride >= (int64_t)kv_heads * vdim);
  SP_CHECK_ARG(!gate || gate_stride >= (int64_t)heads * vdim);
  SP_CHECK_ARG(!sigmoid_weights || !sinks);
  if (vdim > 64 * kMaxPerLane) return SP_ERR_UNSUPPORTED;
  const int nw = extend_seq_lens ? 4 : 16;       // waves per (token, head): see the kernel
  const size_t lds = ((size_t)dim + 64 * nw + (size_t)nw * vdim + 2 * nw) * sizeof(float);
  if (lds > 64 * 1024) return SP_ERR_UNSUPPORTED;
  SEQ_BATCH(s);
  // portions of prompts in 16-bit types: the matrix-core kernel where its tile shapes and 16-byte row loads apply
  const bool al16 = (((uintptr_t)q | (uintptr_t)kpool | (uintptr_t)vpool | (uintptr_t)kpooled | (uintptr_t)vpooled) & 15) == 0 &&
                    ((uintptr_t)out & 7) == 0;
  if (matrix && extend_seq_lens && num_tokens > batch_size && (dtype == SP_BF16 || dtype == SP_F16) && (dim == 64 || dim == 128) &&
      (vdim == 64 || vdim == 128) && al16 && q_stride % 8 == 0 && kp_stride % 8 == 0 && vp_stride % 8 == 0 && out_stride % 4 == 0 &&
      (!gate || (((uintptr_t)gate & 7) == 0 && gate_stride % 4 == 0))) {
    const dim3 mgrid((unsigned)((num_tokens + 15) / 16 + batch_size), (unsigned)kv_heads);
#define SP_WM2(T, DS, DT, SG)                                                                                            \
  window_attention_mfma_kernel<T, DS, DT, SG><<<mgrid, 256, 64 * 2 * (2 * 32 * DS + 16 * DT), (hipStream_t)stream>>>(                                     \
      out, out_stride, q, q_stride, kpool, vpool, kpooled, vpooled, kp_stride, vp_stride, req_to_token, table_stride, s, heads, \
      kv_heads, window, block, lead, scale, sinks, softcap, head_bias, gate, gate_stride)
#define SP_WM(T, DS, DT)                    \
  do {                                      \
    if (sigmoid_weights) SP_WM2(T, DS, DT, true); \
    else SP_WM2(T, DS, DT, false);          \
  } while (0)
#define SP_WM_SHAPES(T)                                   \
  do {                                                    \
    if (dim == 64 && vdim == 64) SP_WM(T, 2, 4);          \
    else if (dim == 64) SP_WM(T, 2, 8);                   \
    else if (vdim == 64) SP_WM(T, 4, 4);                  \
    else SP_WM(T, 4, 8);                                  \
  } while (0)
    if (dtype == SP_BF16) SP_WM_SHAPES(bf16_tag);
    else SP_WM_SHAPES(f16_tag);
#undef SP_WM_SHAPES
#undef SP_WM
#undef SP_WM2
    SP_LAUNCH_CHECK();
    return SP_OK;
  }
  const dim3 grid((unsigned)num_tokens, (unsigned)heads);
  const int vecn = dtype == SP_F32 ? 4 : 8;
  const bool vec = dim % vecn == 0 && kp_stride % vecn == 0 && ((uintptr_t)kpool & 15) == 0 &&
                   (!kpooled || ((uintptr_t)kpooled & 15) == 0);
#define SP_WA(V, SG)                                                                                                   \
  SP_DISPATCH_DTYPE(dtype, (window_attention_kernel<Tag, V, SG><<<grid, 64 * nw, lds, (hipStream_t)stream>>>(           \
                               out, out_stride, q, q_stride, kpool, vpool, kpooled, vpooled, kp_stride, vp_stride,      \
                               req_to_token, table_stride, s, heads, kv_heads, dim, vdim, window, block, lead, scale, sinks, \
                               softcap, head_bias, gate, gate_stride)))
  if (vec && sigmoid_weights) SP_WA(true, true);
  else if (vec) SP_WA(true, false);
  else if (sigmoid_weights) SP_WA(false, true);
  else SP_WA(false, false);
#undef SP_WA
  SP_LAUNCH_CHECK();
  return SP_OK;
}
