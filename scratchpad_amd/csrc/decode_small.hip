// One launch for the attention of a small decode step: rotation of q and k, the new rows' way into the pool, and the attention itself.
//
// Call site: LlamaAttention.forward's decode branch (nn/models/llama/llama.py:139-154: rotary_emb, then RadixAttention, whose backend
// stores k and v and runs split decode attention and its merge, nn/attention/triton_backend.py:157-196).
//
// What bounds it: nothing but latency.  A step of one request of 300 keys moves 0.6 MB per layer, and rotation, range attention and merge took 13 us
// of it: three launches, each a chain of dependent loads (positions -> table; plan -> request -> slots -> keys; plan -> sums).  Here the chain is
// lengths and rows, then slots and the rotation's table, then keys and values, whose loads are all on their way together (64 keys a wave at heads
// of 64, 32 at 128) while q is rotated; the sums of the eight waves meet in LDS.  A workgroup has a request's keys of one kv head to itself, so nothing
// is left to merge - and long requests are slower than where many share them (SMALL_MAX_ROWS' line in attention.py has both sides).
// us under graph replay, rotation + attention + merge -> this, bf16, 32 query and 8 kv heads: heads of 64, 1 request of 64 / 300 / 600 keys 8.7 ->
// 4.6, 10.2 -> 6.2, 10.4 -> 9.0; heads of 128, 1 of 300 12.2 -> 8.3; byte pools 12.8 -> 9.2 and 14.5 -> 12.0.  A decode step of 1
// row (16 layers, hidden 2048): 843 -> 763.
#include "sp_common.h"

#include <type_traits>

namespace sp {
namespace {

typedef float f32x4_s __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8_s __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_s __attribute__((ext_vector_type(8)));
typedef short s16x4_s __attribute__((ext_vector_type(4)));
typedef _Float16 f16x4_s __attribute__((ext_vector_type(4)));

constexpr float kLog2eS = 1.4426950408889634f, kNegBigS = -1.0e30f;
constexpr int kSmallWaves = 8;
template <int D>
constexpr int kSmallTiles = D == 64 ? 4 : 2;                         // of 16 keys, on their way per wave (four of them spill at 128)

struct SmallArgs {
  char* out;
  const char *q, *k, *v;              // the projection's rows, not rotated
  const char* cache;                  // [position][cos half | sin half]
  const int64_t* positions;
  const int64_t* loc;
  char *kbuf, *vbuf;
  const int32_t* r2t;
  const void *req_idx, *seq_lens;
  int64_t r2t_stride, q_stride, k_stride, v_stride, o_stride, kv_stride;      // elements
  int idx64, Hkv, G, max_len;
  float qk_scale, out_scale, k_scale, v_scale;
};

template <typename Tag>
__device__ __forceinline__ f32x4_s dot32(const u32x4& a, const u32x4& b, const f32x4_s& c) {
  if constexpr (std::is_same<Tag, bf16_tag>::value)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_s, a), __builtin_bit_cast(bf16x8_s, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_s, a), __builtin_bit_cast(f16x8_s, b), c, 0, 0, 0);
}
template <typename Tag>
__device__ __forceinline__ f32x4_s dot16(const u32x2& a, const u32x2& b, const f32x4_s& c) {
  if constexpr (std::is_same<Tag, bf16_tag>::value)
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4_s, a), __builtin_bit_cast(s16x4_s, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(f16x4_s, a), __builtin_bit_cast(f16x4_s, b), c, 0, 0, 0);
}
template <typename Tag>
__device__ __forceinline__ uint32_t pack2s(float lo, float hi) {
  if constexpr (std::is_same<Tag, bf16_tag>::value) {
    bf16x2_t b;
    b[0] = (__bf16)lo;
    b[1] = (__bf16)hi;
    return __builtin_bit_cast(uint32_t, b);
  } else {
    f16x2_t b;
    b[0] = (_Float16)lo;
    b[1] = (_Float16)hi;
    return __builtin_bit_cast(uint32_t, b);
  }
}
// over the lanes 16 and 32 apart, every lane of the four ending with the same
__device__ __forceinline__ float max_quarters(float x) {
  const auto h = __builtin_amdgcn_permlane32_swap(as_u32(x), as_u32(x), false, false);
  x = fmaxf(as_f32(h[0]), as_f32(h[1]));
  const auto r = __builtin_amdgcn_permlane16_swap(as_u32(x), as_u32(x), false, false);
  return fmaxf(as_f32(r[0]), as_f32(r[1]));
}
__device__ __forceinline__ float sum_quarters(float x) {
  const auto h = __builtin_amdgcn_permlane32_swap(as_u32(x), as_u32(x), false, false);
  x = as_f32(h[0]) + as_f32(h[1]);
  const auto r = __builtin_amdgcn_permlane16_swap(as_u32(x), as_u32(x), false, false);
  return as_f32(r[0]) + as_f32(r[1]);
}
// 8 neighbouring coordinates of the first half and those of the second, rotated as sp_rotary_embedding does it: every product and sum rounded
template <typename Tag>
__device__ __forceinline__ void rotate8(u32x4& first, u32x4& second, const u32x4& cos, const u32x4& sin) {
  typedef Elem<Tag> E;
  float a[8], b[8], c[8], s[8], u[8], w[8];
  unpack16<Tag>(first, a);
  unpack16<Tag>(second, b);
  unpack16<Tag>(cos, c);
  unpack16<Tag>(sin, s);
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    u[e] = __fsub_rn(E::round(__fmul_rn(a[e], c[e])), E::round(__fmul_rn(b[e], s[e])));
    w[e] = __fadd_rn(E::round(__fmul_rn(b[e], c[e])), E::round(__fmul_rn(a[e], s[e])));
  }
  first = pack16<Tag>(u);
  second = pack16<Tag>(w);
}
// 8 elements as a byte pool holds them: sp_kv_store_fp8's two roundings
template <typename Tag>
__device__ __forceinline__ u32x2 to_bytes(const u32x4& x, float scale) {
  float f[8];
  unpack16<Tag>(x, f);
  u32x2 out = {0u, 0u};
#pragma unroll
  for (int e = 0; e < 8; ++e) out[e >> 2] |= f32_to_e5m2_bits(scale == 1.f ? f[e] : Elem<Tag>::round(f[e] / scale)) << (8 * (e & 3));
  return out;
}

// workgroup = (kv head, request), 8 waves; wave w has the tiles w, w + 8, .. of 16 keys, a few of them on their way at a time
template <typename Tag, int D, bool KV8>
__global__ __launch_bounds__(kSmallWaves * 64, 2) void decode_small_kernel(SmallArgs a) {
  typedef Elem<Tag> E;
  typedef typename std::conditional<KV8, f16_tag, Tag>::type CT;          // of the products
  typedef typename std::conditional<KV8, u32x2, u32x4>::type raw_t;       // 8 elements of the pool
  constexpr int S = D / 32, CPR = D / 8, RPL = 64 / CPR, NV = 16 / RPL, DB = D / 16, EB = KV8 ? 1 : 2, ROW = D * 2;
  constexpr int T = kSmallTiles<D>, kKeys = kSmallWaves * T * 16;         // keys of a pass
  // The weights of a tile of 16 keys are rounded against the tile's own largest, which is 1 then and exact, and its sums join the others' in fp32: with
  // one reference for all tiles of a wave a request of 600 - 1000 keys came out 1.01 - 1.03 times as far from 64 bits as in sp_decode_attention, whose
  // pieces are that short; now 0.96 - 0.98, for 0.3 - 0.8 us.  bf16 queries of a byte pool: their weights are fp16, far below what the output rounds.
  constexpr bool OWN_TOP = std::is_same<CT, Tag>::value;
  __shared__ __attribute__((aligned(16))) char tiles[kSmallWaves][16 * ROW];
  __shared__ float ml[kSmallWaves][8][2];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, col = lane & 15, kq = lane >> 4;
  const int hk = blockIdx.x, b = blockIdx.y, G = a.G;
  const int seq = min((int)load_idx(a.seq_lens, b, a.idx64), a.max_len);
  const int64_t req = load_idx(a.req_idx, b, a.idx64), pos = a.positions[b], fresh = a.loc[b];
  // the rows of this step: q of the head in this lane's column, k and v of the kv head
  u32x4 qf[S], kn[S];
  const char* const qp = a.q + ((int64_t)b * a.q_stride + (int64_t)(hk * G + min(col, G - 1)) * D + 8 * kq) * 2;
  const char* const kp = a.k + ((int64_t)b * a.k_stride + (int64_t)hk * D + 8 * kq) * 2;
#pragma unroll
  for (int s = 0; s < S; ++s) qf[s] = ld16(qp + s * 64);
#pragma unroll
  for (int s = 0; s < S; ++s) kn[s] = ld16(kp + s * 64);
  const u32x4 vn = ld16(a.v + ((int64_t)b * a.v_stride + (int64_t)hk * D + 8 * (lane % CPR)) * 2);
  const int32_t* const row = a.r2t + req * a.r2t_stride;
  // this lane's key of a pass: key col of the wave's tile kq
  const int mine = kq * (kSmallWaves * 16) + wave * 16 + col;
  int idx = kq < T && mine < seq ? row[mine] : -1;
  u32x4 cs[S / 2], sn[S / 2];
  const char* const cp = a.cache + pos * D * 2 + kq * 16;
#pragma unroll
  for (int s = 0; s < S / 2; ++s) cs[s] = ld16(cp + s * 64), sn[s] = ld16(cp + D + s * 64);

  const int64_t tok = a.kv_stride * EB;
  raw_t kr[T][S], vr[T][NV];
  const auto gather_k = [&](int slots) {
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const int slot = __shfl(slots, t * 16 + col);
      const char* const p = a.kbuf + (int64_t)max(slot, 0) * tok + (hk * D + 8 * kq) * EB;
#pragma unroll
      for (int s = 0; s < S; ++s) kr[t][s] = slot >= 0 ? *(const raw_t*)(p + s * 32 * EB) : raw_t{};
    }
  };
  const auto gather_v = [&](int slots) {
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const int R = i * RPL + lane / CPR, slot = __shfl(slots, t * 16 + R);
        const char* const p = a.vbuf + (int64_t)max(slot, 0) * tok + (hk * D + 8 * ((lane % CPR) ^ (R & (CPR - 1)))) * EB;
        vr[t][i] = slot >= 0 ? *(const raw_t*)p : raw_t{};
      }
  };
  gather_k(idx);
  gather_v(idx);
#pragma unroll
  for (int s = 0; s < S / 2; ++s) rotate8<Tag>(qf[s], qf[s + S / 2], cs[s], sn[s]);
  if constexpr (KV8 && std::is_same<Tag, bf16_tag>::value) {
#pragma unroll
    for (int s = 0; s < S; ++s) qf[s] = bf16x8_to_f16x8(qf[s]);
  }
  // the waves that see the new key, and the last one, which puts it into the pool, need it rotated (the pool's row is as old as its slot's last use)
  bool turned = false;
  u32x4 vnew = vn;
  const auto turn = [&]() {
    if (turned) return;
    turned = true;
#pragma unroll
    for (int s = 0; s < S / 2; ++s) rotate8<Tag>(kn[s], kn[s + S / 2], cs[s], sn[s]);
    if constexpr (KV8) {
#pragma unroll
      for (int s = 0; s < S; ++s) kn[s] = expand_e5m2x8(to_bytes<Tag>(kn[s], a.k_scale));
      vnew = expand_e5m2x8(to_bytes<Tag>(vn, a.v_scale));
    }
  };
  const auto put = [&](char* p, const u32x4& x) {
    if constexpr (KV8) {          // the halves' upper bytes
      *(u32x2*)p = u32x2{__builtin_amdgcn_perm(x[1], x[0], 0x07050301u), __builtin_amdgcn_perm(x[3], x[2], 0x07050301u)};
    } else {
      st16(p, x);
    }
  };
  if (wave == kSmallWaves - 1) {
    turn();
    if (col == 0) {
#pragma unroll
      for (int s = 0; s < S; ++s) put(a.kbuf + fresh * tok + (hk * D + 32 * s + 8 * kq) * EB, kn[s]);
    }
    if (lane < CPR) put(a.vbuf + fresh * tok + (hk * D + 8 * lane) * EB, vnew);
  }

  f32x4_s o[DB];
#pragma unroll
  for (int d = 0; d < DB; ++d) o[d] = f32x4_s{0.f, 0.f, 0.f, 0.f};
  float m = kNegBigS, l = 0.f;
  char* const tile = tiles[wave];
  const int tr = 4 * kq + (col >> 2);                                // the row a lane names in a transposed read
  for (int base = wave * 16; base < seq; base += kKeys) {       // (the wave's first key of a pass)
    const int after = base - wave * 16 + kKeys + mine;
    const int next = kq < T && after < seq ? row[after] : -1;
    const uint64_t is_new = __ballot(idx >= 0 && (int64_t)idx == fresh);
    if (is_new) turn();
    f32x4_s x[T];
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const bool own = is_new >> (t * 16 + col) & 1;
      f32x4_s c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < S; ++s) {
        u32x4 kf;
        if constexpr (KV8) kf = expand_e5m2x8(kr[t][s]);
        else kf = kr[t][s];
        if (is_new) {
#pragma unroll
          for (int w = 0; w < 4; ++w) kf[w] = own ? kn[s][w] : kf[w];
        }
        c = dot32<CT>(kf, qf[s], c);
      }
      x[t] = c;
    }
    const bool more = base + kKeys < seq;
    if (more) gather_k(next);
    float top = m, tops[T], part[T];
#pragma unroll
    for (int t = 0; t < T; ++t) {
      tops[t] = kNegBigS;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        x[t][j] = base + t * kSmallWaves * 16 + 4 * kq + j < seq ? x[t][j] * a.qk_scale : -INFINITY;
        tops[t] = fmaxf(tops[t], x[t][j]);
      }
      if constexpr (OWN_TOP) tops[t] = max_quarters(tops[t]);
      top = fmaxf(top, tops[t]);
    }
    if constexpr (!OWN_TOP) top = max_quarters(top);
    const float keep = __builtin_amdgcn_exp2f(m - top);
    float sum = 0.f;
#pragma unroll
    for (int t = 0; t < T; ++t) {
      if constexpr (!OWN_TOP) tops[t] = top;
      part[t] = OWN_TOP ? __builtin_amdgcn_exp2f(tops[t] - top) : 1.f;
      float of = 0.f;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        x[t][j] = Elem<CT>::round(__builtin_amdgcn_exp2f(x[t][j] - tops[t]));      // (as the products take it: the weights sum to one)
        of += x[t][j];
      }
      sum = __builtin_fmaf(of, part[t], sum);
    }
    l = __builtin_fmaf(l, keep, sum_quarters(sum));
    m = top;
#pragma unroll
    for (int d = 0; d < DB; ++d)
#pragma unroll
      for (int r = 0; r < 4; ++r) o[d][r] *= keep;
#pragma unroll
    for (int t = 0; t < T; ++t) {
      if (base + t * kSmallWaves * 16 >= seq) break;
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        u32x4 vf;
        if constexpr (KV8) vf = expand_e5m2x8(vr[t][i]);
        else vf = vr[t][i];
        st16(tile + (i * RPL + lane / CPR) * ROW + (lane % CPR) * 16, vf);
      }
      for (uint32_t left = (uint32_t)(is_new >> (t * 16)) & 0xffffu; left; left &= left - 1) {
        const int R = __builtin_ctz(left);
        if (lane < CPR) st16(tile + R * ROW + ((lane ^ (R & (CPR - 1))) * 16), vnew);
      }
      const u32x2 pf = {pack2s<CT>(x[t][0], x[t][1]), pack2s<CT>(x[t][2], x[t][3])};
#pragma unroll
      for (int d = 0; d < DB; ++d) {
        const int cg = 2 * d + ((col & 3) >> 1);
        const char* const p = tile + tr * ROW + ((cg ^ (tr & (CPR - 1))) * 16) + 8 * (col & 1);
        const u32x2 vf = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4_s*)p));
        if constexpr (OWN_TOP) {
          const f32x4_s c = dot16<CT>(vf, pf, f32x4_s{0.f, 0.f, 0.f, 0.f});
#pragma unroll
          for (int r = 0; r < 4; ++r) o[d][r] = __builtin_fmaf(c[r], part[t], o[d][r]);
        } else {
          o[d] = dot16<CT>(vf, pf, o[d]);
        }
      }
    }
    if (more) gather_v(next);
    idx = next;
  }
  // the waves' sums meet in LDS, each wave's in the place of its tile (G <= 8: as many bytes)
  if (col < G) {
    float* const to = (float*)tile + col * D + 4 * kq;
#pragma unroll
    for (int d = 0; d < DB; ++d) *(f32x4_s*)(to + 16 * d) = o[d];
    if (kq == 0) ml[wave][col][0] = m, ml[wave][col][1] = l;
  }
  lds_barrier();
  if (seq <= 0) return;
  for (int i = threadIdx.x; i < G * D; i += kSmallWaves * 64) {
    const int g = i / D;
    float top = kNegBigS, L = 0.f, sum = 0.f;
#pragma unroll
    for (int w = 0; w < kSmallWaves; ++w) top = fmaxf(top, ml[w][g][0]);
#pragma unroll
    for (int w = 0; w < kSmallWaves; ++w) {
      const float f = __builtin_amdgcn_exp2f(ml[w][g][0] - top);
      L = __builtin_fmaf(ml[w][g][1], f, L);
      sum = __builtin_fmaf(((const float*)tiles[w])[i], f, sum);
    }
    E::store(a.out, (int64_t)b * a.o_stride + (int64_t)hk * G * D + i, sum / L * a.out_scale);
  }
}

template <typename Tag, int D>
int launch_small(const SmallArgs& a, int bs, bool kv8, hipStream_t st) {
  const dim3 grid(a.Hkv, bs);
  if (kv8) decode_small_kernel<Tag, D, true><<<grid, kSmallWaves * 64, 0, st>>>(a);
  else decode_small_kernel<Tag, D, false><<<grid, kSmallWaves * 64, 0, st>>>(a);
  SP_LAUNCH_CHECK();
  return SP_OK;
}

}  // namespace
}  // namespace sp

using namespace sp;

extern "C" int sp_decode_small(void* out, const void* q, const void* k, const void* v, const void* cos_sin_cache, const int64_t* positions,
                               const int64_t* out_cache_loc, void* k_buffer, void* v_buffer, const int32_t* req_to_token, int64_t req_to_token_stride,
                               const void* req_pool_indices, const void* seq_lens, int idx64, int batch_size, int num_q_heads, int num_kv_heads,
                               int head_dim, int64_t q_stride, int64_t k_stride, int64_t v_stride, int64_t out_stride, int64_t kv_buffer_stride,
                               float sm_scale, float k_scale, float v_scale, int64_t max_seq_len, int dtype, int kv_dtype, void* stream) {
  SP_CHECK_ARG(out && q && k && v && cos_sin_cache && positions && out_cache_loc && k_buffer && v_buffer && req_to_token && req_pool_indices && seq_lens);
  SP_CHECK_ARG(batch_size >= 0 && batch_size <= 65535 && num_q_heads > 0 && num_kv_heads > 0 && num_q_heads % num_kv_heads == 0);
  SP_CHECK_ARG(max_seq_len >= 0 && max_seq_len <= 0x7fffffffLL - 4096 && k_scale > 0.f && v_scale > 0.f && kv_buffer_stride > 0);
  const bool kv8 = kv_dtype == SP_FP8_E5M2;
  if ((dtype != SP_F16 && dtype != SP_BF16) || (!kv8 && kv_dtype != dtype)) return SP_ERR_UNSUPPORTED;
  if ((head_dim != 64 && head_dim != 128) || num_q_heads / num_kv_heads > 8) return SP_ERR_UNSUPPORTED;
  const uintptr_t rows = (uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)cos_sin_cache, pool = (uintptr_t)k_buffer | (uintptr_t)v_buffer;
  SP_CHECK_ARG((rows & 15) == 0 && (pool & (kv8 ? 7 : 15)) == 0);
  SP_CHECK_ARG(q_stride % 8 == 0 && k_stride % 8 == 0 && v_stride % 8 == 0 && kv_buffer_stride % 8 == 0);
  if (batch_size == 0) return SP_OK;
  SmallArgs a;
  a.out = (char*)out; a.q = (const char*)q; a.k = (const char*)k; a.v = (const char*)v; a.cache = (const char*)cos_sin_cache;
  a.positions = positions; a.loc = out_cache_loc; a.kbuf = (char*)k_buffer; a.vbuf = (char*)v_buffer;
  a.r2t = req_to_token; a.r2t_stride = req_to_token_stride; a.req_idx = req_pool_indices; a.seq_lens = seq_lens; a.idx64 = idx64;
  a.q_stride = q_stride; a.k_stride = k_stride; a.v_stride = v_stride; a.o_stride = out_stride; a.kv_stride = kv_buffer_stride;
  a.Hkv = num_kv_heads; a.G = num_q_heads / num_kv_heads; a.max_len = (int)max_seq_len;
  // the pool holds k / k_scale and v / v_scale: scores take the one back, the result the other
  a.qk_scale = sm_scale * k_scale * kLog2eS; a.out_scale = v_scale; a.k_scale = k_scale; a.v_scale = v_scale;
  hipStream_t st = (hipStream_t)stream;
  if (dtype == SP_BF16) return head_dim == 64 ? launch_small<bf16_tag, 64>(a, batch_size, kv8, st) : launch_small<bf16_tag, 128>(a, batch_size, kv8, st);
  return head_dim == 64 ? launch_small<f16_tag, 64>(a, batch_size, kv8, st) : launch_small<f16_tag, 128>(a, batch_size, kv8, st);
}
