// Mixture of experts: fp32 routers - sigmoid scores, or softmax scores on ready logits - with a choice correction and
// group-limited top-k; the (token, expert)
// pairs of a step ordered by expert on the device; a grouped matrix product over that order (every expert's weights are
// read once per row tile, fp32 accumulation); the clamped gated activation; and the weighted sum of a token's experts in
// a fixed order, so a token's result does not depend on which other tokens share the step.
#include "lds_ring.h"
#include "seq_batch.h"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace sp {
namespace {

// the lowest of the lanes' indexes that hold the largest value; 0x7fffffff where no lane has one.  A butterfly of value and index through
// LDS took 12 exchanges in a row; the lanes that hold the largest value are usually one.  Top 4 of 32 experts: 4096 tokens 7.6 -> 5.5 us,
// 8 tokens 6.2 -> 4.4.
__device__ __forceinline__ int first_of_largest(float best, int at) {
  const unsigned long long ties = __ballot(best == wave_max(best));
  if (__popcll(ties) == 1) return __builtin_amdgcn_readlane(at, __ffsll(ties) - 1);
  at = ties >> (threadIdx.x & 63) & 1 ? at : 0x7fffffff;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) at = min(at, __shfl_xor(at, off, 64));
  return at;
}

// ---- router: one wave per token ----------------------------------------------------------------------------------
// z = W x (fp32), s = sigmoid(z), choice = s + correction; groups: score = sum of the two largest choices of the group,
// the best `keep` groups stay, the others' choices count as -inf; the `top` largest choices win; weights = their s.
template <typename Tag>
__global__ void moe_route_kernel(int32_t* ids, float* weights, const void* x, int64_t x_stride, const float* router,
                                 const float* correction, int64_t T, int width, int E, int top, int groups, int keep) {
  typedef Elem<Tag> El;
  extern __shared__ float smem[];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t t = (int64_t)blockIdx.x * (blockDim.x >> 6) + wave;
  if (t >= T) return;
  float* score = smem + (size_t)wave * (2 * E + groups);     // s[E], choice[E], group score[groups]
  float* choice = score + E;
  float* gscore = choice + E;
  for (int e = 0; e < E; ++e) {
    float d = 0.f;
    for (int i = lane; i < width; i += 64) d += router[(int64_t)e * width + i] * El::load(x, t * x_stride + i);
    d = wave_sum(d);
    if (lane == 0) {
      const float sg = 1.f / (1.f + expf(-d));
      score[e] = sg;
      choice[e] = sg + correction[e];
    }
  }
  __builtin_amdgcn_wave_barrier();
  if (groups > 1 && keep < groups) {
    const int per = E / groups;
    for (int gidx = lane; gidx < groups; gidx += 64) {
      float a = -INFINITY, b2 = -INFINITY;              // the two largest
      for (int e = gidx * per; e < (gidx + 1) * per; ++e) {
        const float c = choice[e];
        if (c > a) { b2 = a; a = c; }
        else if (c > b2) b2 = c;
      }
      gscore[gidx] = per > 1 ? a + b2 : a;
    }
    __builtin_amdgcn_wave_barrier();
    if (lane == 0) {
      // drop all but the best `keep` groups (ties: the lower index stays)
      for (int gidx = 0; gidx < groups; ++gidx) {
        int better = 0;
        for (int o = 0; o < groups; ++o)
          better += (gscore[o] > gscore[gidx]) || (gscore[o] == gscore[gidx] && o < gidx);
        if (better >= keep)
          for (int e = gidx * per; e < (gidx + 1) * per; ++e) choice[e] = -INFINITY;
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
  for (int k = 0; k < top; ++k) {
    float best = -INFINITY;
    int at = 0x7fffffff;
    for (int e = lane; e < E; e += 64) {
      const float c = choice[e];
      if (c > best || (c == best && e < at && c > -INFINITY)) { best = c; at = e; }
    }
    at = first_of_largest(best, at);
    if (at >= E) at = 0;                                  // fewer finite choices than `top`: cannot happen for top <= kept experts
    if (lane == 0) {
      ids[t * top + k] = at;
      weights[t * top + k] = score[at];
      choice[at] = -INFINITY;
    }
    __builtin_amdgcn_wave_barrier();
  }
}

// ---- softmax scores and choice on ready fp32 logits: one wave per token ---------------------------------------------
// s = softmax(z) over all experts; choice = s + correction (s itself without one); with groups > keep only experts of the
// `keep` groups with the largest single choice can win, whatever the others' signs; the `top` largest choices win (ties:
// the lower index); weights = s * scale.  gate: sigmoid of the logit behind the experts' (column E of the row).
__global__ void moe_softmax_topk_kernel(int32_t* ids, float* weights, float* gate, const float* logits, int64_t z_stride,
                                        const float* correction, int64_t T, int E, int top, int groups, int keep, float scale,
                                        int renorm) {
  extern __shared__ float smem[];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t t = (int64_t)blockIdx.x * (blockDim.x >> 6) + wave;
  if (t >= T) return;
  float* score = smem + (size_t)wave * (2 * E + groups);     // s[E], choice[E], group score[groups]
  float* choice = score + E;
  float* gscore = choice + E;
  const float* z = logits + t * z_stride;
  if (gate && lane == 0) gate[t] = 1.f / (1.f + expf(-z[E]));
  float zmax = -INFINITY;
  for (int e = lane; e < E; e += 64) zmax = fmaxf(zmax, z[e]);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) zmax = fmaxf(zmax, __shfl_xor(zmax, off, 64));
  float part = 0.f;
  for (int e = lane; e < E; e += 64) part += expf(z[e] - zmax);
  const float inv = 1.f / wave_sum(part);
  for (int e = lane; e < E; e += 64) {
    const float sv = expf(z[e] - zmax) * inv;
    score[e] = sv;
    choice[e] = correction ? sv + correction[e] : sv;
  }
  __builtin_amdgcn_wave_barrier();
  if (keep < groups) {
    const int per = E / groups;
    for (int g = lane; g < groups; g += 64) {
      float best = -INFINITY;
      for (int e = g * per; e < (g + 1) * per; ++e) best = fmaxf(best, choice[e]);
      gscore[g] = best;
    }
    __builtin_amdgcn_wave_barrier();
    for (int g = lane; g < groups; g += 64) {             // every lane judges its groups: ties leave the lower index in
      int better = 0;
      for (int o = 0; o < groups; ++o) better += (gscore[o] > gscore[g]) || (gscore[o] == gscore[g] && o < g);
      if (better >= keep)
        for (int e = g * per; e < (g + 1) * per; ++e) choice[e] = -INFINITY;
    }
    __builtin_amdgcn_wave_barrier();
  }
  float chosen = 0.f;                                  // lane 0: the sum of the chosen scores
  for (int k = 0; k < top; ++k) {
    float best = -INFINITY;
    int at = 0x7fffffff;
    for (int e = lane; e < E; e += 64) {
      const float c = choice[e];
      if (c > best) { best = c; at = e; }
    }
    at = first_of_largest(best, at);
    if (at >= E) at = 0;
    if (lane == 0) {
      ids[t * top + k] = at;
      weights[t * top + k] = score[at] * scale;
      chosen += score[at];
      choice[at] = -INFINITY;
    }
    __builtin_amdgcn_wave_barrier();
  }
  // the softmax over the chosen logits only = the chosen scores divided by their sum
  if (renorm && lane == 0)
    for (int k = 0; k < top; ++k) weights[t * top + k] /= chosen;
}

// ---- pairs ordered by expert: offsets[E + 1], order[pos] = pair, place[pair] = pos.  One workgroup. ---------------
// Bound by its chain of latencies.  Up to 16384 pairs a thread's ids are on their way together and stay in registers, and a pair's place
// inside its expert is what the count gave back, so the counters are gone through once; the order is written in rows out of LDS.  More
// pairs go through the counters a second time (the count's answer kept in `place` meanwhile: 65536 pairs of 32 experts 41 us, so 34).  The
// sums over experts go 64 at a time.  16384 pairs of 32 experts: 14.6 -> 8.8 us (scattered stores of the order: 10.5); 32 pairs: 2.9 -> 2.3.
constexpr int kAlignThreads = 1024, kAlignHeld = 16, kAlignPairs = kAlignThreads * kAlignHeld;

__global__ void __launch_bounds__(kAlignThreads) moe_align_kernel(int32_t* offsets, int32_t* order, int32_t* place, const int32_t* ids, int P,
                                                                  int E) {
  extern __shared__ int32_t cnt[];          // counts[E], first positions[E], then the held pairs in their order
  int32_t* first = cnt + E;
  uint16_t* sorted = (uint16_t*)(first + E);
  const int tid = threadIdx.x;
  const bool held = P <= kAlignPairs;
  int32_t id[kAlignHeld], rank[kAlignHeld];
  if (held) {
#pragma unroll
    for (int i = 0; i < kAlignHeld; ++i) {
      if (i * kAlignThreads >= P) break;
      id[i] = ids[min(i * kAlignThreads + tid, P - 1)];
    }
  }
  for (int e = tid; e < E; e += kAlignThreads) cnt[e] = 0;
  __syncthreads();
  if (held) {
#pragma unroll
    for (int i = 0; i < kAlignHeld; ++i) {
      if (i * kAlignThreads >= P) break;
      if (i * kAlignThreads + tid < P) rank[i] = atomicAdd(&cnt[id[i]], 1);
    }
  } else {
    for (int p = tid; p < P; p += kAlignThreads) atomicAdd(&cnt[ids[p]], 1);
  }
  __syncthreads();
  if (tid < 64) {
    int32_t run = 0;
    for (int e0 = 0; e0 < E; e0 += 64) {
      const int e = e0 + tid;
      const int32_t n = e < E ? cnt[e] : 0;
      int32_t sum = n;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const int32_t below = __shfl_up(sum, off, 64);
        if (tid >= off) sum += below;
      }
      if (e < E) offsets[e] = first[e] = run + sum - n;
      run += __shfl(sum, 63, 64);
    }
    if (tid == 0) offsets[E] = run;
  }
  __syncthreads();
  if (held) {
#pragma unroll
    for (int i = 0; i < kAlignHeld; ++i) {
      if (i * kAlignThreads >= P) break;
      const int p = i * kAlignThreads + tid;
      if (p < P) {
        const int pos = first[id[i]] + rank[i];
        sorted[pos] = (uint16_t)p;
        place[p] = pos;
      }
    }
    __syncthreads();
    for (int i = tid; i < P; i += kAlignThreads) order[i] = sorted[i];
  } else {
    for (int p = tid; p < P; p += kAlignThreads) {
      const int pos = atomicAdd(&first[ids[p]], 1);
      order[pos] = p;
      place[p] = pos;
    }
  }
}

// ---- grouped product: out[pos, n] = sum_k a[row(pos), k] * w[expert(pos), n, k] -------------------------------------
// row(pos) = order[pos] / row_div when order is given (the token of a pair), else pos; act 1: max(out, 0)^2 instead (on the
// fp32 sum, rounded once).  Pairs of ids from E on (outputs without a weight) are left alone.  Tiles of 32 rows x 64 columns;
// a tile never spans two experts.  Each output element accumulates over k in the same order wherever its row sits.
constexpr int GM = 32, GN = 64, GK = 32;

__device__ __forceinline__ float gemm_act(float v, int act) {
  if (act == 0) return v;
  const float r = fmaxf(v, 0.f);
  return r * r;
}

template <typename Tag>
__global__ void __launch_bounds__(256)
moe_grouped_gemm_kernel(void* out, const void* a, const void* w, const int32_t* offsets, const int32_t* order, int row_div,
                        int P, int N, int K, int E, int64_t a_stride, int64_t out_stride, int act) {
  typedef Elem<Tag> El;
  __shared__ float As[GK][GM + 1];
  __shared__ float Bs[GK][GN + 4];
  // which expert and which of its row tiles
  int tile = blockIdx.x, e = 0, row0 = 0, rows_end = 0;
  for (; e < E; ++e) {
    const int lo = offsets[e], hi = offsets[e + 1];
    const int tiles = (hi - lo + GM - 1) / GM;
    if (tile < tiles) {
      row0 = lo + tile * GM;
      rows_end = hi;
      break;
    }
    tile -= tiles;
  }
  if (e >= E) return;
  const int n0 = blockIdx.y * GN;
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;       // 16 x 16 threads: 2 rows x 4 columns each
  float acc[2][4] = {};
  const char* wbase = (const char*)w + (int64_t)e * N * K * El::kBytes;
  // loader roles: A tile 32 x 32 (4 per thread), B tile 64 x 32 (8 per thread)
  const int ar = threadIdx.x >> 3, ak = (threadIdx.x & 7) * 4;
  const int br = threadIdx.x >> 2, bk = (threadIdx.x & 3) * 8;
  int64_t arow = -1;
  if (row0 + ar < rows_end) arow = order ? order[row0 + ar] / row_div : row0 + ar;
  for (int k0 = 0; k0 < K; k0 += GK) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int k = k0 + ak + i;
      As[ak + i][ar] = (arow >= 0 && k < K) ? El::load(a, arow * a_stride + k) : 0.f;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int k = k0 + bk + i, n = n0 + br;
      Bs[bk + i][br] = (n < N && k < K) ? El::load(wbase, (int64_t)n * K + k) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < GK; ++k) {
      const float a0 = As[k][ty * 2], a1 = As[k][ty * 2 + 1];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float bv = Bs[k][tx * 4 + j];
        acc[0][j] += a0 * bv;
        acc[1][j] += a1 * bv;
      }
    }
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int pos = row0 + ty * 2 + i;
    if (pos >= rows_end) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + tx * 4 + j;
      if (n < N) El::store(out, (int64_t)pos * out_stride + n, gemm_act(acc[i][j], act));
    }
  }
}

// ---- the same product on the matrix cores (16-bit types, K a multiple of 32, 16-byte aligned rows) -------------------
// v_mfma_f32_16x16x32: lane (r16 = lane & 15, q = lane >> 4) holds 8 k-values of row r16 of each operand and receives
// D[4 q + r][r16], r < 4 - with the weights as the first operand a lane ends up with 4 neighbouring output columns of ONE
// row.  The kernels below (tile, ring, wide, rows, narrow rows) add the k-steps of 32 in ascending order into one accumulator, so an output
// element has the same bits whichever of them - and whichever tile height - computes it: a token's result does not depend on the
// step's size.
//
// ACT: 0 the product, 1 max(., 0)^2 of the fp32 sum; 2 and 3 take w [E, 2 N, K] (gate rows, then up rows), keep the two sums
// of an output column in one lane and store the activation of the ROUNDED sums - bit for bit the plain product followed by
// sp_silu_and_mul (2) or sp_moe_glu (3), without the [P, 2 N] round trip and the launch.
typedef float f32x4_q __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8_q __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_q __attribute__((ext_vector_type(8)));
template <typename Tag>
__device__ __forceinline__ f32x4_q mfma_q(const u32x4& a, const u32x4& b, const f32x4_q& c);
template <>
__device__ __forceinline__ f32x4_q mfma_q<bf16_tag>(const u32x4& a, const u32x4& b, const f32x4_q& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_q, a), __builtin_bit_cast(bf16x8_q, b), c, 0, 0, 0);
}
template <>
__device__ __forceinline__ f32x4_q mfma_q<f16_tag>(const u32x4& a, const u32x4& b, const f32x4_q& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_q, a), __builtin_bit_cast(f16x8_q, b), c, 0, 0, 0);
}

struct GroupedArgs {
  char* out;
  const char* a;
  const char* w;
  const int32_t* offsets;
  const int32_t* order;
  int row_div, N, K, E;              // N: output columns
  int64_t a_stride, out_stride;      // elements
  int vec_out;                       // 8-byte stores of 4 columns are aligned and inside a row
  float limit, alpha;                // ACT 3
  int32_t far;                       // entries of `order` from here on name rows that no 32-bit offset from a's first byte reaches (the ring's)
};

// (shared by the separate launch and the fused epilogue, which agree bit for bit)
template <typename Tag>
__device__ __forceinline__ float moe_glu_value(float g, float u, float limit, float alpha) {
  g = fminf(g, limit);
  u = fminf(fmaxf(u, -limit), limit);
  return mul_round<Tag>(over_one_plus_exp(g, alpha * g), u + 1.f);
}

template <typename Tag, int ACT>
__device__ __forceinline__ float grouped_act(float v, float up, const GroupedArgs& p) {
  typedef Elem<Tag> El;
  if constexpr (ACT == 1) return gemm_act(v, 1);
  if constexpr (ACT == 2) return mul_round<Tag>(El::round(silu_ref(El::round(v))), El::round(up));
  if constexpr (ACT == 3) return moe_glu_value<Tag>(El::round(v), El::round(up), p.limit, p.alpha);
  return v;
}

template <typename Tag>
__device__ __forceinline__ void store4(const GroupedArgs& p, int64_t pos, int n, const float* v) {
  typedef Elem<Tag> El;
  if (p.vec_out && n + 4 <= p.N) {
    const float f[8] = {v[0], v[1], v[2], v[3], 0.f, 0.f, 0.f, 0.f};
    const u32x4 w = pack16<Tag>(f);
    *(u32x2*)(p.out + (pos * p.out_stride + n) * 2) = u32x2{w[0], w[1]};
    return;
  }
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (n + r < p.N) El::store(p.out, pos * p.out_stride + n + r, v[r]);
}

// Row tiles of `bm` rows, expert after expert (a tile never spans two): the expert, first row and end of tile `tile`, found by
// a wave with one load per lane and a scan (E <= 64: one round).  False past the last tile.  `total`: all tiles, if asked for.
__device__ __forceinline__ int wave_inclusive(int v, int lane) {
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int o = __shfl_up(v, off, 64);
    if (lane >= off) v += o;
  }
  return v;
}
__device__ __forceinline__ int grouped_tiles(const int32_t* offsets, int E, int bm, int lane) {
  int run = 0;
  for (int e0 = 0; e0 < E; e0 += 64) {
    const int e = e0 + lane;
    int v = e < E ? (offsets[e + 1] - offsets[e] + bm - 1) / bm : 0;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    run += v;
  }
  return run;
}
__device__ __forceinline__ bool grouped_tile(const int32_t* offsets, int E, int bm, int tile, int lane, int& e_out, int& row0,
                                             int& rows_end) {
  for (int e0 = 0; e0 < E; e0 += 64) {
    const int e = e0 + lane;
    const int lo = e < E ? offsets[e] : 0, hi = e < E ? offsets[e + 1] : 0;
    const int tiles = (hi - lo + bm - 1) / bm, incl = wave_inclusive(tiles, lane);
    const uint64_t hit = __ballot(tile < incl);
    if (hit) {
      const int l = __ffsll((unsigned long long)hit) - 1;
      e_out = e0 + l;
      row0 = __builtin_amdgcn_readfirstlane(__shfl(lo, l, 64) + (tile - __shfl(incl - tiles, l, 64)) * bm);
      rows_end = __builtin_amdgcn_readfirstlane(__shfl(hi, l, 64));
      return true;
    }
    tile -= __builtin_amdgcn_readfirstlane(__shfl(incl, 63, 64));
  }
  return false;
}

// The same for a launch of `cols` column tiles per row tile, an expert's row tiles next to each other: the column tile as well.
__device__ __forceinline__ bool grouped_tile_by_column(const int32_t* offsets, int E, int bm, int cols, int at, int lane, int& e_out,
                                                       int& row0, int& rows_end, int& col, int& rows_tiles) {
  for (int e0 = 0; e0 < E; e0 += 64) {
    const int e = e0 + lane;
    const int lo = e < E ? offsets[e] : 0, hi = e < E ? offsets[e + 1] : 0;
    const int tiles = (hi - lo + bm - 1) / bm, incl = wave_inclusive(tiles * cols, lane);
    const uint64_t hit = __ballot(at < incl);
    if (hit) {
      const int l = __ffsll((unsigned long long)hit) - 1;
      e_out = e0 + l;
      const int n = __builtin_amdgcn_readfirstlane(__shfl(tiles, l, 64));
      const int in = __builtin_amdgcn_readfirstlane(at - __shfl(incl - tiles * cols, l, 64));
      col = in / n;
      rows_tiles = n;
      row0 = __builtin_amdgcn_readfirstlane(__shfl(lo, l, 64)) + (in - col * n) * bm;
      rows_end = __builtin_amdgcn_readfirstlane(__shfl(hi, l, 64));
      return true;
    }
    at -= __builtin_amdgcn_readfirstlane(__shfl(incl, 63, 64));
  }
  return false;
}

// Steps with more than a few rows per expert, any K that is a multiple of 8: BM rows x 128 weight rows per workgroup, k in steps of 64.  Both operands go to LDS by
// direct loads (16 bytes per lane, no registers on the way), one step ahead of the MFMAs, in two buffers; a step costs one
// barrier.  LDS rows are 128 bytes whose eight 16-byte chunks are permuted by the row's number (the SOURCE address is
// permuted: a direct load writes lane after lane), so the 16 rows of a fragment read meet no bank twice in a phase.
// Four waves: BM 128 as 2 x 2 of 64 x 64, smaller tiles as 1 x 4 of BM x 32.  The tiles of a row block lie next to each
// other in one XCD's share of the grid (block b runs on XCD b mod 8), so an XCD's L2 sees each row of `a` once.
constexpr int kGroupedBN = 128, kGroupedBK = 64;

template <typename Tag, int BM, int ACT>
__global__ void __launch_bounds__(256, 2) moe_grouped_tile_kernel(GroupedArgs p) {
  constexpr bool GLU = ACT >= 2;
  constexpr int WN = BM == 128 ? 2 : 4, CPW = kGroupedBN / WN, FM = (BM == 128 ? 64 : BM) / 16, FN = CPW / 16;
  constexpr int OUT_N = GLU ? kGroupedBN / 2 : kGroupedBN;
  constexpr int LA = BM / 32, LB = kGroupedBN / 32;              // direct loads per wave and step
  constexpr int kBuf = (BM + kGroupedBN) * 128;
  __shared__ __attribute__((aligned(16))) char lds0[kBuf];
  __shared__ __attribute__((aligned(16))) char lds1[kBuf];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, r16 = lane & 15, q = lane >> 4;
  const int ntiles = (p.N + OUT_N - 1) / OUT_N;
  const int total = grouped_tiles(p.offsets, p.E, BM, lane) * ntiles, share = (total + 7) / 8;
  const int idx = (int)(blockIdx.x >> 3), at = (int)(blockIdx.x & 7) * share + idx;
  if (idx >= share || at >= total) return;
  int e = 0, row0 = 0, rows_end = 0;
  if (!grouped_tile(p.offsets, p.E, BM, at / ntiles, lane, e, row0, rows_end)) return;
  e = __builtin_amdgcn_readfirstlane(e);
  const int n0 = (at % ntiles) * OUT_N;
  const int wm = wave / WN, wn = wave % WN;
  const int wrows = GLU ? 2 * p.N : p.N;
  // sources of this wave's direct loads: lane -> row lane / 8 of the 8 rows of a load, chunk lane % 8 of LDS
  const int chunk = (lane & 7) ^ (lane >> 3);
  const char* src[LA + LB];
#pragma unroll
  for (int i = 0; i < LA; ++i) {
    const int pos = min(row0 + (wave * LA + i) * 8 + (lane >> 3), rows_end - 1);      // rows past the end: never stored
    const int64_t arow = p.order ? p.order[pos] / p.row_div : pos;
    src[i] = p.a + arow * p.a_stride * 2 + chunk * 16;
  }
  const char* wbase = p.w + (int64_t)e * wrows * p.K * 2 + chunk * 16;
#pragma unroll
  for (int i = 0; i < LB; ++i) {
    const int br = (wave * LB + i) * 8 + (lane >> 3);
    int row;
    if constexpr (GLU) {
      const int in = br % CPW, col = n0 + (br / CPW) * (CPW / 2) + in % (CPW / 2);
      row = min(col, p.N - 1) + (in >= CPW / 2 ? p.N : 0);
    } else {
      row = min(n0 + br, p.N - 1);
    }
    src[LA + i] = wbase + (int64_t)row * p.K * 2;
  }
  const auto stage = [&](char* lds, int k0) {
    // the last step of a K that is no multiple of 64: chunks past the row's end are read from its start and never used
    const int back = k0 + chunk * 8 >= p.K ? chunk * 16 : -k0 * 2;
#pragma unroll
    for (int i = 0; i < LA + LB; ++i) {
      char* dst = lds + (i < LA ? (wave * LA + i) : (BM / 8 + wave * LB + i - LA)) * 1024;
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src[i] - back),
                                       (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
    }
  };
  f32x4_q acc[FM][FN];
#pragma unroll
  for (int f = 0; f < FM; ++f)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[f][j] = f32x4_q{0.f, 0.f, 0.f, 0.f};
  const int arow0 = (wm * (BM == 128 ? 64 : 0) + r16) * 128, brow0 = (BM + wn * CPW + r16) * 128;
  const auto compute = [&](const char* lds, auto halves) {
#pragma unroll
    for (int kk = 0; kk < decltype(halves)::value; ++kk) {
      const int c = ((kk * 4 + q) ^ (r16 & 7)) * 16;
      u32x4 xf[FM], wf[FN];
#pragma unroll
      for (int f = 0; f < FM; ++f) xf[f] = ld16(lds + arow0 + f * 2048 + c);
#pragma unroll
      for (int j = 0; j < FN; ++j) wf[j] = ld16(lds + brow0 + j * 2048 + c);
#pragma unroll
      for (int f = 0; f < FM; ++f)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[f][j] = mfma_q<Tag>(wf[j], xf[f], acc[f][j]);
    }
  };
  const auto ready = [&]() {           // this wave's loads have landed, then everyone's; the other buffer is free
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
  };
  const std::integral_constant<int, 2> whole;
  const int full = p.K & ~(kGroupedBK - 1);
  int k0 = 0;
  stage(lds0, 0);
  for (; k0 + 2 * kGroupedBK <= full; k0 += 2 * kGroupedBK) {
    ready();
    stage(lds1, k0 + kGroupedBK);
    compute(lds0, whole);
    ready();
    if (k0 + 2 * kGroupedBK < p.K) stage(lds0, k0 + 2 * kGroupedBK);
    compute(lds1, whole);
  }
  const std::integral_constant<int, 1> half;
  if (k0 < full) {                     // one more whole step, then perhaps half a one
    ready();
    if (full < p.K) stage(lds1, full);
    compute(lds0, whole);
    if (full < p.K) {
      ready();
      compute(lds1, half);
    }
  } else if (full < p.K) {
    ready();
    compute(lds0, half);
  }
  constexpr int FO = GLU ? FN / 2 : FN;
#pragma unroll
  for (int f = 0; f < FM; ++f) {
    const int pos = row0 + wm * (BM == 128 ? 64 : 0) + 16 * f + r16;
    if (pos >= rows_end) continue;
#pragma unroll
    for (int j = 0; j < FO; ++j) {
      float v[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = grouped_act<Tag, ACT>(acc[f][j][r], GLU ? acc[f][j + FN - FO][r] : 0.f, p);
      store4<Tag>(p, pos, n0 + wn * (GLU ? CPW / 2 : CPW) + 16 * j + 4 * q, v);
    }
  }
}

// The sums of a wave's part of a ring tile straight from memory, in the ring's order: for tiles with a row that a load's 32-bit offset does not
// reach.  (An order may name any rows of `a`, and only the device knows which; those that moe_align makes lie in its first pairs / row_div + 1,
// which the launcher looks at.)
template <typename Tag, typename T, bool GLU>
__device__ __forceinline__ void far_product(f32x4_q (&acc)[T::FM][T::FN], const GroupedArgs& p, const char* we, int pos0, int rows_end, int n0, int col0,
                                            int lane) {
  const int r16 = lane & 15, q = lane >> 4;
#pragma unroll 1
  for (int k = 8 * q; k < p.K; k += 32) {
    u32x4 wf[T::FN];
#pragma unroll
    for (int j = 0; j < T::FN; ++j) {
      const int c = col0 + 16 * j;                         // (a multiple of 16)
      const int64_t row = GLU ? min(n0 + c / 2 + r16 % 8, p.N - 1) + (r16 >= 8 ? p.N : 0) : min(n0 + c + r16, p.N - 1);
      wf[j] = ld16(we + (row * p.K + k) * 2);
    }
#pragma unroll
    for (int f = 0; f < T::FM; ++f) {
      const int64_t row = p.order[min(pos0 + 16 * f + r16, rows_end - 1)] / p.row_div;
      const u32x4 xf = ld16(p.a + (row * p.a_stride + k) * 2);
#pragma unroll
      for (int j = 0; j < T::FN; ++j) acc[f][j] = mfma32<Tag>(wf[j], xf, acc[f][j]);
    }
  }
}

// The same for K a multiple of 64, by ring_product's loop.  Two workgroups share a CU (of all tiles but the largest) and fill each other's beginnings
// and ends.  GLU: 8 gate rows and the up rows of the same 8 columns in one operand, their sums 32 lanes apart.  ONCE: an expert with one row tile reads
// its weights past the L2.  The row tiles of one column tile follow each other: the weights they share are in the L2.
// Width 2048, 32 experts of ff 1024, up + down in us, the kernels before (64 x 128, 128 x 128 and 128 x 256 tiles, one wave per 16 rows) -> these: mean rows
// 3: 63 + 27 -> 55 + 24, 16: 67 + 28 -> 55 + 23, 32: 68 + 29 -> 59 + 25, 50: 69 + 30 -> 60 + 30, 88: 72 + 32 -> 74 + 32, 125: 97 + 51 -> 82 + 34, 188: 98 + 52 ->
// 102 + 53, 250: 134 + 70 -> 111 + 58, 512: 180 + 107 -> 171 + 92; width 4096, 128 experts of 1536, 4: 560 + 270 -> 481 + 239, 256: 1344 + 735 -> 1110 + 617;
// 16 experts of 1408, 50: 50 + 26 -> 52 + 21, 750: 172 + 107 -> 173 + 85; 8 of 1536, 40: 38 + 20 -> 31 + 12, 1024: 142 + 86 -> 131 + 58.
template <typename Tag, typename T, bool ONCE, int ACT>
__global__ void __launch_bounds__(T::W * 64, T::kWaves) moe_grouped_ring_kernel(GroupedArgs p) {
  constexpr bool GLU = ACT >= 2;
  constexpr int BM = T::BM, RB = T::RB, RPL = T::RPL, CH = T::CH, L = T::L, FM = T::FM, FN = T::FN, OUT_N = GLU ? T::BN / 2 : T::BN;
  extern __shared__ __attribute__((aligned(1024))) char ring_lds[];
  char* const lds = ring_lds;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, r16 = lane & 15, q = lane >> 4;
  const int ntiles = (p.N + OUT_N - 1) / OUT_N;
  const int total = grouped_tiles(p.offsets, p.E, BM, lane) * ntiles, share = (total + 7) / 8;
  const int idx = (int)(blockIdx.x >> 3), at = (int)(blockIdx.x & 7) * share + idx;
  if (idx >= share || at >= total) return;
  int e = 0, row0 = 0, rows_end = 0, col = 0, row_tiles = 0;
  if (!grouped_tile_by_column(p.offsets, p.E, BM, ntiles, at, lane, e, row0, rows_end, col, row_tiles)) return;
  e = __builtin_amdgcn_readfirstlane(e);
  const int n0 = col * OUT_N, wrows = GLU ? 2 * p.N : p.N, steps = p.K / T::BK;
  const int wm = wave / T::WN, wn = wave % T::WN;
  // this wave's direct loads: lane -> row lane / CH of a load, chunk lane % CH
  uint32_t off[L];
  const char* base[L];
  const char* const we = p.w + (int64_t)e * wrows * p.K * 2;
  bool far = false;                                        // (of the tile, the same in every wave)
  if (p.order)
#pragma unroll
    for (int r = 0; r < BM; r += 64) far |= p.order[min(row0 + r + lane, rows_end - 1)] >= p.far;
#pragma unroll
  for (int i = 0; i < L; ++i) {
    const int g = min(i * T::W + wave, T::G - 1), r = g * RPL + lane / CH, chunk = (lane % CH) ^ (r & 7);
    const bool is_x = g * RPL < BM;
    int64_t row;                                         // rows and columns past the end: the last one again, never stored
    if (is_x) {
      const int pos = min(row0 + r, rows_end - 1);
      row = p.order ? p.order[pos] / p.row_div : pos;
    } else if constexpr (GLU) {
      const int in = (r - BM) % 16;
      row = min(n0 + (r - BM) / 16 * 8 + in % 8, p.N - 1) + (in >= 8 ? p.N : 0);
    } else {
      row = min(n0 + r - BM, p.N - 1);
    }
    off[i] = (uint32_t)(row * (is_x ? p.a_stride : p.K) * 2) + chunk * 16;
    base[i] = is_x ? p.a : we;
  }
  f32x4_q acc[FM][FN];
#pragma unroll
  for (int f = 0; f < FM; ++f)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[f][j] = f32x4_q{0.f, 0.f, 0.f, 0.f};
  if (__any(far)) far_product<Tag, T, GLU>(acc, p, we, row0 + wm * T::TM, rows_end, n0, wn * T::TN, lane);
  else if (ONCE && row_tiles == 1) ring_product<Tag, T, ONCE, 2>(acc, off, base, lds, steps, wave, lane);
  else ring_product<Tag, T, 0, 2>(acc, off, base, lds, steps, wave, lane);
#pragma unroll
  for (int f = 0; f < FM; ++f) {
    const int pos = row0 + wm * T::TM + 16 * f + r16;
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      float v[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const auto both = __builtin_amdgcn_permlane32_swap(as_u32(acc[f][j][r]), as_u32(acc[f][j][r]), false, false);      // [1]: lanes 32-63 twice
        v[r] = grouped_act<Tag, ACT>(acc[f][j][r], GLU ? as_f32(both[1]) : 0.f, p);
      }
      if (pos < rows_end && !(GLU && q >= 2)) store4<Tag>(p, pos, GLU ? n0 + wn * (T::TN / 2) + 8 * j + 4 * q : n0 + wn * T::TN + 16 * j + 4 * q, v);
    }
  }
}

template <typename Tag, typename T, bool ONCE, int ACT>
int launch_grouped_ring(const GroupedArgs& p, int pairs, int held, hipStream_t st) {
  constexpr int per = ACT >= 2 ? T::BN / 2 : T::BN;
  static PerDevice<int> raised;
  int ok = 0;
  raised.get(ok, [&](int) {
    return hipFuncSetAttribute((const void*)moe_grouped_ring_kernel<Tag, T, ONCE, ACT>, hipFuncAttributeMaxDynamicSharedMemorySize, T::kLds) ==
                   hipSuccess ? 1 : 0;
  });
  if (!ok) return SP_ERR_LAUNCH;
  const int64_t ntiles = (p.N + per - 1) / per;
  const unsigned blocks = (unsigned)(((pairs / T::BM + held) * ntiles + 7) / 8 * 8);
  moe_grouped_ring_kernel<Tag, T, ONCE, ACT><<<dim3(blocks), dim3(T::W * 64), T::kLds, st>>>(p);
  SP_LAUNCH_CHECK();
  return SP_OK;
}

// The tiles, and what one costs: us per step of BK where two workgroups share a unit and where one has it alone, and us besides.
#define SP_RING_TILES(F)                                        \
  F(0, 0.979f, 0.454f, 1.63f, true, 32, 128, 64, 1, 4, 4)       \
  F(1, 0.801f, 0.389f, 2.88f, true, 32, 64, 128, 1, 4, 3)       \
  F(2, 0.967f, 0.519f, 2.19f, true, 64, 128, 64, 2, 2, 3)       \
  F(3, 0.529f, 0.129f, 4.16f, false, 64, 128, 64, 1, 4, 3)      \
  F(4, 0.680f, 0.290f, 4.94f, false, 80, 128, 64, 1, 4, 3)      \
  F(5, 0.455f, 0.118f, 3.98f, false, 96, 64, 64, 2, 2, 4)       \
  F(6, 1.102f, 0.533f, 4.92f, false, 128, 128, 64, 2, 4, 2)     \
  F(7, 1.269f, 0.664f, 5.16f, false, 160, 128, 64, 2, 2, 2)     \
  F(8, 1.432f, 0.658f, 5.84f, false, 192, 128, 64, 4, 2, 2)     \
  F(9, 3.326f, 1.018f, 5.36f, false, 192, 192, 64, 2, 4, 3)

struct RingCost {
  float two, one, fixed;
  int bm, bn, bk, lds;
  bool once;
};
#define SP_RING_ROW(I, TWO, ONE, FIXED, ONCE, ...) \
  {TWO, ONE, FIXED, RingTile<__VA_ARGS__>::BM, RingTile<__VA_ARGS__>::BN, RingTile<__VA_ARGS__>::BK, RingTile<__VA_ARGS__>::kLds, ONCE},
constexpr RingCost kRingTiles[] = {SP_RING_TILES(SP_RING_ROW)};

// Expected row tiles of one expert of `experts`, each pair choosing each of them alike
inline double ring_row_tiles(int pairs, int experts, int bm) {
  const double mean = (double)pairs / experts, sd = sqrt(mean * (1. - 1. / experts));
  double tiles = 1. - exp(-mean);
  for (double edge = bm; edge < mean + 4. * sd; edge += bm) tiles += edge < mean - 4. * sd ? 1. : .5 * erfc((edge + .5 - mean) / (1.41421356 * sd));
  return tiles;
}

// The time of a product with tile `t`: the longest of the chains of tiles that a unit works through, of what it loads into its LDS and of the
// weights' way from memory, the two lesser ones added softly.  The last, not full round of tiles counts by the chance that it is there and that
// some unit holds two of it.  Costs by least squares
// from 20 tiles' timings of 58 products (widths 1024 and 2048, 8 to 128 experts, 8 to 4096 rows: 11 % rms), those of the smaller tiles then moved to what picks the
// fastest tile: 2 - 3 % behind the best of the 20 on average (70 other row counts: 1 % faster than by the plain fit, 0.96 - 1.10).
inline double ring_us(const RingCost& t, int pairs, int experts, int64_t wrows, int K) {
  const double cols = (double)((wrows + t.bn - 1) / t.bn), tiles = experts * ring_row_tiles(pairs, experts, t.bm) * cols, steps = K / t.bk;
  const bool pair = t.lds <= 80 * 1024;
  const double slots = pair ? 512. : 256., one = t.fixed + steps * t.one, two = t.fixed + steps * t.two;
  const double full = floor(tiles / slots), rest = tiles - full * slots, round = pair ? two : one;
  double last = one;
  if (pair && rest > 256.) last += (two - one) * (1. - exp((256. - rest) / cols)) * (.8 + .2 * std::min(1., std::max(0., rest / 256. - 1.)));
  last *= 1. - exp(-rest / cols);
  const double chain = full * round + (full > 0. ? .88 * last + .12 * std::min(last, rest / slots * round) : last);
  const double fill = std::max(1., tiles / 256.) * steps * (t.bm + t.bn) * t.bk * 2. / 76.8e3;              // bytes per us of a unit
  const double stream = experts * (1. - exp(-(double)pairs / experts)) * (double)wrows * K * 2. / (t.once ? 6.11e6 : 5.15e6);
  const double c2 = chain * chain, f2 = fill * fill, s2 = stream * stream;
  return c2 * c2 + f2 * f2 + s2 * s2;                                                                         // (its fourth power)
}

// (2 us of the host: the layers of a model ask for the same sizes one after the other, so a thread's last answers are kept)
inline int ring_tile(int pairs, int experts, int64_t wrows, int K) {
  struct Answer {
    int64_t wrows;
    int pairs, experts, K, tile;
  };
  thread_local Answer kept[16] = {};
  Answer& a = kept[((unsigned)pairs * 5u + (unsigned)experts * 3u + (unsigned)(wrows >> 4) + (unsigned)(K >> 6)) % 16];
  if (a.pairs == pairs && a.experts == experts && a.wrows == wrows && a.K == K) return a.tile;
  int best = -1;
  double least = 0.;
  for (int i = 0; i < (int)(sizeof(kRingTiles) / sizeof(kRingTiles[0])); ++i) {
    if (K % kRingTiles[i].bk) continue;
    const double us = ring_us(kRingTiles[i], pairs, experts, wrows, K);
    if (best < 0 || us < least) best = i, least = us;
  }
  a = Answer{wrows, pairs, experts, K, best};
  return best;
}

// Gated products of hundreds of rows per expert, and plain ones whose K the ring does not take: 128 rows x 256 weight rows per workgroup, a wave
// 64 x 128 of them, k in steps of 32, any K that is a multiple of 32.  What the 128 x 128 tiles wait for is LDS (a wave reads 8 KB for 16 products of
// 16 cycles: 128 bytes per cycle for the four of them, all there is) and the L2 (64 bytes per cycle and CU); here it is 96 and 48.  A step's operands
// are 24 KB, double-buffered, so three workgroups share a CU and fill each other's waits.  The row tiles of one column tile follow each other: the
// weights they share are in the L2 once.  LDS rows are 64 bytes; the chunk of a row is permuted by its number / 4, so that the 16 rows of a
// fragment read lie in 64 banks.
// Against the ring's tiles, gated, past a mean of 320 rows, 67 sizes (4 to 256 experts, widths 1024 to 7168), each routed evenly, by expert weights
// of spread e^0.5 and by 1 / rank: the ring 0.67 - 1.8 of this one's speed, 2 % faster on average but more than 5 % slower in 70 of 201, where
// counts above 192 or 384 rows cost a row tile more.  Width 2048, 32 experts of ff 1024, up product in us, ring | this, evenly and by weights: 4096 tokens
// 170 | 186, 195 | 180; 6000: 256 | 251, 296 | 251; 8192: 323 | 318, 322 | 320.
constexpr int kWideBM = 128, kWideBN = 256, kWideBK = 32;
template <typename Tag, int ACT>
__global__ void __launch_bounds__(256, 3) moe_grouped_wide_kernel(GroupedArgs p) {
  constexpr bool GLU = ACT >= 2;
  constexpr int CPW = kWideBN / 2, FM = 4, FN = CPW / 16, OUT_N = GLU ? kWideBN / 2 : kWideBN;
  constexpr int LA = kWideBM / 64, LB = kWideBN / 64;            // direct loads per wave and step
  constexpr int kBuf = (kWideBM + kWideBN) * kWideBK * 2;
  extern __shared__ __attribute__((aligned(16))) char wide_lds[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, r16 = lane & 15, q = lane >> 4;
  const int ntiles = (p.N + OUT_N - 1) / OUT_N;
  const int total = grouped_tiles(p.offsets, p.E, kWideBM, lane) * ntiles, share = (total + 7) / 8;
  const int idx = (int)(blockIdx.x >> 3), at = (int)(blockIdx.x & 7) * share + idx;
  if (idx >= share || at >= total) return;
  int e = 0, row0 = 0, rows_end = 0, col = 0, row_tiles = 0;
  if (!grouped_tile_by_column(p.offsets, p.E, kWideBM, ntiles, at, lane, e, row0, rows_end, col, row_tiles)) return;
  e = __builtin_amdgcn_readfirstlane(e);
  const int n0 = col * OUT_N;
  const int wm = wave >> 1, wn = wave & 1;
  const int wrows = GLU ? 2 * p.N : p.N;
  // sources of this wave's direct loads: lane -> row lane / 4 of the 16 rows of a load, chunk lane % 4 of LDS
  const int chunk = (lane & 3) ^ (lane >> 4);
  const char* src[LA + LB];
#pragma unroll
  for (int i = 0; i < LA; ++i) {
    const int pos = min(row0 + (wave * LA + i) * 16 + (lane >> 2), rows_end - 1);     // rows past the end: never stored
    const int64_t arow = p.order ? p.order[pos] / p.row_div : pos;
    src[i] = p.a + arow * p.a_stride * 2 + chunk * 16;
  }
  const char* wbase = p.w + (int64_t)e * wrows * p.K * 2 + chunk * 16;
#pragma unroll
  for (int i = 0; i < LB; ++i) {
    const int br = (wave * LB + i) * 16 + (lane >> 2);
    int row;
    if constexpr (GLU) {
      const int in = br % CPW, n = n0 + (br / CPW) * (CPW / 2) + in % (CPW / 2);
      row = min(n, p.N - 1) + (in >= CPW / 2 ? p.N : 0);
    } else {
      row = min(n0 + br, p.N - 1);
    }
    src[LA + i] = wbase + (int64_t)row * p.K * 2;
  }
  const int steps = p.K / kWideBK;
  const auto stage = [&](char* lds, int step) {
#pragma unroll
    for (int i = 0; i < LA + LB; ++i) {
      char* dst = lds + (i < LA ? (wave * LA + i) : (kWideBM / 16 + wave * LB + i - LA)) * 1024;
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src[i] + step * (kWideBK * 2)),
                                       (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
    }
  };
  f32x4_q acc[FM][FN];
#pragma unroll
  for (int f = 0; f < FM; ++f)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[f][j] = f32x4_q{0.f, 0.f, 0.f, 0.f};
  const int c = (q ^ (r16 >> 2)) * 16;
  const int arow0 = (wm * 64 + r16) * 64 + c, brow0 = (kWideBM + wn * CPW + r16) * 64 + c;
  char *now = wide_lds, *next = wide_lds + kBuf;
  stage(now, 0);
  for (int s = 0; s < steps; ++s) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    lds_barrier();
    if (s + 1 < steps) stage(next, s + 1);
    u32x4 xf[FM], wf[FN];
#pragma unroll
    for (int f = 0; f < FM; ++f) xf[f] = ld16(now + arow0 + f * 1024);
#pragma unroll
    for (int j = 0; j < FN; ++j) wf[j] = ld16(now + brow0 + j * 1024);
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int f = 0; f < FM; ++f) acc[f][j] = mfma_q<Tag>(wf[j], xf[f], acc[f][j]);
    char* const t = now;
    now = next, next = t;
  }
  constexpr int FO = GLU ? FN / 2 : FN;
#pragma unroll
  for (int f = 0; f < FM; ++f) {
    const int pos = row0 + wm * 64 + 16 * f + r16;
    if (pos >= rows_end) continue;
#pragma unroll
    for (int j = 0; j < FO; ++j) {
      float v[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = grouped_act<Tag, ACT>(acc[f][j][r], GLU ? acc[f][j + FN - FO][r] : 0.f, p);
      store4<Tag>(p, pos, n0 + wn * (GLU ? CPW / 2 : CPW) + 16 * j + 4 * q, v);
    }
  }
}

// Steps with a few rows per expert (decode): a stream of the chosen experts' weights.  One wave per 16 rows x 32 weight rows
// (GLU: 16 gate rows and their 16 up rows), operands straight from global memory, kRowsUnroll k-steps of loads in flight.
// Single waves spread evenly over the 1024 SIMDs whatever the number of chosen experts; nothing is shared between them.
constexpr int kRowsUnroll = 8;

template <typename Tag, int ACT>
__global__ void __launch_bounds__(64) moe_grouped_rows_kernel(GroupedArgs p) {
  constexpr bool GLU = ACT >= 2;
  const int lane = threadIdx.x, r16 = lane & 15, q = lane >> 4;
  int e = 0, row0 = 0, rows_end = 0;
  if (!grouped_tile(p.offsets, p.E, 16, (int)blockIdx.y, lane, e, row0, rows_end)) return;
  e = __builtin_amdgcn_readfirstlane(e);
  const int n0 = blockIdx.x * (GLU ? 16 : 32);
  const int pos = min(row0 + r16, rows_end - 1);                 // rows past the end: never stored
  const int64_t arow = p.order ? p.order[pos] / p.row_div : pos;
  const char* xp = p.a + (arow * p.a_stride + 8 * q) * 2;
  const char* wbase = p.w + ((int64_t)e * (GLU ? 2 * p.N : p.N) * p.K + 8 * q) * 2;
  const char* wp[2];
#pragma unroll
  for (int j = 0; j < 2; ++j)
    wp[j] = wbase + (int64_t)(GLU ? j * p.N + min(n0 + r16, p.N - 1) : min(n0 + 16 * j + r16, p.N - 1)) * p.K * 2;
  f32x4_q acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
  const int ksteps = p.K / 32;
  int ks = 0;
  for (; ks + kRowsUnroll <= ksteps; ks += kRowsUnroll) {
    u32x4 wf[kRowsUnroll][2], xf[kRowsUnroll];
#pragma unroll
    for (int u = 0; u < kRowsUnroll; ++u) {
      wf[u][0] = ld16(wp[0] + (ks + u) * 64);
      wf[u][1] = ld16(wp[1] + (ks + u) * 64);
      xf[u] = ld16(xp + (ks + u) * 64);
    }
    __builtin_amdgcn_sched_barrier(0);      // all loads of the round first: the scheduler would trade them for registers
#pragma unroll
    for (int u = 0; u < kRowsUnroll; ++u) {
      acc[0] = mfma_q<Tag>(wf[u][0], xf[u], acc[0]);
      acc[1] = mfma_q<Tag>(wf[u][1], xf[u], acc[1]);
    }
  }
  for (; ks < ksteps; ++ks) {
    const u32x4 xf = ld16(xp + ks * 64);
    acc[0] = mfma_q<Tag>(ld16(wp[0] + ks * 64), xf, acc[0]);
    acc[1] = mfma_q<Tag>(ld16(wp[1] + ks * 64), xf, acc[1]);
  }
  if (row0 + r16 >= rows_end) return;
#pragma unroll
  for (int j = 0; j < (GLU ? 1 : 2); ++j) {
    float v[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = grouped_act<Tag, ACT>(acc[j][r], acc[1][r], p);
    store4<Tag>(p, row0 + r16, n0 + 16 * j + 4 * q, v);
  }
}

// The same with half the weight rows per wave (16; GLU: 8 gate rows and their 8 up rows) and twice the k-steps on their way, where
// narrow_pays below.
constexpr int kNarrowUnroll = 16;

template <typename Tag, int ACT>
__global__ void __launch_bounds__(64) moe_grouped_narrow_rows_kernel(GroupedArgs p) {
  constexpr bool GLU = ACT >= 2;
  const int lane = threadIdx.x, r16 = lane & 15, q = lane >> 4;
  int e = 0, row0 = 0, rows_end = 0;
  if (!grouped_tile(p.offsets, p.E, 16, (int)blockIdx.y, lane, e, row0, rows_end)) return;
  e = __builtin_amdgcn_readfirstlane(e);
  const int n0 = blockIdx.x * (GLU ? 8 : 16);
  const int pos = min(row0 + r16, rows_end - 1);                 // rows past the end: never stored
  const int64_t arow = p.order ? p.order[pos] / p.row_div : pos;
  const char* xp = p.a + (arow * p.a_stride + 8 * q) * 2;
  const char* wp = p.w + ((int64_t)e * (GLU ? 2 * p.N : p.N) * p.K + 8 * q) * 2 +
                   (int64_t)(GLU ? (r16 >> 3) * p.N + min(n0 + (r16 & 7), p.N - 1) : min(n0 + r16, p.N - 1)) * p.K * 2;
  f32x4_q acc = {0.f, 0.f, 0.f, 0.f};
  const int ksteps = p.K / 32;
  int ks = 0;
  for (; ks + kNarrowUnroll <= ksteps; ks += kNarrowUnroll) {
    u32x4 wf[kNarrowUnroll], xf[kNarrowUnroll];
#pragma unroll
    for (int u = 0; u < kNarrowUnroll; ++u) {
      wf[u] = ld16(wp + (ks + u) * 64);
      xf[u] = ld16(xp + (ks + u) * 64);
    }
    __builtin_amdgcn_sched_barrier(0);      // all loads of the round first: the scheduler would trade them for registers
#pragma unroll
    for (int u = 0; u < kNarrowUnroll; ++u) acc = mfma_q<Tag>(wf[u], xf[u], acc);
  }
  for (; ks < ksteps; ++ks) acc = mfma_q<Tag>(ld16(wp + ks * 64), ld16(xp + ks * 64), acc);
  float v[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const float up = GLU ? __shfl_xor(acc[r], 32, 64) : 0.f;     // (gates in the lanes below 32, their up sums 32 above)
    v[r] = grouped_act<Tag, ACT>(acc[r], up, p);
  }
  if (row0 + r16 >= rows_end || (GLU && lane >= 32)) return;
  store4<Tag>(p, row0 + r16, n0 + 4 * q, v);
}

// Half the weight rows per wave, of a product with `blocks` column blocks of the wider kernel:
//   * at most one wave per compute unit, were every pair another expert's: units are idle.  us of the up and down product, wider -> narrow,
//     top 4 of 32 experts: 1 token of 2048 x 1024 (256 waves each) 10.7 + 6.8 -> 10.0 + 6.2, of 1024 x 512 (128 waves) 6.7 + 4.1 -> 5.4 + 3.5;
//   * one to one and a half waves per SIMD (four to a unit) of the experts that so many pairs are expected to choose: the SIMDs with a second
//     wave set the time, and half a wave more does less to them.  Layers, mean of 8 routings (single ones 0.91 - 1.07): 32 experts of
//     2048 x 1024, 6 - 8 tokens 59.9 -> 58.9, 64 experts, top 4, 6 tokens 61.5 -> 60.8, of 1024 x 512, top 8, 8 tokens 43.8 -> 43.2.
// Elsewhere the second reading of x's rows costs as much as the evener shares give, or more: 2 tokens of 2048 x 1024 (512 waves) 13.3 + 7.8
// -> 15.4 + 8.2; 64 experts, top 8, 4 tokens (1660) 80.3 -> 85.5; 16 tokens of 32 experts 39.2 + 21.3 -> 44.1 + 23.0.
static bool narrow_pays(int pairs, int experts, int blocks) {
  if (pairs > experts) return false;
  const double chosen = experts * (1. - pow(1. - 1. / experts, pairs)) * blocks;
  return (long)pairs * blocks <= 256 || (chosen > 1024. && chosen <= 1536.);
}

// Which kernel: by the mean rows per expert, pairs / experts (the counts themselves are on the device).  The rows kernel up to a mean of
//   * 0 - it reads half a line at a time, the ring's loads whole ones past the L2 - where the chosen experts' weights are a stream out of HBM (220 MB and
//     700 tiles of 64 weight rows): width 4096, 128 experts of ff 1536, 2 / 4 / 16 tokens, top 8: 70 + 33 | 63 + 33, 134 + 62 | 114 + 58, 366 + 173 | 309 + 151;
//     8 of 14336, 2 / 6 tokens, top 2, up 137 | 117, 303 | 265; with fewer tiles 1 token of the former, up 37.5 | 39.7, of the latter, down 45 | 64;
//   * 1.5.  Width 2048, 16 experts of ff 1408, up + down in us, rows kernel | ring tiles: mean 2: 44 + 18 | 40 + 18, 4: 43 + 19 | 39 + 18, 10: 43 + 19 |
//     38 + 18; 32 experts of ff 1024, 3: 63 + 27 | 55 + 24, 16: 67 + 28 (64-row tiles) | 55 + 23; 128 of 512, width 1024, 4: 50 + 28 | 45 + 26;
//   * 10 where it is at most one wave per SIMD: width 1024, 16 experts of ff 512, mean 2: 9.2 + 6.7 | 10.5 + 7.3, 10: 10.0 + 7.0 | 10.5 + 7.7; 32 experts,
//     2 - 8: 14.5 + 9.2 | 15.0 + 9.6; 8 of 1536, width 2048, 2: 24.6 + 11.5 | 26.4 + 12.7, 10: 22.9 + 12.3 | 23.7 + 12.1 - and 12: 35 + 20 | 24 + 12;
//   * 10 where the ring does not take the product (K no multiple of 64, 2^31 bytes of offsets), the 64-row tiles from there, the 128-row tiles from 56.
// Else the ring tiles, the tile by ring_tile, and from a mean of 320 rows on the wide kernel for gated products (its comment has both sides) and for
// what the ring does not take (K of 1056, 512 rows: 379 by the 128-row tiles, 337 by it, both of K 1024).
// The mean says nothing of a skewed step: a row tile chosen for the mean may be taller than most experts' rows, or one row too short for some.  Over 350
// sizes (4 to 256 experts, widths 1024 to 7168, means 1 to 2000), each routed evenly, by expert weights of spread e^0.5 and by 1 / rank, against the
// kernels before (64 x 128, 128 x 128 and 128 x 256 tiles, one wave per 16 rows): up products 1.16 and down products 1.16 times as fast on average, one in
// twenty more than 5 % slower (0.60 - 0.95; 16 experts, width 2560, mean 135, by 1 / rank: 18 -> 30), most of them at means just below a tile's height.
// No choice by sizes alone does better: costs fitted to uneven routings, or expected counts spread by any width, lose as often.  Every pair on
// top_k experts, both products together: 32 experts of ff 1024, 24 tokens 25.4 -> 29.2, 48: 33.3 -> 22.5, 200: 42.2 -> 31.8; 128 of 1536, width 4096,
// 200: 114 -> 143, 800: 405 -> 316.
// (sizes alone: the plan is the same for every step of them)
enum : int { kGroupedRows = 0, kGroupedNarrow = 1, kGrouped64 = 2, kGrouped128 = 3, kGroupedWide = 4, kGroupedRing = 16 };      // + its tile
inline int grouped_plan(bool gated, bool ordered, int row_div, int pairs, int n, int k, int experts, int64_t a_stride) {
  const int held = pairs < experts ? pairs : experts;           // experts with a row, at most
  const int row_tiles = pairs / 16 + held;
  // (moe_align takes 4096 experts, 6656 tiles; more than a grid's second dimension holds go to the 64-row tiles)
  // (a ring's loads have 32-bit offsets from the operand's first byte; rows further on that an order names: far_product)
  const int64_t last_row = ordered ? (int64_t)pairs / row_div + 1 : pairs, wide_rows = (gated ? 2 : 1) * (int64_t)n;
  const bool ring = k % 64 == 0 && last_row * a_stride < (int64_t)1 << 31 && wide_rows * k < (int64_t)1 << 31;
  const int blocks_of_rows = (n + (gated ? 15 : 31)) / (gated ? 16 : 32);
  const double wrows = experts * (1. - exp(-(double)pairs / experts)) * wide_rows;                  // of the experts expected to be chosen
  const bool streams = wrows * k >= 110e6 && wrows >= 700. * 64.;
  const int most = !ring ? 20 : streams ? 0 : (int64_t)experts * blocks_of_rows > 1024 ? 3 : 20;      // half rows per expert
  if (2 * (int64_t)pairs <= most * (int64_t)experts && row_tiles <= 65535) return narrow_pays(pairs, experts, blocks_of_rows) ? kGroupedNarrow : kGroupedRows;
  if (pairs > 320 * (int64_t)experts && (gated || !ring)) return kGroupedWide;
  if (ring) return kGroupedRing + ring_tile(pairs, experts, wide_rows, k);
  return pairs > 56 * (int64_t)experts ? kGrouped128 : kGrouped64;
}

template <typename Tag, int ACT>
int launch_grouped_mfma(const GroupedArgs& p, int pairs, hipStream_t st) {
  const int held = pairs < p.E ? pairs : p.E;
  const int plan = grouped_plan(ACT >= 2, p.order, p.row_div, pairs, p.N, p.K, p.E, p.a_stride);
  if (plan == kGroupedRows || plan == kGroupedNarrow) {
    const int per = (ACT >= 2 ? 16 : 32) / (plan == kGroupedNarrow ? 2 : 1);
    const dim3 grid((unsigned)((p.N + per - 1) / per), (unsigned)(pairs / 16 + held));
    if (plan == kGroupedNarrow) moe_grouped_narrow_rows_kernel<Tag, ACT><<<grid, 64, 0, st>>>(p);
    else moe_grouped_rows_kernel<Tag, ACT><<<grid, 64, 0, st>>>(p);
    SP_LAUNCH_CHECK();
    return SP_OK;
  }
  if (plan >= kGroupedRing) {
#define SP_RING_CASE(I, TWO, ONE, FIXED, ONCE, ...) \
  case I: return launch_grouped_ring<Tag, RingTile<__VA_ARGS__>, ONCE, ACT>(p, pairs, held, st);
    switch (plan - kGroupedRing) { SP_RING_TILES(SP_RING_CASE) }
    return SP_ERR_INVALID_ARG;
  }
  const int bm = plan == kGrouped64 ? 64 : 128, bn = plan == kGroupedWide ? kWideBN : kGroupedBN, per = ACT >= 2 ? bn / 2 : bn;
  const int64_t ntiles = (p.N + per - 1) / per;
  const dim3 blocks((unsigned)(((pairs / bm + held) * ntiles + 7) / 8 * 8));
  if (plan == kGroupedWide) {
    constexpr int lds = 2 * (kWideBM + kWideBN) * kWideBK * 2;
    static PerDevice<int> raised;
    int ok = 0;
    raised.get(ok, [&](int) {
      return hipFuncSetAttribute((const void*)moe_grouped_wide_kernel<Tag, ACT>, hipFuncAttributeMaxDynamicSharedMemorySize, lds) ==
             hipSuccess ? 1 : 0;
    });
    if (!ok) return SP_ERR_LAUNCH;
    moe_grouped_wide_kernel<Tag, ACT><<<blocks, 256, lds, st>>>(p);
  } else if (plan == kGrouped128) {
    moe_grouped_tile_kernel<Tag, 128, ACT><<<blocks, 256, 0, st>>>(p);
  } else {
    moe_grouped_tile_kernel<Tag, 64, ACT><<<blocks, 256, 0, st>>>(p);
  }
  SP_LAUNCH_CHECK();
  return SP_OK;
}

// GroupedArgs::far: all of a row below 2^31 / a_stride is within 2^32 bytes of the first one's beginning
inline int32_t far_pairs(int row_div, int64_t a_stride) {
  return (int32_t)std::min<int64_t>((((int64_t)1 << 31) / a_stride) * row_div, INT32_MAX);
}

// ---- y = g' * sigmoid(alpha g') * (u' + 1), g' = min(g, limit), u' = clamp(u, -limit, limit); gu = [g | u] per row -----
template <typename Tag>
__global__ void moe_glu_kernel(void* out, const void* gu, int64_t P, int F, float limit, float alpha) {
  typedef Elem<Tag> El;
  const int64_t n = P * (int64_t)F;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t p = i / F;
    const int f = (int)(i % F);
    El::store(out, i, moe_glu_value<Tag>(El::load(gu, p * 2 * F + f), El::load(gu, p * 2 * F + F + f), limit, alpha));
  }
}

// ---- out[t] = sum_k weights[t, k] * z[place[t * top + k]] ----------------------------------------------------------
// A thread holds V neighbouring columns of a token (V = 16 bytes where the rows allow it, else 1): the rows of up to
// kCombineAhead experts are in flight together, added in the order of k.
constexpr int kCombineAhead = 4;

template <typename Tag, int V>
__global__ void __launch_bounds__(kBlock)
moe_combine_kernel(void* out, const void* z, const int32_t* place, const float* weights, int width, int top,
                   int64_t out_stride) {
  typedef Elem<Tag> El;
  const int64_t t = blockIdx.x;
  const int i = (blockIdx.y * kBlock + threadIdx.x) * V;
  if (i >= width) return;
  float acc[V];
#pragma unroll
  for (int c = 0; c < V; ++c) acc[c] = 0.f;
  for (int k0 = 0; k0 < top; k0 += kCombineAhead) {
    const int n = min(top - k0, kCombineAhead);
    float zv[kCombineAhead][V], w[kCombineAhead];
#pragma unroll
    for (int k = 0; k < kCombineAhead; ++k) {
      const int64_t at = t * top + k0 + min(k, n - 1);
      w[k] = weights[at];
      const int64_t row = (int64_t)place[at] * width + i;
      if constexpr (V == 1) zv[k][0] = El::load(z, row);
      else unpack16<Tag>(ld16((const char*)z + row * El::kBytes), zv[k]);
    }
#pragma unroll
    for (int k = 0; k < kCombineAhead; ++k)
      if (k < n) {
#pragma unroll
        for (int c = 0; c < V; ++c) acc[c] += w[k] * zv[k][c];
      }
  }
  if constexpr (V == 1) El::store(out, t * out_stride + i, acc[0]);
  else st16((char*)out + (t * out_stride + i) * El::kBytes, pack16<Tag>(acc));
}

template <typename Tag>
int launch_combine(void* out, const void* z, const int32_t* place, const float* weights, int64_t T, int width, int top,
                   int64_t out_stride, hipStream_t st) {
  constexpr int V = Elem<Tag>::kVec;
  if (width % V == 0 && out_stride % V == 0 && ((uintptr_t)out & 15) == 0 && ((uintptr_t)z & 15) == 0)
    moe_combine_kernel<Tag, V><<<dim3((unsigned)T, (unsigned)((width / V + kBlock - 1) / kBlock)), kBlock, 0, st>>>(
        out, z, place, weights, width, top, out_stride);
  else
    moe_combine_kernel<Tag, 1><<<dim3((unsigned)T, (unsigned)((width + kBlock - 1) / kBlock)), kBlock, 0, st>>>(
        out, z, place, weights, width, top, out_stride);
  SP_LAUNCH_CHECK();
  return SP_OK;
}

}  // namespace
}  // namespace sp

using namespace sp;

extern "C" int sp_moe_route(int32_t* ids, float* weights, const void* x, int64_t x_stride, const float* router,
                            const float* correction, int64_t num_tokens, int width, int experts, int top, int groups,
                            int keep, int dtype, void* stream) {
  SP_CHECK_ARG(num_tokens >= 0 && width > 0 && experts > 0 && top > 0 && top <= experts);
  SP_CHECK_ARG(groups >= 1 && keep >= 1 && keep <= groups && experts % groups == 0);
  SP_CHECK_ARG((int64_t)top <= (int64_t)keep * (experts / groups));
  if (num_tokens == 0) return SP_OK;
  SP_CHECK_ARG(ids && weights && x && router && correction && x_stride >= width);
  const size_t lds = 4 * (size_t)(2 * experts + groups) * sizeof(float);
  if (lds > 64 * 1024) return SP_ERR_UNSUPPORTED;
  SP_DISPATCH_DTYPE(dtype, (moe_route_kernel<Tag><<<dim3((unsigned)((num_tokens + 3) / 4)), 256, lds, (hipStream_t)stream>>>(
                               ids, weights, x, x_stride, router, correction, num_tokens, width, experts, top, groups, keep)));
  SP_LAUNCH_CHECK();
  return SP_OK;
}

extern "C" int sp_moe_softmax_topk(int32_t* ids, float* weights, float* gate, const float* logits, int64_t logits_stride,
                                   const float* correction, int64_t num_tokens, int experts, int top, int groups, int keep,
                                   float scale, int renorm, void* stream) {
  SP_CHECK_ARG(num_tokens >= 0 && experts > 0 && top > 0 && top <= experts);
  SP_CHECK_ARG(groups >= 1 && keep >= 1 && keep <= groups && experts % groups == 0);
  SP_CHECK_ARG((int64_t)top <= (int64_t)keep * (experts / groups));
  if (num_tokens == 0) return SP_OK;
  SP_CHECK_ARG(ids && weights && logits && logits_stride >= experts + (gate ? 1 : 0));
  const size_t lds = 4 * (size_t)(2 * experts + groups) * sizeof(float);
  if (lds > 64 * 1024) return SP_ERR_UNSUPPORTED;
  moe_softmax_topk_kernel<<<dim3((unsigned)((num_tokens + 3) / 4)), 256, lds, (hipStream_t)stream>>>(
      ids, weights, gate, logits, logits_stride, correction, num_tokens, experts, top, groups, keep, scale, renorm);
  SP_LAUNCH_CHECK();
  return SP_OK;
}

extern "C" int sp_moe_align(int32_t* offsets, int32_t* order, int32_t* place, const int32_t* ids, int pairs, int experts,
                            void* stream) {
  SP_CHECK_ARG(pairs >= 0 && experts > 0 && experts <= 4096);
  SP_CHECK_ARG(offsets && (pairs == 0 || (order && place && ids)));
  // (at most 32 + 32 KB)
  const size_t lds = 2 * (size_t)experts * sizeof(int32_t) + (pairs <= kAlignPairs ? (size_t)pairs * sizeof(uint16_t) : 0);
  moe_align_kernel<<<1, kAlignThreads, lds, (hipStream_t)stream>>>(offsets, order, place, ids, pairs, experts);
  SP_LAUNCH_CHECK();
  return SP_OK;
}

extern "C" int sp_moe_grouped_gemm(void* out, const void* a, const void* w, const int32_t* offsets, const int32_t* order,
                                   int row_div, int pairs, int n, int k, int experts, int64_t a_stride,
                                   int64_t out_stride, int act, int dtype, void* stream) {
  SP_CHECK_ARG(pairs >= 0 && n > 0 && k > 0 && experts > 0 && row_div >= 1 && (act == 0 || act == 1));
  if (pairs == 0) return SP_OK;
  SP_CHECK_ARG(out && a && w && offsets && a_stride >= k && out_stride >= n);
  const bool aligned = k % 32 == 0 && a_stride % 8 == 0 && ((uintptr_t)a & 15) == 0 && ((uintptr_t)w & 15) == 0;
  if ((dtype == SP_BF16 || dtype == SP_F16) && aligned) {
    const GroupedArgs p{(char*)out, (const char*)a, (const char*)w, offsets, order, row_div, n, k, experts, a_stride, out_stride,
                        out_stride % 4 == 0 && ((uintptr_t)out & 7) == 0, 0.f, 0.f, far_pairs(row_div, a_stride)};
    hipStream_t st = (hipStream_t)stream;
    if (dtype == SP_BF16)
      return act ? launch_grouped_mfma<bf16_tag, 1>(p, pairs, st) : launch_grouped_mfma<bf16_tag, 0>(p, pairs, st);
    return act ? launch_grouped_mfma<f16_tag, 1>(p, pairs, st) : launch_grouped_mfma<f16_tag, 0>(p, pairs, st);
  }
  const dim3 grid((unsigned)((pairs + GM - 1) / GM + experts), (unsigned)((n + GN - 1) / GN));
  SP_DISPATCH_DTYPE(dtype, (moe_grouped_gemm_kernel<Tag><<<grid, 256, 0, (hipStream_t)stream>>>(
                               out, a, w, offsets, order, row_div, pairs, n, k, experts, a_stride, out_stride, act)));
  SP_LAUNCH_CHECK();
  return SP_OK;
}

extern "C" int sp_moe_grouped_glu(void* out, const void* a, const void* w, const int32_t* offsets, const int32_t* order,
                                  int row_div, int pairs, int ff, int k, int experts, int64_t a_stride, int64_t out_stride,
                                  int act, float limit, float alpha, int dtype, void* stream) {
  SP_CHECK_ARG(pairs >= 0 && ff > 0 && k > 0 && experts > 0 && row_div >= 1 && (act == 0 || act == 1));
  if (pairs == 0) return SP_OK;
  SP_CHECK_ARG(out && a && w && offsets && a_stride >= k && out_stride >= ff);
  if (dtype != SP_BF16 && dtype != SP_F16) return SP_ERR_UNSUPPORTED;
  if (k % 32 || a_stride % 8 || ((uintptr_t)a & 15) || ((uintptr_t)w & 15)) return SP_ERR_UNSUPPORTED;
  const GroupedArgs p{(char*)out, (const char*)a, (const char*)w, offsets, order, row_div, ff, k, experts, a_stride, out_stride,
                      out_stride % 4 == 0 && ((uintptr_t)out & 7) == 0, limit, alpha, far_pairs(row_div, a_stride)};
  hipStream_t st = (hipStream_t)stream;
  if (dtype == SP_BF16)
    return act ? launch_grouped_mfma<bf16_tag, 3>(p, pairs, st) : launch_grouped_mfma<bf16_tag, 2>(p, pairs, st);
  return act ? launch_grouped_mfma<f16_tag, 3>(p, pairs, st) : launch_grouped_mfma<f16_tag, 2>(p, pairs, st);
}

extern "C" int sp_moe_grouped_plan(int gated, int row_div, int pairs, int n, int k, int experts, int64_t a_stride) {
  if (pairs <= 0 || n <= 0 || k <= 0 || k % 32 || experts <= 0 || row_div < 0 || a_stride < k || a_stride % 8) return -1;
  return grouped_plan(gated != 0, row_div > 0, row_div, pairs, n, k, experts, a_stride);
}

extern "C" int sp_moe_glu(void* out, const void* gu, int64_t pairs, int ff, float limit, float alpha, int dtype,
                          void* stream) {
  SP_CHECK_ARG(pairs >= 0 && ff > 0);
  if (pairs == 0) return SP_OK;
  SP_CHECK_ARG(out && gu);
  int64_t blocks = (pairs * ff + kBlock - 1) / kBlock;
  if (blocks > 4096) blocks = 4096;
  SP_DISPATCH_DTYPE(dtype, (moe_glu_kernel<Tag><<<dim3((unsigned)blocks), kBlock, 0, (hipStream_t)stream>>>(out, gu, pairs, ff,
                                                                                                         limit, alpha)));
  SP_LAUNCH_CHECK();
  return SP_OK;
}

extern "C" int sp_moe_combine(void* out, const void* z, const int32_t* place, const float* weights, int64_t num_tokens,
                              int width, int top, int64_t out_stride, int dtype, void* stream) {
  SP_CHECK_ARG(num_tokens >= 0 && width > 0 && top > 0);
  if (num_tokens == 0) return SP_OK;
  SP_CHECK_ARG(out && z && place && weights && out_stride >= width);
  SP_DISPATCH_DTYPE(dtype, return (launch_combine<Tag>(out, z, place, weights, num_tokens, width, top, out_stride,
                                                       (hipStream_t)stream)));
}
