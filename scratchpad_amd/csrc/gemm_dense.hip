// out[M, N] = x[M, K] . w[N, K]^T for steps of 17 - 256 rows (a server's decode batch, a short prompt; to 1024 rows where K is long and twice N)
// and of 5 - 16 rows over large weights, 16-bit types.
//
// Call sites: the projections of every layer and the LM head (QKVParallelLinear / RowParallelLinear / MergedColumnParallelLinear.forward,
// nn/layers/linear.py:696-760, 423-470, 1033-1155 -> F.linear; LogitsProcessor._get_logits, nn/layers/logits_processor.py:340-376).
//
// What bounds it: at 64 rows a product is still a stream of its weights, at 256 rows the matrix cores need half the stream's time.
// The library's kernels for these sizes are tiles of 128 - 256 rows without a split of K: too few workgroups to pull the weights
// in (4096 x 14336 at 128 rows: 32 tiles), or rows computed for nothing.  Here
//   * the tile follows the rows (16 - 256) and is narrow (16 - 128 weight rows), so that about one workgroup per compute unit streams;
//     where K is long, its shares go to workgroups of their own and a second launch adds them (2 us + the sums' traffic);
//   * both operands go to LDS by direct loads, into rings of steps; up to about 128 rows the first waves load x, the others w, each with its own count of
//     steps in flight (loads retire in order: in one wave, x out of the L2 would wait behind weights out of HBM);
//   * weights are loaded past the L2 (nt): a stream of 235 MB takes 37 us with it and 42 without;
//   * a step is one barrier, in front of its last products: the next step's first operands are read behind it, under them;
//   * small tiles split every 64 of k over two groups of waves (WK): twice the waves to hide LDS behind, one exchange at the end.
// From about 128 rows on the matrix cores and the stream take as long as each other, and a wave's direct loads hold its products up: there
// dense_wide_kernel, whose waves all load both operands and spread the loads between their products (the best tile and shares of dense_kernel and
// of it: 28672 x 4096 at 256 rows 106 and 65 us; 4096 x 14336 58.9 and 45.6, at 640 rows 113 and 78; 2048 x 8192 23.9 and 22.7).
// us under graph replay, cold weights, library -> this, as it is planned:
//                                                         rows 17           64           128          256
//   3072 x 2048 (qkv, hidden 2048)                          8.9 ->  7.6   9.5 ->  7.8   12.1 ->  9.6   11.0 -> 12.2
//   2048 x 2048                                             8.6 ->  7.4   9.2 ->  7.5    8.8 ->  7.5    9.8 ->  9.6
//   16384 x 2048 (gate and up)                             18.6 -> 16.2  18.3 -> 17.0   22.4 -> 20.7   30.6 -> 26.1
//   2048 x 8192 (down)                                     14.2 -> 12.2  22.5 -> 13.9   21.4 -> 17.3   26.9 -> 21.4
//   6144 x 4096 (qkv, hidden 4096)                         16.3 -> 13.4  18.3 -> 17.0   25.4 -> 21.3   41.0 -> 28.3
//   4096 x 4096                                            14.2 -> 11.9  15.3 -> 12.6   24.7 -> 16.2   22.9 -> 20.4
//   28672 x 4096                                           55.4 -> 48.5  54.7 -> 48.6   60.3 -> 53.1   74.2 -> 66.2
//   4096 x 14336                                           30.0 -> 23.8  38.9 -> 28.6   76.2 -> 34.2   61.2 -> 47.5
// 5 / 8 / 16 rows (the library or sp_gemm_skinny, whichever was faster): 28672 x 4096 49 -> 42, 54 -> 43, 61 -> 44; 128256 x 4096 190 -> 161,
// 193 -> 162, 193 -> 164.  From 512 rows on the library's 256 x 256 tiles are 10 - 30 % faster where N is large.
#include "lds_ring.h"

namespace sp {
namespace {

struct DenseArgs {
  char* out;
  float* part;                        // [splits][M][N] sums of the shares of K, when there is more than one
  const char* x;
  const char* w;
  int M, N, K, splits, mblocks, nblocks;   // N: output columns
  int64_t x_stride, w_stride, out_stride;  // elements
  int vec;                            // 4 neighbouring output columns are one aligned store
};

// BM x BN outputs per workgroup, BK of k a step, WK x WM x WN waves, the first WX of which load x and the others w; SX and SW steps of
// x and w in LDS
template <int BM_, int BN_, int BK_, int WK_, int WM_, int WN_, int WX_, int SX_, int SW_>
struct Tile {
  static constexpr int BM = BM_, BN = BN_, BK = BK_, WK = WK_, WM = WM_, WN = WN_, WX = WX_, SX = SX_, SW = SW_;
  static constexpr int kWaves = WK * WM * WN, kX = BM * BK * 2, kW = BN * BK * 2;
  static constexpr int kRing = SX * kX + SW * kW, kSums = WK > 1 ? BM * BN * 4 : 0;
  static constexpr int kLds = kRing > kSums ? kRing : kSums;
  static constexpr int kOcc = kLds <= 80 * 1024 && kWaves <= 4 ? 2 : kWaves / 4;      // waves per SIMD
};

// acc[f][j][r] = out[row 16 f + lane % 16][column 16 j + 4 (lane / 16) + r] of a wave's FM x FN tiles at m0, n0 (EPI: the lanes below 32 the gate
// sums of column 8 j + 4 q + r, the lanes 32 above them its up sums)
template <typename Tag, int FM, int FN, int EPI, bool SPLIT>
__device__ __forceinline__ void dense_store(const DenseArgs& p, const ring_f32x4 (&acc)[FM][FN], int m0, int n0, int split, int lane) {
  typedef Elem<Tag> E;
  const int r16 = lane & 15, q = lane >> 4;
#pragma unroll
  for (int f = 0; f < FM; ++f) {
    const int m = m0 + 16 * f + r16;
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const int n = n0 + (EPI ? 8 : 16) * j + 4 * q;
      const bool mine = m < p.M && n < p.N && !(EPI && q >= 2);
      if constexpr (SPLIT) {
        float* const to = p.part + ((int64_t)split * p.M + m) * p.N + n;
        if (mine && p.vec) *(ring_f32x4*)to = acc[f][j];
        else if (mine)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (n + r < p.N) to[r] = acc[f][j][r];
      } else {
        uint32_t h[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float v = acc[f][j][r];
          if constexpr (EPI) {
            const auto both = __builtin_amdgcn_permlane32_swap(as_u32(v), as_u32(v), false, false);      // lanes 0-31 twice, 32-63 twice
            v = mul_round<Tag>(E::round(silu_ref(E::round(v))), E::round(as_f32(both[1])));
          }
          if constexpr (std::is_same<Tag, bf16_tag>::value) h[r] = f32_to_bf16_bits(v);
          else h[r] = f32_to_f16_bits(v);
        }
        char* const to = p.out + ((int64_t)m * p.out_stride + n) * 2;
        if (mine && p.vec) *(u32x2*)to = u32x2{h[0] | h[1] << 16, h[2] | h[3] << 16};
        else if (mine)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (n + r < p.N) ((uint16_t*)to)[r] = (uint16_t)h[r];
      }
    }
  }
}

// EPI: 0 the product; 1 w is [2 N, K], gate rows then up rows, and the output silu(gate) * up of the rounded sums
template <typename Tag, typename T, int EPI, bool SPLIT>
__global__ void __launch_bounds__(T::kWaves * 64, T::kOcc) dense_kernel(DenseArgs p) {
  constexpr int RB = T::BK * 2, RPL = 1024 / RB, CH = T::BK / 8;          // bytes of a row, rows and chunks of 16 bytes a load
  constexpr int TM = T::BM / T::WM, TN = T::BN / T::WN, FM = TM / 16, FN = TN / 16, KS = T::BK / 32 / T::WK;
  constexpr int GX = T::BM / RPL, GW = T::BN / RPL, WW = T::kWaves - T::WX;
  constexpr int LX = (GX + T::WX - 1) / T::WX, LW = (GW + WW - 1) / WW, LM = LX > LW ? LX : LW;
  static_assert(T::BM % RPL == 0 && T::BN % RPL == 0 && TM % 16 == 0 && TN % 16 == 0 && T::BK % (64 * T::WK) == 0 && T::WK <= 2, "tile");
  static_assert(LX * (T::SX - 1) <= 63 && LW * (T::SW - 1) <= 63 && T::SX >= 2 && T::SW >= 2 && T::kLds <= 160 * 1024, "ring");
  extern __shared__ __attribute__((aligned(1024))) char dense_lds[];
  char* const lds = dense_lds;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, r16 = lane & 15, q = lane >> 4;
  const int total = p.mblocks * p.nblocks * p.splits, share = (total + 7) / 8;
  const int idx = (int)(blockIdx.x >> 3), t = (int)(blockIdx.x & 7) * share + idx;
  if (idx >= share || t >= total) return;
  const int mb = t % p.mblocks, split = t / p.mblocks % p.splits, nb = t / (p.mblocks * p.splits);
  const int m0 = mb * T::BM, n0 = nb * (EPI ? T::BN / 2 : T::BN);
  const int ksteps = p.K / T::BK, first = ksteps * split / p.splits, steps = ksteps * (split + 1) / p.splits - first;
  const int wk = wave / (T::WM * T::WN), wmn = wave % (T::WM * T::WN), wm = wmn / T::WN, wn = wmn % T::WN;
  const bool loads_x = wave < T::WX;
  // this wave's direct loads: lane -> row lane / CH of a load's rows, chunk lane % CH of LDS
  uint32_t off[LM];
#pragma unroll
  for (int i = 0; i < LM; ++i) {
    const int g = loads_x ? min(wave * LX + i, GX - 1) : min((wave - T::WX) * LW + i, GW - 1);
    const int r = g * RPL + lane / CH, chunk = (lane % CH) ^ (r & 7);
    int row;                                             // rows and columns past the end: the last one again, never stored
    if (loads_x) {
      row = min(m0 + r, p.M - 1);
    } else if constexpr (EPI) {
      const int in = r % 16;                             // 8 gate rows, then the up rows of the same 8 columns
      row = min(n0 + r / 16 * 8 + in % 8, p.N - 1) + (in >= 8 ? p.N : 0);
    } else {
      row = min(n0 + r, p.N - 1);
    }
    off[i] = (uint32_t)row * (uint32_t)((loads_x ? p.x_stride : p.w_stride) * 2) + chunk * 16;
  }
  const char* const src = (loads_x ? p.x : p.w) + (int64_t)first * RB;
  const uint32_t lds0 = lds_address(lds);
  const auto stage_x = [&](int s, int buf) {
#pragma unroll
    for (int i = 0; i < LX; ++i) ring_load<false>(off[i], src + (int64_t)s * RB, lds0 + buf + min(wave * LX + i, GX - 1) * 1024);
  };
  const auto stage_w = [&](int s, int buf) {
#pragma unroll
    for (int i = 0; i < LW; ++i)
      ring_load<true>(off[i], src + (int64_t)s * RB, lds0 + T::SX * T::kX + buf + min((wave - T::WX) * LW + i, GW - 1) * 1024);
  };
  ring_f32x4 acc[FM][FN];
#pragma unroll
  for (int f = 0; f < FM; ++f)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[f][j] = ring_f32x4{0.f, 0.f, 0.f, 0.f};
  const int arow = (wm * TM + r16) * RB, brow = T::SX * T::kX + (wn * TN + r16) * RB;
  u32x4 xf[2][FM], wf[2][FN];
  const auto read = [&](int bx, int bw, int kk, int to) {
    const int c = ((kk * 4 + q) ^ (r16 & 7)) * 16;
#pragma unroll
    for (int j = 0; j < FN; ++j) wf[to][j] = ld16(lds + bw + brow + j * 16 * RB + c);
#pragma unroll
    for (int f = 0; f < FM; ++f) xf[to][f] = ld16(lds + bx + arow + f * 16 * RB + c);
  };
  if (loads_x) {
    for (int s = 0; s < T::SX && s < steps; ++s) stage_x(s, s * T::kX);
    ring_wait<LX, T::SX - 1>(steps - 1);
  } else {
    for (int s = 0; s < T::SW && s < steps; ++s) stage_w(s, s * T::kW);
    ring_wait<LW, T::SW - 1>(steps - 1);
  }
  ring_barrier();
  read(0, 0, wk, 0);
  int cx = 0, cw = 0;
  // a step's products, behind the reads of the next one's first operands
  for (int s = 0; s < steps; ++s) {
    const int nx = cx == (T::SX - 1) * T::kX ? 0 : cx + T::kX, nw = cw == (T::SW - 1) * T::kW ? 0 : cw + T::kW;
#pragma unroll
    for (int j = 0; j < KS; ++j) {
      const int at = j & 1;
      if (j < KS - 1) {
        read(cx, cw, (j + 1) * T::WK + wk, at ^ 1);
      } else if (s + 1 < steps) {
        // the step's last operands are in registers: when every wave is here its buffers are free, and the next step's are full
        if (loads_x) ring_wait<LX, T::SX - 2>(steps - 2 - s);
        else ring_wait<LW, T::SW - 2>(steps - 2 - s);
        ring_barrier();
        if (loads_x) {
          if (s + T::SX < steps) stage_x(s + T::SX, cx);
        } else if (s + T::SW < steps) {
          stage_w(s + T::SW, cw);
        }
        read(nx, nw, wk, at ^ 1);
      }
#pragma unroll
      for (int n = 0; n < FN; ++n)
#pragma unroll
        for (int f = 0; f < FM; ++f) acc[f][n] = mfma32<Tag>(wf[at][n], xf[at][f], acc[f][n]);
    }
    cx = nx, cw = nw;
  }
  if constexpr (T::WK > 1) {                              // the two halves of every 64 of k meet in LDS, the first wave's plus the second's
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    ring_barrier();
    ring_f32x4* const sums = (ring_f32x4*)lds + wmn * FM * FN * 64 + lane;
    if (wk) {
#pragma unroll
      for (int f = 0; f < FM; ++f)
#pragma unroll
        for (int n = 0; n < FN; ++n) sums[(f * FN + n) * 64] = acc[f][n];
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    ring_barrier();
    if (wk) return;
#pragma unroll
    for (int f = 0; f < FM; ++f)
#pragma unroll
      for (int n = 0; n < FN; ++n) acc[f][n] += sums[(f * FN + n) * 64];
  }
  dense_store<Tag, FM, FN, EPI, SPLIT>(p, acc, m0 + wm * TM, n0 + wn * (EPI ? TN / 2 : TN), split, lane);
}

// The same by ring_product's loop, for more rows: every wave loads both operands, its loads spread between its products.  Past the L2 only the weights of
// an unsplit product with one row block: at 256 rows 28672 x 4096 66 us with it and 72 without, 4096 x 14336 in 8 shares (the fastest
// there; four of 128 x 128 tiles are planned) 44 and 45, at 192 41 and 39.
// Four row blocks share the columns they pass: their rows of x and a few columns stay in an XCD's L2.
constexpr int kRowGroup = 4;

template <typename Tag, typename T, int EPI, bool SPLIT>
__global__ void __launch_bounds__(T::W * 64, T::kWaves) dense_wide_kernel(DenseArgs p) {
  extern __shared__ __attribute__((aligned(1024))) char dense_lds[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int total = p.mblocks * p.nblocks * p.splits, share = (total + 7) / 8;
  const int idx = (int)(blockIdx.x >> 3), at = (int)(blockIdx.x & 7) * share + idx;
  if (idx >= share || at >= total) return;
  const int blocks = p.mblocks * p.nblocks, split = at / blocks, t = at % blocks;
  const int group = t / (kRowGroup * p.nblocks), high = min(kRowGroup, p.mblocks - group * kRowGroup), in = t - group * kRowGroup * p.nblocks;
  const int m0 = (group * kRowGroup + in % high) * T::BM, n0 = in / high * (EPI ? T::BN / 2 : T::BN);
  const int ksteps = p.K / T::BK, first = ksteps * split / p.splits, steps = ksteps * (split + 1) / p.splits - first;
  uint32_t off[T::L];
  const char* base[T::L];
#pragma unroll
  for (int i = 0; i < T::L; ++i) {
    const int g = min(i * T::W + wave, T::G - 1), r = g * T::RPL + lane / T::CH, chunk = (lane % T::CH) ^ (r & 7);
    const bool is_x = g * T::RPL < T::BM;
    int row;                                               // rows and columns past the end: the last one again, never stored
    if (is_x) {
      row = min(m0 + r, p.M - 1);
    } else if constexpr (EPI) {
      const int pos = (r - T::BM) % 16;                    // 8 gate rows, then the up rows of the same 8 columns
      row = min(n0 + (r - T::BM) / 16 * 8 + pos % 8, p.N - 1) + (pos >= 8 ? p.N : 0);
    } else {
      row = min(n0 + r - T::BM, p.N - 1);
    }
    off[i] = (uint32_t)row * (uint32_t)((is_x ? p.x_stride : p.w_stride) * 2) + chunk * 16;
    base[i] = (is_x ? p.x : p.w) + (int64_t)first * T::RB;
  }
  ring_f32x4 acc[T::FM][T::FN];
#pragma unroll
  for (int f = 0; f < T::FM; ++f)
#pragma unroll
    for (int j = 0; j < T::FN; ++j) acc[f][j] = ring_f32x4{0.f, 0.f, 0.f, 0.f};
  if (!SPLIT && p.mblocks == 1) ring_product<Tag, T, 2, 1>(acc, off, base, dense_lds, steps, wave, lane);
  else ring_product<Tag, T, 0, 1>(acc, off, base, dense_lds, steps, wave, lane);
  dense_store<Tag, T::FM, T::FN, EPI, SPLIT>(p, acc, m0 + wave / T::WN * T::TM, n0 + wave % T::WN * (EPI ? T::TN / 2 : T::TN), split, lane);
}

// the shares of K summed in their order, 4 columns of a row a thread
template <typename Tag, int S>
__global__ void __launch_bounds__(256) dense_sum_kernel(DenseArgs p) {
  typedef Elem<Tag> E;
  const int per_row = (p.N + 3) / 4;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int m = (int)(i / per_row), n = (int)(i % per_row) * 4;
  if (m >= p.M) return;
  const float* from = p.part + (int64_t)m * p.N + n;
  const int64_t step = (int64_t)p.M * p.N;
  if (p.vec) {
    ring_f32x4 v[S];
#pragma unroll
    for (int s = 0; s < S; ++s) v[s] = *(const ring_f32x4*)(from + s * step);
#pragma unroll
    for (int by = 1; by < S; by *= 2)                          // in pairs: each share is rounded log2 S times
#pragma unroll
      for (int s = 0; s + by < S; s += 2 * by) v[s] += v[s + by];
    u32x2 o;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const float a = v[0][2 * h], b = v[0][2 * h + 1];
      if constexpr (std::is_same<Tag, bf16_tag>::value) o[h] = f32_to_bf16_bits(a) | f32_to_bf16_bits(b) << 16;
      else o[h] = f32_to_f16_bits(a) | f32_to_f16_bits(b) << 16;
    }
    *(u32x2*)(p.out + ((int64_t)m * p.out_stride + n) * 2) = o;
  } else {
    for (int r = 0; r < 4 && n + r < p.N; ++r) {
      float v[S];
#pragma unroll
      for (int s = 0; s < S; ++s) v[s] = from[s * step + r];
#pragma unroll
      for (int by = 1; by < S; by *= 2)
#pragma unroll
        for (int s = 0; s + by < S; s += 2 * by) v[s] += v[s + by];
      E::store(p.out, (int64_t)m * p.out_stride + n + r, v[0]);
    }
  }
}

template <typename T, typename = void>
struct IsRing : std::false_type {};
template <typename T>
struct IsRing<T, std::enable_if_t<(T::ST > 0)>> : std::true_type {};

template <typename Tag, typename T, int EPI, bool SPLIT>
int launch_dense_kernel(const DenseArgs& p, hipStream_t st) {
  void (*kernel)(DenseArgs);
  int threads;
  if constexpr (IsRing<T>::value) kernel = dense_wide_kernel<Tag, T, EPI, SPLIT>, threads = T::W * 64;
  else kernel = dense_kernel<Tag, T, EPI, SPLIT>, threads = T::kWaves * 64;
  const int64_t groups = ((int64_t)p.mblocks * p.nblocks * p.splits + 7) / 8 * 8;
  if (groups * threads >= (int64_t)1 << 32) return SP_ERR_UNSUPPORTED;          // (what a launch holds)
  static PerDevice<int> raised;
  int ok = 0;
  raised.get(ok, [&](int) {
    return hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, T::kLds) == hipSuccess ? 1 : 0;
  });
  if (!ok) return SP_ERR_LAUNCH;
  kernel<<<dim3((unsigned)groups), dim3(threads), T::kLds, st>>>(p);
  SP_LAUNCH_CHECK();
  return SP_OK;
}

template <typename Tag, typename T>
int launch_dense_tile(DenseArgs p, int epilogue, hipStream_t st) {
  if (p.K % T::BK) return SP_ERR_UNSUPPORTED;
  const int per = epilogue ? T::BN / 2 : T::BN;
  p.mblocks = (p.M + T::BM - 1) / T::BM;
  p.nblocks = (p.N + per - 1) / per;
  if (epilogue) return p.splits == 1 ? launch_dense_kernel<Tag, T, 1, false>(p, st) : SP_ERR_UNSUPPORTED;
  if (p.splits == 1) return launch_dense_kernel<Tag, T, 0, false>(p, st);
  const int64_t quads = (int64_t)p.M * ((p.N + 3) / 4);
  if (quads >= ((int64_t)1 << 32) - 256) return SP_ERR_UNSUPPORTED;
  const int rc = launch_dense_kernel<Tag, T, 0, true>(p, st);
  if (rc != SP_OK) return rc;
  const dim3 grid((unsigned)((quads + 255) / 256));
  switch (p.splits) {
    case 2: dense_sum_kernel<Tag, 2><<<grid, 256, 0, st>>>(p); break;
    case 3: dense_sum_kernel<Tag, 3><<<grid, 256, 0, st>>>(p); break;
    case 4: dense_sum_kernel<Tag, 4><<<grid, 256, 0, st>>>(p); break;
    case 6: dense_sum_kernel<Tag, 6><<<grid, 256, 0, st>>>(p); break;
    default: dense_sum_kernel<Tag, 8><<<grid, 256, 0, st>>>(p);
  }
  SP_LAUNCH_CHECK();
  return SP_OK;
}

// ---- which tile, how many shares of K
// Every tile's cost: us of one step of one workgroup and of a workgroup's beginning and end, both fitted (with the constants below) to
// 7600 timings over 23 shapes of 1 - 1050 MB at 5 - 640 rows.  A product takes the chain of its busiest unit, the traffic into
// that unit's LDS or the weights' stream, whichever is longest; the choice is within 1.2 % of the fastest tile and split on average.
#define SP_DENSE_TILES(F)                                \
  F(0, 0.655f, 2.26f, 16, 64, 256, 2, 1, 4, 2, 3, 4)     \
  F(1, 0.588f, 2.04f, 16, 128, 128, 1, 1, 8, 1, 4, 4)    \
  F(2, 0.293f, 2.39f, 32, 16, 256, 2, 2, 1, 2, 4, 8)     \
  F(3, 0.404f, 2.17f, 32, 32, 256, 2, 2, 2, 4, 3, 6)     \
  F(4, 0.933f, 1.78f, 32, 64, 256, 2, 1, 4, 2, 2, 4)     \
  F(5, 0.627f, 2.62f, 32, 128, 128, 1, 1, 8, 2, 3, 4)    \
  F(6, 0.474f, 2.86f, 48, 32, 256, 2, 1, 2, 2, 3, 5)     \
  F(7, 0.258f, 2.62f, 64, 32, 128, 2, 2, 2, 4, 4, 6)     \
  F(8, 0.228f, 2.55f, 64, 64, 64, 1, 2, 2, 2, 4, 6)      \
  F(9, 0.578f, 3.53f, 64, 64, 256, 2, 2, 2, 4, 2, 3)     \
  F(10, 0.648f, 3.52f, 64, 128, 128, 1, 2, 4, 4, 2, 4)   \
  F(11, 0.565f, 2.63f, 96, 64, 128, 1, 2, 4, 4, 3, 4)    \
  F(12, 0.395f, 3.12f, 96, 128, 64, 1, 2, 4, 4, 4, 6)    \
  F(13, 0.398f, 2.98f, 128, 96, 64, 1, 4, 2, 4, 4, 6)
// and of dense_wide_kernel, from 2300 timings over 10 shapes at 96 - 1024 rows; the choice among all tiles is within 0.9 % of the fastest there
#define SP_WIDE_TILES(F)                        \
  F(14, 0.315f, 1.07f, 128, 64, 64, 2, 2, 3)    \
  F(15, 0.372f, 2.90f, 128, 128, 64, 2, 4, 4)   \
  F(16, 0.428f, 4.44f, 192, 128, 64, 4, 2, 4)   \
  F(17, 0.511f, 4.85f, 256, 128, 64, 4, 2, 3)   \
  F(18, 0.426f, 3.97f, 256, 96, 64, 4, 2, 3)    \
  F(19, 0.768f, 4.95f, 160, 256, 64, 2, 4, 3)   \
  F(20, 0.548f, 5.27f, 192, 192, 64, 2, 4, 3)
constexpr int kDenseTiles = 21, kFirstWide = 14;
constexpr float kLaunch = 1.72f, kStream = 5.43e6f, kFill = 67.72e3f;     // us, bytes per us
constexpr int kUnits = 256;

struct TileCost {
  int bm, bn, bk, wk, lds;
  float step, fixed, sum, rate;       // the launch that adds the shares: us, and bytes per us
};
#define SP_DENSE_COST(I, STEP, FIXED, ...) \
  {Tile<__VA_ARGS__>::BM, Tile<__VA_ARGS__>::BN, Tile<__VA_ARGS__>::BK, Tile<__VA_ARGS__>::WK, Tile<__VA_ARGS__>::kLds, STEP, FIXED, 2.f, 3.76e6f},
#define SP_WIDE_COST(I, STEP, FIXED, ...) \
  {RingTile<__VA_ARGS__>::BM, RingTile<__VA_ARGS__>::BN, RingTile<__VA_ARGS__>::BK, 1, RingTile<__VA_ARGS__>::kLds, STEP, FIXED, 4.03f, 5.9e6f},
constexpr TileCost kCosts[kDenseTiles] = {SP_DENSE_TILES(SP_DENSE_COST) SP_WIDE_TILES(SP_WIDE_COST)};

float dense_us(const TileCost& c, int M, int64_t rows, int K, int splits) {
  const int64_t wgs = (M + c.bm - 1) / c.bm * ((rows + c.bn - 1) / c.bn) * splits;
  const int held = c.lds <= 80 * 1024 ? 2 : 1;                         // workgroups that a unit holds
  const float steps = (float)((K / c.bk + splits - 1) / splits);
  const float chain = (float)((wgs + kUnits * held - 1) / (kUnits * held)) * (c.fixed + steps * c.step);
  const float fill = (float)((wgs + kUnits - 1) / kUnits) * steps * (float)((c.bm + c.bn) * c.bk * 2) / kFill;
  const float stream = 2.f * (float)rows * (float)K / kStream;
  const float c2 = chain * chain, f2 = fill * fill, s2 = stream * stream;
  float us = kLaunch + sqrtf(sqrtf(c2 * c2 + f2 * f2 + s2 * s2));
  if (splits > 1) us += c.sum + 8.f * (float)splits * (float)M * (float)rows / c.rate;
  return us;
}

template <typename Tag>
int launch_dense(const DenseArgs& p, int tile, int epilogue, hipStream_t st) {
#define SP_DENSE_CASE(I, STEP, FIXED, ...) \
  case I: return launch_dense_tile<Tag, Tile<__VA_ARGS__>>(p, epilogue, st);
#define SP_WIDE_CASE(I, STEP, FIXED, ...) \
  case I: return launch_dense_tile<Tag, RingTile<__VA_ARGS__>>(p, epilogue, st);
  switch (tile) { SP_DENSE_TILES(SP_DENSE_CASE) SP_WIDE_TILES(SP_WIDE_CASE) }
  return SP_ERR_INVALID_ARG;
}

}  // namespace
}  // namespace sp

// tile + 256 * shares of K, or -1: no tile takes the product.  With the activation in the epilogue: the tile is one that adds in the
// order of the plain product's, so that a step's bits do not depend on whether it is fused.
extern "C" int sp_gemm_dense_plan(int M, int N, int K, int epilogue) {
  if (M <= 0 || N <= 0 || K <= 0 || K % 64 || epilogue < 0 || epilogue > 1 || (epilogue && N >= 1 << 30)) return -1;
  const int rows = epilogue ? 2 * N : N;
  const int plain = epilogue ? sp_gemm_dense_plan(M, rows, K, 0) : 0;
  if (epilogue && plain >> 8 != 1) return -1;
  int best = -1;
  float least = 0.f;
  for (int i = 0; i < sp::kDenseTiles; ++i) {
    const sp::TileCost& c = sp::kCosts[i];
    // (the first tiles' costs hold up to 256 rows: 3072 x 3072 at 777 they promise less than the 29 us that they take, dense_wide_kernel 25 - 30)
    if (K % c.bk || (M > 256 && i < sp::kFirstWide) || (epilogue && c.wk != sp::kCosts[plain & 255].wk)) continue;
    for (int splits : {1, 2, 3, 4, 6, 8}) {
      if (splits > 1 && epilogue) break;
      if (i < sp::kFirstWide && splits % 3 == 0) continue;
      // shares of at least three steps, for launches that would leave units idle, with sums that stay in the caches
      if (splits > 1 && (K / c.bk / splits < 3 || (M + c.bm - 1) / c.bm * (int64_t)((rows + c.bn - 1) / c.bn) * splits > 600 ||
                         4 * (int64_t)splits * M * N > (int64_t)128 << 20))
        break;
      const float us = sp::dense_us(c, M, rows, K, splits);
      if (best < 0 || us < least) best = i + 256 * splits, least = us;
    }
  }
  return best;
}

extern "C" int sp_gemm_dense(void* out, const void* x, const void* w, float* sums, int64_t sums_floats, int M, int N, int K, int64_t x_stride,
                             int64_t w_stride, int64_t out_stride, int epilogue, int plan, int dtype, void* stream) {
  SP_CHECK_ARG(M >= 0 && N >= 0 && K > 0 && epilogue >= 0 && epilogue <= 1);
  if (M == 0 || N == 0) return SP_OK;
  SP_CHECK_ARG(out && x && w && plan >= 0);
  const int tile = plan & 255, splits = plan >> 8;
  SP_CHECK_ARG(tile < sp::kDenseTiles && (splits <= 4 || splits == 6 || splits == 8) && splits >= 1);
  SP_CHECK_ARG(splits == 1 || (sums && ((uintptr_t)sums & 15) == 0 && sums_floats >= (int64_t)splits * M * N));
  const int64_t rows = epilogue ? 2 * (int64_t)N : N;
  SP_CHECK_ARG(x_stride % 8 == 0 && w_stride % 8 == 0 && x_stride >= K && w_stride >= K && out_stride >= N);
  SP_CHECK_ARG(((uintptr_t)x & 15) == 0 && ((uintptr_t)w & 15) == 0 && ((uintptr_t)out & 1) == 0);
  if (dtype != SP_BF16 && dtype != SP_F16) return SP_ERR_UNSUPPORTED;
  if (K % sp::kCosts[tile].bk || K / sp::kCosts[tile].bk < splits) return SP_ERR_UNSUPPORTED;
  // a load's place is a 32-bit offset from the operand's first byte
  if ((int64_t)M * x_stride * 2 >= (int64_t)1 << 32 || rows * w_stride * 2 >= (int64_t)1 << 32) return SP_ERR_UNSUPPORTED;
  const int vec = N % 4 == 0 && out_stride % 4 == 0 && ((uintptr_t)out & 7) == 0;
  const sp::DenseArgs p{(char*)out, sums, (const char*)x, (const char*)w, M, N, K, splits, 0, 0, x_stride, w_stride, out_stride, vec};
  return dtype == SP_BF16 ? sp::launch_dense<sp::bf16_tag>(p, tile, epilogue, (hipStream_t)stream)
                          : sp::launch_dense<sp::f16_tag>(p, tile, epilogue, (hipStream_t)stream);
}
