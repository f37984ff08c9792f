// Direct loads into LDS, in rings of steps: what the tiled products share.
#pragma once
#include "sp_common.h"

#include <type_traits>

namespace sp {

// 16 bytes per lane from base + off to lds + 16 lane, without a register on the way.  (The builtin of the same makes every later read of
// LDS wait for it.  m0 is named, so that no value another instruction needs in it is carried past; the compiler calls that reserved.)
// ONCE: past the L2's other lines.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
template <bool ONCE>
__device__ __forceinline__ void ring_load(uint32_t off, const char* base, uint32_t lds) {
  if constexpr (ONCE)
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 nt" ::"v"(off), "s"(base), "s"(lds) : "memory", "m0");
  else
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(lds) : "memory", "m0");
}
#pragma clang diagnostic pop

// Waits until at most min(later, MOST) steps of L loads each are on their way, and for this wave's reads of LDS
template <int L, int MOST>
__device__ __forceinline__ void ring_wait(int later) {
  if constexpr (MOST == 0) {
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  } else {
    if (later >= MOST) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(L* MOST) : "memory");
    else ring_wait<L, MOST - 1>(later);
  }
}

__device__ __forceinline__ void ring_barrier() {
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// f(0), f(1) .. f(N - 1) as constants
template <int N, int I = 0, typename F>
__device__ __forceinline__ void each(const F& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>());
    each<N, I + 1>(f);
  }
}

typedef float ring_f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 ring_bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 ring_f16x8 __attribute__((ext_vector_type(8)));

template <typename Tag>
__device__ __forceinline__ ring_f32x4 mfma32(const u32x4& a, const u32x4& b, const ring_f32x4& c) {
  if constexpr (std::is_same<Tag, bf16_tag>::value)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(ring_bf16x8, a), __builtin_bit_cast(ring_bf16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(ring_f16x8, a), __builtin_bit_cast(ring_f16x8, b), c, 0, 0, 0);
}

__device__ __forceinline__ uint32_t lds_address(const char* p) { return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) char*)p; }

// A product of BM rows x BN weight rows whose waves all load both operands: k in steps of BK, ST of them in a ring of LDS buffers of BM, then BN
// rows whose 16-byte chunks are permuted by the row's number.  One barrier a step, in front of its last products: behind it the next step's first
// operands are read, and the loads into the buffer that has become free are spread between those products - in one piece they hold a wave's
// products up (an instruction a wave can't issue stops the ones behind it): a 256 x 256 tile's loop, operands in the L2, 1245 -> 1480 TFLOP/s
// with the loads spread and the waves in their products ahead of the others.
template <int BM_, int BN_, int BK_, int WM_, int WN_, int ST_>
struct RingTile {
  static constexpr int BM = BM_, BN = BN_, BK = BK_, WM = WM_, WN = WN_, ST = ST_, W = WM * WN;
  static constexpr int RB = BK * 2, RPL = 1024 / RB, CH = BK / 8;                            // a row's bytes; rows and 16-byte chunks of a load
  static constexpr int TM = BM / WM, TN = BN / WN, FM = TM / 16, FN = TN / 16, KK = BK / 32;
  static constexpr int G = (BM + BN) / RPL, L = (G + W - 1) / W, kStage = (BM + BN) * RB, kLds = ST * kStage;
  static constexpr int kWaves = (kLds <= 80 * 1024 ? 2 : 1) * W / 4;                          // of a SIMD: at most two workgroups in a unit
  static_assert(BM % RPL == 0 && BN % RPL == 0 && TM % 16 == 0 && TN % 16 == 0 && KK % 2 == 0 && kLds <= 160 * 1024 && L * (ST - 1) <= 63, "tile");
};

// acc[f][j][r] += sum over k of x[row 16 f + lane % 16] w[column 16 j + 4 (lane / 16) + r] of the wave's TM x TN, ascending k.  Load i of a
// wave is the (i W + wave)-th of the tile's RPL rows each, x's first: base[i] + off[i], 64 lanes.  ONCE: past the L2 none of the loads (0), all
// (1), those of w (2).  Loads are spread from SPREAD products a load on.
template <typename Tag, typename T, int ONCE, int SPREAD>
__device__ __forceinline__ void ring_product(ring_f32x4 (&acc)[T::FM][T::FN], const uint32_t (&off)[T::L], const char* const (&base)[T::L], char* lds,
                                             int steps, int wave, int lane) {
  constexpr int PER = T::FM * T::FN / T::L, KK = T::KK, ST = T::ST;
  const int r16 = lane & 15, q = lane >> 4, wm = wave / T::WN, wn = wave % T::WN;
  const uint32_t lds0 = lds_address(lds);
  const auto load = [&](auto at, int s, int buf) {
    constexpr int i = decltype(at)::value;
    ring_load<(ONCE == 1 || (ONCE == 2 && i * T::W * T::RPL >= T::BM))>(off[i], base[i] + (int64_t)s * T::RB,
                                                                       lds0 + buf + min(i * T::W + wave, T::G - 1) * 1024);
  };
  const auto load_all = [&](int s, int buf) { each<T::L>([&](auto i) { load(i, s, buf); }); };
  const int arow = (wm * T::TM + r16) * T::RB, brow = (T::BM + wn * T::TN + r16) * T::RB;
  u32x4 xf[2][T::FM], wf[2][T::FN];
  const auto read = [&](int buf, int kk) {
    const int c = ((kk * 4 + q) ^ (r16 & 7)) * 16;
#pragma unroll
    for (int j = 0; j < T::FN; ++j) wf[kk & 1][j] = ld16(lds + buf + brow + j * 16 * T::RB + c);
#pragma unroll
    for (int f = 0; f < T::FM; ++f) xf[kk & 1][f] = ld16(lds + buf + arow + f * 16 * T::RB + c);
  };
  for (int s = 0; s < ST && s < steps; ++s) load_all(s, s * T::kStage);
  ring_wait<T::L, ST - 1>(steps - 1);
  ring_barrier();
  read(0, 0);
  int cur = 0;
  const auto step = [&](int s, auto more) {               // more: there is a step ST ahead to load
    constexpr bool MORE = decltype(more)::value;
    const int next = cur == (ST - 1) * T::kStage ? 0 : cur + T::kStage;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      if (kk < KK - 1) {
        read(cur, kk + 1);
      } else if (MORE || s + 1 < steps) {
        ring_wait<T::L, ST - 2>(MORE ? ST : steps - 2 - s);
        ring_barrier();
        if constexpr (MORE && PER < SPREAD) load_all(s + ST, cur);
        read(next, 0);
      }
      __builtin_amdgcn_s_setprio(1);
      each<T::FN * T::FM>([&](auto at) {
        constexpr int i = decltype(at)::value, n = i / T::FM, f = i % T::FM;
        if constexpr (MORE && PER >= SPREAD) {
          if constexpr (i % PER == 0 && i / PER < T::L) {
            if (kk == KK - 1) {
              __builtin_amdgcn_sched_barrier(0);
              load(std::integral_constant<int, i / PER>(), s + ST, cur);
              __builtin_amdgcn_sched_barrier(0);
            }
          }
        }
        acc[f][n] = mfma32<Tag>(wf[kk & 1][n], xf[kk & 1][f], acc[f][n]);
      });
      __builtin_amdgcn_s_setprio(0);
    }
    cur = next;
  };
  int s = 0;
  for (; s + ST < steps; ++s) step(s, std::true_type());
  for (; s < steps; ++s) step(s, std::false_type());
}

}  // namespace sp
