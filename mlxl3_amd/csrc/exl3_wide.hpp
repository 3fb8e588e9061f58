// The decode-in-registers QMM loop: NW waves, 16*R rows x 32*NW columns, one
// K-range, for the linear at more than 16 rows (qmm_tensor,
// linear.rs:1874-2083).
//
// Wave w owns 32 columns.  It decodes their trellis tiles into MFMA B fragments
// in registers, as the QMV does, and multiplies them with all 16*R rows, so a
// weight never passes through LDS and is decoded once per 16*R rows.  Everything
// that comes from memory goes global -> LDS directly, into two rings of one slot
// per step of 64 inputs: the A rows (xhat, one 128-byte line per row, swizzled)
// and the trellis words of the step's 4 tile rows x 2*NW tiles.  In step q a wave
//   * issues the copies of steps q + SA - 1 (A) and q + SW - 1 (trellis),
//   * decodes the trellis words of step q + 1 in pieces between the MFMAs, and
//     reads those of step q + 2, and
//   * multiplies step q: slot (h, rb) takes the A fragment of row block rb and
//     half h, read some slots earlier, against the two B fragments of that half;
// one barrier ends the step.  The source order fixes that interleaving, so VALU
// and MFMA overlap inside a wave and not only between the two waves of a SIMD.
//
// What bounds it: the SIMD's VALU port.  A 16x16x32 MFMA keeps it for 8 of its 16
// cycles (measured: n VALU instructions beside each, two waves per SIMD, cycles
// per MFMA: n=2 16.8, 4 25.0, 5 28.8), the decode of K = 4 adds 4.5 per MFMA at R =
// 8 and 2.25 at R = 16; past that the card's power: the same loop with the decode
// left out (timing only) runs its MFMAs at ~1260 TFLOP/s and a lower clock.
// Measured, 4096 -> 14336, K = 4 (a call, us): 2048 rows, R = 16, 236 to 239 (1007 to 1019
// TFLOP/s; the producer/consumer kernel 285); 512 rows, R = 8, 77 to 78, where that kernel
// with the same epilogue takes 75 to 76 and keeps the launch.  Forms that were no faster: 32x32x16 MFMAs with 64 columns per wave and two K halves (714
// TFLOP/s at 512 rows, fewer cycles at a lower clock), the same with one wave per
// SIMD and 256 rows (878 at 2048 rows), trellis words read one step later.
#pragma once

#include "exl3_device.hpp"
#include "exl3_params.hpp"
#include "exl3_qmm.hpp"

namespace exl3 {

// NW waves, 32 * NW columns.
template <int K, int R, int NW>
struct WideShape {
  static constexpr int kRows = 16 * R, kCols = 32 * NW;
  static constexpr int kA = kRows * 128, kW = 256 * K * NW;  // bytes of a ring's slot
  static constexpr int kAJobs = kA / 1024, kWJobs = kW / 1024;  // 1 KB copies per step
  static constexpr int PA = (kAJobs + NW - 1) / NW, PW = (kWJobs + NW - 1) / NW;  // per wave
  // ring depths: with 4 waves, and up to 64 rows, two workgroups share a CU
  static constexpr int kBudget = NW == 4 || R <= 4 ? 79 * 1024 : 158 * 1024;
  static constexpr int SA = 4 * (kA + kW) <= kBudget ? 4 : 3;
  static constexpr int kFitW = (kBudget - SA * kA) / kW;
  static constexpr int SW = kFitW < 3 ? 3 : kFitW > 6 ? 6 : kFitW;
  // kAhead: the first A fragments of a step are read in the step before, which
  // costs a ring slot (the copy has one step less to land in)
  static constexpr bool kAhead = SA >= 4;
  // trellis words are read two steps ahead (else one) where the ring is deep enough
  static constexpr int kLead = SW >= 5 ? 2 : 1;
  // copies that may be outstanding at a step's end where a wave issues pa A copies
  // per step: what the next step reads must have landed, A of step q + 1 (+ 1 with
  // kAhead) and trellis of step q + 1 + kLead
  static constexpr int out(int pa) {
    const int a = PW + (SA - (kAhead ? 3 : 2)) * (pa + PW), w = (SW - kLead - 2) * (pa + PW);
    return a < w ? a : w;
  }
  static constexpr int kStride = kCols + 8;  // halves per staged output row
  static constexpr int kY = kRows * kStride * 2;
  static constexpr int kRings = SA * kA + SW * kW;
  static constexpr int kLds = kRings > kY ? kRings : kY;
};

// One of the two sources of a step's copies, as a buffer: step q starts q *
// `step` bytes past the base.  Reads past `bytes` return zeros.
struct WideSource {
  u32x4 rsrc;     // wave-uniform
  uint32_t step;  // bytes per step (uniform)
};
__device__ __forceinline__ WideSource wide_source(const void* base, size_t bytes, uint32_t step) {
  const uint64_t a = (uint64_t)base;
  WideSource s;
  s.rsrc = u32x4{(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)a),
                 (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(a >> 32) & 0xffff),
                 (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)min(bytes, (size_t)0xffffffffu)),
                 (uint32_t)kBufferRsrcWord3};
  s.step = step;
  return s;
}
// Lane l copies the 16 bytes at src + soff + off to LDS bytes lds + add + 16l
// (soff, lds, add uniform).  The compiler sees neither the load nor the LDS
// write: the caller waits (vmcnt) before the barrier that publishes the bytes.
// m0 is a reserved register, which a clobber list may not name; the compiler writes it
// only right before an instruction of its own that reads it, and the kernels that
// copy this way have none.
__device__ __forceinline__ void wide_copy(const u32x4& rsrc, uint32_t off, uint32_t soff,
                                          uint32_t lds, uint32_t add) {
  asm volatile("s_add_u32 m0, %3, %4\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds"
               :
               : "v"(off), "s"(rsrc), "s"(soff), "s"(lds), "s"(add)
               : "memory", "scc");
}

// The windows of states S, S + 1 of a lane into src (shared windows are taken
// from the state that owns them, decoded earlier).
template <int K, int S>
__device__ __forceinline__ void state_window(const uint32_t (&B)[K + 1], uint32_t (&src)[32]) {
  if constexpr (16 % K == 0) {
    constexpr int d = 16 / K;
    if constexpr ((S / d) % 2 == 0)
      src[S] = window32<K, S>(B);
    else
      src[S] = src[S - d];
  } else {
    src[S] = window16<K, S>(B);
  }
}

// The decode of a step's weights beside MFMAs.  Every inline-assembly
// instruction here writes a register that already holds a live value ("+v"): an
// MFMA may get other registers for its result than for its addend, a VALU
// instruction that reuses the addend's registers has to come 3 wait states
// later, and the compiler keeps that distance only for instructions it sees as
// VALU.  A register that is live across the MFMA cannot be its addend's.
template <int HI>
__device__ __forceinline__ void mad16_into(uint32_t& d, uint32_t w, uint32_t b, uint32_t c) {
  if constexpr (HI)
    asm("v_mad_u32_u16 %0, %1, %2, %3 op_sel:[1,0,0,0]" : "+v"(d) : "v"(w), "v"(b), "v"(c));
  else
    asm("v_mad_u32_u16 %0, %1, %2, %3" : "+v"(d) : "v"(w), "v"(b), "v"(c));
}
template <int HI>
__device__ __forceinline__ void mul24_hi16_into(uint32_t& d, uint32_t w, uint32_t b) {
  if constexpr (HI)
    asm("v_mul_u32_u24_sdwa %0, %1, %2 dst_sel:WORD_1 dst_unused:UNUSED_PAD src0_sel:WORD_1 "
        "src1_sel:DWORD"
        : "+v"(d)
        : "v"(w), "v"(b));
  else
    asm("v_mul_u32_u24_sdwa %0, %1, %2 dst_sel:WORD_1 dst_unused:UNUSED_PAD src0_sel:WORD_0 "
        "src1_sel:DWORD"
        : "+v"(d)
        : "v"(w), "v"(b));
}
// codeword_product in two instructions on d.
template <int CB, int HI>
__device__ __forceinline__ void product_first(uint32_t& d, uint32_t w) {
  if constexpr (CB == 0)
    mad16_into<HI>(d, w, 6u, 0u);
  else
    mul24_hi16_into<HI>(d, w, CB == 1 ? 0xcbacu : 0x83dcu);
}
template <int CB, int HI>
__device__ __forceinline__ void product_second(uint32_t& d, uint32_t w) {
  if constexpr (CB == 0)
    asm("v_mad_u32_u24 %0, %0, %1, %2" : "+v"(d) : "s"(14871059u), "v"(64248484u));
  else
    mad16_into<HI>(d, w, CB == 1 ? 0x1fedu : 0xd12du, d);
}

// One step's decode as 34 pieces, each to be preceded by an MFMA: piece 2D
// finishes pair D - 1's masks, writes its low half and starts the products of
// pair D, piece 2D + 1 completes those products and writes pair D - 1's high
// half.  So an inline-assembly result is never read without an instruction in
// between that the compiler counts as a wait state (it counts none for inline
// assembly and would add an s_nop at each).  Pair D = 4p + 2cg + h is dword p of
// fragment (h, cg); states that share a 32-bit window follow each other.
template <int K, int CB>
struct StepDecode {
  uint32_t src[32];
  template <int D>
  static constexpr int state() {
    return 8 * (D >> 2) + 4 * ((D >> 1) & 1) + 2 * (D & 1);
  }
  // the fragment (h, cg) of pair D
  template <int D>
  static constexpr int of() {
    return 2 * (D & 1) + ((D >> 1) & 1);
  }
  template <int D>
  __device__ __forceinline__ void masks(uint32_t (&z)[2][2], u32x4 (&frag)[4]) {
    uint32_t &z0 = z[D & 1][0], &z1 = z[D & 1][1];
    if constexpr (CB < 2) {
      z0 = (z0 & 0x8fff8fffu) ^ 0x3b603b60u;
      z1 = (z1 & 0x8fff8fffu) ^ 0x3b603b60u;
      uint32_t d = frag[of<D>()][D >> 2];
      asm("v_add_f16_sdwa %0, %1, %1 dst_sel:WORD_0 dst_unused:UNUSED_PAD src0_sel:WORD_0 "
          "src1_sel:WORD_1"
          : "+v"(d)
          : "v"(z0));
      frag[of<D>()][D >> 2] = d;
    } else {
      asm("v_sad_u8 %0, %0, 0, %1" : "+v"(z0) : "v"(0x6400u));
      asm("v_sad_u8 %0, %0, 0, %1" : "+v"(z1) : "v"(0x6400u));
    }
  }
  template <int D>
  __device__ __forceinline__ void high_half(uint32_t (&z)[2][2], u32x4 (&frag)[4]) {
    const uint32_t z0 = z[D & 1][0], z1 = z[D & 1][1];
    if constexpr (CB < 2) {
      uint32_t d = frag[of<D>()][D >> 2];
      asm("v_add_f16_sdwa %0, %1, %1 dst_sel:WORD_1 dst_unused:UNUSED_PRESERVE src0_sel:WORD_0 "
          "src1_sel:WORD_1"
          : "+v"(d)
          : "v"(z1));
      frag[of<D>()][D >> 2] = d;
    } else {
      const half2v sum = __builtin_bit_cast(half2v, z0 | (z1 << 16));
      const half2v inv = __builtin_bit_cast(half2v, 0x1eee1eeeu);
      const half2v bias = __builtin_bit_cast(half2v, 0xc931c931u);
      frag[of<D>()][D >> 2] =
          __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(sum, inv, bias));
    }
  }
  template <int I>
  __device__ __forceinline__ void piece(const uint32_t (&B)[K + 1], uint32_t (&z)[2][2],
                                        u32x4 (&frag)[4]) {
    constexpr int D = I >> 1, S0 = state<D>();
    uint32_t &z0 = z[D & 1][0], &z1 = z[D & 1][1];
    if constexpr (I % 2 == 0) {
      if constexpr (D < 16) {
        state_window<K, S0>(B, src);
        state_window<K, S0 + 1>(B, src);
      }
      if constexpr (D > 0) masks<D - 1>(z, frag);
      if constexpr (D < 16) {
        product_first<CB, state_half<K, S0>()>(z0, src[S0]);
        product_first<CB, state_half<K, S0 + 1>()>(z1, src[S0 + 1]);
      }
    } else {
      if constexpr (D > 0) high_half<D - 1>(z, frag);
      if constexpr (D < 16) {
        product_second<CB, state_half<K, S0>()>(z0, src[S0]);
        product_second<CB, state_half<K, S0 + 1>()>(z1, src[S0 + 1]);
      }
    }
  }
};
constexpr int kDecodePieces = 34;

// acc[rb][cg] += A (16*R rows) x this wave's 32 columns over nq steps.  lds: the
// rings; aoff, woff: the lane's byte offset of each of the wave's copies in its
// source.  Register r of lane (g = lane / 16, n = lane % 16) of acc[rb][cg] is row
// 16rb + 4g + r, column 16*(n / 8) + n % 8 + 8cg of the wave's 32.  With SOME, only
// the first `live` row blocks (uniform, 1..R) are copied and, rounded up to a pair,
// multiplied.
template <int K, int CB, int R, int NW, bool SOME>
__device__ __forceinline__ void wide_mm(uint8_t* lds, const WideSource& asrc, const WideSource& wsrc,
                                        const uint32_t (&aoff)[WideShape<K, R, NW>::PA],
                                        const uint32_t (&woff)[WideShape<K, R, NW>::PW], int nq,
                                        int live, int wave, int lane, float4v (&acc)[R][2]) {
  using C = WideShape<K, R, NW>;
  constexpr int kRing = R == 8 ? 4 : 2;  // slot pairs of A fragments in registers
  const int g = lane >> 4, am = lane & 15, hsel = (lane >> 3) & 1, j = lane & 7;
  const uint32_t lds0 = lds_offset(lds);
  // copy i of the wave is the step's copy wave + NW * i; past the last one it
  // repeats that
  const int ajobs = SOME ? 2 * live : C::kAJobs;
  const int pa = SOME ? (max(ajobs - wave, 0) + NW - 1) / NW : C::PA;  // A copies per step
  auto wait_copies = [&]() {
    static_for<C::PA + 1>([&](auto pa_) {
      constexpr int n = decltype(pa_)::value;
      if (SOME ? pa == n : n == C::PA) __builtin_amdgcn_s_waitcnt(vmcnt_only(C::out(n)));
    });
  };
  uint32_t alds[C::PA], wlds[C::PW];
#pragma unroll
  for (int i = 0; i < C::PA; ++i)
    alds[i] = __builtin_amdgcn_readfirstlane(lds0 + min(wave + NW * i, C::kAJobs - 1) * 1024);
#pragma unroll
  for (int i = 0; i < C::PW; ++i)
    wlds[i] = __builtin_amdgcn_readfirstlane(lds0 + C::SA * C::kA +
                                             min(wave + NW * i, C::kWJobs - 1) * 1024);
  const uint32_t a_end = (uint32_t)(nq - 1) * asrc.step, w_end = (uint32_t)(nq - 1) * wsrc.step;
  uint32_t a_at = 0, w_at = 0;  // byte offsets of the next step to copy
  // past the end: the last step again, into a slot that is not read
  auto copy_a = [&](uint32_t slot) {
#pragma unroll
    for (int i = 0; i < C::PA; ++i)
      if (!SOME || wave + NW * i < ajobs) wide_copy(asrc.rsrc, aoff[i], a_at, slot, alds[i]);
    a_at = min(a_at + asrc.step, a_end);
  };
  auto copy_w = [&](uint32_t slot) {
#pragma unroll
    for (int i = 0; i < C::PW; ++i) wide_copy(wsrc.rsrc, woff[i], w_at, slot, wlds[i]);
    w_at = min(w_at + wsrc.step, w_end);
  };
  // fragment (rb, h): row 16rb + am, chunk 2g + h, at its swizzled slot (the
  // swizzle depends on the row's low 4 bits only)
  int foff[2];
#pragma unroll
  for (int h = 0; h < 2; ++h)
    foff[h] = am * 128 + (((2 * g + h) ^ a_swizzle(am)) << 4);
  auto read_a = [&](half8& dst, uint32_t at, auto slot_) {
    constexpr int slot = decltype(slot_)::value, h = slot / R, rb = slot % R;
    dst = *(const half8*)(lds + at + foff[h] + rb * 2048);
  };
  // both fragments of slot pair `pr`; the first one used is read last, so one
  // wait serves both
  auto pair_live = [&](auto pr_) {
    constexpr int rb = 2 * decltype(pr_)::value % R;
    return !SOME || rb == 0 || rb < live;
  };
  auto read_pair = [&](half8(&dst)[2], uint32_t at, auto pr_) {
    constexpr int pr = decltype(pr_)::value;
    if (!pair_live(pr_)) return;
    read_a(dst[1], at, std::integral_constant<int, 2 * pr + 1>{});
    read_a(dst[0], at, std::integral_constant<int, 2 * pr>{});
  };
  const int wbase = C::SA * C::kA + ((g * 2 * NW + 2 * wave + hsel) * 8 * K + j * K) * 4;
  const int wprev = wbase + (j == 0 ? 8 * K - 1 : -1) * 4;
  auto read_w = [&](uint32_t(&w)[K + 1], uint32_t at) {
    w[0] = *(const uint32_t*)(lds + at + wprev);
    if constexpr (K == 4 || K == 8) {
#pragma unroll
      for (int i = 0; i < K / 4; ++i) {
        const u32x4 v = *(const u32x4*)(lds + at + wbase + 16 * i);
        w[4 * i + 1] = v[0], w[4 * i + 2] = v[1], w[4 * i + 3] = v[2], w[4 * i + 4] = v[3];
      }
    } else if constexpr (K == 2 || K == 6) {
#pragma unroll
      for (int i = 0; i < K / 2; ++i) {
        const u32x2 v = *(const u32x2*)(lds + at + wbase + 8 * i);
        w[2 * i + 1] = v[0], w[2 * i + 2] = v[1];
      }
    } else {
#pragma unroll
      for (int i = 0; i < K; ++i) w[i + 1] = *(const uint32_t*)(lds + at + wbase + 4 * i);
    }
  };

  // the copies that steps before the first would have issued, in their order
#pragma unroll
  for (int i = 1 - (C::SA > C::SW ? C::SA : C::SW); i < 0; ++i) {
    if (i + C::SA - 1 >= 0) copy_a((i + C::SA - 1) * C::kA);
    if (i + C::SW - 1 >= 0) copy_w((i + C::SW - 1) * C::kW);
  }
  wait_copies();
  __syncthreads();

  u32x4 b[2][4] = {};
  uint32_t z[2][2] = {}, w[2][K + 1];
  half8 a[kRing][2];
  {
    StepDecode<K, CB> dec;
    read_w(w[0], 0);
    static_for<kDecodePieces>([&](auto i) { dec.template piece<decltype(i)::value>(w[0], z, b[0]); });
    if (C::kLead == 2) read_w(w[0], C::kW);
    if (C::kAhead)
      static_for<kRing>([&](auto i) { read_pair(a[decltype(i)::value], 0, i); });
  }
  // ring positions: A of steps q, q + 1 and q + SA - 1 (= q - 1), trellis of steps
  // q + kLead and q + SW - 1 (= q - 1)
  uint32_t at = 0, at1 = C::kA, atd = (C::SA - 1) * C::kA;
  uint32_t wt = C::kLead * C::kW, wtd = (C::SW - 1) * C::kW;
  auto step = [&](auto phase) {
    constexpr int ph = decltype(phase)::value;
    copy_a(atd);
    copy_w(wtd);
    constexpr int wi = C::kLead == 2 ? ph : 0;
    StepDecode<K, CB> dec;
    if (C::kLead == 1) read_w(w[0], wt);
    if constexpr (!C::kAhead)
      static_for<kRing>([&](auto i) { read_pair(a[decltype(i)::value], at, i); });
    u32x4(&cur)[4] = b[ph];
    u32x4(&nxt)[4] = b[ph ^ 1];
    // written by inline assembly: 2 wait states before the MFMAs
    asm volatile("s_nop 1" : "+v"(cur[0]), "+v"(cur[1]), "+v"(cur[2]), "+v"(cur[3]));
    // without fragments read ahead, some of the decode covers their latency
    constexpr int kFirst = C::kAhead ? 0 : 4;
    static_for<kFirst>([&](auto i) {
      dec.template piece<decltype(i)::value>(w[wi], z, nxt);
      __builtin_amdgcn_sched_barrier(0);
    });
    static_for<R>([&](auto pr_) {
      constexpr int pr = decltype(pr_)::value;
      auto pieces = [&](auto m_) {
        constexpr int m = decltype(m_)::value;
        constexpr int kRest = kDecodePieces - kFirst;
        constexpr int i0 = kFirst + kRest * m / (4 * R), i1 = kFirst + kRest * (m + 1) / (4 * R);
        static_for<i1 - i0>([&](auto i) {
          dec.template piece<i0 + decltype(i)::value>(w[wi], z, nxt);
        });
      };
      auto read_next = [&]() {
        if constexpr (pr + kRing < R)
          read_pair(a[pr % kRing], at, std::integral_constant<int, pr + kRing>{});
        else if constexpr (C::kAhead)
          read_pair(a[pr % kRing], at1, std::integral_constant<int, pr + kRing - R>{});
        if constexpr (C::kLead == 2 && pr == R / 2) read_w(w[wi ^ 1], wt);
      };
      if (pair_live(pr_)) {
        static_for<4>([&](auto i_) {
          constexpr int i = decltype(i_)::value, slot = 2 * pr + (i >> 1), cg = i & 1;
          constexpr int h = slot / R, rb = slot % R;
          acc[rb][cg] = mfma16(a[pr % kRing][slot & 1],
                               __builtin_bit_cast(half8, cur[2 * h + cg]), acc[rb][cg]);
          if constexpr (i == 3) read_next();
          pieces(std::integral_constant<int, 4 * pr + i>{});
          __builtin_amdgcn_sched_barrier(0);
        });
      } else {
        // no rows: this pair's share of the decode alone, the compiler's own
        // wait states between the pieces
        read_next();
        static_for<4>([&](auto i_) {
          pieces(std::integral_constant<int, 4 * pr + decltype(i_)::value>{});
          __builtin_amdgcn_sched_barrier(0);
        });
      }
    });
    // what the next step reads has landed; every wave is done with the slots that
    // the next step's copies overwrite, whose reads its MFMAs and decode have
    // waited for
    wait_copies();
    asm volatile("s_barrier" ::: "memory");
    atd = at;
    at = at1;
    at1 = at1 == (C::SA - 1) * C::kA ? 0 : at1 + C::kA;
    wt = wt == (C::SW - 1) * C::kW ? 0 : wt + C::kW;
    wtd = wtd == (C::SW - 1) * C::kW ? 0 : wtd + C::kW;
  };
  int left = nq;
  for (; left >= 2; left -= 2) {
    step(std::integral_constant<int, 0>{});
    step(std::integral_constant<int, 1>{});
  }
  if (left) step(std::integral_constant<int, 0>{});
  // the copies of past-the-end steps must not land on what the caller stores next
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
}

// f16 rows of the tile in LDS from the accumulators of wide_mm.
template <int R>
__device__ __forceinline__ void wide_stage_rows(const float4v (&acc)[R][2], uint16_t* ys, int stride,
                                                int wave, int lane) {
  const int g = lane >> 4, n = lane & 15;
  uint16_t* y = ys + 4 * g * stride + 32 * wave + 16 * (n >> 3) + 2 * (n & 7);
  static_for<R>([&](auto rb_) {
    constexpr int rb = decltype(rb_)::value;
#pragma unroll
    for (int r = 0; r < 4; ++r)
      *(half2v*)(y + (16 * rb + r) * stride) = pack_f16(acc[rb][0][r], acc[rb][1][r]);
  });
}

// Linear at more than 16 rows: tiles of 16*R rows x 32*NW columns (a column unit)
// of one member.
template <int K, int CB, int R, int NW>
__global__ __launch_bounds__(64 * NW) void wide_qmm_kernel(WideParams p) {
  using C = WideShape<K, R, NW>;
  __shared__ __attribute__((aligned(16))) uint8_t lds[C::kLds];
  __shared__ __attribute__((aligned(16))) uint16_t s_svh[C::kCols], s_bias[C::kCols];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

  // Workgroup -> (row tile, column unit, split): each XCD takes a contiguous
  // run, in which four row tiles of one column unit come together, so its L2
  // serves both the trellis (read once per four row tiles) and the A rows.
  const int nwg = p.mtiles * p.units * p.splits;
  const int id = blockIdx.x, xcd = id & 7, rem = nwg & 7;
  const int lin = xcd * (nwg >> 3) + min(xcd, rem) + (id >> 3);
  const int per_split = p.mtiles * p.units;
  const int split = lin / per_split, in_split = lin - split * per_split;
  const int band = in_split / (4 * p.units), in_band = in_split - band * 4 * p.units;
  const int bh = min(4, p.mtiles - 4 * band);
  const int unit = in_band / bh, mtile = 4 * band + (in_band - unit * bh);
  const WideMember mm = select_wide(p, unit);
  const int pl = unit - mm.unit0;  // column unit inside the member
  const int TN = mm.out >> 4;
  // the unit's second 128 columns exist
  const bool whole = NW == 4 || pl * 256 + 128 < mm.out;
  const int nq_all = p.in >> 6;
  const int qa = split * nq_all / p.splits, nq = (split + 1) * nq_all / p.splits - qa;
  const int row0 = mtile * C::kRows;

  if (threadIdx.x < C::kCols) {
    const int c = pl * C::kCols + (whole ? (int)threadIdx.x : (int)threadIdx.x & 127);
    s_svh[threadIdx.x] = mm.svh[c];
    s_bias[threadIdx.x] = mm.bias ? mm.bias[c] : 0;
  }
  const uint8_t* abase = (const uint8_t*)(mm.xhat + (size_t)row0 * p.in + (size_t)qa * 64);
  const WideSource asrc =
      wide_source(abase, (size_t)((const uint8_t*)(mm.xhat + (size_t)p.M * p.in) - abase), 128);
  const size_t wfirst = ((size_t)4 * qa * TN + pl * 2 * NW) * (32 * K);
  const WideSource wsrc = wide_source((const uint8_t*)mm.trellis + wfirst,
                                      (size_t)(p.in >> 4) * TN * (32 * K) - wfirst,
                                      (uint32_t)TN * (128u * K));
  uint32_t aoff[C::PA], woff[C::PW];
#pragma unroll
  for (int i = 0; i < C::PA; ++i) {
    // rows 8*jid..: lane l copies chunk (l & 7) ^ swizzle of row l >> 3; rows past
    // M repeat the last one (never stored)
    const int r = 8 * min(wave + NW * i, C::kAJobs - 1) + (lane >> 3);
    const int rg = min(row0 + r, p.M - 1) - row0;
    aoff[i] = (uint32_t)((rg * p.in + ((lane & 7) ^ a_swizzle(r)) * 8) * 2);
  }
#pragma unroll
  for (int i = 0; i < C::PW; ++i) {
    // bytes v*1024 + 16*lane of the step's [4 tile rows][2 * NW tiles]
    const uint32_t at = (uint32_t)min(wave + NW * i, C::kWJobs - 1) * 1024u + 16u * lane;
    const uint32_t tr = at / (64u * NW * K);
    uint32_t rest = at - tr * (64u * NW * K);
    if (!whole && rest >= 256u * K) rest -= 256u * K;  // the missing half repeats the first
    woff[i] = tr * (uint32_t)TN * (32u * K) + rest;
  }
  float4v acc[R][2];
#pragma unroll
  for (int rb = 0; rb < R; ++rb) acc[rb][0] = acc[rb][1] = float4v{0.f, 0.f, 0.f, 0.f};
  wide_mm<K, CB, R, NW, false>(lds, asrc, wsrc, aoff, woff, nq, R, wave, lane, acc);

  if (p.splits > 1) {
    // split-K: the f32 sums, [split][unit][row block][wave][cg][lane] of 16 bytes,
    // for wide_reduce_kernel (row blocks past M are left out)
    const int blocks = (p.M + 15) >> 4;
    float* dst = p.partials + ((size_t)split * p.units + unit) * blocks * (16 * C::kCols) +
                 (size_t)mtile * R * (16 * C::kCols) + wave * 512 + lane * 4;
#pragma unroll
    for (int rb = 0; rb < R; ++rb)
      if (mtile * R + rb < blocks)
#pragma unroll
        for (int cg = 0; cg < 2; ++cg)
          *(float4v*)(dst + rb * (16 * C::kCols) + cg * 256) = acc[rb][cg];
    return;
  }
  uint16_t* ys = (uint16_t*)lds;
  wide_stage_rows<R>(acc, ys, C::kStride, wave, lane);
  __syncthreads();
  // R row blocks x the unit's 128-column blocks over the waves
  const QmmOut out{mm.y, mm.y_dtype, mm.bias != nullptr};
  constexpr int kH = NW / 4;
  for (int u = wave; u < kH * R; u += NW) {
    const int half = u % kH, rl = 16 * (u / kH), row = row0 + rl;
    if ((half && !whole) || row >= p.M) continue;  // uniform
    qmm_finish16(ys + rl * C::kStride + 128 * half, C::kStride, s_svh + 128 * half,
                 s_bias + 128 * half, lane, p.M - row, out, p.x_dtype,
                 (size_t)row * mm.out + pl * C::kCols + 128 * half, mm.out);
  }
}

// Split-K sums of wide_qmm_kernel and their epilogue: one wave per 16 rows x 128
// columns adds the parts in split order.  A launch of its own: every CU takes
// part and the partials go through the caches, where the last arriver of a tile
// summing them alone (coherent loads, one workgroup per tile) was the larger
// half of such calls.  grid ceil(units * ceil(M / 16) * NW / 4 / 4), 256 threads.
static __global__ __launch_bounds__(256) void wide_reduce_kernel(WideParams p, int NW) {
  __shared__ __attribute__((aligned(16))) uint16_t ys[4][16 * kYStride];
  __shared__ __attribute__((aligned(16))) uint16_t s_svh[4][128], s_bias[4][128];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kh = NW / 4, blocks = (p.M + 15) >> 4, job = blockIdx.x * 4 + wave;
  const int half = job % kh, ub = job / kh;  // ub = unit * blocks + row block
  const int unit = ub / blocks, row0 = (ub - unit * blocks) * 16;
  if (unit >= p.units) return;  // uniform per wave
  const WideMember mm = select_wide(p, unit);
  const int col0 = (unit - mm.unit0) * 32 * NW + 128 * half;
  if (col0 >= mm.out) return;
#pragma unroll
  for (int i = lane; i < 128; i += 64) {
    s_svh[wave][i] = mm.svh[col0 + i];
    s_bias[wave][i] = mm.bias ? mm.bias[col0 + i] : 0;
  }
  const size_t sstride = (size_t)p.units * blocks * 512 * NW;
  const float* src = p.partials + ((size_t)ub * NW + 4 * half) * 512 + lane * 4;
  float4v sum[8];
#pragma unroll
  for (int f = 0; f < 8; ++f) sum[f] = *(const float4v*)(src + f * 256);
  for (int s = 1; s < p.splits; ++s) {
    float4v t[8];
#pragma unroll
    for (int f = 0; f < 8; ++f) t[f] = *(const float4v*)(src + s * sstride + f * 256);
#pragma unroll
    for (int f = 0; f < 8; ++f) sum[f] += t[f];
  }
  const int g = lane >> 4, n = lane & 15;
  uint16_t* y = ys[wave] + 4 * g * kYStride + 16 * (n >> 3) + 2 * (n & 7);
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      *(half2v*)(y + r * kYStride + 32 * i) = pack_f16(sum[2 * i][r], sum[2 * i + 1][r]);
  const QmmOut out{mm.y, mm.y_dtype, mm.bias != nullptr};
  // a wave's own rows: its LDS accesses stay in order
  qmm_finish16(ys[wave], kYStride, s_svh[wave], s_bias[wave], lane, p.M - row0, out, p.x_dtype,
               (size_t)row0 * mm.out + col0, mm.out);
}

}  // namespace exl3
