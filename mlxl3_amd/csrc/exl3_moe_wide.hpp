// Grouped expert QMMs for many rows per expert (prefill): the decode-in-registers
// loop of exl3_wide.hpp over blocks of up to 16*R rows of one expert, in place of
// moe_mm_kernel's 64-row blocks (which decode a 125-row expert's weights twice,
// between barriers that the decode and the MFMAs do not overlap across).
//
//   moe_wide_kernel:  per (block, 128 columns of the gate, the up or the down bank)
//     four waves, two workgroups per CU, so that one's ring fill and epilogue run
//     beside the other's loop (an expert's K-ranges are 12 to 32 steps).  Gate and up
//     leave their f16 sums, the down's epilogue is finish_and_reduce's per-slot
//     part (moe.rs:586-609);
//   moe_glu_kernel:   glu_down_input (moe.rs:435-563; GELU banks: forward_gelu,
//     moe.rs:1087-1153) on 16 rows x 128 columns per wave.
//
// Every Hadamard of the epilogues is an MFMA per 16 columns and adds between a
// lane's results (qmm_finish16): by lane exchanges, as moe_finish_row has them,
// the epilogues of 16 000 routed rows took about as long as the weights.
#pragma once

#include "exl3_moe.hpp"
#include "exl3_wide.hpp"

namespace exl3 {

// Row blocks of 16 per workgroup: as many as two workgroups' rings leave room for
// (K = 8's trellis ring is the largest).
template <int K>
constexpr int kMoeWideR = K == 8 ? 8 : 10;

constexpr int kGluStride = 264;  // halves per staged row of a gate/up pair

// The staged rows' operand of group i: row n, positions 16i + 4g + 0..3.
__device__ __forceinline__ void load_staged(const uint16_t* ys, int stride, int lane,
                                            half4 (&in)[8]) {
#pragma unroll
  for (int i = 0; i < 8; ++i)
    in[i] = *(const half4*)(ys + (lane & 15) * stride + 16 * i + 4 * (lane >> 4));
}

// glu_down_input / forward_gelu's glue for 16 staged rows: gate columns 0..127 and
// up columns 128..255 at `ys`, scales of the 128 columns in LDS, the down
// projection's xhat to dst (row n's first of the 128 columns).
template <bool GELU>
__device__ __forceinline__ void moe_glu16(const uint16_t* ys, const uint16_t* gsv,
                                          const uint16_t* usv, const uint16_t* dsu, int col0,
                                          int logical_hidden, uint16_t* dst, int width, int rows,
                                          int lane) {
  const int g = lane >> 4;
  const half4 hs = h16_row<true>(lane);
  half4 in[8];
  float a[8][4], u[8][4];
  load_staged(ys, kGluStride, lane, in);
  h128_mfma<GELU>(in, hs, a);
  load_staged(ys + 128, kGluStride, lane, in);
  h128_mfma<GELU>(in, hs, u);
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int c = 16 * i + 4 * g;
    const half4 gs = *(const half4*)(gsv + c), us = *(const half4*)(usv + c);
    const half4 ds = *(const half4*)(dsu + c);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float act;
      if constexpr (GELU) {
        const float gv = round_f16(round_f16(a[i][r] * kHadScale) * (float)gs[r]);
        const float uv = round_f16(round_f16(u[i][r] * kHadScale) * (float)us[r]);
        act = col0 + c + r < logical_hidden ? geglu_f16(gv, uv) : 0.f;
      } else {
        const float gv = round_f16(a[i][r] * kHadScale * (float)gs[r]);
        const float uv = round_f16(u[i][r] * kHadScale * (float)us[r]);
        act = round_f16((gv / (1.0f + expf(-gv))) * uv);
      }
      in[i][r] = (_Float16)(act * (float)ds[r]);
    }
  }
  h128_mfma<GELU>(in, h16_row<false>(lane), a);
  const int n = lane & 15;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const half2v lo = pack_f16(a[i][0] * kHadScale, a[i][1] * kHadScale);
    const half2v hi = pack_f16(a[i][2] * kHadScale, a[i][3] * kHadScale);
    *(half4*)(ys + n * kGluStride + 16 * i + 4 * g) = half4{lo[0], lo[1], hi[0], hi[1]};
  }
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const int row = 4 * t + g;
    const half8 o = *(const half8*)(ys + row * kGluStride + 8 * n);
    if (row < rows) *(half8*)(dst + (size_t)row * width + 8 * n) = o;
  }
}

// finish_and_reduce's per-slot part for 16 staged rows x 128 columns: z of the
// first `rows` rows at their slots (slots: the block's sorted positions from this
// row group on).
__device__ __forceinline__ void moe_down16(uint16_t* ys, int stride, const uint16_t* svh,
                                           const MoeMmParams& p, const int* slots, int col0, int rows, int lane) {
  const int g = lane >> 4, n = lane & 15;
  half4 in[8];
  float v[8][4];
  load_staged(ys, stride, lane, in);
  const int slot = slots[min(n, rows - 1)];
  h128_mfma<true>(in, h16_row<true>(lane), v);
  const float sc = load_score(p.scores, p.scores_dtype, slot);
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int c = 16 * i + 4 * g;
    const half4 sv = *(const half4*)(svh + c);
    float o[4];
#pragma unroll
    for (int r = 0; r < 4; ++r)
      o[r] = weighted(round_f16(round_f16(v[i][r] * kHadScale) * (float)sv[r]), sc, p.scores_dtype);
    if (p.scores_dtype == DT_F16) {
      const half2v lo = pack_f16(o[0], o[1]), hi = pack_f16(o[2], o[3]);
      *(half4*)(ys + n * stride + c) = half4{lo[0], lo[1], hi[0], hi[1]};
    } else if (n < rows) {
      *(float4v*)((float*)p.z + (size_t)slot * p.width + col0 + c) =
          float4v{o[0], o[1], o[2], o[3]};
    }
  }
  if (p.scores_dtype != DT_F16) return;
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const int row = 4 * t + g;
    const half8 o = *(const half8*)(ys + row * stride + 8 * n);
    if (row < rows) *(half8*)((uint16_t*)p.z + (size_t)slots[row] * p.width + col0 + 8 * n) = o;
  }
}

// Launch 1 of the forward where the expert QMMs are these: the route plan
// (moe_route_kernel's) beside the gather of the gate/up inputs, one wave per (16
// slots, projection, 128-block) with the Hadamard by MFMA (~30 -> ~9 VALU
// instructions per element).  grid 1 + ceil(ceil(slots / 16) * 2 * blocks / 4), 256
// threads, (3 * experts + 1) ints of dynamic LDS.
template <bool VEC>
__global__ __launch_bounds__(256) void moe_route16_kernel(MoePlanParams pp, MoeGatherParams p) {
  if (blockIdx.x == 0) {
    moe_plan_block<256>(pp);
    return;
  }
  __shared__ __attribute__((aligned(16))) uint16_t ys[4][16 * kYStride];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int job = (blockIdx.x - 1) * 4 + wave;
  const int nb = p.in >> 7, pair = job / nb, b = job - pair * nb;
  const int proj = pair & 1, slot0 = 16 * (pair >> 1) + (lane >> 4);
  if (16 * (pair >> 1) >= p.slots) return;  // uniform per wave
  const size_t c0 = (size_t)b * 128 + 8 * (lane & 15);
  uint32_t e[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) e[t] = p.selected[min(slot0 + 4 * t, p.slots - 1)];
  half8 io[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const int slot = min(slot0 + 4 * t, p.slots - 1);
    const size_t ex = e[t] < (uint32_t)p.experts ? e[t] : 0u;
    io[t] = scaled8<VEC>(p.x, p.x_dtype, (size_t)(slot / p.top_k) * p.in + c0,
                         p.gu_suh + (ex * 2 + proj) * p.in + c0);
  }
  h128_rows16(io, ys[wave], lane);
#pragma unroll
  for (int t = 0; t < 4; ++t)
    if (slot0 + 4 * t < p.slots && e[t] < (uint32_t)p.experts)
      store8<VEC>(io[t], p.xgu + ((size_t)proj * p.slots + slot0 + 4 * t) * p.in + c0);
}

// Workgroup -> (block, column unit): XCD x takes blocks x, x + 8, ... whole, as in
// moe_mm_kernel, so a block's rows are read into one L2.  grid: blocks rounded up
// to 8, times `units` (NPROJ * width / 128).
template <int K, int CB, int NPROJ>
__global__ __launch_bounds__(256) void moe_wide_kernel(MoeMmParams p, int units, uint16_t* raw) {
  constexpr int R = kMoeWideR<K>, NW = 4;
  using C = WideShape<K, R, NW>;
  __shared__ __attribute__((aligned(16))) uint8_t lds[C::kLds];
  __shared__ __attribute__((aligned(16))) uint16_t s_sv[128];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wk = blockIdx.x >> 3;
  const int blk = (wk / units) * 8 + (blockIdx.x & 7), unit = wk % units;
  if (blk >= p.counts[0]) return;  // uniform
  const int4 ent = p.table[blk];
  const int e = __builtin_amdgcn_readfirstlane(ent.x), pos0 = __builtin_amdgcn_readfirstlane(ent.y);
  const int nrows = __builtin_amdgcn_readfirstlane(ent.z);
  const int live = (nrows + 15) >> 4, nq = p.k_in >> 6;
  const int tpe = p.width / 16;
  const int proj = NPROJ == 2 && unit >= p.col_blocks ? 1 : 0;
  const int cblk = unit - proj * p.col_blocks;
  const int tcol = (proj * p.experts + e) * tpe + cblk * 8;
  if (NPROJ == 1 && threadIdx.x < 128)
    s_sv[threadIdx.x] = p.down_svh[(size_t)e * p.width + cblk * 128 + threadIdx.x];
  const WideSource asrc =
      wide_source(p.xa, (size_t)NPROJ * p.slots_pad * p.k_in * sizeof(uint16_t), 128);
  const size_t row_bytes = (size_t)p.tn_total * (32 * K), wfirst = (size_t)tcol * (32 * K);
  const WideSource wsrc =
      wide_source((const uint8_t*)p.trellis + wfirst, row_bytes * (p.k_in >> 4) - wfirst,
                  (uint32_t)(4 * row_bytes));
  uint32_t aoff[C::PA], woff[C::PW];
#pragma unroll
  for (int i = 0; i < C::PA; ++i) {
    // rows past the block's end repeat its last one (never stored)
    const int r = 8 * min(wave + NW * i, C::kAJobs - 1) + (lane >> 3);
    const int at = pos0 + min(r, nrows - 1);
    const int arow = p.a_rows ? p.a_rows[at] : at;
    aoff[i] = (uint32_t)((((size_t)proj * p.slots_pad + arow) * p.k_in +
                          ((lane & 7) ^ a_swizzle(r)) * 8) * 2);
  }
#pragma unroll
  for (int i = 0; i < C::PW; ++i) {
    const uint32_t at = (uint32_t)min(wave + NW * i, C::kWJobs - 1) * 1024u + 16u * lane;
    const uint32_t tr = at / (256u * K);
    woff[i] = tr * (uint32_t)row_bytes + (at - tr * (256u * K));
  }
  float4v acc[R][2];
#pragma unroll
  for (int rb = 0; rb < R; ++rb) acc[rb][0] = acc[rb][1] = float4v{0.f, 0.f, 0.f, 0.f};
  wide_mm<K, CB, R, NW, true>(lds, asrc, wsrc, aoff, woff, nq, live, wave, lane, acc);
  uint16_t* ys = (uint16_t*)lds;
  wide_stage_rows<R>(acc, ys, C::kStride, wave, lane);
  __syncthreads();
  for (int u = wave; u < live; u += NW) {
    uint16_t* y = ys + 16 * u * C::kStride;
    if constexpr (NPROJ == 2) {
      // the staged rows as they are (moe_glu_kernel reads their order)
      uint16_t* dst = raw + ((size_t)proj * p.slots_pad + pos0 + 16 * u) * p.width + cblk * 128 +
                      8 * (lane & 15);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int row = 4 * t + (lane >> 4);
        const half8 o = *(const half8*)(y + row * C::kStride + 8 * (lane & 15));
        if (16 * u + row < nrows) *(half8*)(dst + (size_t)row * p.width) = o;
      }
    } else {
      moe_down16(y, C::kStride, s_sv, p, p.sorted_slot + pos0 + 16 * u, cblk * 128,
                 nrows - 16 * u, lane);
    }
  }
}

// The GLU edge between moe_wide_kernel's gate/up and down launches: raw
// [2][slots_pad][width] (the staged rows' column order) -> xd.  grid: (blocks, width
// / 128), 256 threads, 16 rows per wave and pass.
template <bool GELU>
__global__ __launch_bounds__(256) void moe_glu_kernel(MoeMmParams p, const uint16_t* raw) {
  __shared__ __attribute__((aligned(16))) uint16_t ys[4][16 * kGluStride];
  __shared__ __attribute__((aligned(16))) uint16_t s_sv[256], s_dsu[128];
  const int lane = threadIdx.x & 63, g = lane >> 4, n = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int blk = blockIdx.x, cblk = blockIdx.y;
  if (blk >= p.counts[0]) return;  // uniform
  const int4 ent = p.table[blk];
  const int e = ent.x, pos0 = ent.y, nrows = ent.z, live = (nrows + 15) >> 4;
  const int c = threadIdx.x & 127, h = threadIdx.x >> 7;
  s_sv[threadIdx.x] = p.gu_svh[((size_t)e * 2 + h) * p.width + cblk * 128 + c];
  if (h == 0) s_dsu[c] = p.down_suh[(size_t)e * p.width + cblk * 128 + c];
  __syncthreads();
  for (int u = wave; u < live; u += 4) {
    const size_t at = (size_t)(pos0 + 16 * u) * p.width + cblk * 128;
    half8 io[2][4];
#pragma unroll
    for (int pj = 0; pj < 2; ++pj)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int row = min(4 * t + g, nrows - 16 * u - 1);
        io[pj][t] = *(const half8*)(raw + (size_t)pj * p.slots_pad * p.width + at +
                                    (size_t)row * p.width + 8 * n);
      }
#pragma unroll
    for (int pj = 0; pj < 2; ++pj)
#pragma unroll
      for (int t = 0; t < 4; ++t)
        *(half8*)(ys[wave] + (4 * t + g) * kGluStride + 128 * pj + 8 * n) = io[pj][t];
    moe_glu16<GELU>(ys[wave], s_sv, s_sv + 128, s_dsu, cblk * 128, p.logical_hidden, p.xd + at,
                    p.width, nrows - 16 * u, lane);
  }
}

}  // namespace exl3
