// fmxq_moe_walk.hpp -- the shared-x segment walk of the grouped MoE product
// (moe_qmvw_kernel) for one weight format, and its launcher.  fmxq_moe_gemm.hip
// builds it for 4 bits in groups of 64, fmxq_moe_walk_q4.hip and
// fmxq_moe_walk_q8.hip for the other formats.
#pragma once
#include "fmxq_common.hpp"
#include "fmxq_internal.hpp"
#include "fmxq_qmvs.hpp"

namespace fmxq {
namespace {

__device__ __forceinline__ float r16(float v) { return bf16_bits_to_f32(f32_to_bf16_rne(v)); }

// Store a segment's rows.  C layout of a 16x16 tile: register r of lane l is row
// 4 (l / 16) + r, column l % 16.  Row m of tile mt is slot start + 16 mt + m; nb
// is the wave's first column.
template <int MT, int NTT, int NMAT>
__device__ __forceinline__ void store_segment(const MoeArgs& a, int64_t start, int64_t len,
                                              bool bad_e, int64_t nb,
                                              const f32x4 (&acc)[NMAT][MT][NTT]) {
  const int lane = threadIdx.x & 63;
  const int c16 = lane & 15, q = lane >> 4;
  bool raise = false;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = 16 * mt + 4 * q + r;
      if (m >= len) continue;
      const int64_t slot = start + m;
      const int64_t xr = a.lhs ? (int64_t)a.lhs[slot] : slot / a.lhs_div;
      const bool bad = bad_e || xr >= a.x_rows;
      raise |= bad;
      const int64_t orow = a.yrow ? (int64_t)a.yrow[slot] : slot;
      uint16_t* yr = a.y + orow * a.N;
#pragma unroll
      for (int t = 0; t < NTT; ++t) {
        const int64_t n = nb + 16 * t + c16;
        if (n >= a.N) continue;
        uint16_t v;
        if (bad) {
          v = 0;
        } else if constexpr (NMAT == 2) {
          const float g = r16(acc[0][mt][t][r]), u = r16(acc[1][mt][t][r]);
          const float sg_ = r16(1.f / (1.f + __expf(-g)));
          v = (uint16_t)f32_to_bf16_rne(r16(r16(g * sg_) * u));
        } else {
          v = (uint16_t)f32_to_bf16_rne(acc[0][mt][t][r]);
        }
        yr[n] = v;
      }
    }
  if (raise) atomicOr(a.err_flag, 1u);
}

#ifndef FMXQ_MOE_DEQ_MIN_MT
#define FMXQ_MOE_DEQ_MIN_MT 2
#endif
// Walks of at least this many 16-row x tiles dequantize the weights (DEQ of
// qmvs_walk_xlds) instead of folding the bias term: the 32-slot segments with
// more than 16 slots.  Measured per layer: configuration 4 at M=256 1529-1541 ->
// 1492 us, at M=32 581-583 -> 575-579 us; configuration 3 at M=512 254-259 ->
// 249-252 us, at M=128 unchanged.
constexpr int kMoeDeqMinMT = FMXQ_MOE_DEQ_MIN_MT;

// Fixed-length (16 or 32 slot) x-in-LDS form of moe_qmvs_kernel for blocks whose
// 4 waves walk the whole K range side by side (16 NTT columns each): the
// segment's x rows go to LDS once per step for all four (qmvs_walk_xlds), so a
// step's texture-unit traffic is the weights plus a quarter of x instead of the
// weights plus all of x per wave.
template <int MT, int NTT, int NMAT, int WV, int BITS, int GS>
__global__ __launch_bounds__(WV * 64) __attribute__((amdgpu_waves_per_eu(MT == 1 && NTT == 1 && !(BITS == 8 && NMAT == 2) ? 3 : 2))) void moe_qmvw_kernel(
    MoeArgs a) {
  using G = QmvsGeom<NTT, 4, BITS, GS>;
  constexpr bool kDeq = BITS == 4 && GS == 64 && MT >= kMoeDeqMinMT;
  __shared__ __attribute__((aligned(1024))) uint8_t xs[2][16 * MT * kXStageRow];
  __shared__ __attribute__((aligned(16))) uint8_t stage[WV][NMAT * G::STAGE];

  const int64_t sg = blockIdx.y;
  if (sg >= (a.seg ? (int64_t)*a.nseg : a.S)) return;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t start = a.seg ? (int64_t)a.seg[2 * sg] : sg;
  const int64_t len = a.seg ? (int64_t)a.seg[2 * sg + 1] : 1;
  const uint32_t e = a.rhs[start];
  const int64_t nb = (int64_t)blockIdx.x * (16 * NTT * WV) + wave * (16 * NTT);
  const bool sh = a.sh_seg && (int64_t)e == a.E;
  const bool bad_e = (int64_t)e >= a.E && !sh;

  f32x4 acc[NMAT][MT][NTT];
#pragma unroll
  for (int p = 0; p < NMAT; ++p)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int t = 0; t < NTT; ++t) acc[p][mt][t] = f32x4{};
  if (!bad_e) {
    const int64_t wpr = a.K * BITS / 32, gpr = a.K / GS;
    const uint32_t* w[NMAT];
    const uint16_t* sc[NMAT];
    const uint16_t* bi[NMAT];
#pragma unroll
    for (int p = 0; p < NMAT; ++p) {
      w[p] = sh ? a.sh_w[p] : a.w[p] + (int64_t)e * a.N * wpr;
      sc[p] = sh ? a.sh_s[p] : a.s[p] + (int64_t)e * a.N * gpr;
      bi[p] = sh ? a.sh_b[p] : a.b[p] + (int64_t)e * a.N * gpr;
    }
    // moe_xlds_supported keeps x_rows * K * 2 below 2^31.
    const __amdgpu_buffer_rsrc_t xres = __builtin_amdgcn_make_buffer_rsrc(
        (void*)a.x, (short)0, (int)(a.x_rows * a.K * 2), 0x00020000);
    // Byte offset of the x chunk lane `lane` fetches for DMA instruction j (see
    // qmvs_walk_xlds): stage row r is slot start + r (the first slot for a row past
    // the segment that shares an issued instruction), a bad x row reads row 0 (its
    // output is zeroed).
    auto x_offsets = [&](uint32_t* xo, int ax) {
      for (int j = 0; j < ax; ++j) {
        const int r = 2 * (wave * ax + j) + (lane >> 5);
        const int c = (lane & 31) ^ (r & 15);
        const int64_t slot = start + (r < len ? r : 0);
        int64_t xr = a.lhs ? (int64_t)a.lhs[slot] : slot / a.lhs_div;
        if (xr >= a.x_rows) xr = 0;
        xo[j] = (uint32_t)(xr * a.K * 2 + c * 16);
      }
    };
    // One matrix with K <= 512 (the down projection of 512-wide experts): a walk
    // of one or two steps, so every load is issued first (qmvs_walk_xall).
    const bool upfront = NMAT == 1 && a.K <= 512;
    if (MT == 2 && len <= 16) {
      // Short segment of a 32-slot window: 16 stage rows, one tile walked.
      uint32_t xo[8 / WV];
      x_offsets(xo, 8 / WV);
      if (upfront) {
        f32x4 acc1[1][1][NTT];
#pragma unroll
        for (int t = 0; t < NTT; ++t) acc1[0][0][t] = f32x4{};
        qmvs_walk_xall<1, NTT, WV, 2, false, BITS, GS>(&xs[0][0], stage[wave], xres, xo, wave,
                                                       w[0], sc[0], bi[0], nb, a.N, a.K, 0,
                                                       a.K / 256, acc1);
#pragma unroll
        for (int t = 0; t < NTT; ++t) acc[0][0][t] = acc1[0][0][t];
      } else {
        qmvs_walk_xlds<1, MT, NTT, NMAT, WV, true, false, BITS, GS>(
            xs[0], xs[1], stage[wave], xres, xo, wave, len, w, sc, bi, nb, a.N, a.K, 0,
            a.K / 256, acc);
      }
    } else {
      uint32_t xo[8 * MT / WV];
      x_offsets(xo, 8 * MT / WV);
      if constexpr (NMAT == 1) {
        if (upfront)
          qmvs_walk_xall<MT, NTT, WV, 2, false, BITS, GS>(&xs[0][0], stage[wave], xres, xo, wave,
                                                          w[0], sc[0], bi[0], nb, a.N, a.K, 0,
                                                          a.K / 256, acc);
      }
      if (!upfront)
        qmvs_walk_xlds<MT, MT, NTT, NMAT, WV, !kDeq, kDeq, BITS, GS>(
            xs[0], xs[1], stage[wave], xres, xo, wave, len, w, sc, bi, nb, a.N, a.K, 0,
            a.K / 256, acc);
    }
  }
  store_segment<MT, NTT, NMAT>(a, start, len, bad_e, nb, acc);
}

template <int MT, int NTT, int NMAT, int BITS, int GS>
hipError_t launch_moe_qmvw_cfg(const MoeArgs& a, int64_t max_seg, hipStream_t stream) {
  // Four waves per block: an 8-wave block (128 columns per x fetch, two blocks
  // per CU) measured slower (configuration 4 at M=256: 1871 -> 1971 us, and again
  // with the dequantizing walk: 1463-1478 -> 1553-1604 us; at M=32 with one-tile
  // segments too: 556-561 -> 620 us), unlike the dense walk's 64-row tiles.
  constexpr int64_t cols = 16 * NTT * 4;
  dim3 grid((unsigned)((a.N + cols - 1) / cols), (unsigned)max_seg);
  moe_qmvw_kernel<MT, NTT, NMAT, 4, BITS, GS><<<grid, 256, 0, stream>>>(a);
  return hipGetLastError();
}

// nmat matrices (2: gate and up), segments of at most `window` (16 or 32) slots,
// 16 ntt columns per wave (1 for two matrices).
template <int BITS, int GS>
hipError_t launch_moe_qmvw_fmt(const MoeArgs& a, int nmat, int window, int ntt, int64_t max_seg,
                               hipStream_t stream) {
  if (nmat == 2)
    return window == 16 ? launch_moe_qmvw_cfg<1, 1, 2, BITS, GS>(a, max_seg, stream)
                        : launch_moe_qmvw_cfg<2, 1, 2, BITS, GS>(a, max_seg, stream);
  if (ntt == 1)
    return window == 16 ? launch_moe_qmvw_cfg<1, 1, 1, BITS, GS>(a, max_seg, stream)
                        : launch_moe_qmvw_cfg<2, 1, 1, BITS, GS>(a, max_seg, stream);
  return window == 16 ? launch_moe_qmvw_cfg<1, 2, 1, BITS, GS>(a, max_seg, stream)
                      : launch_moe_qmvw_cfg<2, 2, 1, BITS, GS>(a, max_seg, stream);
}

}  // namespace
}  // namespace fmxq
