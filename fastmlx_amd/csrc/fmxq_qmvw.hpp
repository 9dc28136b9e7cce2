// fmxq_qmvw.hpp -- the skinny product with x shared through LDS (qmvw_kernel) for one
// group size, and its launcher.  Block: WV waves side by side over WV * 16 NTT rows of W
// and one K part (steps [s0, s1) of 256 values); the block's x rows (16 MT of them) go
// to LDS once per step for all its waves (qmvs_walk_xlds), so x costs the texture units
// a 1 / WV share of what it costs qmvs, where every wave loads its own.
// Grid: (row blocks, K parts).  One part stores bf16 outputs; several write fp32
// partials [part][M][N] to a.ws and qmvw_fixup_kernel sums them in part order.
// fmxq_skinny.hip builds it for groups of 64, fmxq_qmvw_fmt.hip for 32 and 128.
#pragma once
#include "fmxq_common.hpp"
#include "fmxq_internal.hpp"
#include "fmxq_qmvs.hpp"

namespace fmxq {
namespace {

// The pipelined walk dequantizes the weights (qmvs_walk_xlds DEQ) from this many
// 16-row x tiles: at M = 64, 30.3 -> 24.2 us on 14336x4096 and 29.3 -> 23.6 us on
// 4096x14336; at M = 32 on 4096x14336 19.5 -> 17.9 us.
#ifndef FMXQ_QMVW_DEQ_MIN_MT
#define FMXQ_QMVW_DEQ_MIN_MT 2
#endif
constexpr int kQmvwDeqMinMT = FMXQ_QMVW_DEQ_MIN_MT;
// The up-front walk likewise from 2 tiles (C1 stack at M = 24 / 32: 3.03 -> 2.99 ms,
// 3.09 -> 3.01 ms); at one tile the exponent-trick form is quicker (M = 16 on
// 14336x4096: 16.0 against 17.7 us dequantized).
#ifndef FMXQ_QMVW_XALL_DEQ_MIN_MT
#define FMXQ_QMVW_XALL_DEQ_MIN_MT 2
#endif
constexpr int kQmvwXallDeqMinMT = FMXQ_QMVW_XALL_DEQ_MIN_MT;

// int8 weights in groups of 64 always take the dequantizing walks.  Groups of 32 and
// 128 keep the exact affine form for one x tile (at 8 bits and few rows they came from
// the exact dot2 GEMV) and dequantize from two, as the prefill GEMM they came from does.
// That GEMM also answers rows of x with infinities, so the affine form takes its
// non-finite outputs again, dequantized (deq_row_dot, over the block's own K part).
template <int MT, int NTT, int WV, int D, int BITS, int GS>
__global__ __launch_bounds__(WV * 64) __attribute__((amdgpu_waves_per_eu(MT == 1 && NTT == 1 && !(BITS == 8 && GS == 32) ? 3 : 2)))
void qmvw_kernel(QmmArgs a) {
  using G = QmvsGeom<NTT, 4, BITS, GS>;
  constexpr bool kDeqXlds = (BITS == 8 && GS == 64) || MT >= kQmvwDeqMinMT;
  constexpr bool kDeqXall = (BITS == 8 && GS == 64) || MT >= kQmvwXallDeqMinMT;
  constexpr int AX = 8 * MT / WV;
  constexpr int XSLOTS = D > 0 ? D : 2;
  __shared__ __attribute__((aligned(1024))) uint8_t xs[XSLOTS][16 * MT * kXStageRow];
  __shared__ __attribute__((aligned(16))) uint8_t stage[WV][G::STAGE];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c16 = lane & 15, q = lane >> 4;
  const int64_t nb = (int64_t)blockIdx.x * (16 * NTT * WV) + wave * (16 * NTT);
  const int parts = a.splits > 1 ? a.splits : 1;
  const int part = (int)blockIdx.y;
  const int64_t nst = a.K / 256;
  const int64_t s0 = part * nst / parts, s1 = (part + 1) * nst / parts;

  // x through a buffer resource (qmvw_supported keeps its byte size below 2^31).
  // DMA instruction j of this wave fills stage rows 2 (AX wave + j) and the next
  // (qmvs_walk_xlds); a row past M reads row M - 1 and reaches no stored output.
  const __amdgpu_buffer_rsrc_t xres = __builtin_amdgcn_make_buffer_rsrc(
      (void*)a.x, (short)0, (int)(((a.M - 1) * a.ldx + a.K) * 2), 0x00020000);
  uint32_t xo[AX];
#pragma unroll
  for (int j = 0; j < AX; ++j) {
    const int r = 2 * (wave * AX + j) + (lane >> 5);
    const int c = (lane & 31) ^ (r & 15);
    const int64_t xr = r < a.M ? r : a.M - 1;
    xo[j] = (uint32_t)(xr * a.ldx * 2 + c * 16);
  }
  f32x4 acc[1][MT][NTT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int t = 0; t < NTT; ++t) acc[0][mt][t] = f32x4{};
  if constexpr (D > 0) {
    qmvs_walk_xall<MT, NTT, WV, D, kDeqXall, BITS, GS>(&xs[0][0], stage[wave], xres, xo, wave,
                                                              a.w, a.scales, a.biases,
                                   nb, a.N, a.K, s0, s1, acc);
  } else {
    const uint32_t* const w[1] = {a.w};
    const uint16_t* const sc[1] = {a.scales};
    const uint16_t* const bi[1] = {a.biases};
    qmvs_walk_xlds<MT, MT, NTT, 1, WV, false, kDeqXlds, BITS, GS>(xs[0], xs[1], stage[wave], xres, xo,
                                                                     wave, a.M, w, sc, bi,
                                       nb, a.N, a.K, s0, s1, acc);
  }

  // C layout of a 16x16 tile: register r of lane l is row 4 (l / 16) + r, column
  // l % 16.
  constexpr bool kRedo = GS != 64 && !(D > 0 ? kDeqXall : kDeqXlds);
  static_assert(!kRedo || NTT * MT * 4 <= 32, "one bit per output of a lane");
  uint32_t odd = 0;
  auto put = [&](int64_t m, int64_t n, float v) {
    if (parts == 1) a.y[m * a.ldy + n] = finish_out(v, a.bias, n);
    else a.ws[((int64_t)part * a.M + m) * a.N + n] = v;
  };
#pragma unroll
  for (int t = 0; t < NTT; ++t) {
    const int64_t n = nb + 16 * t + c16;
    if (n >= a.N) continue;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t m = 16 * mt + 4 * q + r;
        if (m >= a.M) continue;
        const float v = acc[0][mt][t][r];
        if constexpr (kRedo) odd |= __builtin_isfinite(v) ? 0u : 1u << ((t * MT + mt) * 4 + r);
        put(m, n, v);
      }
  }
  if constexpr (kRedo) {
    while (odd) {
      const int i = __builtin_ctz(odd);
      odd &= odd - 1;
      const int64_t m = 16 * ((i >> 2) % MT) + 4 * q + (i & 3), n = nb + 16 * ((i >> 2) / MT) + c16;
      put(m, n, deq_row_dot<BITS, GS>(a.x + m * a.ldx, a.w + n * (a.K * BITS / 32), a.scales + n * (a.K / GS),
                                      a.biases + n * (a.K / GS), s0 * 256, s1 * 256));
    }
  }
}

// Grid (ceil(N / 1024), M): thread t of block x sums the parts of outputs
// 4 (256 x + t) .. +4 of row blockIdx.y (N % 4 == 0, so 16-byte pieces), or of
// output 256 x + t alone when N % 4 != 0 (grid x then ceil(N / 256)).  All parts
// are loaded before the first add (at most kQmvwMaxParts), so a thread waits for
// one round trip instead of one per part; the sum runs in part order.

__global__ __launch_bounds__(256) void qmvw_fixup_kernel(QmmArgs a) {
  const int64_t m = blockIdx.y;
  const int64_t mn = a.M * a.N;
  const float* src = a.ws + m * a.N;
  uint16_t* dst = a.y + m * a.ldy;
  const int parts = a.splits;
  if ((a.N & 3) == 0) {
    const int64_t n = 4 * ((int64_t)blockIdx.x * 256 + threadIdx.x);
    if (n >= a.N) return;
    f32x4 v[kQmvwMaxParts];
#pragma unroll
    for (int p = 0; p < kQmvwMaxParts; ++p)
      if (p < parts) v[p] = *reinterpret_cast<const f32x4*>(src + p * mn + n);
    f32x4 t = v[0];
#pragma unroll
    for (int p = 1; p < kQmvwMaxParts; ++p)
      if (p < parts) t += v[p];
#pragma unroll
    for (int i = 0; i < 4; ++i) dst[n + i] = finish_out(t[i], a.bias, n + i);
  } else {
    const int64_t n = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (n >= a.N) return;
    float v[kQmvwMaxParts];
#pragma unroll
    for (int p = 0; p < kQmvwMaxParts; ++p)
      if (p < parts) v[p] = src[p * mn + n];
    float t = v[0];
#pragma unroll
    for (int p = 1; p < kQmvwMaxParts; ++p)
      if (p < parts) t += v[p];
    dst[n] = finish_out(t, a.bias, n);
  }
}

template <int MT, int NTT, int WV, int D, int GS>
hipError_t launch_qmvw_cfg(const QmmArgs& a, hipStream_t stream) {
  const int parts = a.splits > 1 ? a.splits : 1;
  const dim3 grid((unsigned)((a.N + 16 * NTT * WV - 1) / (16 * NTT * WV)), (unsigned)parts);
  if (a.bits == 8) {
    // int8: 16-row W tiles, pipelined walk only (qmvw_plan)
    if constexpr (NTT == 1 && D == 0) qmvw_kernel<MT, 1, WV, 0, 8, GS><<<grid, WV * 64, 0, stream>>>(a);
    else return hipErrorInvalidValue;
  } else {
    qmvw_kernel<MT, NTT, WV, D, 4, GS><<<grid, WV * 64, 0, stream>>>(a);
  }
  if (parts > 1) {
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const int64_t per = (a.N & 3) == 0 ? 1024 : 256;
    qmvw_fixup_kernel<<<dim3((unsigned)((a.N + per - 1) / per), (unsigned)a.M), 256, 0, stream>>>(a);
  }
  return hipGetLastError();
}

template <int MT, int NTT, int WV, int GS>
hipError_t launch_qmvw_d(const QmmArgs& a, int d, hipStream_t stream) {
  if (d == 2) return launch_qmvw_cfg<MT, NTT, WV, 2, GS>(a, stream);
  if constexpr (MT <= 2) {
    if (d == 4) return launch_qmvw_cfg<MT, NTT, WV, 4, GS>(a, stream);
  }
  return launch_qmvw_cfg<MT, NTT, WV, 0, GS>(a, stream);
}

template <int MT, int GS>
hipError_t launch_qmvw_mt(const QmmArgs& a, int ntt, int d, hipStream_t stream) {
  if constexpr (MT <= 2) {
    if (ntt == 2) return launch_qmvw_d<MT, 2, 4, GS>(a, d, stream);
  }
  return launch_qmvw_d<MT, 1, 4, GS>(a, d, stream);
}

template <int GS>
hipError_t launch_qmvw_gs(const QmmArgs& a, const QmvwPlan& p, hipStream_t stream) {
  if (p.mt == 1) return launch_qmvw_mt<1, GS>(a, p.ntt, p.d, stream);
  if (p.mt == 2) return launch_qmvw_mt<2, GS>(a, p.ntt, p.d, stream);
  // 64-row x tiles use 16-row W tiles only (32-row ones would spill), and at most
  // two up-front steps (LDS); the pipelined walk runs 8-wave blocks.
  if (p.wv == 8) return launch_qmvw_cfg<4, 1, 8, 0, GS>(a, stream);
  return launch_qmvw_mt<4, GS>(a, 1, p.d, stream);
}

}  // namespace
}  // namespace fmxq
