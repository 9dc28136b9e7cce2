// fmxq_route.hip -- MoE routers: the expert choice and weights that feed
// switchGLU (switch_glu.go:107-153) and the weighted combine.
//
//   - route_kernel<.., GROUP=false>: the softmax router of qwen3NextMoE
//     (qwen3next_forward.go:513-518): gates = softmax(logits), the top_k gates,
//     optionally renormalized over the selection.
//   - route_kernel<.., GROUP=true>: DeepSeek-V3's group-limited router
//     (routeExperts, deepseekv3_forward.go:452-491; CPU restatement
//     GroupExpertSelect, deepseekv3.go:305-384): sigmoid scores plus the
//     correction bias, the topk_group groups with the best sum of their two
//     best biased scores kept (the others' biased scores set to 0), the top_k
//     experts by biased score, their unbiased sigmoid scores optionally
//     renormalized over the selection and scaled by routed_scaling_factor.
//
// One wave per token row.  Element e of the row sits in lane e % 64, slot
// e / 64.  Selection is k rounds of a wave-wide maximum; equal values go to the
// lower index, which is the order the reference's stable sorts produce.  The
// arithmetic is fp32 (the reference fixture for the group router is a float32
// sigmoid compared at 1e-5).  Outputs are written in selection order (highest
// first): inds [T, k] uint32 and weights [T, k] fp32 or bf16.
//
// The row's E values are a few KB, so the kernel is one chain of dependent
// cross-lane steps and nothing else: its time is that chain's latency at any T
// that fits the chip.  So a round holds as few steps as it can: the values are
// compared as order-preserving uint32 keys, the wave's maximum is six DPP steps
// (ds_bpermute shuffles of (value, index) pairs take an LDS round trip each), and
// the winner's index comes from a ballot per slot (the lowest slot, then the
// lowest lane holding the maximum) instead of travelling with the value.  The
// picked source values are read back from LDS once, after the last round.  The
// group scores use 64 / n_group lanes for each group at once instead of a
// wave-wide reduction per group.  Measured (rocprof medians): E = 512, k = 10 softmax
// at T = 1 10.8 -> 6.6 us; E = 256, k = 8 of 4 of 8 groups at T = 1024 15.6 -> 8.1 us.
#include "fmxq_common.hpp"
#include "fmxq_internal.hpp"

namespace fmxq {
namespace {

constexpr float kNegInf = -__builtin_inff();

template <int CTRL, int RMASK>
__device__ __forceinline__ uint32_t dpp_or(uint32_t old, uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp((int)old, (int)v, CTRL, RMASK, 0xf, false);
}

// The wave's maximum on DPP: quad swaps, half-row and row mirrors, then the row
// broadcasts, which leave it in lane 63.
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
  v = max(v, dpp_or<0xb1, 0xf>(0, v));
  v = max(v, dpp_or<0x4e, 0xf>(0, v));
  v = max(v, dpp_or<0x141, 0xf>(0, v));
  v = max(v, dpp_or<0x140, 0xf>(0, v));
  v = max(v, dpp_or<0x142, 0xa>(0, v));
  v = max(v, dpp_or<0x143, 0xc>(0, v));
  return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// The wave's sum in every lane, added as __shfl_xor by 32, 16, .. 1 adds it (wave_sum),
// so that the weights do not depend on how the lanes are read: half and row swaps for
// the first two steps, then DPP.  After the step of distance d a lane's value depends on
// its number mod d only, so a rotation within the row of 16 reads the same value as xor.
__device__ __forceinline__ float wave_add(float v) {
  const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(h[0]) + __uint_as_float(h[1]);
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  v += __uint_as_float(dpp_or<0x128, 0xf>(0, __float_as_uint(v)));  // row_ror:8
  v += __uint_as_float(dpp_or<0x124, 0xf>(0, __float_as_uint(v)));  // row_ror:4
  v += __uint_as_float(dpp_or<0x4e, 0xf>(0, __float_as_uint(v)));   // quad_perm [2,3,0,1]
  v += __uint_as_float(dpp_or<0xb1, 0xf>(0, __float_as_uint(v)));   // quad_perm [1,0,3,2]
  return v;
}

// Order-preserving key: a < b as floats exactly when key(a) < key(b), -0 equal to
// +0; 0 (below every number's key) for NaN, which is never picked.
__device__ __forceinline__ uint32_t order_key(float f) {
  const uint32_t u = __float_as_uint(f + 0.f);
  const uint32_t k = u ^ ((uint32_t)((int32_t)u >> 31) | 0x80000000u);
  return f == f ? k : 0u;
}
__device__ __forceinline__ float key_value(uint32_t k) {
  return __uint_as_float(k ^ (k & 0x80000000u ? 0x80000000u : 0xffffffffu));
}

template <typename TIn>
__device__ __forceinline__ float load_in(const TIn* p, int64_t i);
template <>
__device__ __forceinline__ float load_in<float>(const float* p, int64_t i) { return p[i]; }
template <>
__device__ __forceinline__ float load_in<uint16_t>(const uint16_t* p, int64_t i) {
  return bf16_bits_to_f32(p[i]);
}

template <typename TIn, int EPL, bool GROUP, bool OUT_BF16>
__global__ __launch_bounds__(256) void route_kernel(RouteArgs a) {
  // Per wave: the values the weights are taken from, by expert (GROUP: first the
  // biased scores the groups are scored from), and the group scores.
  __shared__ float vals[4][64 * EPL];
  __shared__ float gscore[GROUP ? 4 : 1][64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t row = (int64_t)blockIdx.x * 4 + wave;
  if (row >= a.T) return;  // whole waves only: T rows, 4 per block
  const TIn* in = static_cast<const TIn*>(a.logits) + row * a.E;
  const int E = (int)a.E;
  float* const mine = vals[wave];

  float v[EPL];    // selection value
  float src[EPL];  // value the weight is taken from
#pragma unroll
  for (int j = 0; j < EPL; ++j) {
    const int e = lane + 64 * j;
    v[j] = e < E ? load_in<TIn>(in, e) : kNegInf;
  }

  if constexpr (!GROUP) {
    float m = kNegInf;
#pragma unroll
    for (int j = 0; j < EPL; ++j) m = fmaxf(m, v[j]);
    // The maximum number among the logits (a NaN gives key 0 and is passed over,
    // as fmaxf does; with no number at all the sum below is NaN either way).
    m = key_value(max(wave_max_u32(order_key(m)), order_key(kNegInf)));
    float s = 0.f;
#pragma unroll
    for (int j = 0; j < EPL; ++j) {
      const int e = lane + 64 * j;
      v[j] = e < E ? expf(v[j] - m) : 0.f;
      s += v[j];
    }
    s = wave_add(s);
    const float inv = 1.f / s;
#pragma unroll
    for (int j = 0; j < EPL; ++j) {
      v[j] *= inv;
      src[j] = v[j];
    }
  } else {
#pragma unroll
    for (int j = 0; j < EPL; ++j) {
      const int e = lane + 64 * j;
      src[j] = 1.f / (1.f + expf(-v[j]));
      v[j] = src[j] + (a.bias && e < E ? a.bias[e] : 0.f);
    }
    if (a.n_group > 1) {
      const int ng = a.n_group, per = E / ng;
#pragma unroll
      for (int j = 0; j < EPL; ++j) mine[lane + 64 * j] = v[j];
      __builtin_amdgcn_wave_barrier();
      // Group score: the sum of the group's two best biased scores (one when a
      // group holds a single expert).  L lanes (a power of two) work on each group.
      const int L = 1 << (31 - __builtin_clz(64 / ng));
      const int g = lane / L, sub = lane % L;
      float t1 = kNegInf, t2 = kNegInf;
      if (g < ng)
        for (int i = sub; i < per; i += L) {
          const float x = mine[g * per + i];
          t2 = fmaxf(t2, fminf(t1, x));
          t1 = fmaxf(t1, x);
        }
      for (int off = L >> 1; off >= 1; off >>= 1) {
        const float o1 = __shfl_xor(t1, off, 64), o2 = __shfl_xor(t2, off, 64);
        const float hi = fmaxf(t1, o1);
        t2 = fmaxf(fminf(t1, o1), fmaxf(t2, o2));
        t1 = hi;
      }
      if (g < ng && sub == 0) gscore[wave][g] = per > 1 ? t1 + t2 : t1;
      __builtin_amdgcn_wave_barrier();
      // Keep the topk_group best groups (ties to the lower group index): those
      // that fewer than topk_group others beat.
      bool kept = false;
      if (lane < ng) {
        const uint32_t ks = order_key(gscore[wave][lane]);
        int better = 0;
        for (int h = 0; h < ng; ++h) {
          const uint32_t kh = order_key(gscore[wave][h]);
          better += kh > ks || (kh == ks && h < lane);
        }
        kept = ks != 0 && better < a.topk_group;
      }
      const uint64_t keep = __ballot(kept);
      // e / per as a multiplication: exact for e < 1024 and per <= 512.
      const uint32_t inv_per = (1u << 20) / (uint32_t)per + 1u;
#pragma unroll
      for (int j = 0; j < EPL; ++j)
        if (!((keep >> ((lane + 64 * j) * inv_per >> 20 & 63u)) & 1)) v[j] = 0.f;
      __builtin_amdgcn_wave_barrier();
    }
  }
#pragma unroll
  for (int j = 0; j < EPL; ++j) mine[lane + 64 * j] = src[j];

  // Top-k: lane r keeps the r-th pick's index (0xffffffff when no candidate is
  // left: the callers' id check reports it).
  uint32_t key[EPL];
#pragma unroll
  for (int j = 0; j < EPL; ++j) key[j] = lane + 64 * j < E ? order_key(v[j]) : 0u;
  const int k = a.k;
  uint32_t my_idx = 0xffffffffu;
  for (int r = 0; r < k; ++r) {
    uint32_t best = key[0];
#pragma unroll
    for (int j = 1; j < EPL; ++j) best = max(best, key[j]);
    best = wave_max_u32(best);
    if (best == 0) break;
    uint32_t idx = 0;
    uint64_t found = 0;
#pragma unroll
    for (int j = EPL - 1; j >= 0; --j) {
      const uint64_t at = __ballot(key[j] == best);
      found = at ? at : found;
      idx = at ? 64u * j : idx;
    }
    const uint32_t wl = (uint32_t)__builtin_ctzll(found);
    idx += wl;
#pragma unroll
    for (int j = 0; j < EPL; ++j)
      if ((uint32_t)(lane + 64 * j) == idx) key[j] = 0;
    if (lane == r) my_idx = idx;
  }
  __builtin_amdgcn_wave_barrier();
  float my_w = my_idx != 0xffffffffu ? mine[my_idx] : 0.f;
  // GroupExpertSelect renormalizes only a selection of two or more
  // (deepseekv3.go:363); qwen3NextMoE renormalizes any selection
  // (qwen3next_forward.go:517-518).
  if (a.norm && (!GROUP || k > 1)) {
    const float s = wave_add(lane < k ? my_w : 0.f);
    if (s != 0.f) my_w = my_w / s;
  }
  my_w *= a.scale;
  if (lane < k) {
    a.inds[row * k + lane] = my_idx;
    if constexpr (OUT_BF16)
      static_cast<uint16_t*>(a.weights)[row * k + lane] = (uint16_t)f32_to_bf16_rne(my_w);
    else
      static_cast<float*>(a.weights)[row * k + lane] = my_w;
  }
}

template <typename TIn, bool GROUP, bool OUT_BF16>
hipError_t launch_epl(const RouteArgs& a, hipStream_t stream) {
  const unsigned blocks = (unsigned)((a.T + 3) / 4);
  if (a.E <= 64) route_kernel<TIn, 1, GROUP, OUT_BF16><<<blocks, 256, 0, stream>>>(a);
  else if (a.E <= 128) route_kernel<TIn, 2, GROUP, OUT_BF16><<<blocks, 256, 0, stream>>>(a);
  else if (a.E <= 256) route_kernel<TIn, 4, GROUP, OUT_BF16><<<blocks, 256, 0, stream>>>(a);
  else if (a.E <= 512) route_kernel<TIn, 8, GROUP, OUT_BF16><<<blocks, 256, 0, stream>>>(a);
  else route_kernel<TIn, 16, GROUP, OUT_BF16><<<blocks, 256, 0, stream>>>(a);
  return hipGetLastError();
}

template <bool GROUP>
hipError_t launch_route_kind(const RouteArgs& a, hipStream_t stream) {
  if (a.in_bf16)
    return a.out_bf16 ? launch_epl<uint16_t, GROUP, true>(a, stream)
                      : launch_epl<uint16_t, GROUP, false>(a, stream);
  return a.out_bf16 ? launch_epl<float, GROUP, true>(a, stream)
                    : launch_epl<float, GROUP, false>(a, stream);
}

}  // namespace

hipError_t launch_route(const RouteArgs& a, bool group, hipStream_t stream) {
  if (a.T <= 0) return hipSuccess;
  if (a.E < 1 || a.E > kRouteMaxExperts || a.k < 1 || a.k > 64 || a.k > a.E)
    return hipErrorInvalidValue;
  if (group && (a.n_group < 1 || a.n_group > 64 || a.E % a.n_group != 0 || a.topk_group < 1))
    return hipErrorInvalidValue;
  return group ? launch_route_kind<true>(a, stream) : launch_route_kind<false>(a, stream);
}

}  // namespace fmxq
