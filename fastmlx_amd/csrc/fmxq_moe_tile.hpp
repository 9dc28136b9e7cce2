// fmxq_moe_tile.hpp -- the grouped MoE product for longer expert runs: tiles of up to
// 64 slots of one expert by 4 x 32 columns of two matrices (gate and up), or 4 x 64
// columns of one (down).  Same products, segment table, roundings and error handling
// as the segment walk (fmxq_moe_walk.hpp), in exact affine arithmetic for every run
// (the walk dequantizes pieces of 17 and more slots to bf16).  Outputs that come out
// infinite or NaN so (an infinity in x, sums past the fp32 range) are taken again with
// the dequantized weights.
//
// What bounds it: with few slots per expert the weight stream, with many the MFMA and
// VALU work.  The walk's blocks (64 columns, 16 or 32 slots) are bound by the vector
// memory path instead: each loads its slots' x rows again for 64 columns and an
// expert's weights again for every 32 slots, so at 1024 tokens over 256 experts x
// and weights make 16 GB of L1 traffic for 4.1 GB of gate/up weights.  A tile reads x
// once per 128 (256) columns and the weights once per 64 slots.  Layers before and
// after: moe_window (fmxq_moe_gemm.hip).
//
// Block: 4 waves, two blocks per CU (one block of 8 waves and twice the columns had
// every wave of a CU at the same barrier: 512 experts, 2000 tokens 473 -> 427 us).
// Wave w owns 32 columns in each of two column groups.  A step is 128 values of K:
//   - weights: whole-segment loads (8 rows x 128 bytes an instruction: two steps of 4
//     bits, one of 8) one load ahead in registers, then through the wave's own LDS
//     stage into MFMA operand order (64-byte rows, a step of 4 bits each, made the
//     256-expert layer at 1024 tokens 2377 -> 2927 us);
//   - x: the tile's rows DMA'd (buffer_load ... lds) one step ahead into one of two
//     stages shared by the waves, 16-byte chunk c of row r at position c ^ (r & 15);
//   - one barrier per step.
// v_mfma_f32_32x32x16_bf16 with x as the A operand and the weights as B, so that a
// lane's accumulators all belong to one weight row: per group P = sum x (OFF + q)
// from zero, then acc += s P with one scale per lane (16 FMAs per 32 x 32 tile).
//
// The bias term sum_g (b - OFF s) xs_g, xs_g the x row's sum over group g, is a
// product over groups: tile_prep_kernel sums every x row once, splits each fp32 sum
// into three bf16 (24 bits: hi + mid + lo), and one MFMA adds two groups, slots
// (b b b s' s' s') against (hi mid lo hi mid lo), s' = -OFF s.  (Summed in the tile
// by the block's threads, from the x stage, the sums cost 14-16% of the layer.)
// b and s' are exact in bf16, so the products carry the sums' fp32 precision.  For 4
// bits the same pass puts x into the exponent trick's pair order, which every wave of
// every tile would otherwise permute again.
//
// Groups of 32: MFMA i of a unit must stay inside one group, so the lane halves
// exchange words (v_permlane32_swap) to hold chunks 2 i + h instead of 4 h + i.
#pragma once
#include <type_traits>

#include "fmxq_common.hpp"
#include "fmxq_internal.hpp"
#include "fmxq_mfma_frag.hpp"

namespace fmxq {
namespace {

typedef __attribute__((address_space(3))) void tile_lds_t;

constexpr int kTileWaves = 4;

template <int BITS, int GS>
struct TileGeom {
  static constexpr int SU = 2;                     // 64-value units per step
  static constexpr int WS = BITS == 4 ? 2 : 1;     // steps per weight load
  static constexpr int RB = 128;                   // bytes of a weight row per load (WS steps)
  static constexpr int LPR = RB / 16;              // lanes per weight row of a load
  static constexpr int NI = 32 * RB / 1024;        // weight loads per column group
  static constexpr int XROW = SU * 128;            // bytes of an x row per step
  static constexpr int GPS = SU * 64 / GS;         // groups per step
  static constexpr int SPAN = 8 / GPS;             // steps per scale load (8 groups)
  static constexpr int XI = kMoeTileRows * XROW / 1024 / kTileWaves;  // x DMAs per wave
  static constexpr int XR = 1024 / XROW;           // x rows per DMA instruction
  static constexpr float OFF = BITS == 4 ? 128.f : 0.f;
  static constexpr int SRB = tile_sum_bytes(GS);   // bytes of a row's group sums per step
  static constexpr int SI = kMoeTileRows * SRB / 1024;  // sums DMAs (one a wave)
};

// Place of chunk c (16 bytes) in weight-stage row r (128 bytes): 16 rows read at one
// chunk fall on distinct banks.
__device__ __forceinline__ int tile_wpos(int c, int r) { return c ^ ((r & 7) ^ ((r >> 3) & 1)); }

__device__ __forceinline__ float tile_r16(float v) { return bf16_bits_to_f32(f32_to_bf16_rne(v)); }

// Low and high half-wave values of v, each in both halves.
struct HalfPair {
  uint32_t lo, hi;
};
__device__ __forceinline__ HalfPair tile_halves(uint32_t v) {
  const auto p = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  return {p[0], p[1]};
}

// This lane's packed words of unit j of a stage row, in MFMA order: chunk 4 h + i (of 8
// values: one word of 4 bits, two of 8) for MFMA i, or chunk 2 i + h for groups of 32.
// wb: byte offset of the lane's row and of chunk (BITS / 4) h in it, swizzled.
template <int BITS, int GS>
__device__ __forceinline__ void tile_words(const uint8_t* stage, int wb, int j, uint32_t (&w)[BITS]) {
  constexpr int W = BITS / 4;  // words per chunk
#pragma unroll
  for (int t = 0; t < W; ++t) {
    const u32x4 v = *reinterpret_cast<const u32x4*>(stage + (wb ^ ((2 * W * j + t) << 4)));
#pragma unroll
    for (int i = 0; i < 4; ++i) w[4 * t + i] = v[i];
  }
  if constexpr (GS == 32) {
    // Half h holds chunks 4 h .. + 4; exchanging chunk 1 (3) of the low half with
    // chunk 0 (2) of the high one leaves 2 i + h.
    uint32_t o[BITS];
#pragma unroll
    for (int t = 0; t < W; ++t) {
      const auto a = __builtin_amdgcn_permlane32_swap(w[t], w[W + t], false, false);
      const auto b = __builtin_amdgcn_permlane32_swap(w[2 * W + t], w[3 * W + t], false, false);
      o[t] = a[0], o[2 * W + t] = a[1], o[W + t] = b[0], o[3 * W + t] = b[1];
    }
#pragma unroll
    for (int i = 0; i < BITS; ++i) w[i] = o[i];
  }
}

// Everything a wave needs for its walk over K.
template <int BITS, int GS>
struct TileWave {
  using G = TileGeom<BITS, GS>;
  const void *x, *sums, *w[2];  // the buffers, below 2^31 bytes each
  int x_bytes, s_bytes, w_bytes;
  uint32_t xo[G::XI];        // x DMA byte offsets (row and swizzled chunk; past x, which
                             // loads zeros without a memory access, past the slots)
  uint32_t so;               // sums DMA byte offset (waves below SI)
  uint32_t wo[2];            // weight byte offset (row L / LPR of the wave's 32, chunk L % LPR)
  int wstep;                 // bytes of 64 / LPR weight rows
  const uint16_t* sb[2];     // this lane's scale (low half) or bias (high half) row
  int steps, groups;         // steps, groups per row
};

// s_waitcnt operand for vmcnt(n), lgkmcnt left alone (gfx9 encoding).
template <int N>
constexpr int wait_vm() {
  return (N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8);
}

template <int RT, int BITS, int GS>
__device__ __forceinline__ void tile_walk(const TileWave<BITS, GS>& tw, uint8_t* xs0, uint8_t* xs1,
                                          uint8_t* stage, uint8_t* sums0, uint8_t* sums1, int wave,
                                          f32x16 (&acc)[2][RT]) {
  using G = TileGeom<BITS, GS>;
  constexpr int SU = G::SU, GPS = G::GPS, XROW = G::XROW, SPAN = G::SPAN, NI = G::NI, LPR = G::LPR, WS = G::WS;
  constexpr int SRB = G::SRB;
  auto buffer = [](const void* p, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc((void*)p, (short)0, bytes, 0x00020000);
  };
  const __amdgpu_buffer_rsrc_t xres = buffer(tw.x, tw.x_bytes), sres = buffer(tw.sums, tw.s_bytes);
  const __amdgpu_buffer_rsrc_t wres0 = buffer(tw.w[0], tw.w_bytes), wres1 = buffer(tw.w[1], tw.w_bytes);
  constexpr int wait_lgkm0 = (15 | (3 << 14)) | (7 << 4);  // vmcnt left alone
  const int tid = threadIdx.x, lane = tid & 63;
  const int r32 = lane & 31, h = lane >> 5;

  // This lane's place in the weight stage: load i covers rows i (64 / LPR) + L / LPR.
  int sw[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int r = i * (64 / LPR) + lane / LPR;
    sw[i] = r * G::RB + (tile_wpos(lane % LPR, r) << 4);
  }
  u32x4 wbuf[2][NI];
  // Scales and biases of 8 groups: current, and (loaded ahead) the next.
  u32x4 sbn[2], sbc[2];
  constexpr int NW = GPS > 1 ? GPS / 2 : 1;  // scale pairs per step

  // The x rows and scales of step k; the weights of steps k .. k + WS.
  auto issue_x = [&](int k, uint8_t* xs, uint8_t* sums) {
    if (wave < G::SI)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(sres, (tile_lds_t*)(sums + wave * 1024), 16,
                                               (int)tw.so + k * SRB, 0, 0, 0);
#pragma unroll
    for (int j = 0; j < G::XI; ++j)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          xres, (tile_lds_t*)(xs + (wave * G::XI + j) * 1024), 16, (int)tw.xo[j] + k * XROW, 0, 0, 0);
    if (k % SPAN == 0) {
      const int g = k * GPS, left = tw.groups - g;
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const uint16_t* p = tw.sb[c] + g;
        if (left >= 8) {
          // 4-byte aligned at least (groups per row is even for every size and K a
          // multiple of 256).
          __builtin_memcpy(&sbn[c], __builtin_assume_aligned(p, 4), 16);
        } else {
#pragma unroll
          for (int w = 0; w < 4; ++w) {
            uint32_t v = 0;
            if (2 * w < left) __builtin_memcpy(&v, __builtin_assume_aligned(p + 2 * w, 4), 4);
            sbn[c][w] = v;
          }
        }
      }
    }
  };
  auto issue_w = [&](int k) {
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int i = 0; i < NI; ++i)
        wbuf[c][i] = __builtin_bit_cast(
            u32x4, __builtin_amdgcn_raw_buffer_load_b128(c ? wres1 : wres0, (int)tw.wo[c],
                                                         k / WS * G::RB + i * tw.wstep, 2));
  };
  // The step's scale (sv) and bias (bv) words of each column group, in every lane:
  // groups 2 w and 2 w + 1 of the step (one group per step: the low half of the word).
  uint32_t sv[2][NW], bv[2][NW];
  auto pairs = [&](int k) {
    const int o = (k % SPAN) * GPS;  // the step's first of the 8 loaded groups
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        uint32_t v = sbc[c][w];
#pragma unroll
        for (int q = w + 1; q < 4; ++q) v = (o >> 1) + w == q ? sbc[c][q] : v;
        if constexpr (GPS == 1) v = (o & 1) ? v >> 16 : v;
        const HalfPair p = tile_halves(v);
        sv[c][w] = p.lo;
        bv[c][w] = p.hi;
      }
  };
  // acc += the bias term of one step's groups, two per MFMA (lane half h: group 2 f + h).
  auto fold = [&](const uint8_t* sums) {
#pragma unroll
    for (int f = 0; f < NW; ++f) {
      const bool have = 2 * f + h < GPS;
      bf16x8 A[RT];
#pragma unroll
      for (int i = 0; i < RT; ++i) {
        const u32x2 v = *reinterpret_cast<const u32x2*>(sums + (32 * i + r32) * SRB +
                                                        (have ? 2 * f + h : 0) * 8);
        A[i] = BITS == 4 ? as_bf16x8(v[0], v[1] | (v[0] << 16), (v[0] >> 16) | (v[1] << 16), 0u)
                         : as_bf16x8(v[0], v[1], 0u, 0u);
      }
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const uint32_t b = have ? (h ? bv[c][f] >> 16 : bv[c][f] & 0xffffu) : 0u;
        bf16x8 B;
        if constexpr (BITS == 4) {
          const float sf = h ? bf16_hi(sv[c][f]) : bf16_lo(sv[c][f]);
          const uint32_t s = have ? f32_to_bf16_rne(-G::OFF * sf) : 0u;
          B = as_bf16x8(b | (b << 16), b | (s << 16), s | (s << 16), 0u);
        } else {
          B = as_bf16x8(b | (b << 16), b, 0u, 0u);
        }
#pragma unroll
        for (int i = 0; i < RT; ++i)
          acc[c][i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A[i], B, acc[c][i], 0, 0, 0);
      }
    }
  };

  auto step = [&](auto ec, int k) {
    constexpr int e = decltype(ec)::value;
    uint8_t* const xc = e ? xs1 : xs0;
    uint8_t* const xn = e ? xs0 : xs1;
    uint8_t* const sc = e ? sums1 : sums0;
    uint8_t* const sn = e ? sums0 : sums1;
    // This step's x and scales, issued one step ago, and where a load's steps begin its
    // weights, issued WS steps ago (in the other steps the next ones stay in flight).
    constexpr bool fresh = WS == 1 || e == 0;
    if (fresh || k + 1 >= tw.steps) __builtin_amdgcn_s_waitcnt(wait_vm<0>());
    else __builtin_amdgcn_s_waitcnt(wait_vm<2 * NI>());
    if constexpr (fresh) {
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int i = 0; i < NI; ++i)
          *reinterpret_cast<u32x4*>(stage + c * 32 * G::RB + sw[i]) = wbuf[c][i];
    }
    if (k % SPAN == 0) {
      sbc[0] = sbn[0];
      sbc[1] = sbn[1];
    }
    // Every wave's x and sums DMAs have landed; every wave has left the stages that
    // the next ones fill.
    __builtin_amdgcn_s_waitcnt(wait_lgkm0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    if (k + 1 < tw.steps) issue_x(k + 1, xn, sn);
    __builtin_amdgcn_sched_barrier(0);
    if (fresh && k + WS < tw.steps) issue_w(k + WS);
    __builtin_amdgcn_sched_barrier(0);
    pairs(k);
    // LDS offsets of the lane's weight and x row with its half's chunk bits; opaque, so
    // that the swizzled offset of each read is one xor here and not a register held
    // across the loop.
    int wb = r32 * G::RB + (tile_wpos((BITS / 4) * h, r32) << 4);
    int xb = r32 * XROW + (((GS == 32 ? h : 4 * h) ^ (r32 & 15)) << 4);
    asm volatile("" : "+v"(wb), "+v"(xb));
    // Products are taken per block: a unit, or a group of 32 (a group of 128 scales
    // its two units' products apart).
    constexpr int GB = GS == 32 ? 2 : 1;       // blocks of a unit
    constexpr int MB = 4 / GB;                 // MFMAs of a block's product
    constexpr int NB = SU * GB;                // blocks of the step
    constexpr int AB = RT == 1 ? 2 : RT;       // x fragment sets
    bf16x8 A[AB][MB], B[2][MB];
    uint32_t wv[2][BITS];  // packed words of a unit: chunks 4 h + i (groups of 32: 2 i + h)
    f32x16 P[2];
    float ps = 0.f;
    auto load_a = [&](int i, int b) {
#pragma unroll
      for (int m = 0; m < MB; ++m) {
        const int i4 = (b % GB) * MB + m;
        const int chunk = 8 * (b / GB) + (GS == 32 ? 2 * i4 : i4);  // (+ h or 4 h, in xb)
        A[RT == 1 ? b & 1 : i][m] = __builtin_bit_cast(
            bf16x8, *reinterpret_cast<const u32x4*>(xc + 32 * i * XROW + (chunk >> 4) * 256 +
                                                    (xb ^ ((chunk & 15) << 4))));
      }
    };
    auto load_w = [&](int j) {
#pragma unroll
      for (int c = 0; c < 2; ++c) tile_words<BITS, GS>(stage + c * 32 * G::RB, wb, j + (WS == 2 ? SU * e : 0), wv[c]);
    };
    auto unpack = [&](int c, int b) {
#pragma unroll
      for (int m = 0; m < MB; ++m) {
        const int i4 = (b % GB) * MB + m;
        if constexpr (BITS == 4) B[c][m] = wfrag<4>(wv[c][i4]);
        else B[c][m] = cvt_frag8(wv[c][2 * i4], wv[c][2 * i4 + 1]);
      }
    };
    // (The empty asm keeps the FMAs here: left alone, the compiler sinks them into
    // the next step, past the products' registers it has.)
    auto correct = [&](int c, int i, int o) {
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[c][i][r] = __builtin_fmaf(ps, P[o][r], acc[c][i][r]);
      asm volatile("" : "+v"(acc[c][i]));
    };
    auto scale = [&](int c, int g) {
      return (GPS > 1 && (g & 1)) ? bf16_hi(sv[c][g >> 1]) : bf16_lo(sv[c][g >> 1]);
    };
    load_w(0);
#pragma unroll
    for (int i = 0; i < RT; ++i) load_a(i, 0);
    fold(sc);
    unpack(0, 0);
    __builtin_amdgcn_sched_barrier(0);
    // Tiles in order (block, column group, x tile).  While a tile's MFMAs run, the wave
    // scales the tile before it, unpacks the next weights and reads ahead from LDS.
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int i = 0; i < RT; ++i) {
          const int t = (b * 2 + c) * RT + i;  // tile number in the step
          const bool last = i == RT - 1;
          // Reads ahead: the x fragments a tile earlier has done with, and the next
          // unit's words once both columns' are unpacked.
          if (RT == 2 && c == 1 && i == 1 && b + 1 < NB) load_a(0, b + 1);
          if (RT == 2 && c == 0 && i == 0 && b > 0) load_a(1, b);
          if (RT == 1 && c == 0 && b + 1 < NB) load_a(0, b + 1);
          if (c == 1 && i == 0 && b + 1 < NB && (b + 1) % GB == 0) load_w((b + 1) / GB);
          f32x16 p = {};
#pragma unroll
          for (int m = 0; m < MB; ++m)
            p = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A[RT == 1 ? b & 1 : i][m], B[c][m], p, 0, 0, 0);
          if (t > 0) correct((t - 1) / RT % 2, (t - 1) % RT, (t - 1) & 1);
          P[t & 1] = p;
          ps = scale(c, (64 * b / GB) / GS);
          if (last && c == 0) unpack(1, b);
          if (last && c == 1 && b + 1 < NB) unpack(0, b + 1);
          // Per MFMA: LDS reads and a share of the tile's VALU work (16 FMAs, and with
          // the last x tile a column group's unpacking).
          constexpr int kFma = 20 / MB, kAll = kFma + (BITS == 4 ? 7 : 12);
#pragma unroll
          for (int m = 0; m < MB; ++m) {
            __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            if (last) __builtin_amdgcn_sched_group_barrier(0x002, kAll, 0);
            else __builtin_amdgcn_sched_group_barrier(0x002, kFma, 0);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
    correct(1, RT - 1, (NB * 2 * RT - 1) & 1);
  };

  issue_x(0, xs0, sums0);
  __builtin_amdgcn_sched_barrier(0);
  issue_w(0);
  __builtin_amdgcn_sched_barrier(0);
  // K is a multiple of 256 (moe_qmvs_supported), two steps.
#pragma clang loop unroll(disable)
  for (int k = 0; k < tw.steps; k += 2) {
    step(std::integral_constant<int, 0>{}, k);
    step(std::integral_constant<int, 1>{}, k + 1);
  }
}

template <int RT, int NMAT, int BITS, int GS>
__device__ __forceinline__ void tile_store(const MoeArgs& a, int64_t start, int64_t eo, bool sh, int64_t n0,
                                           int wave, int len, bool bad_e, const uint32_t* rows,
                                           const f32x16 (&acc)[2][RT]) {
  const int lane = threadIdx.x & 63, r32 = lane & 31, h = lane >> 5;
  constexpr int NC = NMAT == 2 ? 1 : 2;  // stored columns per lane
  auto column = [&](int c) { return n0 + 32 * kTileWaves * c + 32 * wave + r32; };
  auto silu_mul = [&](float v0, float v1) {
    const float g = tile_r16(v0), u = tile_r16(v1);
    const float sg = tile_r16(1.f / (1.f + __expf(-g)));
    return (uint16_t)f32_to_bf16_rne(tile_r16(tile_r16(g * sg) * u));
  };
  // C layout: register r of lane l is row 8 (r / 4) + 4 (l / 32) + r % 4, column l % 32.
  auto row_of = [&](int i, int r) { return 32 * i + 8 * (r / 4) + 4 * h + (r % 4); };
  // Infinite and NaN outputs, bit 16 i + r: one FMA per sum (0 times it, NaN then) tells
  // a lane without any from the others.
  uint32_t odd[NC] = {};
  float zero = 0.f;
#pragma unroll
  for (int c = 0; c < 2; ++c)
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) zero = __builtin_fmaf(acc[c][i][r], 0.f, zero);
  if (__builtin_expect(zero != 0.f, 0)) {
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int m = row_of(i, r);
          if (m < len && !bad_e && !(rows[m] >> 31) && column(c % NC) < a.N && !__builtin_isfinite(acc[c][i][r]))
            odd[c % NC] |= 1u << (16 * i + r);
        }
  }
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int m = row_of(i, r);
      if (m >= len) continue;
      const uint32_t row = rows[m];
      const bool bad = bad_e || (row >> 31);
      uint16_t* yr = a.y + (int64_t)(row & 0x7fffffffu) * a.N;
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const int64_t n = column(c);
        if (n >= a.N) continue;
        const uint16_t v = NMAT == 2 ? silu_mul(acc[0][i][r], acc[1][i][r]) : (uint16_t)f32_to_bf16_rne(acc[c][i][r]);
        yr[n] = bad ? 0 : v;
      }
    }
  // The walk's dequantized answers for rows whose sums are not finite (deq_row_dot).
#pragma unroll
  for (int c = 0; c < NC; ++c)
    while (odd[c]) {
      const int i = __builtin_ctz(odd[c]), r = i & 15;
      odd[c] &= odd[c] - 1;
      const int m = row_of(i >> 4, r);
      const int64_t slot = start + m, n = eo + column(c);
      const uint16_t* x = a.x + (a.lhs ? (int64_t)a.lhs[slot] : slot / a.lhs_div) * a.K;
      float v[2] = {0.f, 0.f};
#pragma unroll
      for (int p = 0; p < NMAT; ++p)
        v[p] = deq_row_dot<BITS, GS>(x, (sh ? a.sh_w[p] : a.w[p]) + n * (a.K * BITS / 32),
                                     (sh ? a.sh_s[p] : a.s[p]) + n * (a.K / GS),
                                     (sh ? a.sh_b[p] : a.b[p]) + n * (a.K / GS), 0, a.K);
      a.y[(int64_t)rows[m] * a.N + column(c)] = NMAT == 2 ? silu_mul(v[0], v[1]) : (uint16_t)f32_to_bf16_rne(v[0]);
    }
}

// The group sums of x rows (see the top of the file) and, for 4 bits, the rows with each
// 8-value chunk in pair order.  Thread: 32 values (4 chunks) of a row; 4 threads make a
// step of 128 values, whose sums are SRB bytes (8 per group: hi, mid, lo, 0).
template <int BITS, int GS>
__global__ __launch_bounds__(256) void tile_prep_kernel(const uint16_t* __restrict__ x,
                                                        uint16_t* __restrict__ xp,
                                                        uint8_t* __restrict__ xsum, int64_t n32) {
  constexpr int TPG = GS / 32;  // threads per group
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const bool in = t < n32;  // whole groups of 4 threads
  const u32x4* src = reinterpret_cast<const u32x4*>(x) + 4 * (in ? t : 0);
  u32x4 v[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) v[c] = src[c];
  float s = 0.f;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
#pragma unroll
    for (int i = 0; i < 4; ++i) s = dot2_bf16(v[c][i], 0x3F803F80u, s);
    if (BITS == 4 && in)
      reinterpret_cast<u32x4*>(xp)[4 * t + c] = __builtin_bit_cast(u32x4, xfrag4(v[c]));
  }
  auto add = [&](auto ctrl) {
    s += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(s), decltype(ctrl)::value, 0xf, 0xf, false));
  };
  if constexpr (TPG >= 2) add(std::integral_constant<int, 0xb1>{});
  if constexpr (TPG >= 4) add(std::integral_constant<int, 0x4e>{});
  const uint32_t hi = f32_to_bf16_rne(s);
  const float r1 = s - bf16_bits_to_f32(hi);
  const uint32_t mid = f32_to_bf16_rne(r1);
  const uint32_t lo = f32_to_bf16_rne(r1 - bf16_bits_to_f32(mid));
  if (in && t % TPG == 0)
    *reinterpret_cast<u32x2*>(xsum + (t >> 2) * tile_sum_bytes(GS) + (t & 3) / TPG * 8) =
        u32x2{hi | (mid << 16), lo};
}

// Grid: (column tiles, segment bound).  The caller checks the sizes (moe_window):
// x and each expert's matrix below 2^31 bytes, fewer than 2^31 rows.
template <int NMAT, int BITS, int GS>
__global__ __launch_bounds__(kTileWaves * 64) __attribute__((amdgpu_waves_per_eu(2, 2))) void moe_tile_kernel(
    MoeArgs a) {
  using G = TileGeom<BITS, GS>;
  __shared__ __attribute__((aligned(1024))) uint8_t xs0[kMoeTileRows * G::XROW];
  __shared__ __attribute__((aligned(1024))) uint8_t xs1[kMoeTileRows * G::XROW];
  __shared__ __attribute__((aligned(16))) uint8_t stage[kTileWaves][2 * 32 * G::RB];
  __shared__ __attribute__((aligned(1024))) uint8_t sums0[kMoeTileRows * G::SRB];
  __shared__ __attribute__((aligned(1024))) uint8_t sums1[kMoeTileRows * G::SRB];
  __shared__ uint32_t rows[kMoeTileRows];  // output row of each slot, top bit: bad x row

  const int64_t sg = blockIdx.y;
  if (sg >= (int64_t)*a.nseg) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // One value per block: in scalar registers, which the walk has to spare.
  const int64_t start = (uint32_t)__builtin_amdgcn_readfirstlane((int)a.seg[2 * sg]);
  const int len = __builtin_amdgcn_readfirstlane((int)a.seg[2 * sg + 1]);
  const uint32_t e = (uint32_t)__builtin_amdgcn_readfirstlane((int)a.rhs[start]);
  const bool sh = a.sh_seg && (int64_t)e == a.E;
  const bool bad_e = (int64_t)e >= a.E && !sh;
  const int64_t n0 = (int64_t)blockIdx.x * (32 * kTileWaves * (NMAT == 2 ? 1 : 2));

  if (tid < kMoeTileRows) {
    uint32_t v = 0;
    if (tid < len) {
      const int64_t slot = start + tid;
      const int64_t xr = a.lhs ? (int64_t)a.lhs[slot] : slot / a.lhs_div;
      v = (a.yrow ? a.yrow[slot] : (uint32_t)slot) | (xr >= a.x_rows ? 0x80000000u : 0u);
      if (bad_e || xr >= a.x_rows) atomicOr(a.err_flag, 1u);
    }
    rows[tid] = v;
  }

  TileWave<BITS, GS> tw;
  tw.steps = (int)(a.K / (G::SU * 64));
  tw.groups = (int)(a.K / GS);
  const int64_t wpr = a.K * BITS / 32, gpr = a.K / GS;
  tw.wstep = (int)(64 / G::LPR * wpr * 4);
  const int64_t eo = sh || bad_e ? 0 : (int64_t)e * a.N;
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const int p = NMAT == 2 ? c : 0;
    const uint32_t* w = (sh ? a.sh_w[p] : a.w[p]) + eo * wpr;
    tw.w[c] = w;
    // N is a multiple of 32: a wave past the columns re-reads the last 32.
    int64_t nb = n0 + (NMAT == 2 ? 0 : 32 * kTileWaves * c) + 32 * wave;
    nb = nb < a.N ? nb : a.N - 32;
    tw.wo[c] = (uint32_t)((nb + lane / G::LPR) * wpr * 4 + (lane % G::LPR) * 16);
    tw.sb[c] = ((lane >> 5) ? (sh ? a.sh_b[p] : a.b[p]) : (sh ? a.sh_s[p] : a.s[p])) +
               (eo + nb + (lane & 31)) * gpr;
  }
  const int64_t srow = a.K / 128 * G::SRB;  // bytes of a row's sums
  tw.x = a.xp;
  tw.sums = a.xsum;
  tw.x_bytes = (int)(a.x_rows * a.K * 2);
  tw.s_bytes = (int)(a.x_rows * srow);
  tw.w_bytes = (int)(a.N * wpr * 4);
#pragma unroll
  for (int j = 0; j < G::XI; ++j) {
    constexpr int CPR = G::XROW / 16;  // chunks per x row and step
    const int r = G::XR * (wave * G::XI + j) + lane / CPR;
    const int c = (lane % CPR) ^ (r & 15);
    const int64_t slot = start + (r < len ? r : 0);
    int64_t xr = a.lhs ? (int64_t)a.lhs[slot] : slot / a.lhs_div;
    if (xr >= a.x_rows) xr = 0;
    tw.xo[j] = r < len ? (uint32_t)(xr * a.K * 2 + c * 16) : 0x80000000u;
  }
  {
    constexpr int LPS = G::SRB / 16;  // lanes per row's sums
    const int r = 64 / LPS * wave + lane / LPS;
    const int64_t slot = start + (r < len ? r : 0);
    int64_t xr = a.lhs ? (int64_t)a.lhs[slot] : slot / a.lhs_div;
    if (xr >= a.x_rows) xr = 0;
    tw.so = r < len ? (uint32_t)(xr * srow + lane % LPS * 16) : 0x80000000u;
  }
  __syncthreads();

  if (len <= 32) {
    f32x16 acc[2][1] = {};
    if (!bad_e) tile_walk<1, BITS, GS>(tw, xs0, xs1, stage[wave], sums0, sums1, wave, acc);
    tile_store<1, NMAT, BITS, GS>(a, start, eo, sh, n0, wave, len, bad_e, rows, acc);
  } else {
    f32x16 acc[2][2] = {};
    if (!bad_e) tile_walk<2, BITS, GS>(tw, xs0, xs1, stage[wave], sums0, sums1, wave, acc);
    tile_store<2, NMAT, BITS, GS>(a, start, eo, sh, n0, wave, len, bad_e, rows, acc);
  }
}

template <int BITS, int GS>
hipError_t launch_moe_tile_fmt(MoeArgs a, int nmat, int64_t max_seg, hipStream_t stream) {
  // The x rows' sums, then (4 bits) their pair order, in the caller's scratch.
  const int64_t n32 = a.x_rows * a.K / 32;
  uint16_t* xp = BITS == 4 ? reinterpret_cast<uint16_t*>(a.xprep + moe_tile_sum_bytes(a.x_rows * a.K, GS))
                           : nullptr;
  tile_prep_kernel<BITS, GS><<<(unsigned)((n32 + 255) / 256), 256, 0, stream>>>(a.x, xp, a.xprep, n32);
  a.xsum = a.xprep;
  a.xp = BITS == 4 ? xp : a.x;
  const int64_t cols = 32 * kTileWaves * (nmat == 2 ? 1 : 2);
  const dim3 grid((unsigned)((a.N + cols - 1) / cols), (unsigned)max_seg);
  if (nmat == 2) moe_tile_kernel<2, BITS, GS><<<grid, kTileWaves * 64, 0, stream>>>(a);
  else moe_tile_kernel<1, BITS, GS><<<grid, kTileWaves * 64, 0, stream>>>(a);
  return hipGetLastError();
}

}  // namespace
}  // namespace fmxq
