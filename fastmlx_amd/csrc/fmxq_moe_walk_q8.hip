// fmxq_moe_walk_q8.hip -- the grouped MoE walk for 8-bit weights.
// Bound by the weight stream, like the 4-bit form.  8-bit experts ran the general
// gather kernels before (32 x 32 MFMA tiles whose waves each load 32 rows at 32
// bytes): 512 experts of 512 columns, K = 2048, top-10: 200 tokens 1425 -> 333 us a
// layer, 24 tokens (the GEMV forms of fmxq_moe_gemm.hip) 1013 -> 171 us.
#include "fmxq_moe_walk.hpp"

namespace fmxq {

hipError_t launch_moe_qmvw_q8(const MoeArgs& a, int nmat, int window, int ntt, int64_t max_seg,
                              hipStream_t stream) {
  switch (a.group_size) {
    case 32: return launch_moe_qmvw_fmt<8, 32>(a, nmat, window, ntt, max_seg, stream);
    case 64: return launch_moe_qmvw_fmt<8, 64>(a, nmat, window, ntt, max_seg, stream);
    case 128: return launch_moe_qmvw_fmt<8, 128>(a, nmat, window, ntt, max_seg, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace fmxq
