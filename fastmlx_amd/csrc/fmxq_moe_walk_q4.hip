// fmxq_moe_walk_q4.hip -- the grouped MoE walk for 4-bit weights in groups of 32 and 128.
// Bound by the weight stream, like the groups-of-64 form.  These formats ran the
// general gather kernels before (one slot's GEMV, or 32 x 32 MFMA tiles whose waves
// each load 32 rows at 32 bytes): 512 experts of 512 columns, K = 2048, top-10:
// 40 tokens in groups of 32 423 -> 152 us a layer, 300 tokens in groups of 128
// 907 -> 226 us.
#include "fmxq_moe_walk.hpp"

namespace fmxq {

hipError_t launch_moe_qmvw_q4(const MoeArgs& a, int nmat, int window, int ntt, int64_t max_seg,
                              hipStream_t stream) {
  switch (a.group_size) {
    case 32: return launch_moe_qmvw_fmt<4, 32>(a, nmat, window, ntt, max_seg, stream);
    case 128: return launch_moe_qmvw_fmt<4, 128>(a, nmat, window, ntt, max_seg, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace fmxq
