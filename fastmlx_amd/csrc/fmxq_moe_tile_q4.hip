// fmxq_moe_tile_q4.hip -- the 64-slot MoE tiles for 4-bit weights.
#include "fmxq_moe_tile.hpp"

namespace fmxq {

hipError_t launch_moe_tile_q4(const MoeArgs& a, int nmat, int64_t max_seg, hipStream_t stream) {
  switch (a.group_size) {
    case 32: return launch_moe_tile_fmt<4, 32>(a, nmat, max_seg, stream);
    case 64: return launch_moe_tile_fmt<4, 64>(a, nmat, max_seg, stream);
    case 128: return launch_moe_tile_fmt<4, 128>(a, nmat, max_seg, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace fmxq
