// fmxq_qmvw_fmt.hip -- the shared-x skinny product for groups of 32 and 128.
// Bound as the groups-of-64 form is (fmxq_skinny.hip).  These products ran the prefill
// GEMM's 64-row tile from M = 5 (9 at 8 bits): 14336x4096 in groups of 32 at M = 5 / 24
// 34.0 / 35.7 -> 15.3 / 20.2 us, 4096x14336 at M = 60 37.9 -> 24.3 us, 14336x4096 in
// groups of 128 at M = 16 27.0 -> 14.4 us; 8 bits, groups of 128, 14336x4096 at M = 30
// 30.6 -> 21.7 us, 4096x14336 at M = 3 (dot2 GEMV before) 28.9 -> 15.7 us.
#include "fmxq_qmvw.hpp"

namespace fmxq {

hipError_t launch_qmvw_fmt(const QmmArgs& a, const QmvwPlan& p, hipStream_t stream) {
  switch (a.group_size) {
    case 32: return launch_qmvw_gs<32>(a, p, stream);
    case 128: return launch_qmvw_gs<128>(a, p, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace fmxq
