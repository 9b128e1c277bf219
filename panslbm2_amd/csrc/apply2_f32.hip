// panslbm2_amd/csrc/apply2_f32.hip -- eager boundary programs on the 2D lattices, FP32 storage.
#include "apply.h"

namespace lbm {
template hipError_t program_apply_nd<2, kF32>(const ApplyLaunch &al, const ProgView &pv);
}  // namespace lbm
