// panslbm2_amd/csrc/apply3_f32.hip -- eager boundary programs on the 3D lattices, FP32 storage.
#include "apply.h"

namespace lbm {
template hipError_t program_apply_nd<3, kF32>(const ApplyLaunch &al, const ProgView &pv);
}  // namespace lbm
