// panslbm2_amd/csrc/apply3_f16.hip -- eager boundary programs on the 3D lattices, FP16 storage.
#include "apply.h"

namespace lbm {
template hipError_t program_apply_nd<3, kF16>(const ApplyLaunch &al, const ProgView &pv);
}  // namespace lbm
