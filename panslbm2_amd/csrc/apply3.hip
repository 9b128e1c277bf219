// panslbm2_amd/csrc/apply3.hip -- eager boundary programs on the 3D lattices, FP64 storage.
#include "apply.h"

namespace lbm {
template hipError_t program_apply_nd<3, kF64>(const ApplyLaunch &al, const ProgView &pv);
}  // namespace lbm
