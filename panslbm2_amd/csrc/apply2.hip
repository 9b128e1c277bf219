// panslbm2_amd/csrc/apply2.hip -- eager boundary programs on the 2D lattices, FP64 storage.
#include "apply.h"

namespace lbm {
template hipError_t program_apply_nd<2, kF64>(const ApplyLaunch &al, const ProgView &pv);
}  // namespace lbm
