// panslbm2_amd/csrc/apply2_f16.hip -- eager boundary programs on the 2D lattices, FP16 storage.
#include "apply.h"

namespace lbm {
template hipError_t program_apply_nd<2, kF16>(const ApplyLaunch &al, const ProgView &pv);
}  // namespace lbm
