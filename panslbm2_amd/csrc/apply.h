// panslbm2_amd/csrc/apply.h -- eager boundary programs (one in-place pass per segment), instantiated
// per dimension and storage precision in apply_*.hip.
#pragma once
#include "collide.h"

namespace lbm {

// ------------------------------------------------------------------------------------------
// Boundary program, applied in place: one thread per boundary node runs that node's operators of
// segment `seg` in call order (segments are separated by SmoothCorner calls).
// ------------------------------------------------------------------------------------------
template <class LA, class LB, class S>
__global__ void __launch_bounds__(kBlock) k_program_apply(S *a, S *b, int N, ProgView pv, int seg, Enc ea, Enc eb) {
    int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= pv.nentry) return;
    int n = pv.entry_node[e];
    int2 r = pv.entry_ops[e];
    double fa[LA::nc], fb[LB::nc > 0 ? LB::nc : 1];
    load_node<LA>(a, N, n, fa, ea);
    load_node<LB>(b, N, n, fb, eb);
    const NodeFields pre = load_fields(pv.fm, n);
    for (int t = r.x; t < r.x + r.y; ++t) {
        Op op = pv.ops[t];
        if (op.code != OP_SMOOTH && (int)op.seg == seg)
            apply_op<LA, LB>(OpWord{op.code, op.face, op.lat, op.fset, op.arg, 0}, op_in(op), fa, fb, pv, n, pre);
    }
    store_node<LA>(a, N, n, fa, ea);
    store_node<LB>(b, N, n, fb, eb);
}

template <int ND, int P>
hipError_t program_apply_nd(const ApplyLaunch &al, const ProgView &pv) {
    using S = typename PrecT<P>::S;
    auto go = [&](auto la, auto lb) -> hipError_t {
        using LA = decltype(la);
        using LB = decltype(lb);
        LBM_LAUNCH((k_program_apply<LA, LB, S>), nblocks(pv.nentry), al.stream, static_cast<S *>(al.a),
                   static_cast<S *>(al.b), al.N, pv, al.seg, al.ea, al.eb);
        return hipGetLastError();
    };
    return al.kb < 0 ? dispatch_single_nd<ND>(al.ka, go) : dispatch_coupled_nd<ND>(al.ka, al.kb, go);
}

}  // namespace lbm
