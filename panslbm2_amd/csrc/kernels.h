// panslbm2_amd/csrc/kernels.h -- node-state assembly shared by the stream, boundary-program,
// corner-smoothing and collide kernels.
//
// A node's post-stream state is pulled from the source buffer (periodic wrap as in d2q9.h:80-84),
// then the node's boundary operators run in call order.  The lanes that own smoothed nodes
// (SmoothCorner) rebuild the neighbours' states the same way and average them.
#pragma once
#include "bc2d.h"
#include "bc3d.h"
#include "lattice.h"
#include "physics.h"
#include "program.h"

namespace lbm {

// Placeholder for "no second lattice".
struct NoLat {
    static constexpr int kind = -1, nc = 0, nd = 0;
    static constexpr int cx[1] = {0}, cy[1] = {0}, cz[1] = {0};
    static constexpr double w[1] = {0.0};
};

// compile-time velocity-set helpers
template <class L>
constexpr int comp_of(int c, int ax) {
    return ax == 0 ? L::cx[c] : (ax == 1 ? L::cy[c] : L::cz[c]);
}
template <class L>
constexpr int opposite_of(int c) {
    for (int e = 0; e < L::nc; ++e)
        if (L::cx[e] == -L::cx[c] && L::cy[e] == -L::cy[c] && L::cz[e] == -L::cz[c]) return e;
    return 0;
}
template <class L>
constexpr int mirror_of(int c, int ax) {
    int v0 = L::cx[c], v1 = L::cy[c], v2 = L::cz[c];
    if (ax == 0) v0 = -v0;
    else if (ax == 1) v1 = -v1;
    else v2 = -v2;
    for (int e = 0; e < L::nc; ++e)
        if (L::cx[e] == v0 && L::cy[e] == v1 && L::cz[e] == v2) return e;
    return 0;
}

// Bounce-back (type 1) or specular reflection (type 2) of the populations streaming left
// undefined on face FACE: incoming ones (c_axis == -dir) after Stream, outgoing ones
// (c_axis == dir) after iStream.  d2q9.h:429-575, d3q15.h:982-1239.
template <class L, int FACE, bool ADJ>
__device__ __forceinline__ void bounce_face(double *f, int type) {
    constexpr int AX = FACE / 2;
    constexpr int DIR = (FACE % 2) ? 1 : -1;
    constexpr int WANT = ADJ ? DIR : -DIR;
    sfor<1, L::nc>([&](auto c) {
        constexpr int C = decltype(c)::value;
        if constexpr (comp_of<L>(C, AX) == WANT) {
            constexpr int OPP = opposite_of<L>(C);
            constexpr int MIR = mirror_of<L>(C, AX);
            f[C] = (type == 1) ? f[OPP] : f[MIR];
        }
    });
}
template <class L, bool ADJ>
__device__ __forceinline__ void bounce(double *f, int face, int type) {
    switch (face) {
    case 0: bounce_face<L, 0, ADJ>(f, type); break;
    case 1: bounce_face<L, 1, ADJ>(f, type); break;
    case 2: bounce_face<L, 2, ADJ>(f, type); break;
    case 3: bounce_face<L, 3, ADJ>(f, type); break;
    default:
        if constexpr (L::nd == 3) {
            if (face == 4) bounce_face<L, 4, ADJ>(f, type);
            else bounce_face<L, 5, ADJ>(f, type);
        }
    }
}

// Field values one node's boundary operators read (one field set, at the node).
struct NodeFields {
    double rho, ux, uy, uz, tem, diff;
    bool has_diff;  // the set has a diffusivity field (else AD_SET_Q uses its constant)
};
__device__ __forceinline__ NodeFields load_fields(const FieldSet &s, int n) {
    NodeFields v;
    v.rho = s.rho ? gat(s.rho, n) : 0.0;
    v.ux = s.ux ? gat(s.ux, n) : 0.0;
    v.uy = s.uy ? gat(s.uy, n) : 0.0;
    v.uz = s.uz ? gat(s.uz, n) : 0.0;
    v.tem = s.tem ? gat(s.tem, n) : 0.0;
    v.diff = s.diff ? gat(s.diff, n) : 0.0;
    v.has_diff = s.diff != nullptr;
    return v;
}

// Apply one boundary operator to lattice L's populations `f`; `o` holds the other lattice's
// populations (lattice LO), read by the coupled adjoint pressure operator.
template <class L, class LO>
__device__ __forceinline__ void apply_on(const OpWord &op, const OpIn &q, double *f, const double *o,
                                         const NodeFields &s) {
    const int face = (int)op.face, arg = (int)op.arg;
    switch (op.code) {
    case OP_BOUNCE: bounce<L, false>(f, face, arg); break;
    case OP_IBOUNCE: bounce<L, true>(f, face, arg); break;
    case OP_NS_SET_U:
        if constexpr (L::kind == kD2Q9) ns_set_u_2d(f, face, q.a[0], q.a[1]);
        else if constexpr (L::kind == kD3Q15 || L::kind == kD3Q27)
            ns_set_u_3d<L>(f, face, q.a[0], q.a[1], q.a[2]);
        break;
    case OP_NS_SET_RHO:
        if constexpr (L::kind == kD2Q9) ns_set_rho_2d(f, face, q.a[0], q.a[1]);
        else if constexpr (L::kind == kD3Q15 || L::kind == kD3Q27)
            ns_set_rho_3d<L>(f, face, q.a[0], q.a[1], q.a[2]);
        break;
    case OP_AD_SET_T:  // (the host rejects advection-diffusion operators on D3Q27)
        if constexpr (L::nd == 2) ad_set_t_2d<L>(f, face, q.b[0], s.ux, s.uy);
        else if constexpr (L::nd == 3 && L::kind != kD3Q27) ad_set_t_3d<L>(f, face, q.b[0], s.ux, s.uy, s.uz);
        break;
    case OP_AD_SET_Q: {
        double d = s.has_diff ? s.diff : q.b[1];
        if constexpr (L::nd == 2) ad_set_q_2d<L>(f, face, q.b[0], s.ux, s.uy, d);
        else if constexpr (L::nd == 3 && L::kind != kD3Q27) ad_set_q_3d<L>(f, face, q.b[0], s.ux, s.uy, s.uz, d);
    } break;
    case OP_ANS_ISET_U:
        if constexpr (L::kind == kD2Q9) ans_iset_u_2d(f, face, q.a[0], q.a[1], q.a[3], arg);
        else if constexpr (L::kind == kD3Q15 || L::kind == kD3Q27)
            ans_iset_u_3d<L>(f, face, q.a[0], q.a[1], q.a[2], q.a[3]);
        break;
    case OP_ANS_ISET_RHO:
        if constexpr (L::kind == kD2Q9) ans_iset_rho_2d(f, face);
        else if constexpr (L::kind == kD3Q15 || L::kind == kD3Q27) ans_iset_rho_3d<L>(f, face);
        break;
    case OP_AAD_ISET_T:
        if constexpr (L::nd == 2) aad_iset_t_2d<L>(f, face, s.ux, s.uy);
        else if constexpr (L::nd == 3 && L::kind != kD3Q27) aad_iset_t_3d<L>(f, face, s.ux, s.uy, s.uz);
        break;
    case OP_AAD_ISET_Q:
        if constexpr (L::nd == 2) aad_iset_q_2d<L>(f, face, s.ux, s.uy, q.b[1]);
        else if constexpr (L::nd == 3 && L::kind != kD3Q27) aad_iset_q_3d<L>(f, face, s.ux, s.uy, s.uz, q.b[1]);
        break;
    case OP_AAD_ISET_RHO:
        if constexpr (L::kind == kD2Q9 && LO::nd == 2)
            aad_iset_rho_2d<LO>(f, o, face, arg, s.rho, s.ux, s.uy, s.tem, q.b[1]);
        else if constexpr (L::kind == kD3Q15 && LO::nd == 3)
            aad_iset_rho_3d<LO>(f, o, face, arg, s.rho, s.ux, s.uy, s.uz, s.tem, q.b[1]);
        break;
    default: break;
    }
}

// Field set k of a program.  Selected with constant indices: a runtime index into the by-value
// kernel argument would make the compiler copy the argument to private (scratch) memory.
__device__ __forceinline__ FieldSet field_set(const ProgView &pv, int k) {
    static_assert(kMaxFieldSets == 4, "field_set covers four sets");
    return k == 0 ? pv.fs[0] : (k == 1 ? pv.fs[1] : (k == 2 ? pv.fs[2] : pv.fs[3]));
}

// pre: the merged set's fields (pv.fm) at node n; a set outside it is loaded at use.
template <class LA, class LB>
__device__ __forceinline__ void apply_op(const OpWord &op, const OpIn &q, double *a, double *b, const ProgView &pv,
                                         int n, const NodeFields &pre) {
    NodeFields s = pre;
    if (__builtin_expect(!((pv.fmerged >> op.fset) & 1u), 0)) s = load_fields(field_set(pv, (int)op.fset), n);
    s.has_diff = (pv.has_diff >> op.fset) & 1u;
    if (((int)op.lat ^ pv.latswap) == 0) apply_on<LA, LB>(op, q, a, b, s);
    else if constexpr (LB::nc > 0) apply_on<LB, LA>(op, q, b, a, s);
}
// What node n needs for its boundary operators: its list (NodeList) with the values, and the fields of the
// merged set.  The fused kernels load it before the node's pull, so that the operators wait for no
// memory of their own.  Four things keep the pull from waiting for it: the list's header stays as it was
// loaded (taken apart inside the boundary lanes' branch, it was waited for there) and has no unused half
// (whose register the pull's addresses took, and waited for), run_ops begins with a scheduling
// barrier (or the header's first use is moved up between the pull's loads), and the arguments that the
// branch needs are read together ahead of it (one after the other inside it, each was waited for).
// FP64 step, us, before and after: heat sink 200x400 7.73 -> 7.63, 141x161 7.09 -> 6.82; ducts forward /
// adjoint 113x36x43 17.75 / 21.07 -> 17.44 / 20.61, 96x96x48 33.5 / 38.9 -> 32.5 / 37.9.
struct NodeOps {
    uint64_t list_count;
    uint64_t w[2];
    ListVals vals;
    NodeFields f;
    __device__ __forceinline__ size_t list() const { return list_count >> 24; }
    __device__ __forceinline__ int count() const { return (int)((uint32_t)list_count & 0xffffffu); }
};
__device__ __forceinline__ NodeOps ops_of_node(const ProgView &pv, const Grid &g, int i, int j, int k, int n, int nd,
                                               bool wanted = true) {
    const int place = place_of(i, j, k, g.nx, g.ny, g.nz, nd);
    NodeOps no{0, {0, 0}, {}, {}};
    const FieldSet &fm = pv.fm;
    asm volatile("" ::"s"(fm.rho), "s"(fm.ux), "s"(fm.uy), "s"(fm.uz), "s"(fm.tem), "s"(fm.diff), "s"(pv.place_list),
                 "s"(pv.slot_list));
    asm volatile("" ::"s"(pv.nsym), "s"(pv.fmerged), "s"(pv.has_diff), "s"(pv.latswap), "s"(pv.pull[0]),
                 "s"(pv.pull[1]));
    if (wanted && ((pv.shared | pv.by_slot) >> place & 1u)) {
        const NodeList *e = pv.place_list + place;
        if (pv.by_slot >> place & 1u) e = pv.slot_list + boundary_slot(i, j, k, g.nx, g.ny, g.nz, nd);
        const uint64_t *p = reinterpret_cast<const uint64_t *>(e);
        no.list_count = gat(p, 0);
        no.w[0] = gat(p, 1);
        no.w[1] = gat(p, 2);
        const double *v = reinterpret_cast<const double *>(e) + offsetof(NodeList, vals) / sizeof(double);
#pragma unroll
        for (int c = 0; c < 4; ++c) no.vals.a[c] = gat(v, c);
#pragma unroll
        for (int c = 0; c < 4; ++c) no.vals.b[c >> 1][c & 1] = gat(v, 4 + c);
        no.f = load_fields(fm, n);
    }
    return no;
}

__device__ __forceinline__ uint64_t readlane64(uint64_t v, int lane) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, lane);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), lane);
    return (uint64_t)hi << 32 | lo;
}
// One register for each population, whichever operator wrote it (without it the register allocator
// has spilled the single-lattice kernels: up to 2.6 kB per lane).
template <class L>
__device__ __forceinline__ void settle(double *f) {
#pragma unroll
    for (int c = 0; c < L::nc; ++c) asm volatile("" : "+v"(f[c]));
}
struct NoSmooth {};  // SMOOTH operators do nothing
// Run a node's operators in record order; smooth(kernel lattice 0 / 1) stands for a SMOOTH operator.
// Called with the boundary lanes (and any others: no operators) active.
//
// What bounds it is latency, not throughput: a wavefront of 64 consecutive nodes holds one or two
// x-face nodes, on small grids the step waits for the wavefront with the most operators, and each of
// them is a chain of branches, instruction fetches and divisions of some 0.15 us.  So the wavefront
// takes the program's symbols that its lanes have one after the other, each once for all lanes that
// have it, with scalar branches over one copy of the operators.  FP64 step, us, against each lane
// deciding for itself, which walked every branch of a decision tree per operator in four inlined copies
// after three dependent memory round trips: 200x400 D2Q9 + D2Q5 heat sink 7.6 (7.8), smoothed 7.7 (9.1),
// 101x101 6.4 (6.8), 200x400 with six calls whose masks are drawn per node 12.6 (13.2; 91 with each list
// run by itself); ducts forward / adjoint 44x40x30 10.9 / 11.6 (11.2 / 12.7), 113x36x43 17.4 / 20.6
// (18.0 / 21.0), 96x96x48 32.5 / 37.9 (36.2 / 43.3).  Slower: 200x400 with two calls on all four faces 7.5
// (7.2), and 101x101 with both bounce types, T and Q alternating along the walls 7.9 (6.4).
// More than kSymbols symbols (11 calls that each reach six faces): position by position of the lists, at
// each the words that the lanes have, each once.
template <class LA, class LB, class Smooth = NoSmooth>
__device__ __forceinline__ void run_ops(const ProgView &pv, const NodeOps &no, int n, double *a, double *b,
                                        Smooth &&smooth = Smooth{}) {
    __builtin_amdgcn_sched_barrier(0);
    const bool merged = pv.nsym > 0;
    unsigned long long all = 0;  // merged: the symbols left; else the lanes whose operator at position t is left
    int t = 0;
    uint32_t word = (uint32_t)no.w[0] & 0xffffu, next = 0;
    if (merged) {
        for (unsigned long long left = __ballot(no.w[0] != 0); left;) {
            all |= readlane64(no.w[0], __builtin_ctzll(left));
            left = __ballot((no.w[0] & ~all) != 0);
        }
        if (all) next = pv.sym[__builtin_ctzll(all) >> 1];
    } else {
        all = __ballot(no.count() > 0);
    }
    while (all) {
        uint32_t w;
        int bit = 0;
        bool mine;
        if (merged) {
            bit = __builtin_ctzll(all);
            all &= all - 1;
            w = next >> (bit & 1) * 16;  // loaded one operator ahead
            next = pv.sym[(all ? __builtin_ctzll(all) : bit) >> 1];
            mine = no.w[0] >> bit & 1u;
        } else {
            w = (uint32_t)__builtin_amdgcn_readlane((int)word, __builtin_ctzll(all));
            mine = t < no.count() && word == w;
            all &= ~__ballot(mine);
        }
        const OpWord op = op_fields(w);
        if (mine) {
            const bool second = op.src == kFromSecond;
            OpIn q{{no.vals.a[0], no.vals.a[1], no.vals.a[2], no.vals.a[3]},
                   {second ? no.vals.b[1][0] : no.vals.b[0][0], second ? no.vals.b[1][1] : no.vals.b[0][1]}};
            if (__builtin_expect(op.src == kFromList, 0)) {
                const int at = merged ? __popcll(no.w[0] & ((1ull << bit) - 1)) : t;
                q = op_in(pv.list_ops[no.list() + at]);
            }
            if constexpr (std::is_same_v<std::decay_t<Smooth>, NoSmooth>) {
                apply_op<LA, LB>(op, q, a, b, pv, n, no.f);
            } else {
                if (op.code == OP_SMOOTH) smooth((int)op.lat ^ pv.latswap);
                else apply_op<LA, LB>(op, q, a, b, pv, n, no.f);
            }
            settle<LA>(a);
            settle<LB>(b);
        }
        if (!merged && all == 0) {
            ++t;
            all = __ballot(t < no.count());
            word = (uint32_t)((t < 4 ? no.w[0] : no.w[1]) >> 16 * (t & 3)) & 0xffffu;
            if (t >= kWordOps && t < no.count()) word = pv.list_words[no.list() + t];
        }
    }
}

// E_c of a shift, in FP64
template <class L, int C>
__device__ __forceinline__ double shift_c(const Enc &e) {
    return e.rest * L::w[C];
}
// decode a stored value of node n (FP64 storage: the value itself)
template <class L, int C, class S>
__device__ __forceinline__ double dec(S x, const Enc &e) {
    if constexpr (std::is_same_v<S, double>) return x;
    else return double(x) + shift_c<L, C>(e);
}
template <class L, int C, class S>
__device__ __forceinline__ S enc(double v, const Enc &e) {
    if constexpr (std::is_same_v<S, double>) return v;
    else return S(v - shift_c<L, C>(e));
}

// One value at a byte offset of a plane, loaded non-temporal with NT (see pull_pair).
template <bool NT, class S>
__device__ __forceinline__ S pull_load(const S *plane, uint32_t off) {
    if constexpr (NT) return gload_nt(plane, off);
    else return gload(plane, off);
}

// Pull node n's populations: pull = +1 from x - c (Stream), -1 from x + c (iStream), 0 in place.
// S: storage type; values are decoded with the source node's shift.  The byte offsets of the three
// columns, rows and planes a pull can come from are formed once; each population then costs one
// three-way add beside its load (64-bit addresses per population took about 300 of the 1,200
// vector instructions of a D3Q15 + D3Q7 step).
template <class L, bool NT = false, class S, class R>
__device__ __forceinline__ void load_pull(const S *src, const Grid &g, int i, int j, int k, int n,
                                          int pull, R *f, const Enc &e = Enc{}) {
    if constexpr (L::nc > 0) {
        // its own value of the pointer, or the two forms' loads are merged into plain ones
        if constexpr (NT) asm volatile("" : "+s"(src));
        constexpr uint32_t E = sizeof(S);
        const uint32_t row = (uint32_t)g.nx * E, lay = row * (uint32_t)g.ny;
        const int lo = pull, hi = -pull;  // displacement of the source for c = -1 and c = +1
        const uint32_t x[3] = {(uint32_t)wrap(i, lo, g.nx) * E, (uint32_t)i * E, (uint32_t)wrap(i, hi, g.nx) * E};
        const uint32_t y[3] = {(uint32_t)wrap(j, lo, g.ny) * row, (uint32_t)j * row, (uint32_t)wrap(j, hi, g.ny) * row};
        uint32_t z[3] = {0u, 0u, 0u};
        if constexpr (L::nd == 3) {
            z[0] = (uint32_t)wrap(k, lo, g.nz) * lay;
            z[1] = (uint32_t)k * lay;
            z[2] = (uint32_t)wrap(k, hi, g.nz) * lay;
        }
        f[0] = R(dec<L, 0>(pull_load<NT>(src, (uint32_t)n * E), e));
        sfor<1, L::nc>([&](auto c) {
            constexpr int C = decltype(c)::value;
            const uint32_t off = x[L::cx[C] + 1] + y[L::cy[C] + 1] + z[L::cz[C] + 1];
            f[C] = R(dec<L, C>(pull_load<NT>(src + (size_t)C * g.N, off), e));
        });
    }
}
template <class L, class S>
__device__ __forceinline__ void load_node(const S *__restrict__ src, int N, int n, double *f, const Enc &e = Enc{}) {
    sfor<0, L::nc>([&](auto c) {
        constexpr int C = decltype(c)::value;
        f[C] = dec<L, C>(gat(src + (size_t)C * N, n), e);
    });
}
template <class L, class S>
__device__ __forceinline__ void store_node(S *__restrict__ dst, int N, int n, const double *f, const Enc &e = Enc{}) {
    sfor<0, L::nc>([&](auto c) {
        constexpr int C = decltype(c)::value;
        gput(dst + (size_t)C * N, n, enc<L, C, S>(f[C], e));
    });
}

// register type of a storage type, and a lattice's shift as moments (FP64 storage: none)
template <class S>
using RegOf = std::conditional_t<std::is_same_v<S, double>, double, float>;
template <class S>
__device__ __forceinline__ Sh4 own_shift(const Enc &e) {
    if constexpr (std::is_same_v<S, double>) return Sh4{};
    else return Sh4{float(e.rest), 0.0f, 0.0f, 0.0f};
}
// Values as stored, without decoding (the hot path keeps FP32 deviations of the node's own shift).
template <class L, class S, class R>
__device__ __forceinline__ void load_raw(const S *__restrict__ src, int N, int n, R *f) {
    sfor<0, L::nc>([&](auto c) { f[decltype(c)::value] = R(gat(src + (size_t)decltype(c)::value * N, n)); });
}
template <class L, bool NT = false, class S, class R>
__device__ __forceinline__ void store_raw(S *dst, int N, int n, const R *f) {
    if constexpr (L::nc > 0 && NT) asm volatile("" : "+s"(dst));  // as in load_pull
    sfor<0, L::nc>([&](auto c) {
        constexpr int C = decltype(c)::value;
        if constexpr (NT) gstore_nt(dst + (size_t)C * N, (uint32_t)n * (uint32_t)sizeof(S), S(f[C]));
        else gput(dst + (size_t)C * N, n, S(f[C]));
    });
}
// Register state <-> FP64 populations (identity in FP64; deviations of shift o in FP32)
template <class L>
__device__ __forceinline__ void put_state(double *dst, const double *v, const Enc &, const Sh4 &) {
    sfor<0, L::nc>([&](auto c) { dst[decltype(c)::value] = v[decltype(c)::value]; });
}
template <class L>
__device__ __forceinline__ void put_state(double *dst, const float *v, const Enc &e, const Sh4 &o);
template <class L>
__device__ __forceinline__ void get_state(double *v, const double *src, const Enc &, const Sh4 &) {
    sfor<0, L::nc>([&](auto c) { v[decltype(c)::value] = src[decltype(c)::value]; });
}
template <class L>
__device__ __forceinline__ void get_state(float *v, const double *src, const Enc &e, const Sh4 &o);
// FP32 deviations <-> FP64 populations, for the boundary operators and smoothing
template <class L>
__device__ __forceinline__ void dev_to_f64(const float *d, double *f, const Enc &e, const Sh4 &) {
    sfor<0, L::nc>([&](auto c) {
        constexpr int C = decltype(c)::value;
        f[C] = double(d[C]) + shift_c<L, C>(e);
    });
}
template <class L>
__device__ __forceinline__ void f64_to_dev(const double *f, float *d, const Enc &e, const Sh4 &) {
    sfor<0, L::nc>([&](auto c) {
        constexpr int C = decltype(c)::value;
        d[C] = float(f[C] - shift_c<L, C>(e));
    });
}
template <class L>
__device__ __forceinline__ void put_state(double *dst, const float *v, const Enc &e, const Sh4 &o) {
    dev_to_f64<L>(v, dst, e, o);
}
template <class L>
__device__ __forceinline__ void get_state(float *v, const double *src, const Enc &e, const Sh4 &o) {
    f64_to_dev<L>(src, v, e, o);
}

// Smoothed states (d2q9.h:577-587, d3q15.h:1241-1303) across the lanes of a wavefront.  Lanes come in
// groups: 4 per 2D corner or 3D edge node (two face neighbours' states, then the node's own, then a
// spare), 8 per 3D corner (the neighbours of its three edge nodes in x, y, z order, then its own,
// then a spare).  Lane 2 of a group of 4 gets 0.5 (a + b); lane 6 of a group of 8 the mean of the
// three edge means.  The means are of FP64 populations.
template <class L, class R>
__device__ __forceinline__ void smooth_lanes_mean(R *f, const Enc &e, bool corner3) {
    const int base = (int)(threadIdx.x & 56u);
    sfor<0, L::nc>([&](auto c) {
        constexpr int C = decltype(c)::value;
        double v;
        if constexpr (is_f64<R>) v = f[C];
        else v = double(f[C]) + shift_c<L, C>(e);
        const double m = 0.5 * (v + __shfl_xor(v, 1));
        double s;
        if (corner3) s = (__shfl(m, base) + __shfl(m, base + 2) + __shfl(m, base + 4)) / 3.0;
        else s = __shfl_xor(m, 2);
        if constexpr (is_f64<R>) f[C] = s;
        else f[C] = float(s - shift_c<L, C>(e));
    });
}

__device__ __forceinline__ void coords(int n, const Grid &g, int &i, int &j, int &k) {
    const int t = (int)div_by((uint32_t)n, g.by_nx);
    i = n - t * g.nx;
    k = (int)div_by((uint32_t)t, g.by_ny);
    j = t - k * g.ny;
}
__device__ __forceinline__ int nboundary(int i, int j, int k, const Grid &g, int nd) {
    int c = (i == 0 || i == g.nx - 1) + (j == 0 || j == g.ny - 1);
    if (nd == 3) c += (k == 0 || k == g.nz - 1);
    return c;
}

// Both lattices' pulls of node n.  With kNtLoads the pulled loads are non-temporal, with kNtStores the
// stores (3D launches whose populations do not fit the Infinity Cache; the host's rule has the sizes):
// a step reads each source population once and writes each once, in an order the next step repeats, so
// lines kept behind only displace each other.  D3Q15 + D3Q7 FP64 forward step: 128x128x64 (369 MB) 92 us
// with plain accesses, 78 to 82 with the loads non-temporal, 76 to 80 with the stores too; 104x100x50
// (183 MB, half of it cached from step to step) 36, 43 and 51 us.  In 2D a source row is reused from L2
// for the rows beside it (4096^2 step 773 -> 837 us with the loads non-temporal), so 2D stays plain.
template <class LA, class LB, class S, class R>
__device__ __forceinline__ void pull_pair(const S *sa, const S *sb, const Grid &g, int i, int j, int k, int n,
                                          const ProgView &pv, R *a, R *b, const Enc &, const Enc &) {
    if (LA::nd == 3 && (g.nt & kNtLoads)) {
        load_pull<LA, true>(sa, g, i, j, k, n, pv.pull[0], a);
        load_pull<LB, true>(sb, g, i, j, k, n, pv.pull[1], b);
    } else {
        load_pull<LA>(sa, g, i, j, k, n, pv.pull[0], a);
        load_pull<LB>(sb, g, i, j, k, n, pv.pull[1], b);
    }
}

// Post-stream, post-boundary state of node n; SMOOTH operators are skipped (callers that own
// smoothed nodes apply them), and all are without ops.  FP64: the populations.  FP32: their deviations from node n's shift
// (oa, ob); the boundary operators run on FP64 populations.
template <class LA, class LB>
__device__ __forceinline__ void node_state(const double *sa, const double *sb, const Grid &g, const ProgView &pv, int n,
                                           double *a, double *b, const Enc &, const Enc &, const Sh4 &, const Sh4 &,
                                           bool ops = true) {
    int i, j, k;
    coords(n, g, i, j, k);
    const NodeOps no = ops_of_node(pv, g, i, j, k, n, LA::nd, ops);
    pull_pair<LA, LB>(sa, sb, g, i, j, k, n, pv, a, b, Enc{}, Enc{});
    run_ops<LA, LB>(pv, no, n, a, b);
}
template <class LA, class LB, class S, std::enable_if_t<!std::is_same_v<S, double>, int> = 0>
__device__ __forceinline__ void node_state(const S *sa, const S *sb, const Grid &g, const ProgView &pv, int n,
                                           float *a, float *b, const Enc &ea, const Enc &eb, const Sh4 &oa,
                                           const Sh4 &ob, bool ops = true) {
    int i, j, k;
    coords(n, g, i, j, k);
    const NodeOps no = ops_of_node(pv, g, i, j, k, n, LA::nd, ops);
    pull_pair<LA, LB>(sa, sb, g, i, j, k, n, pv, a, b, Enc{}, Enc{});
    if (no.count() > 0) {
        double xa[LA::nc], xb[LB::nc > 0 ? LB::nc : 1];
        dev_to_f64<LA>(a, xa, ea, oa);
        if constexpr (LB::nc > 0) dev_to_f64<LB>(b, xb, eb, ob);
        run_ops<LA, LB>(pv, no, n, xa, xb);
        f64_to_dev<LA>(xa, a, ea, oa);
        if constexpr (LB::nc > 0) f64_to_dev<LB>(xb, b, eb, ob);
    }
}

}  // namespace lbm
