// panslbm2_amd/csrc/program.h -- boundary programs: the reference's sequence of boundary calls
// for one time step, tabulated per boundary node.
//
// The reference applies boundary conditions as a sequence of host loops over the domain faces
// (e.g. production/heatsink.cpp:153-168), each loop evaluating a lambda per face node and
// rewriting that node's populations in place.  Every operator is node-local, so the sequence is
// equivalent to running, at each boundary node, that node's operators in call order.  A program
// stores exactly that: per node, the ordered list of operators with their tabulated lambda
// values.  Corner smoothing (SmoothCorner) is the one non-local step and is handled by the
// kernels that own smoothed nodes.
#pragma once
#include <cstdint>

namespace lbm {

enum OpCode : uint8_t {
    OP_NONE = 0,
    OP_BOUNCE = 1,        // d2q9.h:429-501 / d3q15.h:982-1110; arg 1 = BARRIER, 2 = MIRROR
    OP_IBOUNCE = 2,       // d2q9.h:503-575 / d3q15.h:1112-1239
    OP_NS_SET_U = 3,      // navierstokes.h:92-257; v = (ux, uy, uz)
    OP_NS_SET_RHO = 4,    // navierstokes.h:261-426; v = (rho, us, ut)
    OP_AD_SET_T = 5,      // advection.h:99-238; v[0] = T; reads ux, uy, uz
    OP_AD_SET_Q = 6,      // advection.h:242-524; v[0] = qn, v[1] = constant D when the set has no diff
    OP_ANS_ISET_U = 7,    // adjointnavierstokes.h:97-254; v = (ux, uy, uz), v3 = eps; arg = compat
    OP_ANS_ISET_RHO = 8,  // adjointnavierstokes.h:258-392
    OP_AAD_ISET_T = 9,    // adjointadvection.h:154-300; reads ux, uy, uz
    OP_AAD_ISET_Q = 10,   // adjointadvection.h:304-484; v3 = eps
    OP_AAD_ISET_RHO = 11, // adjointadvection.h:488-751; arg = 1 SetT / 2 SetQ, v3 = eps; writes lat, reads the other
    OP_SMOOTH = 12,       // d2q9.h:577-587, d3q15.h:1241-1303 (fix-up kernels only)
};

// One operator at one node, as recorded.
struct Op {
    uint8_t code;
    uint8_t face;  // 0 xmin, 1 xmax, 2 ymin, 3 ymax, 4 zmin, 5 zmax
    uint8_t lat;   // lattice written: 0 = first (NS / adjoint NS), 1 = second (AD / adjoint AD)
    uint8_t arg;
    uint8_t fset;  // index of the field set the operator reads
    uint8_t seg;   // number of SmoothCorner calls recorded before this operator
    uint8_t pad[2];
    double v[3];
    double v3;     // eps where used
};

// Fields a boundary operator reads at its own node (device pointers).  The reference passes
// them as raw arrays to each call (advection.h:1074, adjointadvection.h:1425).
struct FieldSet {
    const double *rho, *ux, *uy, *uz, *tem, *diff;
};
constexpr int kMaxFieldSets = 4;
constexpr size_t kXcdRemapMaxBytes = size_t(640) << 20;  // population bytes read + written per step


// The fused kernels' form of an operator: 16 bits, and its values among the few its node's list holds
// (OpIn: a for the Navier-Stokes operators, b for the advection-diffusion ones), so that a boundary
// node learns all it has to do with one load and has every operand with the next ones.
enum OpSource : uint32_t { kFromFirst = 0, kFromSecond = 1, kFromList = 2 };
constexpr int kWordOps = 8;  // operators in a NodeList of a program without symbols; a longer list's further words sit in list_words
constexpr int kSymbols = 64;  // most symbols of a program (ProgView::sym)
__host__ __device__ constexpr uint32_t op_word(uint32_t code, uint32_t face, uint32_t lat, uint32_t fset, uint32_t arg,
                                               uint32_t src) {
    return code | face << 4 | lat << 7 | fset << 8 | arg << 10 | src << 12;
}
struct OpWord {
    uint32_t code, face, lat, fset, arg, src;
};
__host__ __device__ inline OpWord op_fields(uint32_t w) {
    return OpWord{w & 15u, w >> 4 & 7u, w >> 7 & 1u, w >> 8 & 3u, w >> 10 & 3u, w >> 12 & 3u};
}
// An operator's values: a = (v[0], v[1], v[2], v3); b = (v[0], v[1]) of OP_AD_SET_Q, (v[0], -) of
// OP_AD_SET_T, (-, v3) of the adjoint ones.
struct OpIn {
    double a[4], b[2];
};
// The values of a recorded operator.
__host__ __device__ inline OpIn op_in(const Op &o) {
    return OpIn{{o.v[0], o.v[1], o.v[2], o.v3}, {o.v[0], o.code == OP_AD_SET_Q ? o.v[1] : o.v3}};
}
struct alignas(16) ListVals {  // a list's values: one a, two b
    double a[4], b[2][2];
};

// A boundary node's operators and their values.
struct alignas(16) NodeList {
    uint64_t list_count;         // its first operator in ProgView::list_ops << 24 | operators; 0 without
    uint64_t w[2];               // w[0]: which of ProgView::sym; without symbols: the first kWordOps operators, 16 bits each
    ListVals vals;
};
// The nodes of a grid fall into 27 places: on the low side, between or on the high side of each axis
// (2D: always between in z); 13 is the interior.  Where all nodes of a place share one list, as those
// of a wall or of a uniform inlet do, the fused kernels take it from a table of places, which stays
// in the nearest cache; the nodes of other places look theirs up by slot.
constexpr int kPlaces = 27;
__host__ __device__ inline int place_of(int i, int j, int k, int nx, int ny, int nz, int nd) {
    const int x = i == 0 ? 0 : (i == nx - 1 ? 2 : 1), y = j == 0 ? 0 : (j == ny - 1 ? 2 : 1);
    const int z = nd == 2 ? 1 : (k == 0 ? 0 : (k == nz - 1 ? 2 : 1));
    return x + 3 * y + 9 * z;
}

// Device view of a program.
struct ProgView {
    const int *slot_entry;  // boundary slot -> entry index or -1 (size nslot)
    const int *entry_node;  // entry -> node index
    const int2 *entry_ops;  // entry -> (first op, op count)
    const Op *ops;
    const NodeList *place_list;  // place -> its nodes' list, where they share one
    const NodeList *slot_list;   // boundary slot -> its list (size nslot)
    unsigned shared, by_slot;    // bit p: place p's nodes share a list of operators / have several lists
    const Op *list_ops;         // the lists' operators (for values outside a NodeList)
    const uint32_t *list_words; // their words
    // The program's symbols: its distinct (call, face, word), two words to an element, in the order of
    // the calls and their faces, which every list is in.  They ride in the kernel's arguments: from memory
    // their first use was a round trip of its own (101x101 D2Q9 + D2Q5 step 6.5 us against 6.3).
    // nsym 0: more than kSymbols.
    uint32_t sym[kSymbols / 2];
    int nsym;
    int nentry;
    int nslot;
    FieldSet fs[kMaxFieldSets];
    // The field sets that agree wherever two of them name the same field, as one: a boundary node's
    // fields are loaded once for all of them (bit k of fmerged: set k is in fm; bit k of has_diff:
    // set k has a diffusivity field).
    FieldSet fm;
    unsigned fmerged, has_diff;
    int pull[2];            // per kernel lattice: +1 stream (pull from x - c), -1 iStream (x + c), 0 none
    int latswap;            // 1 when the program's lattice 0 is the kernel's second lattice
    int xcd;                // 1: workgroup -> tile remap that keeps consecutive tiles on one XCD
    // Smoothing after the pass: the fused pass saves the post-boundary state of each
    // smoothed node's inward face neighbours here (kSideStride doubles each: the kernel's first
    // lattice, then its second) and a kernel launched after it averages them (2D corners; 3D edges
    // and corners).  nullptr when unused.
    const int *side_of_slot;  // boundary slot -> side-state index or -1
    double *side;
    // Smoothing inside the fused pass, used when the boundary operators read no array the collide
    // saves: the grid's first lanes rebuild the states of the smoothed nodes' inward neighbours and
    // finish the smoothed nodes, concurrently with the rest of the pass.
    int nsmooth;                // lanes (2D: a wavefront per corner; 3D: the length of smooth_lanes); 0: none
    int smooth_bits;            // bit k: the program's lattice k is smoothed
    const int2 *smooth_lanes;   // 3D: per lane (node whose state it rebuilds, node it finishes or -1)
};
constexpr int kCornerLanes = 512;  // 3D: the first lanes of smooth_lanes, a wavefront per corner
constexpr int kSideStride = 40;  // >= nc(first) + nc(second) of any lattice pair (D3Q27 + D3Q7: 34)

// Boundary slot of node (i, j, k) on an nx*ny*nz grid, -1 for interior nodes.  Surface nodes are
// numbered z-faces first, then the y-faces of the remaining layers, then the x-faces.
__host__ __device__ inline int boundary_slot(int i, int j, int k, int nx, int ny, int nz, int nd) {
    if (nd == 2) {
        if (j == 0) return i;
        if (j == ny - 1) return nx + i;
        if (i == 0) return 2 * nx + (j - 1);
        if (i == nx - 1) return 2 * nx + (ny - 2) + (j - 1);
        return -1;
    }
    if (k == 0) return i + nx * j;
    if (k == nz - 1) return nx * ny + i + nx * j;
    int base = 2 * nx * ny;
    if (j == 0) return base + (k - 1) * nx + i;
    if (j == ny - 1) return base + (nz - 2) * nx + (k - 1) * nx + i;
    base += 2 * (nz - 2) * nx;
    if (i == 0) return base + (k - 1) * (ny - 2) + (j - 1);
    if (i == nx - 1) return base + (nz - 2) * (ny - 2) + (k - 1) * (ny - 2) + (j - 1);
    return -1;
}
__host__ __device__ inline int boundary_slot_count(int nx, int ny, int nz, int nd) {
    if (nd == 2) return 2 * nx + 2 * (ny - 2);
    return 2 * nx * ny + 2 * (nz - 2) * nx + 2 * (nz - 2) * (ny - 2);
}

}  // namespace lbm
