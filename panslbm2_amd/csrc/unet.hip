// panslbm2_amd/csrc/unet.hip -- learned warm start for the steady solves.
//
// A 3-level 3D U-Net (channels c, 2c, 4c with c = 16; two 3x3x3 convolutions + ReLU per level,
// 2x2x2 average pooling, nearest upsampling with skip concatenation [upsampled, skip], a 1x1x1
// linear head) maps the design and the boundary masks to the fields that the InitialCondition
// calls take.  It runs and trains on the GPU:
//
//   * convolutions are implicit GEMMs on the gfx950 matrix cores (v_mfma_f32_16x16x32_bf16):
//     bfloat16 weights and activations, FP32 accumulation.  Activations are channels-last
//     ([voxel][channel], voxel = x + nx (y + ny z)), so the 8 consecutive K values one lane feeds
//     the matrix core (8 channels of one tap) are one 16-byte load, of a brick staged in LDS;
//   * the input gradient of a convolution is the same kernel run on the output gradient with the
//     weights transposed and the taps mirrored;
//   * the weight gradient reduces over voxels: tiles of the output gradient and of the input are
//     staged through LDS as they lie in memory ([voxel][channel]), and the matrix core's operands
//     (eight voxels of one channel) come from transposing LDS reads; partial sums per voxel range are
//     reduced in a fixed order, so the gradient is deterministic;
//   * Adam keeps FP32 master weights and repacks the bfloat16 copies after each update.
//
// The fields the solver uses are FP64 arrays; the network reads and writes them directly
// (normalised by a per-channel mean and scale, optionally relative to base fields, so that it can
// learn the change from a previous solution).  The network has its own HIP stream: its training
// kernels (matrix-core bound) overlap the solver's memory-bound steps on the context stream; the
// calls that read or write solver fields are ordered against the context stream with events.
// The CPU restatement of the same network is oracle/unet_oracle.py.  No reference counterpart:
// the reference starts every solve from rest.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/panslbm2_amd.h"
#include "context.h"
#include "lattice.h"

namespace {

typedef uint16_t bf16_t;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f4;

constexpr int kMaxFields = 16;
constexpr int kTileV = 64;   // voxel ranges of the weight gradient are multiples of this

__host__ __device__ inline bf16_t f2bf(float f) {
    uint32_t u;
    memcpy(&u, &f, 4);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (bf16_t)((u >> 16) | 0x40);  // NaN stays NaN
    u += 0x7fffu + ((u >> 16) & 1u);  // round to nearest even
    return (bf16_t)(u >> 16);
}
__host__ __device__ inline float bf2f(bf16_t h) {
    uint32_t u = (uint32_t)h << 16;
    float f;
    memcpy(&f, &u, 4);
    return f;
}
__device__ inline bf16x8 ld8(const bf16_t *p) { return __builtin_bit_cast(bf16x8, *(const uint4 *)p); }

// ---- convolution (forward, and input gradient with transposed weights) ----------------------------
// y[v][o] = bias[o] + sum_k w[o][k] x[v + off(tap)][ci], k = tap cin + ci.
// The matrix core sums A[m][k] B[k][n] over k: A = weights (row m = lane % 16), B = shifted input
// (column n = lane % 16); both operands give slot j of lane group q the same k = 8q + j, so the
// sum is the same whatever order the hardware pairs slots in.  D[m = 4q + j][n = lane % 16].

// Four output channels of one voxel: bias, ReLU, or the mask of a ReLU's input gradient (act: the
// activation the ReLU gave; y = act > 0 ? value : 0), stored as 8 bytes of bfloat16 or 16 of FP32.
struct ConvOut {
    const float *bias;
    bf16_t *y;
    float *y32;
    const bf16_t *act;
    int cstore, creal, relu;
};
__device__ __forceinline__ void conv_store(const ConvOut &o, size_t v, int co, f4 a) {
    float val[4];
    uint2 on = {0u, 0u};
    if (o.act) on = *(const uint2 *)(o.act + v * o.cstore + co);
    const uint32_t m[4] = {on.x & 0xffffu, on.x >> 16, on.y & 0xffffu, on.y >> 16};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        val[j] = a[j] + (o.bias ? o.bias[co + j] : 0.f);
        if (o.relu) val[j] = fmaxf(val[j], 0.f);
        if (co + j >= o.creal) val[j] = 0.f;  // padded channels stay zero
        if (o.act && !(bf2f((bf16_t)m[j]) > 0.f)) val[j] = 0.f;
    }
    if (o.y) {
        uint2 p;
        p.x = (uint32_t)f2bf(val[0]) | (uint32_t)f2bf(val[1]) << 16;
        p.y = (uint32_t)f2bf(val[2]) | (uint32_t)f2bf(val[3]) << 16;
        *(uint2 *)(o.y + v * o.cstore + co) = p;
    }
    if (o.y32) *(f4 *)(o.y32 + v * o.cstore + co) = f4{val[0], val[1], val[2], val[3]};
}

// 1x1x1 convolution to 16 output channels (the head and its input gradient): one wave computes 16
// channels x 64 voxels; every input is read once, straight from memory.
__global__ void __launch_bounds__(256) k_conv1(const bf16_t *__restrict__ x, int cin, const bf16_t *__restrict__ w,
                                               int kpad, ConvOut out, int V) {
    constexpr int NT = 4;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, r = lane & 15, q = lane >> 4;
    const int v0 = (blockIdx.x * 4 + wv) * (16 * NT), co0 = blockIdx.y * 16;
    f4 acc[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[nt] = f4{0.f, 0.f, 0.f, 0.f};
    for (int kc = 0; kc < kpad; kc += 32) {
        const int k = kc + 8 * q;
        const bf16x8 a = ld8(w + (size_t)(co0 + r) * kpad + k);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            const int v = v0 + nt * 16 + r;
            bf16x8 b = __builtin_bit_cast(bf16x8, uint4{0u, 0u, 0u, 0u});
            if (k < cin && v < V) b = ld8(x + (size_t)v * cin + k);
            acc[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc[nt], 0, 0, 0);
        }
    }
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        const int v = v0 + nt * 16 + r;
        if (v < V) conv_store(out, (size_t)v, co0 + 4 * q, acc[nt]);
    }
}

// d where bit is set, zero where not, without a branch
__device__ __forceinline__ uint4 keep(const uint4 &d, uint32_t bit) {
    const uint32_t m = 0u - (bit & 1u);
    return uint4{d.x & m, d.y & m, d.z & m, d.w & m};
}
// 3x3x3 convolution.  A workgroup of WM x WN waves stages a brick of 18 x 6 x (WN + 2) voxels (its 16
// x 4 x WN outputs and their halo, zero outside the grid) with all CIN channels in LDS once; wave
// (m, n) computes 16 MT output channels of z layer n, 4 rows of 16 voxels.  Read from global memory
// per tap, as it was, every input came through L1 27 times and each of those reads cost an address
// and three bounds checks: at 96x96x48 and 16 -> 16 channels 58 us (109 TFLOP/s), bound by vector
// instructions and L1; 22 us (272 TFLOP/s) now.  Here a K step of 32 costs one LDS read of 16 bytes
// per lane and row at an address the compiler knows up to a per-lane base, and its weights; all K
// steps are unrolled.
// A voxel's row in LDS is 16 bytes longer than its channels (CIN = 8: not), so that the 16 lanes of a
// row fall into different banks.  The products are summed in the order k = 0, 32, ... as before.
template <int CIN>
struct Brick {
    static constexpr int VS = CIN * 2 + (CIN == 8 ? 0 : 16);  // bytes of a voxel in LDS
    static constexpr int KS = (27 * CIN + 31) / 32;           // K steps
    // byte offset of K unit u = 4 step + q (8 values of k) from the voxel at the output's corner (-1, -1, -1)
    static constexpr int off(int u) {
        const int k = 8 * u < 27 * CIN ? 8 * u : 0, t = k / CIN;  // past the end: any voxel of the brick
        return (((t / 9) * 6 + (t / 3) % 3) * 18 + t % 3) * VS + (k % CIN) * 2;
    }
};
template <int CIN, int MT, int WM, int WN>
__global__ void __launch_bounds__(64 * WM * WN) k_conv3(const bf16_t *__restrict__ x, const bf16_t *__restrict__ w,
                                                        ConvOut out, int nx, int ny, int nz, int ntx, int nty) {
    using B = Brick<CIN>;
    constexpr int NT = 4, VS = B::VS, KS = B::KS, KPAD = 32 * KS, NV = 18 * 6 * (WN + 2), THREADS = 64 * WM * WN;
    extern __shared__ __align__(16) unsigned char lds[];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, r = lane & 15, q = lane >> 4;
    const int wm = wv % WM, wn = wv / WM;
    const int bx = blockIdx.x % ntx, by = (blockIdx.x / ntx) % nty, bz = blockIdx.x / (ntx * nty);
    const int x0 = bx * 16, y0 = by * 4, z0 = bz * WN;
    // the weights of the first AHEAD steps; in the loop a step loads those of the step AHEAD later
    constexpr int AHEAD = MT == 1 ? 8 : 4;
    const int co0 = (blockIdx.y * WM + wm) * 16 * MT;
    const bf16_t *wr = w + (size_t)(co0 + r) * KPAD + 8 * q;
    bf16x8 a[AHEAD][MT];
#pragma unroll
    for (int s = 0; s < AHEAD && s < KS; ++s)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) a[s][mt] = ld8(wr + (size_t)mt * 16 * KPAD + 32 * s);
    // loads from clamped addresses, zeroed afterwards, so that a batch of them is in flight at once
    constexpr int CU = CIN / 8, UNITS = NV * CU, IT = (UNITS + THREADS - 1) / THREADS, BATCH = IT < 8 ? IT : 8;
#pragma unroll
    for (int it = 0; it < IT; it += BATCH) {
        uint4 d[BATCH];
        bool in[BATCH];
#pragma unroll
        for (int h = 0; h < BATCH; ++h) {
            const int u = min(tid + (it + h) * THREADS, UNITS - 1), vox = u / CU, c = u - vox * CU;
            const int xx = x0 + vox % 18 - 1, yy = y0 + (vox / 18) % 6 - 1, zz = z0 + vox / 108 - 1;
            in[h] = (unsigned)xx < (unsigned)nx && (unsigned)yy < (unsigned)ny && (unsigned)zz < (unsigned)nz;
            const int v = in[h] ? xx + nx * (yy + ny * zz) : 0;
            d[h] = *(const uint4 *)(x + (size_t)v * CIN + 8 * c);
        }
#pragma unroll
        for (int h = 0; h < BATCH; ++h) {
            const int u = tid + (it + h) * THREADS, vox = u / CU, c = u - vox * CU;
            if (u < UNITS) *(uint4 *)(lds + vox * VS + 16 * c) = keep(d[h], in[h]);
        }
    }
    f4 acc[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = f4{0.f, 0.f, 0.f, 0.f};
    __syncthreads();
    const unsigned char *base = lds + (wn * 108 + r) * VS;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
        // the four lane groups' units: one tap with the next channels, or taps of their own
        const int o0 = B::off(4 * s), o1 = B::off(4 * s + 1), o2 = B::off(4 * s + 2), o3 = B::off(4 * s + 3);
        const int at = (o1 == o0 + 16 && o2 == o0 + 32 && o3 == o0 + 48)
                           ? o0 + 16 * q
                           : (q < 2 ? (q == 0 ? o0 : o1) : (q == 2 ? o2 : o3));
        const bool past = 32 * s + 8 * q >= 27 * CIN;  // the padding of the last step
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            uint4 d = *(const uint4 *)(base + at + nt * 18 * VS);
            if (32 * s + 32 > 27 * CIN && past) d = uint4{0u, 0u, 0u, 0u};
            const bf16x8 b = __builtin_bit_cast(bf16x8, d);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
                acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[s % AHEAD][mt], b, acc[mt][nt], 0, 0, 0);
        }
        if (s + AHEAD < KS) {
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) a[s % AHEAD][mt] = ld8(wr + (size_t)mt * 16 * KPAD + 32 * (s + AHEAD));
            __builtin_amdgcn_sched_barrier(0x38f);  // or the compiler moves the loads down to their use
        }
    }
    const int vx = x0 + r, vz = z0 + wn;
    if (vx >= nx || vz >= nz) return;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        const int vy = y0 + nt;
        if (vy >= ny) continue;
        const size_t v = (size_t)vx + (size_t)nx * (vy + (size_t)ny * vz);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) conv_store(out, v, co0 + mt * 16 + 4 * q, acc[mt][nt]);
    }
}

// ---- weight gradient ----------------------------------------------------------------------------
// part[split][tap][o][i] = sum over the split's voxels v of g[v][o] x[v + off(tap)][i].
// Matrix core: A[m = o][k = v], B[k = v][n = i], K steps of 32 voxels in ascending order.
// bpart[split][o] = sum over the split of g[v][o], as four sums over every fourth 16-voxel run.
//
// 3x3x3: a workgroup takes the three taps along x of one (dy, dz) over one split, a wavefront per tap
// with all of its CG x CX products (the fourth only stages).  Tiles of KT voxels go to LDS as they lie in
// memory, voxel by voxel, so that every load is a run of 16-byte pieces; the matrix core's operands want
// eight voxels of one channel, which the transposing LDS read gives (16 lanes read four voxels of 16
// channels, each lane gets four voxels of one).  The three taps read the same x, one voxel apart; a lane
// whose voxel has no x neighbour reads a row of zeros.  The next tile's loads are issued before the
// products of this one.  What bounds it is the chain of tiles: 38 splits x 9 workgroups on 256 CUs, each
// of a tile's loads, stores and products in turn.  KT: 16384 voxel-channels, 32 kB of loads in flight.
// At 96x96x48, 16 x 16 channels 60 us and 16 x 48 99 us, 3.8e2 us over the ten layers; one tap per
// workgroup with element-wise LDS writes took 178 us a layer, rows transposed in registers with a copy of
// x per tap in LDS 138, 377 and 1.0e3 us.  More splits would fill the chip better (56: a fifth less time
// for the former kernel) but change the order of the sums.
template <int CG, int CX>
struct WgradTile {
    static constexpr int CXP = (CX + 15) & ~15;
    static constexpr int KT = CG + CXP <= 32 ? 512 : (CG + CXP <= 64 ? 256 : 128);
};
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
// four voxels (rows) of 16 channels: lane l of 16 points at channels 4 (l % 4).. of row l / 4 and gets
// the four rows of channel l; two of them are an operand's eight voxels
__device__ __forceinline__ s16x4 tr4(const unsigned char *p) {
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4 *)p);
}
__device__ __forceinline__ bf16x8 tr8(const unsigned char *p, const unsigned char *p4) {
    const s16x4 a = tr4(p), b = tr4(p4);
    return __builtin_bit_cast(bf16x8, __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
}
// TAPS 1 (the head): one tap, one wavefront of products, and a thousand splits of one tile.
template <int CG, int CX, int TAPS>
__global__ void __launch_bounds__(256) k_conv_wgrad(const bf16_t *__restrict__ g, const bf16_t *__restrict__ x,
                                                    int nx, int ny, int nz, lbm::FastDiv by_nx, lbm::FastDiv by_ny,
                                                    int nsplit, int chunk, float *__restrict__ part,
                                                    float *__restrict__ bpart) {
    constexpr int CXP = WgradTile<CG, CX>::CXP, KT = WgradTile<CG, CX>::KT, NM = CG / 16, NN = CXP / 16;
    constexpr int TX = TAPS == 27 ? 3 : 1, NYZ = TAPS / TX;
    constexpr int G8 = CG / 8, X8 = CX / 8;                         // 16-byte pieces of a voxel
    constexpr int GU = KT * G8 / 256, XU = KT * X8 / 256;           // pieces a thread stages per tile
    // K steps at once, so that their LDS reads are under way together (the rows past the split are zeros)
    constexpr int U = NM * NN <= 2 ? 8 : (NM * NN <= 4 ? 4 : 2);
    constexpr int SG = CG * 2, SX = CXP * 2, ZERO = (KT + 2) * SX;  // bytes of an LDS row; the row of zeros
    static_assert(KT * G8 % 256 == 0 && KT * X8 % 256 == 0 && KT / 32 % U == 0, "whole pieces per thread, whole groups of steps");
    __shared__ __align__(16) unsigned char sg[KT * SG];
    __shared__ __align__(16) unsigned char sx[(KT + 3) * SX];  // voxels vb - 1 .. vb + KT, zeros
    const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, q = lane >> 4;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    // the workgroups of a split are on one XCD (workgroup id mod 8), one after another
    const int slot = blockIdx.x >> 3, split = slot / NYZ * 8 + (blockIdx.x & 7), yz = slot % NYZ;
    if (split >= nsplit) return;
    const int V = nx * ny * nz, dy = TAPS == 27 ? yz % 3 - 1 : 0, dz = TAPS == 27 ? yz / 3 - 1 : 0;
    const int off = (dy + ny * dz) * nx;
    const int vbeg = split * chunk, vend = min(V, vbeg + chunk);
    const uint4 none{0u, 0u, 0u, 0u};
    if (tid < SX / 16) *(uint4 *)(sx + ZERO + 16 * tid) = none;
    if constexpr (CX < CXP)  // the channels that pad x
        for (int i = tid; i < (KT + 2) * (CXP - CX) / 8; i += 256)
            *(uint4 *)(sx + i / ((CXP - CX) / 8) * SX + CX * 2 + i % ((CXP - CX) / 8) * 16) = none;
    uint4 dg[GU], dx[XU], dh = none;
    uint32_t in = 0;  // bit i: piece i of g counts; 16 + i: of x; 31: the halo piece
    // x of voxel u + off counts if u is a voxel whose row at (dy, dz) is in the grid
    auto load_x = [&](int u, int c, uint32_t &ok) {
        const int row = (int)lbm::div_by((uint32_t)max(u, 0), by_nx), zz = (int)lbm::div_by((uint32_t)row, by_ny);
        ok = u >= 0 && u < V && (unsigned)(row - zz * ny + dy) < (unsigned)ny && (unsigned)(zz + dz) < (unsigned)nz;
        return *(const uint4 *)(x + (size_t)min(max(u + off, 0), V - 1) * CX + c * 8);
    };
    const int hs = tid / X8;  // threads of the halo: 0 the voxel before the tile, 1 the one after it
    auto load = [&](int vb) {
        in = 0;
#pragma unroll
        for (int i = 0; i < GU; ++i) {
            const int p = tid + 256 * i, v = vb + p / G8;
            dg[i] = *(const uint4 *)(g + (size_t)min(v, V - 1) * CG + p % G8 * 8);
            in |= (uint32_t)(v < vend) << i;
        }
#pragma unroll
        for (int i = 0; i < XU; ++i) {
            const int p = tid + 256 * i;
            uint32_t ok;
            dx[i] = load_x(vb + p / X8, p % X8, ok);
            in |= ok << (16 + i);
        }
        if (hs < 2) {
            uint32_t ok;
            dh = load_x(hs ? vb + KT : vb - 1, tid % X8, ok);
            in |= ok << 31;
        }
    };
    f4 acc[NM][NN];
#pragma unroll
    for (int m = 0; m < NM; ++m)
#pragma unroll
        for (int n = 0; n < NN; ++n) acc[m][n] = f4{0.f, 0.f, 0.f, 0.f};
    const int rot = 32 % nx, none_at = TX == 1 || wv == 1 ? -1 : (wv == 0 ? 0 : nx - 1);  // x without a neighbour at this tap
    const int shift = TX == 1 ? 1 : wv;  // of the tap's x rows against g's
    const int l4 = 8 * q + (r >> 2), lc = (r & 3) * 8;
    const int bt = tid - (256 - 4 * CG);  // the bias's threads, from the fourth wavefront down
    const bool bias = yz == 0 && bt >= 0;
    const int bo = bt & (CG - 1), bq = bt / CG;
    float bsum = 0.f;
    load(vbeg);
    for (int vb = vbeg; vb < vend; vb += KT) {
#pragma unroll
        for (int i = 0; i < GU; ++i) *(uint4 *)(sg + (tid + 256 * i) * 16) = keep(dg[i], in >> i);
#pragma unroll
        for (int i = 0; i < XU; ++i) {
            const int p = tid + 256 * i;
            *(uint4 *)(sx + (1 + p / X8) * SX + p % X8 * 16) = keep(dx[i], in >> (16 + i));
        }
        if (hs < 2) *(uint4 *)(sx + (hs ? KT + 1 : 0) * SX + tid % X8 * 16) = keep(dh, in >> 31);
        __syncthreads();
        if (vb + KT < vend) load(vb + KT);
        const int steps = (min(KT, vend - vb) + 31) / 32;
        if (bias)
            for (int v64 = 0; v64 < 32 * steps; v64 += 64) {
#pragma unroll
                for (int j = 0; j < 16; ++j) bsum += bf2f(*(const bf16_t *)(sg + (v64 + bq * 16 + j) * SG + bo * 2));
            }
        if (wv < TX) {
            int x0 = vb + l4, x4 = x0 + 4;  // the x of the lane's voxels
            x0 -= (int)lbm::div_by((uint32_t)x0, by_nx) * nx;
            x4 -= (int)lbm::div_by((uint32_t)x4, by_nx) * nx;
            for (int k0 = 0; k0 < steps; k0 += U) {
#pragma unroll
                for (int k = k0; k < k0 + U; ++k) {
                    const unsigned char *ga = sg + (32 * k + l4) * SG + lc, *xa = sx + (32 * k + l4 + shift) * SX + lc;
                    const unsigned char *b0 = x0 == none_at ? sx + ZERO + lc : xa;
                    const unsigned char *b4 = x4 == none_at ? sx + ZERO + lc : xa + 4 * SX;
                    bf16x8 a[NM];
#pragma unroll
                    for (int m = 0; m < NM; ++m) a[m] = tr8(ga + 32 * m, ga + 4 * SG + 32 * m);
#pragma unroll
                    for (int n = 0; n < NN; ++n) {
                        const bf16x8 b = tr8(b0 + 32 * n, b4 + 32 * n);
#pragma unroll
                        for (int m = 0; m < NM; ++m)
                            acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[m], b, acc[m][n], 0, 0, 0);
                    }
                    x0 += rot;
                    x0 -= x0 >= nx ? nx : 0;
                    x4 += rot;
                    x4 -= x4 >= nx ? nx : 0;
                }
            }
        }
        __syncthreads();
    }
    if (wv < TX) {
        float *out = part + ((size_t)split * TAPS + 3 * yz + wv) * CG * CXP;
#pragma unroll
        for (int m = 0; m < NM; ++m)
#pragma unroll
            for (int n = 0; n < NN; ++n)
#pragma unroll
                for (int j = 0; j < 4; ++j) out[(size_t)(m * 16 + 4 * q + j) * CXP + n * 16 + r] = acc[m][n][j];
    }
    if (yz == 0) {  // uniform per workgroup
        float *bred = reinterpret_cast<float *>(sg);
        if (bias) bred[4 * bo + bq] = bsum;
        __syncthreads();
        if (tid < CG) bpart[(size_t)split * CG + tid] = (bred[4 * tid] + bred[4 * tid + 1]) + (bred[4 * tid + 2] + bred[4 * tid + 3]);
    }
}

// grad[(o taps + tap) ci + i] = sum over splits (in order) of part[split][tap][o][i]; the bias
// gradient follows the weights: grad[co taps ci + o] = sum over splits of bpart[split][o].  The adds
// are a serial chain per parameter (the order is fixed); its loads are not, so 64 are in flight at
// once, then 16 (the head's 988 splits for 221 parameters: 423 us with one load per add, 46 with 16 in
// flight, now 27; 64 for the other layers' 38, with a clamped rest: 12 us instead of 4.7).
template <int B>
__device__ __forceinline__ void sum_batches(float &s, int &i, const float *__restrict__ &base, uint32_t at,
                                            size_t stride, int n) {
    for (; i + B <= n; i += B) {  // base is the same for all lanes: one scalar add per load
        float v[B];
#pragma unroll
        for (int j = 0; j < B; ++j, base += stride) v[j] = base[at];
#pragma unroll
        for (int j = 0; j < B; ++j) s += v[j];
    }
}
__device__ __forceinline__ float sum_splits(const float *__restrict__ base, uint32_t at, size_t stride, int n) {
    float s = 0.f;
    int i = 0;
    sum_batches<64>(s, i, base, at, stride, n);
    sum_batches<16>(s, i, base, at, stride, n);
    sum_batches<1>(s, i, base, at, stride, n);
    return s;
}
__global__ void __launch_bounds__(64) k_wgrad_reduce(const float *__restrict__ part, const float *__restrict__ bpart,
                                                     int nsplit, int taps, int cg, int cxp, int co, int ci,
                                                     float *__restrict__ grad) {
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    const int nw = co * taps * ci;
    if (n >= nw + co) return;
    if (n < nw) {
        const int i = n % ci, t = (n / ci) % taps, o = n / (ci * taps);
        grad[n] = sum_splits(part, (t * cg + o) * cxp + i, (size_t)taps * cg * cxp, nsplit);
    } else {
        grad[n] = sum_splits(bpart, n - nw, (size_t)cg, nsplit);
    }
}

// ---- weight packing -----------------------------------------------------------------------------
// All convolutions' bfloat16 copies in one launch (blockIdx.y = convolution):
//   forward: wp[o][tap cis + i] = W[o][tap][i] (W is [co][taps][ci] FP32), zero elsewhere;
//   input gradient: wt[i][tap cos + o] = W[o][taps - 1 - tap][i] (mirrored taps, transposed channels);
//   bias: bp[o] = b[o], zero for padded channels.
struct Pack {
    const float *W, *b;
    bf16_t *wp, *wt;
    float *bp;
    int co, taps, ci, cis, cos, kpad, kpadT, rows, rowsT;
};
__global__ void __launch_bounds__(256) k_pack(const Pack *__restrict__ packs) {
    const Pack k = packs[blockIdx.y];
    int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n < k.rows * k.kpad) {
        const int o = n / k.kpad, kk = n - o * k.kpad, t = kk / k.cis, i = kk - t * k.cis;
        k.wp[n] = f2bf(o < k.co && t < k.taps && i < k.ci ? k.W[((size_t)o * k.taps + t) * k.ci + i] : 0.f);
        return;
    }
    n -= k.rows * k.kpad;
    if (n < k.rowsT * k.kpadT) {
        const int i = n / k.kpadT, kk = n - i * k.kpadT, t = kk / k.cos, o = kk - t * k.cos;
        k.wt[n] = f2bf(i < k.ci && t < k.taps && o < k.co ? k.W[((size_t)o * k.taps + (k.taps - 1 - t)) * k.ci + i] : 0.f);
        return;
    }
    n -= k.rowsT * k.kpadT;
    if (n < k.rows) k.bp[n] = n < k.co ? k.b[n] : 0.f;
}

// ---- elementwise pieces ---------------------------------------------------------------------------
struct FieldPtrs {
    const double *f[kMaxFields];
    const double *base[kMaxFields];  // null: no base
    double mean[kMaxFields], scale[kMaxFields];
};
struct FieldOut {
    double *f[kMaxFields];
    const double *base[kMaxFields];
    double mean[kMaxFields], scale[kMaxFields], lo[kMaxFields], hi[kMaxFields];
};

// xs[v][c] = (f_c[v] - base_c[v] - mean_c) / scale_c for c < nf, zero up to cs; bf16 or FP32
__global__ void k_gather(FieldPtrs F, int nf, int cs, int V, bf16_t *__restrict__ xb, float *__restrict__ xf) {
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= V * cs) return;
    const int v = n / cs, c = n - v * cs;
    float val = 0.f;
    if (c < nf) {
        const double b = F.base[c] ? F.base[c][v] : 0.0;
        val = (float)((F.f[c][v] - b - F.mean[c]) / F.scale[c]);
    }
    if (xb) xb[n] = f2bf(val);
    if (xf) xf[n] = val;
}
// f_c[v] = base_c[v] + mean_c + scale_c y[v][c], clamped to [lo_c, hi_c]
__global__ void k_scatter(const float *__restrict__ y, int cs, int nf, int V, FieldOut F) {
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= V * nf) return;
    const int c = n / V, v = n - c * V;
    const double b = F.base[c] ? F.base[c][v] : 0.0;
    const double f = b + F.mean[c] + F.scale[c] * (double)y[(size_t)v * cs + c];
    F.f[c][v] = fmin(fmax(f, F.lo[c]), F.hi[c]);
}

// The elementwise kernels below take 8 channels (16 bytes of bfloat16) per thread: bandwidth-bound
// copies and sums, which 2-byte accesses left at a few hundred GB/s (the level-1 concatenation at
// 96x96x48, 85 MB: 122 us, 13 us now).
__device__ __forceinline__ void unpack8(const bf16_t *p, float (&v)[8]) {
    const uint4 d = *(const uint4 *)p;
    const uint32_t w[4] = {d.x, d.y, d.z, d.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        v[2 * j] = bf2f((bf16_t)(w[j] & 0xffffu));
        v[2 * j + 1] = bf2f((bf16_t)(w[j] >> 16));
    }
}
__device__ __forceinline__ void pack8(bf16_t *p, const float (&v)[8]) {
    uint32_t w[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) w[j] = (uint32_t)f2bf(v[2 * j]) | (uint32_t)f2bf(v[2 * j + 1]) << 16;
    *(uint4 *)p = uint4{w[0], w[1], w[2], w[3]};
}
// 2x2x2 average pooling, fine grid (nx, ny, nz)
__global__ void __launch_bounds__(256) k_pool(const bf16_t *__restrict__ x, int C, int nx, int ny, int nz,
                                              bf16_t *__restrict__ out) {
    const int mx = nx / 2, my = ny / 2, mz = nz / 2, U = C / 8;
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= mx * my * mz * U) return;
    const int c = (n % U) * 8, vc = n / U;
    const int i = vc % mx, j = (vc / mx) % my, k = vc / (mx * my);
    float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ch = 0; ch < 8; ++ch) {  // x fastest
        const int a = ch & 1, b = ch >> 1 & 1, e = ch >> 2;
        float v[8];
        unpack8(x + ((size_t)(2 * i + a) + nx * ((2 * j + b) + ny * (2 * k + e))) * C + c, v);
#pragma unroll
        for (int t = 0; t < 8; ++t) s[t] += v[t];
    }
#pragma unroll
    for (int t = 0; t < 8; ++t) s[t] *= 0.125f;
    pack8(out + (size_t)vc * C + c, s);
}
// out[v] = [coarse[parent(v)] (cu channels), skip[v] (cs channels)]
__global__ void __launch_bounds__(256) k_upcat(const bf16_t *__restrict__ coarse, int cu,
                                               const bf16_t *__restrict__ skip, int cs, int nx, int ny, int nz,
                                               bf16_t *__restrict__ out) {
    const int U = (cu + cs) / 8;
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= nx * ny * nz * U) return;
    const int c = (n % U) * 8, v = n / U;
    uint4 d;
    if (c < cu) {
        const int i = v % nx, j = (v / nx) % ny, k = v / (nx * ny);
        d = *(const uint4 *)(coarse + ((size_t)(i / 2) + (nx / 2) * ((j / 2) + (ny / 2) * (k / 2))) * cu + c);
    } else {
        d = *(const uint4 *)(skip + (size_t)v * cs + (c - cu));
    }
    *(uint4 *)(out + (size_t)n * 8) = d;
}
// g[v][c] = bf16(2 (y - t) / (V nf)) for c < nf, zero to cs; lpart[block] = sum of (y - t)^2
__global__ void __launch_bounds__(256) k_loss(const float *__restrict__ y, const float *__restrict__ t, int cs, int nf,
                                              int V, bf16_t *__restrict__ g, float *__restrict__ lpart) {
    __shared__ float red[256];
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    float sq = 0.f;
    if (n < V * cs) {
        const int c = n % cs;
        float d = 0.f;
        if (c < nf) d = y[n] - t[n];
        sq = d * d;
        g[n] = f2bf(2.f * d / ((float)V * (float)nf));
    }
    red[threadIdx.x] = sq;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) lpart[blockIdx.x] = red[0];
}
// one workgroup of 256: strided partial sums, then a tree (fixed order, deterministic)
__global__ void __launch_bounds__(256) k_loss_final(const float *__restrict__ lpart, int n, double inv,
                                                    double *__restrict__ out) {
    __shared__ double red[256];
    double s = 0.0;
    for (int i = threadIdx.x; i < n; i += 256) s += lpart[i];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int k = 128; k > 0; k >>= 1) {
        if ((int)threadIdx.x < k) red[threadIdx.x] += red[threadIdx.x + k];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[0] = red[0] * inv;
}
__device__ __forceinline__ void unpack8(const float *p, float (&v)[8]) {
    const f4 a = *(const f4 *)p, b = *(const f4 *)(p + 4);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        v[j] = a[j];
        v[4 + j] = b[j];
    }
}
// coarse grid: out[vc][c] = act > 0 ? bf16(sum over the 8 children of d[v][c]) : 0  (fine dims given)
__global__ void __launch_bounds__(256) k_up_bwd(const float *__restrict__ d, int cd, const bf16_t *__restrict__ act,
                                                int C, int nx, int ny, int nz, bf16_t *__restrict__ out) {
    const int mx = nx / 2, my = ny / 2, mz = nz / 2, U = C / 8;
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= mx * my * mz * U) return;
    const int c = (n % U) * 8, vc = n / U;
    const int i = vc % mx, j = (vc / mx) % my, k = vc / (mx * my);
    float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, on[8];
#pragma unroll
    for (int ch = 0; ch < 8; ++ch) {
        const int a = ch & 1, b = ch >> 1 & 1, e = ch >> 2;
        float v[8];
        unpack8(d + ((size_t)(2 * i + a) + nx * ((2 * j + b) + ny * (2 * k + e))) * cd + c, v);
#pragma unroll
        for (int t = 0; t < 8; ++t) s[t] += v[t];
    }
    unpack8(act + (size_t)n * 8, on);
#pragma unroll
    for (int t = 0; t < 8; ++t) s[t] = on[t] > 0.f ? s[t] : 0.f;
    pack8(out + (size_t)n * 8, s);
}
// fine grid: out[v][c] = act > 0 ? bf16(skip[v][off + c] + dc[parent(v)][c] / 8) : 0
__global__ void __launch_bounds__(256) k_pool_bwd(const float *__restrict__ dc, const float *__restrict__ skip,
                                                  int cskip, int off, const bf16_t *__restrict__ act, int C, int nx,
                                                  int ny, int nz, bf16_t *__restrict__ out) {
    const int U = C / 8;
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= nx * ny * nz * U) return;
    const int c = (n % U) * 8, v = n / U;
    const int i = v % nx, j = (v / nx) % ny, k = v / (nx * ny);
    const size_t p = (size_t)(i / 2) + (nx / 2) * ((j / 2) + (ny / 2) * (k / 2));
    float s[8], h[8], on[8];
    unpack8(skip + (size_t)v * cskip + off + c, s);
    unpack8(dc + p * C + c, h);
    unpack8(act + (size_t)n * 8, on);
#pragma unroll
    for (int t = 0; t < 8; ++t) s[t] = on[t] > 0.f ? s[t] + h[t] * 0.125f : 0.f;
    pack8(out + (size_t)n * 8, s);
}
// Adam (Kingma & Ba 2015, Algorithm 1); bc1 = 1 - beta1^t, bc2 = 1 - beta2^t
__global__ void k_adam(float *__restrict__ p, const float *__restrict__ g, float *__restrict__ m,
                       float *__restrict__ v, size_t n, float lr, float b1, float b2, float eps, float bc1, float bc2) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr * (mi / bc1) / (sqrtf(vi / bc2) + eps);
}
__global__ void k_bf_to_f64(const bf16_t *__restrict__ a, int cs, int cr, int V, double *__restrict__ b) {
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= V * cr) return;
    const int v = n / cr, c = n - v * cr;
    b[n] = bf2f(a[(size_t)v * cs + c]);
}
__global__ void k_f_to_f64(const float *__restrict__ a, int cs, int cr, int V, double *__restrict__ b) {
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= V * cr) return;
    const int v = n / cr, c = n - v * cr;
    b[n] = a[(size_t)v * cs + c];
}

inline unsigned blocks(size_t n, int b = 256) { return (unsigned)((n + b - 1) / b); }
inline int r16(int c) { return (c + 15) & ~15; }
inline int r32(int c) { return (c + 31) & ~31; }

}  // namespace

// ==================================================================================================
struct lbm_unet {
    lbm_context *ctx = nullptr;
    hipStream_t s = nullptr;                          // the network's own stream
    hipEvent_t ev_in = nullptr, ev_out = nullptr;     // ordering against the context stream
    int dims[3][3] = {};  // per level: nx, ny, nz
    int V[3] = {};
    int cin = 0, cout = 0, base = 16;
    struct Conv {
        std::string name;
        int ci, co, taps, cis, level;  // real in/out channels, taps, stored input channels, grid level
        size_t wo, bo;                 // offsets of W and b in the parameter vector
        int kpad, kpadT, rowsT;        // packed K (forward), packed K and rows (input gradient)
        bf16_t *wp = nullptr, *wt = nullptr;
        float *bp = nullptr;
    };
    std::vector<Conv> conv;
    size_t np = 0;
    int adam_t = 0;
    std::vector<void *> allocs;
    float *p = nullptr, *g = nullptr, *m = nullptr, *v = nullptr;
    // activations
    bf16_t *x0, *e1a, *e1b, *p1, *e2a, *e2b, *p2, *e3a, *e3b, *cat2, *d2a, *d2b, *cat1, *d1a, *d1b;
    float *y32, *tgt;
    // backward scratch
    bf16_t *gb0, *gb1;
    float *dx1, *dx2, *dxt, *wpart, *bpart, *lpart;
    double *dloss, *hloss;
    size_t wpart_n = 0, bpart_n = 0;
    Pack *packs = nullptr;  // the convolutions' packing tables, on the device
    size_t pack_n = 0;      // the most values one of them packs
    bool have_target = false;
};

namespace {

int hipfail(hipError_t e, const char *what) {
    return lbm::set_error(LBM_ERR_HIP, "%s: %s", what, hipGetErrorString(e));
}
#define UCHK(expr)                                                                                     \
    do {                                                                                               \
        hipError_t e_ = (expr);                                                                        \
        if (e_ != hipSuccess) return hipfail(e_, #expr);                                               \
    } while (0)

template <class T>
int alloc(lbm_unet *N, T **p, size_t n) {
    void *q = nullptr;
    UCHK(hipMalloc(&q, n * sizeof(T) + 16));
    N->allocs.push_back(q);
    *p = (T *)q;
    return LBM_OK;
}

template <int CIN, int MT, int WM, int WN>
int launch_conv3(lbm_unet *N, const bf16_t *x, const bf16_t *w, const ConvOut &out, int tiles, const int *d) {
    const int ntx = (d[0] + 15) / 16, nty = (d[1] + 3) / 4, ntz = (d[2] + WN - 1) / WN;
    const int lds = 18 * 6 * (WN + 2) * Brick<CIN>::VS;
    if (lds > 65536)
        UCHK(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_conv3<CIN, MT, WM, WN>),
                                 hipFuncAttributeMaxDynamicSharedMemorySize, lds));
    k_conv3<CIN, MT, WM, WN><<<dim3(ntx * nty * ntz, tiles / (MT * WM)), 64 * WM * WN, lds, N->s>>>(
        x, w, out, d[0], d[1], d[2], ntx, nty);
    UCHK(hipGetLastError());
    return LBM_OK;
}
// The network's shapes.  The waves of a workgroup share its brick: across the output channels as far
// as there are tiles of 16 (every one of them would otherwise stage the same voxels), the rest along z;
// three tiles to a wave where their number is a multiple of three.  At 96x96x48: 16 -> 16 channels 22 us,
// 16 -> 48 56 us, 48 -> 16 52 us, 32 -> 32 (48x48x24) 11.5 us (25, 58, 76 and 17 with the weights loaded at their use).
int launch_conv(lbm_unet *N, const bf16_t *x, int cin, int taps, const bf16_t *w, int kpad, const ConvOut &out,
                const int *d) {
    const int V = d[0] * d[1] * d[2];
    const int tiles = out.cstore > 0 ? out.cstore / 16 : 0;
    if (cin % 8 || kpad % 32 || tiles <= 0 || out.cstore % 16)
        return lbm::set_error(LBM_ERR_ARG, "conv shape: cin %d kpad %d", cin, kpad);
    if (taps == 1) {
        k_conv1<<<dim3(blocks(V, 256), tiles), 256, 0, N->s>>>(x, cin, w, kpad, out, V);
        UCHK(hipGetLastError());
        return LBM_OK;
    }
    switch (100 * cin + tiles) {
    case 801: return launch_conv3<8, 1, 1, 4>(N, x, w, out, tiles, d);
    case 1601: return launch_conv3<16, 1, 1, 4>(N, x, w, out, tiles, d);
    case 1602: return launch_conv3<16, 1, 2, 2>(N, x, w, out, tiles, d);
    case 1603: return launch_conv3<16, 3, 1, 4>(N, x, w, out, tiles, d);
    case 3201: return launch_conv3<32, 1, 1, 4>(N, x, w, out, tiles, d);
    case 3202: return launch_conv3<32, 1, 2, 2>(N, x, w, out, tiles, d);
    case 3204: return launch_conv3<32, 1, 4, 1>(N, x, w, out, tiles, d);
    case 3206: return launch_conv3<32, 3, 2, 2>(N, x, w, out, tiles, d);
    case 4801: return launch_conv3<48, 1, 1, 4>(N, x, w, out, tiles, d);
    case 6402: return launch_conv3<64, 1, 2, 2>(N, x, w, out, tiles, d);
    case 6404: return launch_conv3<64, 1, 4, 1>(N, x, w, out, tiles, d);
    case 9602: return launch_conv3<96, 1, 2, 1>(N, x, w, out, tiles, d);
    }
    return lbm::set_error(LBM_ERR_ARG, "conv shape: cin %d, %d output tiles", cin, tiles);
}

// splits of a voxel range for the weight gradient: about 1024 workgroups over all taps
void wsplit(int V, int taps, int *nsplit, int *chunk) {
    int want = (1024 + taps - 1) / taps;
    int maxs = (V + kTileV - 1) / kTileV;
    int ns = want < maxs ? want : maxs;
    if (ns < 1) ns = 1;
    int ch = ((V + ns - 1) / ns + kTileV - 1) / kTileV * kTileV;
    *chunk = ch;
    *nsplit = (V + ch - 1) / ch;
}

template <int CG, int CX, int TAPS>
void launch_wgrad(lbm_unet *N, const bf16_t *g, const bf16_t *x, const int *d, int nsplit, int chunk) {
    k_conv_wgrad<CG, CX, TAPS><<<(nsplit + 7) / 8 * 8 * (TAPS == 27 ? 9 : 1), 256, 0, N->s>>>(
        g, x, d[0], d[1], d[2], lbm::fast_div(d[0]), lbm::fast_div(d[1]), nsplit, chunk, N->wpart, N->bpart);
}

// gradient of conv c: g is the output gradient (bf16, r16(co) channels), x its input (cis channels)
int conv_grads(lbm_unet *N, const lbm_unet::Conv &c, const bf16_t *g, const bf16_t *x) {
    const int *d = N->dims[c.level];
    const int V = N->V[c.level], cg = r16(c.co), cxp = r16(c.cis);
    int nsplit, chunk;
    wsplit(V, c.taps, &nsplit, &chunk);
    if ((size_t)nsplit * c.taps * cg * cxp > N->wpart_n) return lbm::set_error(LBM_ERR_ARG, "weight partials overflow");
    if ((size_t)nsplit * cg > N->bpart_n) return lbm::set_error(LBM_ERR_ARG, "bias partials overflow");
    const int shape = (c.taps == 27 ? 0 : 10000) + cg * 100 + c.cis;
    switch (shape) {
    case 1608: launch_wgrad<16, 8, 27>(N, g, x, d, nsplit, chunk); break;
    case 1616: launch_wgrad<16, 16, 27>(N, g, x, d, nsplit, chunk); break;
    case 1648: launch_wgrad<16, 48, 27>(N, g, x, d, nsplit, chunk); break;
    case 3216: launch_wgrad<32, 16, 27>(N, g, x, d, nsplit, chunk); break;
    case 3232: launch_wgrad<32, 32, 27>(N, g, x, d, nsplit, chunk); break;
    case 3296: launch_wgrad<32, 96, 27>(N, g, x, d, nsplit, chunk); break;
    case 6432: launch_wgrad<64, 32, 27>(N, g, x, d, nsplit, chunk); break;
    case 6464: launch_wgrad<64, 64, 27>(N, g, x, d, nsplit, chunk); break;
    case 11616: launch_wgrad<16, 16, 1>(N, g, x, d, nsplit, chunk); break;
    default: return lbm::set_error(LBM_ERR_ARG, "weight gradient: %d x %d channels, %d taps", cg, c.cis, c.taps);
    }
    UCHK(hipGetLastError());
    const int nw = c.co * c.taps * c.ci;  // the bias follows the weights in the parameter vector
    k_wgrad_reduce<<<blocks(nw + c.co, 64), 64, 0, N->s>>>(N->wpart, N->bpart, nsplit, c.taps, cg, cxp, c.co, c.ci,
                                                         N->g + c.wo);
    UCHK(hipGetLastError());
    return LBM_OK;
}

int conv_fwd(lbm_unet *N, int i, const bf16_t *x, bf16_t *y, float *y32, int relu) {
    const auto &c = N->conv[i];
    return launch_conv(N, x, c.cis, c.taps, c.wp, c.kpad, ConvOut{c.bp, y, y32, nullptr, r16(c.co), c.co, relu},
                       N->dims[c.level]);
}
// input gradient of conv i (cis channels): into dx as FP32, or through the ReLU that gave act, into gb
int conv_dx(lbm_unet *N, int i, const bf16_t *g, float *dx, bf16_t *gb = nullptr, const bf16_t *act = nullptr) {
    const auto &c = N->conv[i];
    return launch_conv(N, g, r16(c.co), c.taps, c.wt, c.kpadT, ConvOut{nullptr, gb, dx, act, c.cis, c.cis, 0},
                       N->dims[c.level]);
}

int repack(lbm_unet *N) {
    k_pack<<<dim3(blocks(N->pack_n), (unsigned)N->conv.size()), 256, 0, N->s>>>(N->packs);
    UCHK(hipGetLastError());
    return LBM_OK;
}

enum { E1A, E1B, E2A, E2B, E3A, E3B, D2A, D2B, D1A, D1B, HEAD };

int forward(lbm_unet *N) {
    const int c1 = N->base, c2 = 2 * c1, c3 = 4 * c1;
    int rc;
#define F(call)                                                                                        \
    if ((rc = (call)) != LBM_OK) return rc
    F(conv_fwd(N, E1A, N->x0, N->e1a, nullptr, 1));
    F(conv_fwd(N, E1B, N->e1a, N->e1b, nullptr, 1));
    const int *d1 = N->dims[0], *d2 = N->dims[1];
    k_pool<<<blocks((size_t)N->V[1] * c1 / 8), 256, 0, N->s>>>(N->e1b, c1, d1[0], d1[1], d1[2], N->p1);
    F(conv_fwd(N, E2A, N->p1, N->e2a, nullptr, 1));
    F(conv_fwd(N, E2B, N->e2a, N->e2b, nullptr, 1));
    k_pool<<<blocks((size_t)N->V[2] * c2 / 8), 256, 0, N->s>>>(N->e2b, c2, d2[0], d2[1], d2[2], N->p2);
    F(conv_fwd(N, E3A, N->p2, N->e3a, nullptr, 1));
    F(conv_fwd(N, E3B, N->e3a, N->e3b, nullptr, 1));
    k_upcat<<<blocks((size_t)N->V[1] * (c3 + c2) / 8), 256, 0, N->s>>>(N->e3b, c3, N->e2b, c2, d2[0], d2[1], d2[2], N->cat2);
    F(conv_fwd(N, D2A, N->cat2, N->d2a, nullptr, 1));
    F(conv_fwd(N, D2B, N->d2a, N->d2b, nullptr, 1));
    k_upcat<<<blocks((size_t)N->V[0] * (c2 + c1) / 8), 256, 0, N->s>>>(N->d2b, c2, N->e1b, c1, d1[0], d1[1], d1[2], N->cat1);
    F(conv_fwd(N, D1A, N->cat1, N->d1a, nullptr, 1));
    F(conv_fwd(N, D1B, N->d1a, N->d1b, nullptr, 1));
    F(conv_fwd(N, HEAD, N->d1b, nullptr, N->y32, 0));
    UCHK(hipGetLastError());
    return LBM_OK;
}

int backward(lbm_unet *N) {
    const int c1 = N->base, c2 = 2 * c1, c3 = 4 * c1, co = r16(N->cout);
    const int *d1 = N->dims[0], *d2 = N->dims[1];
    const int V1 = N->V[0], V2 = N->V[1], V3 = N->V[2];
    int rc;
    const int nl = (int)blocks((size_t)V1 * co);
    k_loss<<<nl, 256, 0, N->s>>>(N->y32, N->tgt, co, N->cout, V1, N->gb0, N->lpart);
    k_loss_final<<<1, 256, 0, N->s>>>(N->lpart, nl, 1.0 / ((double)V1 * N->cout), N->dloss);
    // head and level-1 decoder
    F(conv_grads(N, N->conv[HEAD], N->gb0, N->d1b));
    F(conv_dx(N, HEAD, N->gb0, nullptr, N->gb1, N->d1b));
    F(conv_grads(N, N->conv[D1B], N->gb1, N->d1a));
    F(conv_dx(N, D1B, N->gb1, nullptr, N->gb0, N->d1a));
    F(conv_grads(N, N->conv[D1A], N->gb0, N->cat1));
    F(conv_dx(N, D1A, N->gb0, N->dx1));  // [V1][c2 + c1]: upsampled part, then the skip of e1b
    k_up_bwd<<<blocks((size_t)V2 * c2 / 8), 256, 0, N->s>>>(N->dx1, c2 + c1, N->d2b, c2, d1[0], d1[1], d1[2], N->gb1);
    // level-2 decoder
    F(conv_grads(N, N->conv[D2B], N->gb1, N->d2a));
    F(conv_dx(N, D2B, N->gb1, nullptr, N->gb0, N->d2a));
    F(conv_grads(N, N->conv[D2A], N->gb0, N->cat2));
    F(conv_dx(N, D2A, N->gb0, N->dx2));  // [V2][c3 + c2]
    k_up_bwd<<<blocks((size_t)V3 * c3 / 8), 256, 0, N->s>>>(N->dx2, c3 + c2, N->e3b, c3, d2[0], d2[1], d2[2], N->gb1);
    // bottleneck
    F(conv_grads(N, N->conv[E3B], N->gb1, N->e3a));
    F(conv_dx(N, E3B, N->gb1, nullptr, N->gb0, N->e3a));
    F(conv_grads(N, N->conv[E3A], N->gb0, N->p2));
    F(conv_dx(N, E3A, N->gb0, N->dxt));  // [V3][c2]
    k_pool_bwd<<<blocks((size_t)V2 * c2 / 8), 256, 0, N->s>>>(N->dxt, N->dx2, c3 + c2, c3, N->e2b, c2, d2[0], d2[1], d2[2],
                                                         N->gb1);
    // level-2 encoder
    F(conv_grads(N, N->conv[E2B], N->gb1, N->e2a));
    F(conv_dx(N, E2B, N->gb1, nullptr, N->gb0, N->e2a));
    F(conv_grads(N, N->conv[E2A], N->gb0, N->p1));
    F(conv_dx(N, E2A, N->gb0, N->dxt));  // [V2][c1]
    k_pool_bwd<<<blocks((size_t)V1 * c1 / 8), 256, 0, N->s>>>(N->dxt, N->dx1, c2 + c1, c2, N->e1b, c1, d1[0], d1[1], d1[2],
                                                         N->gb1);
    // level-1 encoder
    F(conv_grads(N, N->conv[E1B], N->gb1, N->e1a));
    F(conv_dx(N, E1B, N->gb1, nullptr, N->gb0, N->e1a));
    F(conv_grads(N, N->conv[E1A], N->gb0, N->x0));
#undef F
    UCHK(hipGetLastError());
    return LBM_OK;
}

int adam(lbm_unet *N, double lr, double b1, double b2, double eps) {
    N->adam_t += 1;
    const double bc1 = 1.0 - std::pow(b1, N->adam_t), bc2 = 1.0 - std::pow(b2, N->adam_t);
    k_adam<<<blocks(N->np), 256, 0, N->s>>>(N->p, N->g, N->m, N->v, N->np, (float)lr, (float)b1, (float)b2,
                                            (float)eps, (float)bc1, (float)bc2);
    UCHK(hipGetLastError());
    return repack(N);
}

int fields_in(const double *const *f, const double *const *base, const double *mean, const double *scale, int nf,
              FieldPtrs *F) {
    if (nf < 1 || nf > kMaxFields || !f) return lbm::set_error(LBM_ERR_ARG, "1..%d fields expected", kMaxFields);
    for (int c = 0; c < nf; ++c) {
        if (!f[c]) return lbm::set_error(LBM_ERR_ARG, "field %d is null", c);
        F->f[c] = f[c];
        F->base[c] = base ? base[c] : nullptr;
        F->mean[c] = mean ? mean[c] : 0.0;
        F->scale[c] = scale ? scale[c] : 1.0;
        if (F->scale[c] == 0.0) return lbm::set_error(LBM_ERR_ARG, "field %d has scale 0", c);
    }
    return LBM_OK;
}

void destroy(lbm_unet *N) {
    if (!N) return;
    (void)hipSetDevice(lbm::context_device(N->ctx));
    if (N->s) (void)hipStreamSynchronize(N->s);
    for (void *q : N->allocs) (void)hipFree(q);
    if (N->hloss) (void)hipHostFree(N->hloss);
    if (N->ev_in) (void)hipEventDestroy(N->ev_in);
    if (N->ev_out) (void)hipEventDestroy(N->ev_out);
    if (N->s) (void)hipStreamDestroy(N->s);
    delete N;
}

// the network stream waits for what the context stream has queued so far
int after_ctx(lbm_unet *N) {
    UCHK(hipEventRecord(N->ev_in, lbm::context_stream(N->ctx)));
    UCHK(hipStreamWaitEvent(N->s, N->ev_in, 0));
    return LBM_OK;
}
// the context stream waits for what the network stream has queued so far
int before_ctx(lbm_unet *N) {
    UCHK(hipEventRecord(N->ev_out, N->s));
    UCHK(hipStreamWaitEvent(lbm::context_stream(N->ctx), N->ev_out, 0));
    return LBM_OK;
}

// xorshift64* stream for the initial weights
struct Rng {
    uint64_t s;
    double uniform() {
        s ^= s >> 12;
        s ^= s << 25;
        s ^= s >> 27;
        return (double)((s * 2685821657736338717ull) >> 11) * (1.0 / 9007199254740992.0);
    }
};

}  // namespace

extern "C" {

int lbm_unet_create(lbm_context *ctx, int nx, int ny, int nz, int cin, int cout, int base, unsigned long long seed,
                    lbm_unet **out) {
    if (!ctx || !out) return lbm::set_error(LBM_ERR_ARG, "null argument");
    *out = nullptr;
    if (nx < 4 || ny < 4 || nz < 4 || nx % 4 || ny % 4 || nz % 4)
        return lbm::set_error(LBM_ERR_ARG, "grid %dx%dx%d: each side a multiple of 4 (two poolings)", nx, ny, nz);
    if (cin < 1 || cin > 8) return lbm::set_error(LBM_ERR_ARG, "cin %d: 1..8 input fields", cin);
    if (cout < 1 || cout > 16) return lbm::set_error(LBM_ERR_ARG, "cout %d: 1..16 output fields", cout);
    if (base != 16) return lbm::set_error(LBM_ERR_UNSUPPORTED, "base %d: only 16 (channels 16/32/64)", base);
    if ((size_t)nx * ny * nz > (size_t)1 << 28) return lbm::set_error(LBM_ERR_ARG, "grid too large");
    UCHK(hipSetDevice(lbm::context_device(ctx)));
    lbm_unet *N = new lbm_unet;
    N->ctx = ctx;
    if (hipStreamCreateWithFlags(&N->s, hipStreamNonBlocking) != hipSuccess ||
        hipEventCreateWithFlags(&N->ev_in, hipEventDisableTiming) != hipSuccess ||
        hipEventCreateWithFlags(&N->ev_out, hipEventDisableTiming) != hipSuccess) {
        destroy(N);
        return lbm::set_error(LBM_ERR_HIP, "stream or event creation failed");
    }
    N->cin = cin;
    N->cout = cout;
    N->base = base;
    for (int l = 0; l < 3; ++l) {
        N->dims[l][0] = nx >> l;
        N->dims[l][1] = ny >> l;
        N->dims[l][2] = nz >> l;
        N->V[l] = N->dims[l][0] * N->dims[l][1] * N->dims[l][2];
    }
    const int c1 = base, c2 = 2 * base, c3 = 4 * base;
    struct L {
        const char *name;
        int ci, co, taps, cis, level;
    } layers[] = {
        {"e1a", cin, c1, 27, 8, 0},        {"e1b", c1, c1, 27, c1, 0},      {"e2a", c1, c2, 27, c1, 1},
        {"e2b", c2, c2, 27, c2, 1},        {"e3a", c2, c3, 27, c2, 2},      {"e3b", c3, c3, 27, c3, 2},
        {"d2a", c3 + c2, c2, 27, c3 + c2, 1}, {"d2b", c2, c2, 27, c2, 1},   {"d1a", c2 + c1, c1, 27, c2 + c1, 0},
        {"d1b", c1, c1, 27, c1, 0},        {"head", c1, cout, 1, c1, 0},
    };
    size_t off = 0;
    for (const auto &l : layers) {
        lbm_unet::Conv c;
        c.name = l.name;
        c.ci = l.ci;
        c.co = l.co;
        c.taps = l.taps;
        c.cis = l.cis;
        c.level = l.level;
        c.wo = off;
        c.bo = off + (size_t)l.co * l.taps * l.ci;
        off = c.bo + l.co;
        c.kpad = r32(l.taps * l.cis);
        c.kpadT = r32(l.taps * r16(l.co));
        c.rowsT = r16(l.cis);
        N->conv.push_back(c);
    }
    N->np = off;
    const size_t V1 = N->V[0], V2 = N->V[1], V3 = N->V[2];
    int rc = LBM_OK;
#define A(p, n)                                                                                        \
    if (rc == LBM_OK) rc = alloc(N, &(p), (n))
    A(N->p, N->np);
    A(N->g, N->np);
    A(N->m, N->np);
    A(N->v, N->np);
    for (auto &c : N->conv) {
        A(c.wp, (size_t)r16(c.co) * c.kpad);
        A(c.wt, (size_t)c.rowsT * c.kpadT);
        A(c.bp, (size_t)r16(c.co));
    }
    A(N->x0, V1 * 8);
    A(N->e1a, V1 * c1);
    A(N->e1b, V1 * c1);
    A(N->p1, V2 * c1);
    A(N->e2a, V2 * c2);
    A(N->e2b, V2 * c2);
    A(N->p2, V3 * c2);
    A(N->e3a, V3 * c3);
    A(N->e3b, V3 * c3);
    A(N->cat2, V2 * (c3 + c2));
    A(N->d2a, V2 * c2);
    A(N->d2b, V2 * c2);
    A(N->cat1, V1 * (c2 + c1));
    A(N->d1a, V1 * c1);
    A(N->d1b, V1 * c1);
    A(N->y32, V1 * r16(cout));
    A(N->tgt, V1 * r16(cout));
    size_t gmax = std::max(std::max(V1 * c1, V2 * c2), V3 * c3);
    gmax = std::max(gmax, V1 * (size_t)r16(cout));
    A(N->gb0, gmax);
    A(N->gb1, gmax);
    A(N->dx1, V1 * (c2 + c1));
    A(N->dx2, V2 * (c3 + c2));
    A(N->dxt, gmax);
    size_t wpn = 0;
    for (auto &c : N->conv) {
        int ns, ch;
        wsplit(N->V[c.level], c.taps, &ns, &ch);
        wpn = std::max(wpn, (size_t)ns * c.taps * r16(c.co) * r16(c.cis));
    }
    N->wpart_n = wpn;
    A(N->wpart, wpn);
    size_t bpn = 0;
    for (auto &c : N->conv) {
        int ns, ch;
        wsplit(N->V[c.level], c.taps, &ns, &ch);
        bpn = std::max(bpn, (size_t)ns * r16(c.co));
    }
    N->bpart_n = bpn;
    A(N->bpart, N->bpart_n);
    A(N->lpart, blocks(V1 * r16(cout)));
    A(N->dloss, 1);
    A(N->packs, N->conv.size());
#undef A
    if (rc == LBM_OK && hipHostMalloc(&N->hloss, sizeof(double), hipHostMallocDefault) != hipSuccess)
        rc = lbm::set_error(LBM_ERR_HIP, "hipHostMalloc failed");
    if (rc != LBM_OK) {
        destroy(N);
        return rc;
    }
    // He-uniform initial weights (bound sqrt(6 / fan_in)), zero biases, and a zero linear head:
    // the untrained network outputs zero (the base fields, when it predicts a change)
    std::vector<float> h(N->np, 0.f);
    Rng rng{seed * 0x9E3779B97F4A7C15ull + 0x2545F4914F6CDD1Dull};
    for (auto &c : N->conv) {
        if (c.name == "head") continue;
        const double b = std::sqrt(6.0 / ((double)c.taps * c.ci));
        for (size_t i = c.wo; i < c.bo; ++i) h[i] = (float)((2.0 * rng.uniform() - 1.0) * b);
    }
    hipError_t e = hipMemcpyAsync(N->p, h.data(), N->np * sizeof(float), hipMemcpyHostToDevice, N->s);
    if (e == hipSuccess) e = hipMemsetAsync(N->m, 0, N->np * sizeof(float), N->s);
    if (e == hipSuccess) e = hipMemsetAsync(N->v, 0, N->np * sizeof(float), N->s);
    if (e == hipSuccess) e = hipMemsetAsync(N->g, 0, N->np * sizeof(float), N->s);
    if (e == hipSuccess) e = hipMemsetAsync(N->x0, 0, V1 * 8 * sizeof(bf16_t), N->s);
    if (e == hipSuccess) e = hipMemsetAsync(N->tgt, 0, V1 * r16(cout) * sizeof(float), N->s);
    std::vector<Pack> packs;
    for (const auto &c : N->conv) {
        packs.push_back(Pack{N->p + c.wo, N->p + c.bo, c.wp, c.wt, c.bp, c.co, c.taps, c.ci, c.cis, r16(c.co), c.kpad,
                             c.kpadT, r16(c.co), c.rowsT});
        N->pack_n = std::max(N->pack_n, (size_t)r16(c.co) * (c.kpad + 1) + (size_t)c.rowsT * c.kpadT);
    }
    if (e == hipSuccess)
        e = hipMemcpyAsync(N->packs, packs.data(), packs.size() * sizeof(Pack), hipMemcpyHostToDevice, N->s);
    if (e == hipSuccess) e = hipStreamSynchronize(N->s);
    if (e != hipSuccess) {
        destroy(N);
        return hipfail(e, "initial weights");
    }
    if ((rc = repack(N)) != LBM_OK) {
        destroy(N);
        return rc;
    }
    *out = N;
    return LBM_OK;
}

int lbm_unet_destroy(lbm_unet *net) {
    destroy(net);
    return LBM_OK;
}

int lbm_unet_num_params(lbm_unet *net, size_t *n) {
    if (!net || !n) return lbm::set_error(LBM_ERR_ARG, "null argument");
    *n = net->np;
    return LBM_OK;
}

static int vec_io(lbm_unet *N, float *dev, double *host_out, const double *host_in, size_t n) {
    if (!N || n != N->np) return lbm::set_error(LBM_ERR_ARG, "expected %zu parameters", N ? N->np : (size_t)0);
    UCHK(hipSetDevice(lbm::context_device(N->ctx)));
    std::vector<float> h(n);
    if (host_in) {
        for (size_t i = 0; i < n; ++i) h[i] = (float)host_in[i];
        UCHK(hipMemcpyAsync(dev, h.data(), n * sizeof(float), hipMemcpyHostToDevice, N->s));
        UCHK(hipStreamSynchronize(N->s));
        return repack(N);
    }
    UCHK(hipMemcpyAsync(h.data(), dev, n * sizeof(float), hipMemcpyDeviceToHost, N->s));
    UCHK(hipStreamSynchronize(N->s));
    for (size_t i = 0; i < n; ++i) host_out[i] = h[i];
    return LBM_OK;
}
int lbm_unet_get_params(lbm_unet *net, double *host, size_t n) { return vec_io(net, net ? net->p : nullptr, host, nullptr, n); }
int lbm_unet_set_params(lbm_unet *net, const double *host, size_t n) {
    if (!host) return lbm::set_error(LBM_ERR_ARG, "null argument");
    return vec_io(net, net ? net->p : nullptr, nullptr, host, n);
}
int lbm_unet_get_grads(lbm_unet *net, double *host, size_t n) { return vec_io(net, net ? net->g : nullptr, host, nullptr, n); }

int lbm_unet_reset_optimizer(lbm_unet *N) {
    if (!N) return lbm::set_error(LBM_ERR_ARG, "null argument");
    UCHK(hipSetDevice(lbm::context_device(N->ctx)));
    UCHK(hipMemsetAsync(N->m, 0, N->np * sizeof(float), N->s));
    UCHK(hipMemsetAsync(N->v, 0, N->np * sizeof(float), N->s));
    N->adam_t = 0;
    return LBM_OK;
}

int lbm_unet_set_input(lbm_unet *N, const double *const *fields, const double *mean, const double *scale, int nfields) {
    if (!N) return lbm::set_error(LBM_ERR_ARG, "null argument");
    if (nfields != N->cin) return lbm::set_error(LBM_ERR_ARG, "%d input fields, network takes %d", nfields, N->cin);
    FieldPtrs F;
    int rc = fields_in(fields, nullptr, mean, scale, nfields, &F);
    if (rc != LBM_OK) return rc;
    UCHK(hipSetDevice(lbm::context_device(N->ctx)));
    if ((rc = after_ctx(N)) != LBM_OK) return rc;
    k_gather<<<blocks((size_t)N->V[0] * 8), 256, 0, N->s>>>(F, nfields, 8, N->V[0], N->x0, nullptr);
    UCHK(hipGetLastError());
    return LBM_OK;
}

int lbm_unet_set_target(lbm_unet *N, const double *const *fields, const double *const *base, const double *mean,
                        const double *scale, int nfields) {
    if (!N) return lbm::set_error(LBM_ERR_ARG, "null argument");
    if (nfields != N->cout) return lbm::set_error(LBM_ERR_ARG, "%d target fields, network gives %d", nfields, N->cout);
    FieldPtrs F;
    int rc = fields_in(fields, base, mean, scale, nfields, &F);
    if (rc != LBM_OK) return rc;
    UCHK(hipSetDevice(lbm::context_device(N->ctx)));
    if ((rc = after_ctx(N)) != LBM_OK) return rc;
    const int cs = r16(N->cout);
    k_gather<<<blocks((size_t)N->V[0] * cs), 256, 0, N->s>>>(F, nfields, cs, N->V[0], nullptr, N->tgt);
    UCHK(hipGetLastError());
    N->have_target = true;
    return LBM_OK;
}

int lbm_unet_forward(lbm_unet *N) {
    if (!N) return lbm::set_error(LBM_ERR_ARG, "null argument");
    UCHK(hipSetDevice(lbm::context_device(N->ctx)));
    return forward(N);
}

int lbm_unet_output(lbm_unet *N, double *const *fields, const double *const *base, const double *mean,
                    const double *scale, const double *lo, const double *hi, int nfields) {
    if (!N || !fields) return lbm::set_error(LBM_ERR_ARG, "null argument");
    if (nfields != N->cout) return lbm::set_error(LBM_ERR_ARG, "%d output fields, network gives %d", nfields, N->cout);
    FieldOut F;
    for (int c = 0; c < nfields; ++c) {
        if (!fields[c]) return lbm::set_error(LBM_ERR_ARG, "field %d is null", c);
        F.f[c] = fields[c];
        F.base[c] = base ? base[c] : nullptr;
        F.mean[c] = mean ? mean[c] : 0.0;
        F.scale[c] = scale ? scale[c] : 1.0;
        F.lo[c] = lo ? lo[c] : -HUGE_VAL;
        F.hi[c] = hi ? hi[c] : HUGE_VAL;
        if (!(F.lo[c] <= F.hi[c])) return lbm::set_error(LBM_ERR_ARG, "field %d: empty clamp range", c);
    }
    UCHK(hipSetDevice(lbm::context_device(N->ctx)));
    int rc = after_ctx(N);
    if (rc != LBM_OK) return rc;
    k_scatter<<<blocks((size_t)N->V[0] * nfields), 256, 0, N->s>>>(N->y32, r16(N->cout), nfields, N->V[0], F);
    UCHK(hipGetLastError());
    return before_ctx(N);
}

int lbm_unet_backward(lbm_unet *N, double *loss) {
    if (!N) return lbm::set_error(LBM_ERR_ARG, "null argument");
    if (!N->have_target) return lbm::set_error(LBM_ERR_ARG, "no target set");
    UCHK(hipSetDevice(lbm::context_device(N->ctx)));
    int rc = backward(N);
    if (rc != LBM_OK) return rc;
    if (loss) {
        UCHK(hipMemcpyAsync(N->hloss, N->dloss, sizeof(double), hipMemcpyDeviceToHost, N->s));
        UCHK(hipStreamSynchronize(N->s));
        *loss = *N->hloss;
    }
    return LBM_OK;
}

int lbm_unet_adam(lbm_unet *N, double lr, double beta1, double beta2, double eps) {
    if (!N) return lbm::set_error(LBM_ERR_ARG, "null argument");
    if (!(lr > 0) || !(beta1 >= 0 && beta1 < 1) || !(beta2 >= 0 && beta2 < 1) || !(eps > 0))
        return lbm::set_error(LBM_ERR_ARG, "Adam hyper-parameters out of range");
    UCHK(hipSetDevice(lbm::context_device(N->ctx)));
    return adam(N, lr, beta1, beta2, eps);
}

int lbm_unet_train(lbm_unet *N, int steps, double lr, double *loss) {
    if (!N || steps < 0) return lbm::set_error(LBM_ERR_ARG, "bad argument");
    if (!N->have_target) return lbm::set_error(LBM_ERR_ARG, "no target set");
    if (!(lr > 0)) return lbm::set_error(LBM_ERR_ARG, "lr must be positive");
    UCHK(hipSetDevice(lbm::context_device(N->ctx)));
    int rc;
    for (int s = 0; s < steps; ++s) {
        if ((rc = forward(N)) != LBM_OK) return rc;
        if ((rc = backward(N)) != LBM_OK) return rc;
        if ((rc = adam(N, lr, 0.9, 0.999, 1e-8)) != LBM_OK) return rc;
    }
    if (loss) {
        // loss of the last step's forward pass (before its update)
        UCHK(hipMemcpyAsync(N->hloss, N->dloss, sizeof(double), hipMemcpyDeviceToHost, N->s));
        UCHK(hipStreamSynchronize(N->s));
        *loss = steps ? *N->hloss : NAN;
    }
    return LBM_OK;
}

int lbm_unet_synchronize(lbm_unet *N) {
    if (!N) return lbm::set_error(LBM_ERR_ARG, "null argument");
    UCHK(hipSetDevice(lbm::context_device(N->ctx)));
    UCHK(hipStreamSynchronize(N->s));
    return LBM_OK;
}

int lbm_unet_read(lbm_unet *N, const char *name, double *host, size_t n) {
    if (!N || !name || !host) return lbm::set_error(LBM_ERR_ARG, "null argument");
    const int c1 = N->base, c2 = 2 * c1, c3 = 4 * c1;
    struct T {
        const char *name;
        const void *p;
        int level, cs, cr, f32;
    } tab[] = {
        {"x0", N->x0, 0, 8, N->cin, 0},   {"e1a", N->e1a, 0, c1, c1, 0},   {"e1b", N->e1b, 0, c1, c1, 0},
        {"p1", N->p1, 1, c1, c1, 0},      {"e2a", N->e2a, 1, c2, c2, 0},   {"e2b", N->e2b, 1, c2, c2, 0},
        {"p2", N->p2, 2, c2, c2, 0},      {"e3a", N->e3a, 2, c3, c3, 0},   {"e3b", N->e3b, 2, c3, c3, 0},
        {"cat2", N->cat2, 1, c3 + c2, c3 + c2, 0}, {"d2a", N->d2a, 1, c2, c2, 0}, {"d2b", N->d2b, 1, c2, c2, 0},
        {"cat1", N->cat1, 0, c2 + c1, c2 + c1, 0}, {"d1a", N->d1a, 0, c1, c1, 0}, {"d1b", N->d1b, 0, c1, c1, 0},
        {"y", N->y32, 0, r16(N->cout), N->cout, 1}, {"target", N->tgt, 0, r16(N->cout), N->cout, 1},
    };
    for (const auto &t : tab) {
        if (strcmp(t.name, name)) continue;
        const int V = N->V[t.level];
        const size_t cnt = (size_t)V * t.cr;
        if (n != cnt) return lbm::set_error(LBM_ERR_ARG, "%s holds %zu values, %zu requested", name, cnt, n);
        UCHK(hipSetDevice(lbm::context_device(N->ctx)));
        double *d = nullptr;
        UCHK(hipMalloc(&d, cnt * sizeof(double)));
        if (t.f32)
            k_f_to_f64<<<blocks(cnt), 256, 0, N->s>>>((const float *)t.p, t.cs, t.cr, V, d);
        else
            k_bf_to_f64<<<blocks(cnt), 256, 0, N->s>>>((const bf16_t *)t.p, t.cs, t.cr, V, d);
        hipError_t e = hipMemcpyAsync(host, d, cnt * sizeof(double), hipMemcpyDeviceToHost, N->s);
        if (e == hipSuccess) e = hipStreamSynchronize(N->s);
        (void)hipFree(d);
        if (e != hipSuccess) return hipfail(e, "read");
        return LBM_OK;
    }
    return lbm::set_error(LBM_ERR_ARG, "unknown tensor %s", name);
}

}  // extern "C"
