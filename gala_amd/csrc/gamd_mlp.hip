// gamd_mlp.hip -- the learned SCF surrogate: a 4 -> 256 x 4 (SiLU) -> 4 MLP
// in BF16 on the matrix cores (FP32 accumulation, FP32 master weights), its
// training kernels (forward, backward, Adam) and the surrogate leapfrog with
// a per-orbit energy monitor and exact-SCF fallback.  No counterpart in gala:
// the exact potential it stands in for is the SCF expansion of
// potential/scf/src/bfe.cpp:20-259.
//
// Network, per point q (FP64 in, FP64 out):
//   features  f = (x/r, y/r, z/r, (ln r - mu)/sigma): direction and log
//             radius, so small radii are resolved as finely as large ones
//   hidden    h1 = silu(f W1 + b1), h_l = silu(h_{l-1} W_l + b_l), l = 2..4
//   output    o = h4 W5 + b5   (4 values)
//   physics   Phi_net(q) = Phi_b(r) (1 + c o0), with Phi_b = -G M / (r + r_s)
//             the expansion's Hernquist monopole (smooth, so Phi_net is);
//             the orbit force is -grad Phi_net, the exact gradient of this
//             potential (reverse mode through the network), so a surrogate
//             orbit conserves Phi_net + |v|^2/2 up to the integrator's error
//             and the energy monitor measures a conservative system.
//   o1..o3    auxiliary training targets, s_grad(r) o[1:4] ~ grad Phi (the
//             exact force scaled by a radial profile, piecewise linear in
//             ln r): they shape the hidden features during training; the
//             orbit force does not use them.
//
// Two evaluations of the same network:
//   * training (k_train_tile): BF16 activations and weights, 64-point tiles;
//   * orbits and inference (tile_conservative): the hidden products in
//     three BF16 matrix-core products, hi*hi + hi*lo + lo*hi of the split
//     v = hi + lo (hi = bf16(v), lo = bf16(v - hi)), which carries ~16
//     significant bits: the BF16 network's rounding jitter (~1e-3 of o0)
//     would drift the monitored energy by more than 1e-5 within steps.
//
// Matrix-core mapping (gfx950, v_mfma_f32_16x16x32_bf16; operand layout
// A[i][k] in lane i + 16 (k/8), element k%8; B[k][j] in lane j + 16 (k/8);
// D[i][j] in lane j + 16 (i/4), element i%4):
//   * a workgroup (4 waves) owns a tile of points; a layer's activations
//     live in LDS (rows of 256 BF16 padded to 264 to keep the 16-byte fragment
//     reads conflict-free); wave w computes output units [64w, 64w+64) of all
//     rows, as the transposed product Z^T = W^T H^T: the weight fragment is
//     the A operand, so a lane's four accumulators are four consecutive units
//     of one point (one 8-byte LDS store);
//   * hidden-layer weights are pre-swizzled into fragment order (and, for
//     the reverse pass, their transposes), so each wave reads 1 KB
//     contiguous per (16-unit tile, K step) from L2.
#include <math.h>
#include <string.h>

#include "gamd_host.hpp"

using namespace gamd;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

namespace {

constexpr int H = 256;        // hidden width
constexpr int LDSR = 264;     // padded LDS row (BF16 elements)
// flat FP32 parameter layout
constexpr int OFF_W1 = 0, OFF_B1 = OFF_W1 + 4 * H;
constexpr int OFF_W2 = OFF_B1 + H, OFF_B2 = OFF_W2 + H * H;
constexpr int OFF_W3 = OFF_B2 + H, OFF_B3 = OFF_W3 + H * H;
constexpr int OFF_W4 = OFF_B3 + H, OFF_B4 = OFF_W4 + H * H;
constexpr int OFF_W5 = OFF_B4 + H, OFF_B5 = OFF_W5 + H * 4;
constexpr int NPARAM = OFF_B5 + 4;  // 199,684
// BF16 copies of W2..W4, each block 3 H^2 (one H^2 per layer): fragment
// order of the high and the low parts, and of the transposes (high, low) for
// the reverse passes
constexpr int BF_SW = 0, BF_SWLO = 3 * H * H, BF_TSW = 6 * H * H, BF_TSWLO = 9 * H * H;
constexpr int NBF = 12 * H * H;

// logistic function from the hardware exp2 and reciprocal (v_exp_f32,
// v_rcp_f32, ~1 ulp each): the activations are rounded to BF16 (8 bits)
// right after, so an IEEE divide's extra accuracy is never seen.  Large
// negative z: exp2 overflows to +inf and the reciprocal gives 0, the limit.
__device__ __forceinline__ float sigmoid_fast(float z) {
    return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * z));
}
__device__ __forceinline__ float silu(float z) { return z * sigmoid_fast(z); }
__device__ __forceinline__ float dsilu(float z) {
    const float s = sigmoid_fast(z);
    return s * (1.0f + z * (1.0f - s));
}
__device__ __forceinline__ __bf16 tobf(float f) { return (__bf16)f; }
__device__ __forceinline__ float frombf(__bf16 b) { return (float)b; }

// ---------------------------------------------------------------------------
// features / physics scaling

__device__ __forceinline__ void features(const gamd_mlp_norm &nm, double x, double y, double z,
                                         float *f, double &r) {
    r = sqrt(x * x + y * y + z * z);
    const double ir = 1.0 / r;
    f[0] = (float)(x * ir);
    f[1] = (float)(y * ir);
    f[2] = (float)(z * ir);
    f[3] = (float)((log(r) - nm.mu) * nm.inv_sigma);
}

// the auxiliary heads' scale at radius r: linear interpolation in ln r
// between the profile knots, constant beyond the end knots (numpy.interp's
// convention)
__device__ __forceinline__ double out_scale_grad(const gamd_mlp_norm &nm, double r) {
    double u = (log(r) - nm.lnr0) * nm.inv_dlnr;
    if (!(u > 0.0)) u = 0.0;  // also maps NaN (r = 0 with a zero knot spacing) to the first knot
    if (u > (double)(GAMD_MLP_KNOTS - 1)) u = (double)(GAMD_MLP_KNOTS - 1);
    int k = (int)u;
    k = k > GAMD_MLP_KNOTS - 2 ? GAMD_MLP_KNOTS - 2 : k;
    const double f = u - (double)k;
    const double *sg = nm.scale;
    return sg[k] + f * (sg[k + 1] - sg[k]);
}

// Phi_net and its gradient at q = (x, y, z), |q| = r, from the network's o0
// and its derivatives g[c] = d o0 / d f_c (f the features): with
// f = (q/r, (ln r - mu)/sigma), d(q_i/r)/dq_k = (delta_ik - q_i q_k / r^2) / r
// and d f_3/dq_k = q_k / (r^2 sigma).
__device__ __forceinline__ void net_physics(const gamd_mlp_norm &nm, double x, double y, double z,
                                            double r, float o0, const float *g, double &phi,
                                            double &gx, double &gy, double &gz) {
    const double rb = r + nm.rs;
    const double pb = -nm.gm / rb;            // Phi_b
    const double dpb = nm.gm / (rb * rb);     // d Phi_b / dr
    const double ratio = 1.0 + nm.phi_c * (double)o0;
    phi = pb * ratio;
    const double ir = 1.0 / r;
    const double g0 = (double)g[0], g1 = (double)g[1], g2 = (double)g[2], g3 = (double)g[3];
    const double gq = (g0 * x + g1 * y + g2 * z) * ir * ir;
    const double gr = g3 * nm.inv_sigma * ir * ir;
    // d o0 / dq
    const double ox = (g0 - gq * x) * ir + gr * x;
    const double oy = (g1 - gq * y) * ir + gr * y;
    const double oz = (g2 - gq * z) * ir + gr * z;
    const double a = dpb * ratio * ir, b = pb * nm.phi_c;
    gx = a * x + b * ox;
    gy = a * y + b * oy;
    gz = a * z + b * oz;
}

// ---------------------------------------------------------------------------
// The precise evaluation of one tile of CP = 16 MI points: o0 and d o0 / d f
// (reverse mode), the hidden products in three BF16 matrix-core products of
// the hi/lo split (hi*hi + hi*lo + lo*hi), SiLU and its derivative in FP32,
// the first and last layers in FP32 on the VALU.
//   feat   LDS [CP][4] features;
//   bhi,   LDS [CP][LDSR] BF16 each: a layer's input (activations forward,
//   blo    error signals backward), split;
//   red    LDS [4][CP][5] per-wave partial sums;
//   o0,    LDS [CP] and [CP][4]: results.
//   dfo
// Wave w owns units [64w, 64w + 64) of every layer (forward and backward),
// so the SiLU derivatives it keeps in registers from the forward pass are
// exactly those its reverse-pass products need.  All 256 threads call it.
//
// What bounds it: the matrix products and the SiLU arithmetic (1,152 MFMAs,
// 18.4k cycles, and ~2,700 other vector instructions, ~14k cycles, per wave
// and 32-point tile), with the weights' L2 reads (1.5 MB per tile) close
// behind.  1,048,576 points take 2.41 ms, 1,040 TFLOP/s of executed BF16
// products (a large library BF16 product reaches 1,150 on the same card); 3.91
// ms while the layers were runtime loops, whose per-element branches kept the
// derivatives in scratch memory and the weight reads inside each step.  Hence
// every layer is written out (the derivatives stay in registers), and each
// step's weights are read one step ahead, across the layers' barriers too.
// Larger tiles halve the weight reads but leave one wave per SIMD (64 points:
// 2.39 ms) or spill (48 points); 16-point tiles repeat them (3.58 ms) and only
// pay while there are fewer tiles than compute units (4,096 points: 21 against
// 24 us), see tile_points16.

__device__ __forceinline__ void split_bf(float v, __bf16 &hi, __bf16 &lo) {
    hi = tobf(v);
    lo = tobf(v - frombf(hi));
}

typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));

// this thread's wave in its workgroup, as a scalar: addresses formed from it
// stay in scalar registers
__device__ __forceinline__ unsigned wave_id() {
    return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
}

// The weights and parameters of the tile are read through buffer descriptors:
// a 32-bit lane offset and a scalar offset per read, no 64-bit address
// arithmetic on the vector unit.
struct NetBufs {
    __amdgpu_buffer_rsrc_t w, th;  // BF16 copies; FP32 parameters
};
__device__ __forceinline__ NetBufs net_bufs(const float *theta, const __bf16 *wbf) {
    constexpr int FLAGS = 0x00027000;  // raw buffer, bounds-checked (gfx9 layout)
    return {__builtin_amdgcn_make_buffer_rsrc(const_cast<__bf16 *>(wbf), 0, NBF * 2, FLAGS),
            __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(theta), 0, NPARAM * 4, FLAGS)};
}
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
// four consecutive parameters from index at (scalar) + lane_at
__device__ __forceinline__ f32x4 theta4(const NetBufs &nb, unsigned at, unsigned lane_at) {
    const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(nb.th, lane_at * 4, at * 4, 0);
    return __builtin_bit_cast(f32x4, v);
}

// one K step (32 inputs) of a wave's weight fragments from the layer blocks
// at element offsets hi and lo: hi parts of its four 16-unit tiles in [0, 4),
// lo parts in [4, 8)
__device__ __forceinline__ void load_frags(bf16x8 (&f)[8], const NetBufs &nb, unsigned hi,
                                           unsigned lo, int ks) {
    const unsigned lane = threadIdx.x & 63, w = wave_id();
#pragma unroll
    for (int ni = 0; ni < 4; ni++) {
        const unsigned o = ((4 * w + ni) * 8 + ks) * 64 * 8;
        f[ni] = __builtin_bit_cast(
            bf16x8, __builtin_amdgcn_raw_buffer_load_b128(nb.w, lane * 16, (hi + o) * 2, 0));
        f[4 + ni] = __builtin_bit_cast(
            bf16x8, __builtin_amdgcn_raw_buffer_load_b128(nb.w, lane * 16, (lo + o) * 2, 0));
    }
}

// acc[mi][ni] = sum over the 256 inputs of the layer's weights (fragment
// order: hi parts at element whi of the copies, lo at wlo) times the split
// input in bhi/blo.  The weights of step ks + 1 are loaded before step ks's
// products; those of the first step are in f[0] on entry, and the next
// layer's (nhi, nlo) are in f[0] on return, so that their latency passes
// behind this layer's epilogue.
template <int MI, bool NEXT>
__device__ __forceinline__ void split_layer(const NetBufs &nb, unsigned whi, unsigned wlo,
                                            unsigned nhi, unsigned nlo, const __bf16 *bhi,
                                            const __bf16 *blo, bf16x8 (&f)[2][8],
                                            f32x4 (&acc)[MI][4]) {
    const unsigned lane = threadIdx.x & 63;
#pragma unroll
    for (int mi = 0; mi < MI; mi++)
#pragma unroll
        for (int ni = 0; ni < 4; ni++) acc[mi][ni] = f32x4{0.f, 0.f, 0.f, 0.f};
    // the matrix phase ahead of a neighbouring workgroup's SiLU phase (1 % of an
    // orbit step)
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int ks = 0; ks < 8; ks++) {
        if (ks < 7)
            load_frags(f[(ks + 1) & 1], nb, whi, wlo, ks + 1);
        else if (NEXT)
            load_frags(f[0], nb, nhi, nlo, 0);
        __builtin_amdgcn_sched_barrier(0);  // one step of loads in flight, not all eight
        const bf16x8(&w)[8] = f[ks & 1];
        bf16x8 ah[MI], al[MI];
#pragma unroll
        for (int mi = 0; mi < MI; mi++) {
            const unsigned off = (16 * mi + (lane & 15)) * LDSR + 32 * ks + 8 * (lane >> 4);
            ah[mi] = *reinterpret_cast<const bf16x8 *>(bhi + off);
            al[mi] = *reinterpret_cast<const bf16x8 *>(blo + off);
        }
        // each accumulator takes hi*hi, hi*lo, lo*hi in that order; the three
        // are issued 4 MI products apart, so none waits for the one before it
#pragma unroll
        for (int mi = 0; mi < MI; mi++)
#pragma unroll
            for (int ni = 0; ni < 4; ni++)
                acc[mi][ni] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[ni], ah[mi], acc[mi][ni], 0, 0, 0);
#pragma unroll
        for (int mi = 0; mi < MI; mi++)
#pragma unroll
            for (int ni = 0; ni < 4; ni++)
                acc[mi][ni] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[ni], al[mi], acc[mi][ni], 0, 0, 0);
#pragma unroll
        for (int mi = 0; mi < MI; mi++)
#pragma unroll
            for (int ni = 0; ni < 4; ni++)
                acc[mi][ni] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[4 + ni], ah[mi], acc[mi][ni], 0, 0, 0);
    }
    __builtin_amdgcn_s_setprio(0);
}

// four consecutive units of one point, split, into the layer buffers
__device__ __forceinline__ void store_split(__bf16 *bhi, __bf16 *blo, unsigned at, const float (&v)[4]) {
    __bf16 hh[4], hl[4];
#pragma unroll
    for (int e = 0; e < 4; e++) split_bf(v[e], hh[e], hl[e]);
    *reinterpret_cast<bf16x4 *>(bhi + at) = bf16x4{hh[0], hh[1], hh[2], hh[3]};
    *reinterpret_cast<bf16x4 *>(blo + at) = bf16x4{hl[0], hl[1], hl[2], hl[3]};
}

// epilogue of hidden layer L (2..4): SiLU of acc + bias.  Layers 2 and 3 keep
// their derivatives in ds and write the activations; layer 4 adds the
// output dot to po and writes the output's error signal.
template <int MI, int L>
__device__ __forceinline__ void forward_epilogue(const NetBufs &nb,
                                                 const f32x4 (&acc)[MI][4], __bf16 *bhi,
                                                 __bf16 *blo, f32x4 (&ds)[MI][4],
                                                 float (&po)[MI]) {
    const unsigned lane = threadIdx.x & 63, w = wave_id();
    constexpr unsigned bias = L == 2 ? OFF_B2 : L == 3 ? OFF_B3 : OFF_B4;
    const unsigned lu = 4 * (lane >> 4);  // this lane's first unit of a 16-unit tile
#pragma unroll
    for (int mi = 0; mi < MI; mi++)
#pragma unroll
        for (int ni = 0; ni < 4; ni++) {
            const unsigned unit = 64 * w + 16 * ni + 4 * (lane >> 4);
            const unsigned row = 16 * mi + (lane & 15);
            const f32x4 bc = theta4(nb, bias + 64 * w + 16 * ni, lu);
            float out[4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float z = acc[mi][ni][e] + bc[e];
                const float sg = sigmoid_fast(z);
                const float h = z * sg;
                const float d = sg * (1.0f + z * (1.0f - sg));
                if (L < 4) {
                    ds[mi][ni][e] = d;
                    out[e] = h;
                } else {
                    const float w5 = __builtin_bit_cast(
                        float, __builtin_amdgcn_raw_buffer_load_b32(
                                   nb.th, lu * 16, (OFF_W5 + (64 * w + 16 * ni + e) * 4) * 4, 0));
                    po[mi] += w5 * h;
                    out[e] = w5 * d;
                }
            }
            store_split(bhi, blo, row * LDSR + unit, out);
        }
}

// epilogue of the reverse product into layer L - 1 = 3 or 2: the error signal
template <int MI>
__device__ __forceinline__ void reverse_epilogue(const f32x4 (&acc)[MI][4],
                                                 const f32x4 (&ds)[MI][4], __bf16 *bhi,
                                                 __bf16 *blo) {
    const unsigned lane = threadIdx.x & 63, w = wave_id();
#pragma unroll
    for (int mi = 0; mi < MI; mi++)
#pragma unroll
        for (int ni = 0; ni < 4; ni++) {
            const unsigned unit = 64 * w + 16 * ni + 4 * (lane >> 4);
            const unsigned row = 16 * mi + (lane & 15);
            float out[4];
#pragma unroll
            for (int e = 0; e < 4; e++) out[e] = acc[mi][ni][e] * ds[mi][ni][e];
            store_split(bhi, blo, row * LDSR + unit, out);
        }
}

template <int MI>
__device__ __forceinline__ void tile_conservative(const float *__restrict__ theta,
                                                  const __bf16 *__restrict__ wbf,
                                                  const float (*feat)[4], __bf16 *bhi, __bf16 *blo,
                                                  float (*red)[16 * MI][5], float *o0,
                                                  float (*dfo)[4]) {
    constexpr int NP = 16 * MI;  // points of the tile
    const unsigned t = threadIdx.x, lane = t & 63, w = wave_id();
    constexpr unsigned Fhi = BF_SW, Flo = BF_SWLO;    // forward, layers 2..4
    constexpr unsigned Rhi = BF_TSW, Rlo = BF_TSWLO;  // their transposes
    constexpr unsigned LW = H * H;
    const NetBufs nb = net_bufs(theta, wbf);
    bf16x8 f[2][8];
    load_frags(f[0], nb, Fhi, Flo, 0);
    // layer 1 (FP32): thread t owns units 2j and 2j + 1, j = t % 128, of half
    // of the points
    {
        typedef float f32x2 __attribute__((ext_vector_type(2)));
        typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
        const unsigned j = 2 * (t & 127);
        const f32x2 w0 = *reinterpret_cast<const f32x2 *>(theta + OFF_W1 + 0 * H + j);
        const f32x2 w1 = *reinterpret_cast<const f32x2 *>(theta + OFF_W1 + 1 * H + j);
        const f32x2 w2 = *reinterpret_cast<const f32x2 *>(theta + OFF_W1 + 2 * H + j);
        const f32x2 w3 = *reinterpret_cast<const f32x2 *>(theta + OFF_W1 + 3 * H + j);
        const f32x2 bj = *reinterpret_cast<const f32x2 *>(theta + OFF_B1 + j);
        const unsigned p0 = (t >> 7) * (NP / 2);
#pragma unroll 4
        for (unsigned p = p0; p < p0 + NP / 2; p++) {
            const f32x4 fp = *reinterpret_cast<const f32x4 *>(feat[p]);
            __bf16 hh[2], hl[2];
#pragma unroll
            for (int e = 0; e < 2; e++) {
                const float z = bj[e] + fp[0] * w0[e] + fp[1] * w1[e] + fp[2] * w2[e] + fp[3] * w3[e];
                split_bf(silu(z), hh[e], hl[e]);
            }
            *reinterpret_cast<bf16x2 *>(bhi + p * LDSR + j) = bf16x2{hh[0], hh[1]};
            *reinterpret_cast<bf16x2 *>(blo + p * LDSR + j) = bf16x2{hl[0], hl[1]};
        }
    }
    __syncthreads();
    // SiLU derivatives of layers 2 and 3 at this wave's units, in the
    // accumulator layout: unit 64w + 16ni + 4(lane/16) + e, point 16mi + lane%16
    f32x4 ds2[MI][4], ds3[MI][4];
    float po[MI];  // partial o0 of points 16mi + lane%16
    f32x4 acc[MI][4];
#pragma unroll
    for (int mi = 0; mi < MI; mi++) po[mi] = 0.f;
    // every layer: the products, a barrier (every wave has read the layer's
    // input), the epilogue into the same buffers, a barrier
    split_layer<MI, true>(nb, Fhi, Flo, Fhi + LW, Flo + LW, bhi, blo, f, acc);
    __syncthreads();
    forward_epilogue<MI, 2>(nb, acc, bhi, blo, ds2, po);
    __syncthreads();
    split_layer<MI, true>(nb, Fhi + LW, Flo + LW, Fhi + 2 * LW, Flo + 2 * LW, bhi, blo, f, acc);
    __syncthreads();
    forward_epilogue<MI, 3>(nb, acc, bhi, blo, ds3, po);
    __syncthreads();
    split_layer<MI, true>(nb, Fhi + 2 * LW, Flo + 2 * LW, Rhi + 2 * LW, Rlo + 2 * LW, bhi, blo, f, acc);
    __syncthreads();
    forward_epilogue<MI, 4>(nb, acc, bhi, blo, ds3, po);
    __syncthreads();
    // o0: the four lanes of a point in this wave, then the four waves
#pragma unroll
    for (int mi = 0; mi < MI; mi++) {
        float v = po[mi];
        v += __shfl_xor(v, 16);
        v += __shfl_xor(v, 32);
        if (lane < 16) red[w][16 * mi + lane][4] = v;
    }
    // reverse pass: delta_{l-1} = (W_l^T delta_l) silu'(z_{l-1}), l = 4, 3, 2
    split_layer<MI, true>(nb, Rhi + 2 * LW, Rlo + 2 * LW, Rhi + LW, Rlo + LW, bhi, blo, f, acc);
    __syncthreads();
    reverse_epilogue<MI>(acc, ds3, bhi, blo);
    __syncthreads();
    split_layer<MI, true>(nb, Rhi + LW, Rlo + LW, Rhi, Rlo, bhi, blo, f, acc);
    __syncthreads();
    reverse_epilogue<MI>(acc, ds2, bhi, blo);
    __syncthreads();
    split_layer<MI, false>(nb, Rhi, Rlo, 0, 0, bhi, blo, f, acc);
    // layer 1's derivative, recomputed from its inputs, and d o0 / d f
    float pg[MI][4];
    f32x4 fr[MI];
#pragma unroll
    for (int mi = 0; mi < MI; mi++) {
        fr[mi] = *reinterpret_cast<const f32x4 *>(feat[16 * mi + (lane & 15)]);
#pragma unroll
        for (int c = 0; c < 4; c++) pg[mi][c] = 0.f;
    }
#pragma unroll
    for (int ni = 0; ni < 4; ni++) {
        const unsigned tile = 64 * w + 16 * ni, lu = 4 * (lane >> 4);
        f32x4 w1[4];
#pragma unroll
        for (int c = 0; c < 4; c++) w1[c] = theta4(nb, OFF_W1 + c * H + tile, lu);
        const f32x4 b1 = theta4(nb, OFF_B1 + tile, lu);
#pragma unroll
        for (int mi = 0; mi < MI; mi++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float z = b1[e] + fr[mi][0] * w1[0][e] + fr[mi][1] * w1[1][e] +
                                fr[mi][2] * w1[2][e] + fr[mi][3] * w1[3][e];
                const float d = acc[mi][ni][e] * dsilu(z);
#pragma unroll
                for (int c = 0; c < 4; c++) pg[mi][c] += w1[c][e] * d;
            }
    }
#pragma unroll
    for (int mi = 0; mi < MI; mi++)
#pragma unroll
        for (int c = 0; c < 4; c++) {
            float v = pg[mi][c];
            v += __shfl_xor(v, 16);
            v += __shfl_xor(v, 32);
            if (lane < 16) red[w][16 * mi + lane][c] = v;
        }
    __syncthreads();
    if (t < NP) {
        o0[t] = theta[OFF_B5] + red[0][t][4] + red[1][t][4] + red[2][t][4] + red[3][t][4];
#pragma unroll
        for (int c = 0; c < 4; c++) dfo[t][c] = red[0][t][c] + red[1][t][c] + red[2][t][c] + red[3][t][c];
    }
    __syncthreads();
}

// ---------------------------------------------------------------------------
// inference: q (3,M) FP64 -> Phi_net (M), grad Phi_net (3,M), one tile of
// 16 MI points per workgroup (tile_conservative)
template <int MI>
__global__ __launch_bounds__(256, 2) void k_mlp_forward(const float *__restrict__ theta,
                                                     const __bf16 *__restrict__ wbf,
                                                     gamd_mlp_norm nm,
                                                     const double *__restrict__ q, int64_t M,
                                                     double *__restrict__ phi,
                                                     double *__restrict__ grad) {
    constexpr int CP = 16 * MI;  // points of the workgroup's tile
    __shared__ __align__(16) __bf16 bhi[CP * LDSR];
    __shared__ __align__(16) __bf16 blo[CP * LDSR];
    __shared__ __align__(16) float feat[CP][4];
    __shared__ float red[4][CP][5];
    __shared__ float o0[CP];
    __shared__ float dfo[CP][4];
    const int t = threadIdx.x;
    const int64_t i = (int64_t)blockIdx.x * CP + t;
    double x = nm.pad_r, y = 0, z = 0, r = 1;  // padding rows: a harmless point
    if (t < CP) {
        if (i < M) {
            x = q[i];
            y = q[M + i];
            z = q[2 * M + i];
        }
        float f[4];
        features(nm, x, y, z, f, r);
#pragma unroll
        for (int c = 0; c < 4; c++) feat[t][c] = f[c];
    }
    __syncthreads();
    tile_conservative<MI>(theta, wbf, feat, bhi, blo, red, o0, dfo);
    if (t < CP && i < M) {
        double ph, gx, gy, gz;
        net_physics(nm, x, y, z, r, o0[t], dfo[t], ph, gx, gy, gz);
        phi[i] = ph;
        grad[i] = gx;
        grad[M + i] = gy;
        grad[2 * M + i] = gz;
    }
}

// ---------------------------------------------------------------------------
// Training: loss, its gradient and Adam.
//
// k_train_tile takes 64 points through the network and back: the four hidden
// layers, the output, the loss and the error signals dZ_4 .. dZ_1, with BF16
// weights and activations and FP32 accumulation.  Wave w owns units
// [64w, 64w + 64) of every layer both ways, so the pre-activations it needs
// for the SiLU derivatives stay in its registers (BF16); the activations
// H_1 .. H_3 and the error signals dZ_2 .. dZ_4 that the hidden weights'
// gradients need go to memory, once each; every sum over the tile's points
// (first and output layers' weights, biases, loss) is finished in the tile
// and leaves as one row of 3,080 partial sums.
//
// k_wgrad forms the three hidden weight gradients H_{l-1}^T dZ_l, split over
// slices of the points into partial matrices; k_grad_reduce adds slices and
// tile rows in a fixed order, so gradients are the same in every run.
//
// 32,768 points: k_train_tile 61 us, k_wgrad 26, k_grad_reduce 9 and Adam 5;
// 112 to 118 us per step end to end.  The same step took 450 us as twenty launches:
// a forward pass that wrote every pre-activation and activation (134 MB), a
// product per layer that read them back, and reductions over the points by
// atomic adds from every block (50 us per weight gradient, 31 us for dW5).
// k_train_tile is bound by its vector work (~7,700 instructions per wave beside 768
// matrix ones, two waves per SIMD: VALU 52 % busy) beside 100 MB of stores; k_wgrad and
// k_grad_reduce by their 180 and 39 MB.  64-point tiles of four waves let two
// workgroups share a compute unit, one's products behind the other's SiLU.

constexpr int TP = 64;  // points per workgroup of k_train_tile
// one tile's partial sums: dW1 [4][256], db1..db4 [4][256], dW5 [256][4], db5, loss
constexpr int PT_W1 = 0, PT_B = 4 * H, PT_W5 = 8 * H, PT_B5 = 12 * H, PT_LOSS = PT_B5 + 4;
constexpr int PT_N = 12 * H + 8;

// one K step of a wave's weight fragments (high parts only)
__device__ __forceinline__ void load_frags_hi(bf16x8 (&f)[4], const NetBufs &nb, unsigned hi,
                                              int ks) {
    const unsigned lane = threadIdx.x & 63, w = wave_id();
#pragma unroll
    for (int ni = 0; ni < 4; ni++) {
        const unsigned o = ((4 * w + ni) * 8 + ks) * 64 * 8;
        f[ni] = __builtin_bit_cast(
            bf16x8, __builtin_amdgcn_raw_buffer_load_b128(nb.w, lane * 16, (hi + o) * 2, 0));
    }
}

// acc = weights (fragment order at element offset hi) times the 64 points in
// buf; weights one step ahead as in split_layer (f[0] holds the first step on
// entry and the next block's on return)
template <bool NEXT>
__device__ __forceinline__ void train_layer(const NetBufs &nb, unsigned hi, unsigned nhi,
                                            const __bf16 *buf, bf16x8 (&f)[2][4],
                                            f32x4 (&acc)[4][4]) {
    const unsigned lane = threadIdx.x & 63;
#pragma unroll
    for (int mi = 0; mi < 4; mi++)
#pragma unroll
        for (int ni = 0; ni < 4; ni++) acc[mi][ni] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < 8; ks++) {
        if (ks < 7)
            load_frags_hi(f[(ks + 1) & 1], nb, hi, ks + 1);
        else if (NEXT)
            load_frags_hi(f[0], nb, nhi, 0);
        __builtin_amdgcn_sched_barrier(0);
        bf16x8 a[4];
#pragma unroll
        for (int mi = 0; mi < 4; mi++)
            a[mi] = *reinterpret_cast<const bf16x8 *>(buf + (16 * mi + (lane & 15)) * LDSR +
                                                      32 * ks + 8 * (lane >> 4));
#pragma unroll
        for (int mi = 0; mi < 4; mi++)
#pragma unroll
            for (int ni = 0; ni < 4; ni++)
                acc[mi][ni] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f[ks & 1][ni], a[mi],
                                                                      acc[mi][ni], 0, 0, 0);
    }
}

// the tile's (64, 256) layer in buf to its rows at dst of a (M, 256) matrix,
// 16 bytes per thread and step (through a descriptor of those rows: one
// 32-bit offset serves all steps)
__device__ __forceinline__ void store_tile(const __bf16 *buf, __bf16 *__restrict__ dst) {
    const unsigned t = threadIdx.x;
    const __amdgpu_buffer_rsrc_t out =
        __builtin_amdgcn_make_buffer_rsrc(dst, 0, TP * H * 2, 0x00027000);
    const __bf16 *src = buf + (t >> 5) * LDSR + 8 * (t & 31);
#pragma unroll
    for (int k = 0; k < TP / 8; k++) {
        const u32x4 v = *reinterpret_cast<const u32x4 *>(src + 8 * k * LDSR);
        __builtin_amdgcn_raw_buffer_store_b128(v, out, t * 16, k * 8 * H * 2, 0);
        if (k & 1) __builtin_amdgcn_sched_barrier(0);  // two in flight: registers are scarce
    }
}

// four BF16 values in two registers.  The empty asm makes the pair opaque:
// otherwise each half travels in a register of its own, 64 per layer too many
struct Packed4 {
    unsigned v[2];
    __device__ __forceinline__ void set(const bf16x4 &x) {
        typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
        const u32x2 u = __builtin_bit_cast(u32x2, x);
        v[0] = u[0];
        v[1] = u[1];
        asm("" : "+v"(v[0]), "+v"(v[1]));
    }
    // element e as FP32 (a BF16 value is the top half of its FP32 form)
    __device__ __forceinline__ float get(int e) const {
        const unsigned u = v[e >> 1];
        return __builtin_bit_cast(float, e & 1 ? u & 0xffff0000u : u << 16);
    }
};

// z = acc + bias (BF16 copies kept in z) and silu(z) into buf
template <int L>
__device__ __forceinline__ void train_forward_epilogue(const NetBufs &nb, const f32x4 (&acc)[4][4],
                                                       __bf16 *buf, Packed4 (&z)[4][4]) {
    const unsigned lane = threadIdx.x & 63, w = wave_id(), lu = 4 * (lane >> 4);
    constexpr unsigned bias = L == 2 ? OFF_B2 : L == 3 ? OFF_B3 : OFF_B4;
#pragma unroll
    for (int ni = 0; ni < 4; ni++) {
        const unsigned tile = 64 * w + 16 * ni;
        const f32x4 bc = theta4(nb, bias + tile, lu);
#pragma unroll
        for (int mi = 0; mi < 4; mi++) {
            bf16x4 hv, zv;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float v = acc[mi][ni][e] + bc[e];
                hv[e] = tobf(silu(v));
                zv[e] = tobf(v);
            }
            z[mi][ni].set(zv);
            *reinterpret_cast<bf16x4 *>(buf + (16 * mi + (lane & 15)) * LDSR + tile + lu) = hv;
        }
    }
}

// sum over the 16 lanes (one DPP row) that hold one unit's points, in every
// lane: rotations by 8, 4, 2 and 1 inside the row, no LDS traffic
template <int N>
__device__ __forceinline__ float row_ror(float v) {
    return __builtin_bit_cast(
        float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x120 + N, 0xF, 0xF, true));
}
__device__ __forceinline__ float sum16(float v) {
    v += row_ror<8>(v);
    v += row_ror<4>(v);
    v += row_ror<2>(v);
    v += row_ror<1>(v);
    return v;
}

// dZ = (W^T dZ_next) silu'(z) into buf, its sums over the tile's points to gb
__device__ __forceinline__ void train_reverse_epilogue(const f32x4 (&acc)[4][4],
                                                       const Packed4 (&z)[4][4], __bf16 *buf,
                                                       float *__restrict__ gb) {
    const unsigned lane = threadIdx.x & 63, w = wave_id(), lu = 4 * (lane >> 4);
#pragma unroll
    for (int ni = 0; ni < 4; ni++) {
        const unsigned unit = 64 * w + 16 * ni + lu;
        f32x4 cs = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int mi = 0; mi < 4; mi++) {
            bf16x4 d;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                d[e] = tobf(acc[mi][ni][e] * dsilu(z[mi][ni].get(e)));
                cs[e] += frombf(d[e]);
            }
            *reinterpret_cast<bf16x4 *>(buf + (16 * mi + (lane & 15)) * LDSR + unit) = d;
        }
#pragma unroll
        for (int e = 0; e < 4; e++) cs[e] = sum16(cs[e]);
        if ((lane & 15) == 0) *reinterpret_cast<f32x4 *>(gb + unit) = cs;
    }
}

__global__ __launch_bounds__(256, 2) void k_train_tile(
    const float *__restrict__ theta, const __bf16 *__restrict__ wbf,
    const float *__restrict__ featg, const float *__restrict__ targetg, int64_t M,
    __bf16 *__restrict__ Hs, __bf16 *__restrict__ Ds, float *__restrict__ part) {
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    __shared__ __align__(16) __bf16 buf[TP * LDSR];
    __shared__ __align__(16) float fs[TP][4];   // features
    __shared__ __align__(16) float dy[TP][4];   // d loss / d output
    __shared__ __align__(16) float w5t[4][H];   // output weights, transposed
    __shared__ __align__(16) float half[H][4];  // dW5 of the second half of the points
    __shared__ float red[4];
    const unsigned t = threadIdx.x, lane = t & 63, w = wave_id(), lu = 4 * (lane >> 4);
    const int64_t row0 = (int64_t)blockIdx.x * TP;
    const NetBufs nb = net_bufs(theta, wbf);
    constexpr unsigned LW = H * H;
    const size_t layer = (size_t)M * H;
    __bf16 *Ht = Hs + row0 * H, *Dt = Ds + row0 * H;
    float *pt = part + (size_t)blockIdx.x * PT_N;
    bf16x8 f[2][4];
    load_frags_hi(f[0], nb, BF_SW, 0);
    fs[t >> 2][t & 3] = featg[row0 * 4 + t];
    const float target = targetg[row0 * 4 + t];
    {
        const f32x4 r = theta4(nb, OFF_W5, 4 * t);
#pragma unroll
        for (int o = 0; o < 4; o++) w5t[o][t] = r[o];
    }
    __syncthreads();
    // layer 1: 4 -> 256 in FP32, two units of half of the points per thread
    {
        const unsigned j = 2 * (t & 127), p0 = (t >> 7) * (TP / 2);
        const f32x2 w0 = *reinterpret_cast<const f32x2 *>(theta + OFF_W1 + 0 * H + j);
        const f32x2 w1 = *reinterpret_cast<const f32x2 *>(theta + OFF_W1 + 1 * H + j);
        const f32x2 w2 = *reinterpret_cast<const f32x2 *>(theta + OFF_W1 + 2 * H + j);
        const f32x2 w3 = *reinterpret_cast<const f32x2 *>(theta + OFF_W1 + 3 * H + j);
        const f32x2 bj = *reinterpret_cast<const f32x2 *>(theta + OFF_B1 + j);
#pragma unroll 4
        for (unsigned p = p0; p < p0 + TP / 2; p++) {
            const f32x4 fp = *reinterpret_cast<const f32x4 *>(fs[p]);
            bf16x2 hv;
#pragma unroll
            for (int e = 0; e < 2; e++)
                hv[e] = tobf(silu(bj[e] + fp[0] * w0[e] + fp[1] * w1[e] + fp[2] * w2[e] + fp[3] * w3[e]));
            *reinterpret_cast<bf16x2 *>(buf + p * LDSR + j) = hv;
        }
    }
    __syncthreads();
    f32x4 acc[4][4];
    Packed4 z2[4][4], z3[4][4], z4[4][4];
    store_tile(buf, Ht);
    train_layer<true>(nb, BF_SW, BF_SW + LW, buf, f, acc);
    __syncthreads();
    train_forward_epilogue<2>(nb, acc, buf, z2);
    __syncthreads();
    store_tile(buf, Ht + layer);
    train_layer<true>(nb, BF_SW + LW, BF_SW + 2 * LW, buf, f, acc);
    __syncthreads();
    train_forward_epilogue<3>(nb, acc, buf, z3);
    __syncthreads();
    store_tile(buf, Ht + 2 * layer);
    train_layer<true>(nb, BF_SW + 2 * LW, BF_TSW + 2 * LW, buf, f, acc);
    __syncthreads();
    train_forward_epilogue<4>(nb, acc, buf, z4);
    __syncthreads();
    // output, loss and dY: thread t holds output t % 4 of point t / 4
    {
        const unsigned p = t >> 2, o = t & 3;
        float y = theta[OFF_B5 + o];
        const __bf16 *hrow = buf + p * LDSR;
#pragma unroll 4
        for (int j = 0; j < H; j += 8) {
            const bf16x8 h = *reinterpret_cast<const bf16x8 *>(hrow + j);
            const f32x4 wa = *reinterpret_cast<const f32x4 *>(&w5t[o][j]);
            const f32x4 wb = *reinterpret_cast<const f32x4 *>(&w5t[o][j + 4]);
#pragma unroll
            for (int e = 0; e < 4; e++) y += frombf(h[e]) * wa[e];
#pragma unroll
            for (int e = 0; e < 4; e++) y += frombf(h[4 + e]) * wb[e];
        }
        const float d = y - target;
        const float g = 2.0f * d / (float)M;
        dy[p][o] = g;
        float l = d * d, gs = g;
#pragma unroll
        for (int m = 4; m < 64; m <<= 1) gs += __shfl_xor(gs, m);
#pragma unroll
        for (int m = 1; m < 64; m <<= 1) l += __shfl_xor(l, m);
        // db5 and the loss: this wave's sixteen points, then the four waves
        if (lane < 4) half[w][lane] = gs;
        if (lane == 0) red[w] = l;
    }
    __syncthreads();
    if (t < 4) pt[PT_B5 + t] = half[0][t] + half[1][t] + half[2][t] + half[3][t];
    if (t == 4) pt[PT_LOSS] = red[0] + red[1] + red[2] + red[3];
    __syncthreads();
    // dW5: units j, j + 1 over half of the points, the halves joined in LDS
    {
        const unsigned j = 2 * (t & 127), p0 = (t >> 7) * (TP / 2);
        f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
        for (unsigned p = p0; p < p0 + TP / 2; p++) {
            const bf16x2 h = *reinterpret_cast<const bf16x2 *>(buf + p * LDSR + j);
            const f32x4 g = *reinterpret_cast<const f32x4 *>(dy[p]);
            const float h0 = frombf(h[0]), h1 = frombf(h[1]);
#pragma unroll
            for (int o = 0; o < 4; o++) {
                s0[o] += h0 * g[o];
                s1[o] += h1 * g[o];
            }
        }
        if (t >= 128) {
            *reinterpret_cast<f32x4 *>(half[j]) = s0;
            *reinterpret_cast<f32x4 *>(half[j + 1]) = s1;
        }
        __syncthreads();  // the layer's last readers too: dZ4 overwrites it below
        if (t < 128) {
            *reinterpret_cast<f32x4 *>(pt + PT_W5 + 4 * j) = s0 + *reinterpret_cast<const f32x4 *>(half[j]);
            *reinterpret_cast<f32x4 *>(pt + PT_W5 + 4 * j + 4) =
                s1 + *reinterpret_cast<const f32x4 *>(half[j + 1]);
        }
    }
    // dZ4 = (dY W5^T) silu'(z4)
#pragma unroll
    for (int ni = 0; ni < 4; ni++) {
        const unsigned tile = 64 * w + 16 * ni;
        f32x4 w5[4];
#pragma unroll
        for (int e = 0; e < 4; e++) w5[e] = theta4(nb, OFF_W5 + 4 * (tile + e), 4 * lu);
#pragma unroll
        for (int mi = 0; mi < 4; mi++) {
            const f32x4 g = *reinterpret_cast<const f32x4 *>(dy[16 * mi + (lane & 15)]);
#pragma unroll
            for (int e = 0; e < 4; e++) {
                float s = 0.f;
#pragma unroll
                for (int o = 0; o < 4; o++) s += g[o] * w5[e][o];
                acc[mi][ni][e] = s;
            }
        }
    }
    train_reverse_epilogue(acc, z4, buf, pt + PT_B + 3 * H);
    __syncthreads();
    store_tile(buf, Dt + 2 * layer);
    train_layer<true>(nb, BF_TSW + 2 * LW, BF_TSW + LW, buf, f, acc);
    __syncthreads();
    train_reverse_epilogue(acc, z3, buf, pt + PT_B + 2 * H);
    __syncthreads();
    store_tile(buf, Dt + layer);
    train_layer<true>(nb, BF_TSW + LW, BF_TSW, buf, f, acc);
    __syncthreads();
    train_reverse_epilogue(acc, z2, buf, pt + PT_B + H);
    __syncthreads();
    store_tile(buf, Dt);
    train_layer<false>(nb, BF_TSW, 0, buf, f, acc);
    // layer 1: its pre-activations recomputed, dW1 and db1 summed over the tile
    f32x4 fr[4];
#pragma unroll
    for (int mi = 0; mi < 4; mi++) fr[mi] = *reinterpret_cast<const f32x4 *>(fs[16 * mi + (lane & 15)]);
#pragma unroll
    for (int ni = 0; ni < 4; ni++) {
        const unsigned tile = 64 * w + 16 * ni;
        f32x4 w1[4];
#pragma unroll
        for (int c = 0; c < 4; c++) w1[c] = theta4(nb, OFF_W1 + c * H + tile, lu);
        const f32x4 b1 = theta4(nb, OFF_B1 + tile, lu);
        f32x4 cs = {0.f, 0.f, 0.f, 0.f}, gw[4];
#pragma unroll
        for (int c = 0; c < 4; c++) gw[c] = cs;
#pragma unroll
        for (int mi = 0; mi < 4; mi++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float z = b1[e] + fr[mi][0] * w1[0][e] + fr[mi][1] * w1[1][e] +
                                fr[mi][2] * w1[2][e] + fr[mi][3] * w1[3][e];
                const float d = frombf(tobf(acc[mi][ni][e] * dsilu(frombf(tobf(z)))));
                cs[e] += d;
#pragma unroll
                for (int c = 0; c < 4; c++) gw[c][e] += fr[mi][c] * d;
            }
#pragma unroll
        for (int e = 0; e < 4; e++) {
            cs[e] = sum16(cs[e]);
#pragma unroll
            for (int c = 0; c < 4; c++) gw[c][e] = sum16(gw[c][e]);
        }
        if ((lane & 15) == 0) {
            *reinterpret_cast<f32x4 *>(pt + PT_B + tile + lu) = cs;
#pragma unroll
            for (int c = 0; c < 4; c++) *reinterpret_cast<f32x4 *>(pt + PT_W1 + c * H + tile + lu) = gw[c];
        }
    }
}

// Hidden weight gradients: layer l's (256, 256) matrix H_l^T dZ_l over one
// slice of the points, into that slice's partial matrix.  A workgroup of 8
// waves forms 256 inputs x 128 outputs, 64 x 64 per wave.  Both operands are
// stored point by point while the products run along the points: 64-point
// stages go through LDS as they are stored (the next stage's reads in flight
// in registers meanwhile) and come out transposed (ds_read_b64_tr_b16: four
// points of one unit per lane).  Rows are padded by 32 bytes, which spreads
// the 16 rows of a transposed read over all banks.
constexpr int WG_P = 64;                            // points per stage
// 3 layers x 2 halves x 42: one round of 256 compute units.  Fixed: the order of the sums and the
// size of the workspace are the same on every device.
constexpr int WG_SLICES = 42;
constexpr int WG_LA = H + 16, WG_LB = H / 2 + 16;   // LDS row lengths

typedef short s16x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ bf16x8 tr_frag(const __bf16 *lds, unsigned row, unsigned row_len,
                                          unsigned col) {
    typedef __attribute__((address_space(3))) s16x4 lds_v;
    const unsigned li = threadIdx.x & 15;
    const __bf16 *p = lds + (row + (li >> 2)) * row_len + col + 4 * (li & 3);
    struct {
        s16x4 lo, hi;
    } v;
    v.lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v *)p);
    v.hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v *)(p + 4 * row_len));
    return __builtin_bit_cast(bf16x8, v);
}

// stages [lo, hi) of slice s of n
__host__ __device__ __forceinline__ int slice_begin(int stages, int slices, int s) {
    return (int)((int64_t)stages * s / slices);
}

__global__ __launch_bounds__(512, 2) void k_wgrad(int64_t M, int slices,
                                                  const __bf16 *__restrict__ Hs,
                                                  const __bf16 *__restrict__ Ds,
                                                  float *__restrict__ part) {
    __shared__ __align__(16) __bf16 As[WG_P * WG_LA];
    __shared__ __align__(16) __bf16 Bs[WG_P * WG_LB];
    // consecutive workgroups go to the 8 XCDs in turn: the two halves of one
    // (slice, layer) are 8 apart, so they share their reads of H in one L2
    const unsigned half = (blockIdx.x >> 3) & 1, u = (blockIdx.x & 7) + 8 * (blockIdx.x >> 4);
    if (u >= 3u * slices) return;
    const unsigned l = u % 3, s = u / 3;
    const unsigned t = threadIdx.x, lane = t & 63, w = wave_id();
    const int64_t off = (int64_t)l * M * H;
    const int stages = (int)(M / WG_P);
    const int lo = slice_begin(stages, slices, s), hi = slice_begin(stages, slices, s + 1);
    const __bf16 *A = Hs + off, *B = Ds + off + half * (H / 2);
    bf16x8 ra[4], rb[2];
    auto fetch = [&](int st) {
        const int64_t p0 = (int64_t)st * WG_P;
#pragma unroll
        for (int k = 0; k < 4; k++)
            ra[k] = *reinterpret_cast<const bf16x8 *>(A + (p0 + 16 * k + (t >> 5)) * H + 8 * (t & 31));
#pragma unroll
        for (int k = 0; k < 2; k++)
            rb[k] = *reinterpret_cast<const bf16x8 *>(B + (p0 + 32 * k + (t >> 4)) * H + 8 * (t & 15));
    };
    f32x4 acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    const unsigned mw = 64 * (w >> 1), nw = 64 * (w & 1);
    if (lo < hi) fetch(lo);
    for (int st = lo; st < hi; st++) {
        __syncthreads();  // the previous stage has been read
#pragma unroll
        for (int k = 0; k < 4; k++)
            *reinterpret_cast<bf16x8 *>(As + (16 * k + (t >> 5)) * WG_LA + 8 * (t & 31)) = ra[k];
#pragma unroll
        for (int k = 0; k < 2; k++)
            *reinterpret_cast<bf16x8 *>(Bs + (32 * k + (t >> 4)) * WG_LB + 8 * (t & 15)) = rb[k];
        __syncthreads();
        if (st + 1 < hi) fetch(st + 1);
#pragma unroll
        for (int ks = 0; ks < WG_P; ks += 32) {
            const unsigned row = ks + 8 * (lane >> 4);
            bf16x8 a[4], b[4];
#pragma unroll
            for (int i = 0; i < 4; i++) a[i] = tr_frag(As, row, WG_LA, mw + 16 * i);
#pragma unroll
            for (int j = 0; j < 4; j++) b[j] = tr_frag(Bs, row, WG_LB, nw + 16 * j);
            // outputs as the A operand: a lane's four sums are four
            // consecutive outputs of one input (one 16-byte store below)
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int j = 0; j < 4; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[j], a[i], acc[i][j], 0, 0, 0);
        }
    }
    float *out = part + ((size_t)s * 3 + l) * H * H + half * (H / 2);
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++)
            *reinterpret_cast<f32x4 *>(out + (mw + 16 * i + (lane & 15)) * H + nw + 16 * j +
                                       4 * (lane >> 4)) = acc[i][j];
}

// Gradients from the partial sums: blocks [0, RW) four hidden weights per
// thread over the slices, the others 32 columns of the tiles' rows each (8
// row groups, joined in LDS).
constexpr int RW = 3 * H * H / 1024, RP = (PT_N + 31) / 32;

__global__ __launch_bounds__(256) void k_grad_reduce(const float *__restrict__ wpart, int slices,
                                                     const float *__restrict__ tpart, int tiles,
                                                     float *__restrict__ grad,
                                                     float *__restrict__ loss) {
    const int t = threadIdx.x;
    if (blockIdx.x < RW) {
        const int i = (blockIdx.x * 256 + t) * 4;
        f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 14
        for (int k = 0; k < slices; k++)
            s += *reinterpret_cast<const f32x4 *>(wpart + (size_t)k * 3 * H * H + i);
        const int l = i / (H * H);
        const int o = (l == 0 ? OFF_W2 : l == 1 ? OFF_W3 : OFF_W4) + i % (H * H);
#pragma unroll
        for (int e = 0; e < 4; e++) grad[o + e] = s[e];
        return;
    }
    __shared__ float red[8][32];
    const int c = (blockIdx.x - RW) * 32 + (t & 31), rg = t >> 5;
    float s = 0.f;
    if (c < PT_N)
#pragma unroll 8
        for (int k = rg; k < tiles; k += 8) s += tpart[(size_t)k * PT_N + c];
    red[rg][t & 31] = s;
    __syncthreads();
    if (rg > 0 || c > PT_LOSS) return;
#pragma unroll
    for (int g = 1; g < 8; g++) s += red[g][t];
    if (c < PT_B)
        grad[OFF_W1 + c] = s;
    else if (c < PT_W5) {
        const int l = (c - PT_B) / H;
        grad[(l == 0 ? OFF_B1 : l == 1 ? OFF_B2 : l == 2 ? OFF_B3 : OFF_B4) + (c - PT_B) % H] = s;
    } else if (c < PT_B5)
        grad[OFF_W5 + c - PT_W5] = s;
    else if (c < PT_LOSS)
        grad[OFF_B5 + c - PT_B5] = s;
    else if (loss)
        loss[0] = s;
}

// BF16 copies of W2..W4 (layout at BF_SW .. BF_TSWLO): fragment order of
// the high and the low parts, and of the transposes' high and low parts
__device__ __forceinline__ size_t frag_index(int k, int n) {
    // fragment order of V[k][n] (k input, n output): ((jt * 8 + ks) * 64 +
    // lane) * 8 + e with n = 16 jt + lane % 16, k = 32 ks + 8 (lane / 16) + e
    const int jt = n >> 4, ks = k >> 5, lane = (n & 15) + 16 * ((k & 31) >> 3), e = k & 7;
    return (((size_t)jt * 8 + ks) * 64 + lane) * 8 + e;
}

// the copies of parameter i, if it is a hidden weight
__device__ __forceinline__ void sync_copies(int i, float v, __bf16 *__restrict__ wbf) {
    const int l = i >= OFF_W4 ? 2 : i >= OFF_W3 ? 1 : 0;
    const int rem = i - (l == 0 ? OFF_W2 : l == 1 ? OFF_W3 : OFF_W4);
    if (rem < 0 || rem >= H * H) return;
    const int k = rem / H, n = rem % H;  // W[k][n], row-major [in][out]
    __bf16 hi, lo;
    split_bf(v, hi, lo);
    const size_t lb = (size_t)l * H * H;
    wbf[BF_SW + lb + frag_index(k, n)] = hi;
    wbf[BF_SWLO + lb + frag_index(k, n)] = lo;
    wbf[BF_TSW + lb + frag_index(n, k)] = hi;    // W^T[n][k] = W[k][n]
    wbf[BF_TSWLO + lb + frag_index(n, k)] = lo;
}

__global__ void k_sync_bf16(const float *__restrict__ theta, __bf16 *__restrict__ wbf) {
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i < NPARAM) sync_copies((int)i, theta[i], wbf);
}

// Adam (FP32 masters), and the updated weights' BF16 copies
__global__ void k_adam(float *__restrict__ theta, const float *__restrict__ g,
                       float *__restrict__ m, float *__restrict__ v, float lr, float b1, float b2,
                       float eps, float c1, float c2, __bf16 *__restrict__ wbf) {
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= NPARAM) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.0f - b1) * gi;
    const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float th = theta[i] - lr * (mi * c1) / (sqrtf(vi * c2) + eps);
    theta[i] = th;
    sync_copies((int)i, th, wbf);
}

// training data: positions (3,M) FP64 with exact Phi and grad -> features
// (M,4) and targets (M,4): o0 the potential's departure from the monopole
// in units of c, o1..o3 the force over its radial scale
__global__ void k_make_targets(gamd_mlp_norm nm, const double *__restrict__ q,
                               const double *__restrict__ phi, const double *__restrict__ grad,
                               int64_t M, float *__restrict__ feat, float *__restrict__ target) {
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= M) return;
    const double x = q[i], y = q[M + i], z = q[2 * M + i];
    float f[4];
    double r;
    features(nm, x, y, z, f, r);
#pragma unroll
    for (int c = 0; c < 4; c++) feat[i * 4 + c] = f[c];
    const double sgrad = out_scale_grad(nm, r);
    // o0's target: Phi = Phi_b (1 + c o0) with Phi_b = -G M / (r + r_s)
    target[i * 4 + 0] = (float)((phi[i] / (-nm.gm / (r + nm.rs)) - 1.0) / nm.phi_c);
    target[i * 4 + 1] = (float)(grad[i] / sgrad);
    target[i * 4 + 2] = (float)(grad[M + i] / sgrad);
    target[i * 4 + 3] = (float)(grad[2 * M + i] / sgrad);
}

// ---------------------------------------------------------------------------
// surrogate leapfrog, one step per call (this kernel for the orbits on the
// network, then k_surrogate_fallback for those on the exact force).  Orbit i:
// w (6,N) holds x and the half-step velocity between launches (vsync the
// synchronised velocity after the last step); E0[i] the initial energy;
// fb[i] the step at which the orbit fell back to exact SCF (-1 while on the
// surrogate).  mode 0: initial half kick; mode 1: drift + kick.  The force
// is -grad Phi_net, the gradient of the network's own potential, so the
// monitored energy Phi_net + |v|^2/2 is that of a conservative system; once
// |E - E0| > tol |E0| the orbit switches to the exact SCF force for the rest
// of the run (and for the remainder of this step).
template <int MI>
__global__ __launch_bounds__(256, 2) void k_surrogate_step(
    const float *__restrict__ theta, const __bf16 *__restrict__ wbf, gamd_mlp_norm nm,
    double *__restrict__ wq, double *__restrict__ vsync, double *__restrict__ E0,
    int32_t *__restrict__ fb, double *__restrict__ wsw, int64_t N, double dt, int mode,
    int32_t step, double tol) {
    constexpr int CP = 16 * MI;  // points of the workgroup's tile
    __shared__ __align__(16) __bf16 bhi[CP * LDSR];
    __shared__ __align__(16) __bf16 blo[CP * LDSR];
    __shared__ __align__(16) float feat[CP][4];
    __shared__ float red[4][CP][5];
    __shared__ float o0[CP];
    __shared__ float dfo[CP][4];
    const int t = threadIdx.x;
    const int64_t i = (int64_t)blockIdx.x * CP + t;
    const bool own = t < CP && i < N;
    double x = nm.pad_r, y = 0, z = 0, hx = 0, hy = 0, hz = 0, r = 1;
    int32_t fallback = -1;
    if (own) {
        x = wq[i];
        y = wq[N + i];
        z = wq[2 * N + i];
        hx = wq[3 * N + i];
        hy = wq[4 * N + i];
        hz = wq[5 * N + i];
        fallback = fb[i];
        if (mode == 1) {
            x = x + hx * dt;
            y = y + hy * dt;
            z = z + hz * dt;
        }
    }
    if (t < CP) {
        float f[4];
        features(nm, x, y, z, f, r);
#pragma unroll
        for (int c = 0; c < 4; c++) feat[t][c] = f[c];
    }
    // the tile runs the network unless every orbit in it has fallen back
    // (uniform over the workgroup, so every thread reaches the same barriers)
    const int any_net = __syncthreads_or(own && fallback < 0);
    if (any_net) tile_conservative<MI>(theta, wbf, feat, bhi, blo, red, o0, dfo);
    if (!own || fallback >= 0) return;  // exact-force orbits: k_surrogate_fallback
    double phi, gx, gy, gz;
    net_physics(nm, x, y, z, r, o0[t], dfo[t], phi, gx, gy, gz);
    // energy monitor on the synchronised velocity this force gives
    const double vx = (mode == 0) ? hx : hx - gx * dt / 2.0;
    const double vy = (mode == 0) ? hy : hy - gy * dt / 2.0;
    const double vz = (mode == 0) ? hz : hz - gz * dt / 2.0;
    const double E = phi + 0.5 * (vx * vx + vy * vy + vz * vz);
    if (mode == 0) {
        E0[i] = E;
    } else if (fabs(E - E0[i]) > tol * fabs(E0[i])) {
        // from this step on the exact force: k_surrogate_fallback redoes it
        // from the state before the step, which is recorded when asked
        fb[i] = step;
        if (wsw) {
#pragma unroll
            for (int c = 0; c < 6; c++) wsw[c * N + i] = wq[c * N + i];
        }
        return;
    }
    if (mode == 0) {
        wq[3 * N + i] = hx - gx * dt / 2.0;
        wq[4 * N + i] = hy - gy * dt / 2.0;
        wq[5 * N + i] = hz - gz * dt / 2.0;
    } else {
        wq[i] = x;
        wq[N + i] = y;
        wq[2 * N + i] = z;
        vsync[i] = vx;
        vsync[N + i] = vy;
        vsync[2 * N + i] = vz;
        wq[3 * N + i] = hx - gx * dt;
        wq[4 * N + i] = hy - gy * dt;
        wq[5 * N + i] = hz - gz * dt;
    }
}

// The same leapfrog step for the orbits on the exact SCF force (fb >= 0,
// including those k_surrogate_step has just switched): the drift is redone
// from the stored state, then the force, kick and writes with the
// arithmetic and the SCF evaluator of gamd_leapfrog's loop (k_leapfrog for
// the same potential layout), so from its switch step on an orbit follows
// the exact leapfrog bit for bit.  A kernel of its own keeps the SCF
// evaluator's registers out of the network kernel.
template <int LAY>
__global__ __launch_bounds__(64, scf_waves(LAY)) void k_surrogate_fallback(const DevPot *__restrict__ Pp,
                                                            double *__restrict__ wq,
                                                            double *__restrict__ vsync,
                                                            const int32_t *__restrict__ fb,
                                                            int64_t N, double dt, int mode) {
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= N || fb[i] < 0) return;
    double x = wq[i], y = wq[N + i], z = wq[2 * N + i];
    const double hx = wq[3 * N + i], hy = wq[4 * N + i], hz = wq[5 * N + i];
    if (mode == 1) {
        x = x + hx * dt;
        y = y + hy * dt;
        z = z + hz * dt;
    }
    double gx, gy, gz;
    pot_grad_l<true, LAY>(*Pp, x, y, z, gx, gy, gz);
    if (mode == 0) {
        wq[3 * N + i] = hx - gx * dt / 2.0;
        wq[4 * N + i] = hy - gy * dt / 2.0;
        wq[5 * N + i] = hz - gz * dt / 2.0;
    } else {
        wq[i] = x;
        wq[N + i] = y;
        wq[2 * N + i] = z;
        vsync[i] = hx - gx * dt / 2.0;
        vsync[N + i] = hy - gy * dt / 2.0;
        vsync[2 * N + i] = hz - gz * dt / 2.0;
        wq[3 * N + i] = hx - gx * dt;
        wq[4 * N + i] = hy - gy * dt;
        wq[5 * N + i] = hz - gz * dt;
    }
}

int check_norm(const gamd_mlp_norm *nm) {
    if (!nm || !nm->scale) return GAMD_ERR_INVALID;
    if (!(nm->inv_dlnr > 0.0) || !isfinite(nm->inv_dlnr) || !isfinite(nm->lnr0) ||
        !(nm->pad_r > 0.0) || !(nm->gm > 0.0) || !(nm->rs > 0.0) || !(nm->phi_c > 0.0) ||
        !isfinite(nm->gm) || !isfinite(nm->rs) || !isfinite(nm->phi_c))
        return GAMD_ERR_INVALID;
    return GAMD_OK;
}

// Whether M points go to 16-point tiles (else 32): while every such tile has a
// compute unit of its own the half-sized tile is done sooner (500 points: 19
// against 24 us; 4,096: 21 against 24), from there on it reads every weight
// twice as often (8,192 points: 35 against 27 us).  Same results either way.
bool tile_points16(size_t M) { return M <= (size_t)cu_count() * 16; }

// slices of the points in k_wgrad: whole stages, at most WG_SLICES
int wgrad_slices(int64_t M) { return (int)(M / WG_P < WG_SLICES ? M / WG_P : WG_SLICES); }

int check_params(const float *theta, const uint16_t *wbf) {
    return (theta && wbf) ? GAMD_OK : GAMD_ERR_INVALID;
}

}  // namespace

extern "C" {

int64_t gamd_mlp_param_count(void) { return NPARAM; }
int64_t gamd_mlp_bf16_count(void) { return NBF; }

int64_t gamd_mlp_workspace_bytes(int64_t M) {
    // H1..H3 and dZ2..dZ4 (6 x M x 256 BF16), the hidden gradients' partial
    // matrices, one row of partial sums per tile
    return 6 * M * H * 2 + (int64_t)wgrad_slices(M) * 3 * H * H * 4 + (M / TP) * PT_N * 4 + 256;
}

int gamd_mlp_sync_bf16(const float *theta, uint16_t *wbf, void *stream) {
    if (check_params(theta, wbf)) return GAMD_ERR_INVALID;
    hipLaunchKernelGGL(k_sync_bf16, dim3(grid_for(NPARAM, 256)), dim3(256), 0, as_stream(stream),
                       theta, reinterpret_cast<__bf16 *>(wbf));
    return launch_status();
}

int gamd_mlp_forward(const float *theta, const uint16_t *wbf, const gamd_mlp_norm *norm,
                     const double *q, size_t M, double *phi, double *grad, void *stream) {
    if (check_params(theta, wbf) || check_norm(norm) || (M && (!q || !phi || !grad)))
        return GAMD_ERR_INVALID;
    if (M == 0) return GAMD_OK;
    const bool mi1 = tile_points16(M);
    hipLaunchKernelGGL(mi1 ? k_mlp_forward<1> : k_mlp_forward<2>,
                       dim3(grid_for(M, mi1 ? 16 : 32)), dim3(256), 0,
                       as_stream(stream), theta, reinterpret_cast<const __bf16 *>(wbf), *norm, q,
                       (int64_t)M, phi, grad);
    return launch_status();
}

int gamd_mlp_make_targets(const gamd_mlp_norm *norm, const double *q, const double *phi,
                          const double *grad, size_t M, float *feat, float *target, void *stream) {
    if (check_norm(norm) || (M && (!q || !phi || !grad || !feat || !target)))
        return GAMD_ERR_INVALID;
    if (M == 0) return GAMD_OK;
    hipLaunchKernelGGL(k_make_targets, dim3(grid_for(M, 256)), dim3(256), 0, as_stream(stream),
                       *norm, q, phi, grad, (int64_t)M, feat, target);
    return launch_status();
}

int gamd_mlp_gradients(const float *theta, const uint16_t *wbf, const float *feat,
                       const float *target, size_t M, float *grad, float *loss, void *workspace,
                       size_t workspace_bytes, void *stream) {
    if (check_params(theta, wbf) || !feat || !target || !grad || !workspace) return GAMD_ERR_INVALID;
    if (M == 0 || M % 64) return GAMD_ERR_INVALID;
    if ((int64_t)workspace_bytes < gamd_mlp_workspace_bytes((int64_t)M)) return GAMD_ERR_INVALID;
    hipStream_t s = as_stream(stream);
    const int64_t Mi = (int64_t)M;
    const int slices = wgrad_slices(Mi), tiles = (int)(Mi / TP);
    __bf16 *Hs = static_cast<__bf16 *>(workspace);
    __bf16 *Ds = Hs + 3 * Mi * H;
    float *wpart = reinterpret_cast<float *>(Ds + 3 * Mi * H);
    float *tpart = wpart + (size_t)slices * 3 * H * H;
    const __bf16 *w = reinterpret_cast<const __bf16 *>(wbf);
    hipLaunchKernelGGL(k_train_tile, dim3((unsigned)tiles), dim3(256), 0, s, theta, w, feat,
                       target, Mi, Hs, Ds, tpart);
    hipLaunchKernelGGL(k_wgrad, dim3(16 * grid_for(3 * slices, 8)), dim3(512), 0, s, Mi, slices,
                       Hs, Ds, wpart);
    hipLaunchKernelGGL(k_grad_reduce, dim3(RW + RP), dim3(256), 0, s, wpart, slices, tpart, tiles,
                       grad, loss);
    return launch_status();
}

int gamd_mlp_adam(float *theta, const float *grad, float *m, float *v, int64_t step, float lr,
                  float beta1, float beta2, float eps, uint16_t *wbf, void *stream) {
    if (!theta || !grad || !m || !v || !wbf || step < 1) return GAMD_ERR_INVALID;
    const float c1 = 1.0f / (1.0f - powf(beta1, (float)step));
    const float c2 = 1.0f / (1.0f - powf(beta2, (float)step));
    hipLaunchKernelGGL(k_adam, dim3(grid_for(NPARAM, 256)), dim3(256), 0, as_stream(stream), theta,
                       grad, m, v, lr, beta1, beta2, eps, c1, c2, reinterpret_cast<__bf16 *>(wbf));
    return launch_status();
}

int gamd_surrogate_leapfrog_step(const float *theta, const uint16_t *wbf, const gamd_mlp_norm *norm,
                                 const gamd_potential *scf, double *w, double *vsync, double *E0,
                                 int32_t *fallback_step, double *w_switch, size_t N, double dt,
                                 int mode, int32_t step, double tol, void *stream) {
    if (check_params(theta, wbf) || check_norm(norm) || !scf || !w || !vsync || !E0 ||
        !fallback_step)
        return GAMD_ERR_INVALID;
    if (scf->dev.n != 1 || scf->dev.c[0].type != GAMD_SCF || scf->dev.c[0].shift_rotate)
        return GAMD_ERR_INVALID;
    if (mode != 0 && mode != 1) return GAMD_ERR_INVALID;
    if (N == 0) return GAMD_OK;
    hipStream_t s = as_stream(stream);
    const bool mi1 = tile_points16(N);
    hipLaunchKernelGGL(mi1 ? k_surrogate_step<1> : k_surrogate_step<2>,
                       dim3(grid_for(N, mi1 ? 16 : 32)), dim3(256), 0, s,
                       theta, reinterpret_cast<const __bf16 *>(wbf), *norm, w, vsync, E0,
                       fallback_step, w_switch, (int64_t)N, dt, mode, step, tol);
    int rc = launch_status();
    if (rc) return rc;
    auto fk = scf->dev.layout == LAYOUT_SCF106 ? k_surrogate_fallback<LAYOUT_SCF106>
                                                : k_surrogate_fallback<LAYOUT_SCF>;
    hipLaunchKernelGGL(fk, dim3(grid_for(N, 64)), dim3(64), 0, s, scf->ddev, w, vsync,
                       fallback_step, (int64_t)N, dt, mode);
    return launch_status();
}

}  // extern "C"
