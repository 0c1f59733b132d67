// gamd_row.hpp -- one orbit on a 16-lane DPP row: broadcasts within the row and
// the Milky-Way evaluator shared by its lanes (DOP853's rows, Leapfrog's rows).
#pragma once
#include "gamd_device.hpp"

namespace gamd {

template <int SRC>
__device__ __forceinline__ double row_bcast(double v) {
    // DPP row_newbcast:SRC: every lane of a 16-lane row reads lane SRC of the
    // row (every lane has a source in its row, so the zero is not used); of a
    // double one v_mov_b64_dpp
    return __builtin_amdgcn_update_dpp(0.0, v, 0x150 + SRC, 0xF, 0xF, true);
}

// The Milky-Way evaluator (mw_factors) on a 16-lane row whose lanes 0 to 7
// use its result: the two reciprocal roots that do not wait for each other are
// one, of r^2 in the lower and of z^2 + b^2 in the upper half, and the log's
// polynomial is one chain of three lanes' coefficients instead of three.  The
// same operations on the same values; a wave alone on its SIMD waits for the
// issue of every instruction, of which an evaluation loses 8 in 117.
struct RowMw {
    MwConstants m;
    double lo0, lo1, hi0, hi1;  // lane i: the i-th third of log_poly's coefficients
    bool upper;
    __device__ __forceinline__ RowMw(const DevPot &P, int lane) : m(P), upper(lane >= 8) {
        lo0 = lane == 0 ? 1.0 : (lane == 1 ? 0.1111111111111111 : 0.058823529411764705);
        lo1 = lane == 0 ? 0.3333333333333333
                        : (lane == 1 ? 0.09090909090909091 : 0.05263157894736842);
        hi0 = lane == 0 ? 0.2 : (lane == 1 ? 0.07692307692307693 : 0.047619047619047616);
        hi1 = lane == 0 ? 0.14285714285714285
                        : (lane == 1 ? 0.06666666666666667 : 0.043478260869565216);
        // kept in vector registers: as scalars they were read again from
        // memory, with a wait each, in every attempt
        asm volatile("" : "+v"(m.m1), "+v"(m.c1), "+v"(m.m2), "+v"(m.c2), "+v"(m.m3), "+v"(m.a3),
                     "+v"(m.b3sq), "+v"(m.m4), "+v"(m.irs4));
        asm volatile("" : "+v"(lo0), "+v"(lo1), "+v"(hi0), "+v"(hi1));
    }
    __device__ __forceinline__ void rsqrt_pair(double a, double b, double &ra, double &rb) const {
        ra = rsqrt_nr(upper ? b : a);
        rb = row_bcast<8>(ra);
    }
    __device__ __forceinline__ double operator()(double z, double z2, double z4, double z8) const {
        const double q = fma(z2, fma(z, hi1, hi0), fma(z, lo1, lo0));
        double r;
        asm("s_nop 1\n"
            "v_mov_b64_dpp %0, %1 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
            "v_fmac_f64_dpp %0, %1, %2 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
            "v_fmac_f64_dpp %0, %1, %3 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
            : "=&v"(r)
            : "v"(q), "v"(z4), "v"(z8));
        return r;
    }
};

// the same with the result in all 16 lanes
struct RowMwAll : RowMw {
    using RowMw::RowMw;
    __device__ __forceinline__ void rsqrt_pair(double a, double b, double &ra, double &rb) const {
        const double t = rsqrt_nr(upper ? b : a);
        ra = row_bcast<0>(t);
        rb = row_bcast<8>(t);
    }
};

}  // namespace gamd
