// gamd_rules.hpp -- limits of the dispatch that follow from the number of compute
// units (256 on a whole MI355X, fewer on a partition).  Plain C++: checked on the
// host by tests/test_host.py.
#pragma once
#include <stdint.h>

namespace gamd {

// Most orbits that Leapfrog of the Milky-Way layout integrates one to a 16-lane row
// (k_leapfrog_row), four to a wave: at 16 a compute unit every row's wave has a SIMD
// for itself (two to a SIMD take twice as long).  Measured on 256 units, ns per step
// on rows and one orbit a lane: every step saved, 16 to 1,024 orbits 266-270 and 322,
// 4,096 orbits 300 and 323; final states only, 229-231 and 256, 2,048 orbits 241 and
// 256, 4,096 orbits 264 and 256.
constexpr int64_t leapfrog_row_orbits(int cus, bool saved) {
    return (int64_t)cus * (saved ? 16 : 8);
}

// Most orbits up to which a DOP853 wave keeps all its rows running (wide_tail): one
// wave of single lanes on each of the four SIMDs of a compute unit.
constexpr int64_t filled_row_orbits(int cus) { return (int64_t)cus * 4 * 64; }

}  // namespace gamd
