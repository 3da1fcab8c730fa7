// ppm_lanes.hpp — exchanges between neighbouring lanes of a wavefront on the VALU.
//
// __shfl goes through the LDS crossbar (ds_bpermute): an address instruction and a wait on the LDS
// counter, ~100 cycles on the dependent chain of a relaxation step.  Exchanges within a row of 16
// lanes are DPP moves, which the compiler can also fold into the consuming instruction; rows are
// exchanged by gfx950's v_permlane16_swap / v_permlane32_swap.
#pragma once

#include <hip/hip_runtime.h>

namespace ppm {

template <int CTRL, int BANKS = 0xf>
__device__ __forceinline__ float dpp(float old, float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(old), __float_as_int(v), CTRL, 0xf, BANKS,
                                                      BANKS == 0xf));
}

// Value of lane S of this lane's group of G = 2 or 4 lanes.
template <int G, int S>
__device__ __forceinline__ float from_lane(float v) {
    static_assert((G == 2 || G == 4) && S < G, "groups lie within a quad");
    constexpr int hi = G == 2 ? 2 + S : S;
    return dpp<S | (S << 2) | (hi << 4) | (hi << 6)>(v, v);          // quad_perm
}

// v + the value of lane (lane ^ OFF).  PERIODIC: v repeats with period 2 OFF over the row of 16 (an
// earlier step added lane ^ 2 OFF), so any lane at distance OFF will do.
template <int OFF, bool PERIODIC>
__device__ __forceinline__ float add_xor(float v) {
    if constexpr (OFF == 32) {
        const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
        return __uint_as_float(p[0]) + __uint_as_float(p[1]);
    } else if constexpr (OFF == 16) {
        const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
        return __uint_as_float(p[0]) + __uint_as_float(p[1]);
    } else if constexpr (OFF == 8) {
        return v + dpp<0x128>(v, v);                                  // row_ror:8
    } else if constexpr (OFF == 4 && PERIODIC) {
        return v + dpp<0x124>(v, v);                                  // row_ror:4
    } else if constexpr (OFF == 4) {
        float o = dpp<0x104, 0x5>(v, v);                              // row_shl:4 into lanes 0-3, 8-11
        o = dpp<0x114, 0xa>(o, v);                                    // row_shr:4 into lanes 4-7, 12-15
        return v + o;
    } else if constexpr (OFF == 2) {
        return v + dpp<0x4e>(v, v);                                   // quad_perm [2,3,0,1]
    } else {
        return v + dpp<0xb1>(v, v);                                   // quad_perm [1,0,3,2]
    }
}

// Sum over the G lanes of this lane's group, the butterfly of distances G/2, G/4, ..., 1: every lane
// gets the same bits (the two operands of each addition only trade places).
template <int G, int OFF = G / 2>
__device__ __forceinline__ float group_sum(float v) {
    if constexpr (OFF == 0) return v;
    else return group_sum<G, OFF / 2>(add_xor<OFF, (OFF == 4 && G >= 16)>(v));
}

}  // namespace ppm
