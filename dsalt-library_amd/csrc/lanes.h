// Sums over lanes that avoid the LDS round trips of lane exchanges.
#pragma once

#include "common.h"

namespace dsalt {

// Sum over the aligned groups of W lanes (W a power of two <= 64; every lane of a group
// receives it), with the same tree as a butterfly of lane exchanges by 1, 2, 4, ..., hence
// the same bits: the first four levels are DPP adds (quad permutes and row mirrors: after a
// level the lanes of a pair hold equal sums, so a mirror reaches the partner group as well
// as an exchange does), which cost no LDS round trip; the last two exchange rows through
// v_permlane{16,32}_swap.
template <int CTRL>
__device__ __forceinline__ float dpp_add(float x) {
    return x + __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), CTRL, 0xF, 0xF, false));
}
__device__ __forceinline__ float group_sum_lanes(float x, int width) {
    if (width > 1) x = dpp_add<0xB1>(x);   // quad_perm [1,0,3,2]
    if (width > 2) x = dpp_add<0x4E>(x);   // quad_perm [2,3,0,1]
    if (width > 4) x = dpp_add<0x141>(x);  // row_half_mirror
    if (width > 8) x = dpp_add<0x140>(x);  // row_mirror
    if (width > 16) {
        auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
        x = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
    if (width > 32) x = half_sum(x);
    return x;
}

}  // namespace dsalt
