// fp32 numbers as sums of 16-bit ones for the matrix instructions, and the order of 16-byte pieces within the rows of a wide
// LDS tile: what the kernels of cott_wide.h and cott_split.h have in common.
#pragma once
#include "cott_common.h"
#include <type_traits>

namespace cott {

// Where 16-byte piece c of row r of an A or B tile lies within the row.  A 16-byte read of the wavefront is served 16 lanes
// at a time, not in lane order: 0-3, 12-15 and 20-27 together, then 4-11, 16-19 and 28-31.  Along the contracted dim (lane
// 16g + m reads piece 4ks + g of row m) those are rows 0-3 and 12-15 of one piece and rows 4-11 of its neighbour, or the
// reverse; with rows 4i .. 4i+3 in different groups of four pieces and the rows' upper bits turned by {0, 2, 3, 1} they
// fall on 16 different 16-byte bank groups.  The transposing reads (pieces 4k .. 4k+3 of rows 4i .. 4i+3, one half of each
// piece) cannot do better than two lanes to a bank.  Conflict cycles of the gradients of 16 heads N1024 D256: 2.3 of 10.6
// million LDS cycles, without the turn 5.0 of 13.3, with rows padded by 32 bytes instead 5.4 of 13.7 (2 heads N4096 in one
// group, forward: 190, 197 and 198 us).
__device__ __forceinline__ int wide_piece(int r, int c) {
    const int up = (r >> 1) & 6;  // twice the upper bits of r, carried over into {0, 2, 3, 1}
    return c ^ (4 * (r & 3) + (up & 4 ? up ^ 7 : up));
}

// Two fp32 numbers cut to 16-bit ones of type TR towards zero (so that no finite number becomes infinite).
template <class TR>
__device__ __forceinline__ uint32_t cut2(float a, float b) {
    if constexpr (std::is_same<TR, Fp16>::value)
        return bitcast<uint32_t>(__builtin_amdgcn_cvt_pkrtz(a, b));
    else
        return __builtin_amdgcn_perm(bitcast<uint32_t>(b), bitcast<uint32_t>(a), 0x07060302u);  // the upper halves
}
// fp32 -> three 16-bit numbers of type TR, hi + mid + lo.  Each takes the leading bits of what the ones before it leave: 8
// of bf16 (3 x 8 = 24, exact wherever the last one is a normal number), 11 of fp16 (exact down to 2^-24).
template <class TR>
__device__ __forceinline__ void split3(float a, float b, uint32_t &hi, uint32_t &mid, uint32_t &lo) {
    hi = cut2<TR>(a, b);
    a -= TR::to_float((u16)(hi & 0xffffu));
    b -= TR::to_float((u16)(hi >> 16));
    mid = cut2<TR>(a, b);
    lo = cut2<TR>(a - TR::to_float((u16)(mid & 0xffffu)), b - TR::to_float((u16)(mid >> 16)));
}
__device__ __forceinline__ bool any_nan(f32x4 v) {
    const float s = (v[0] + v[1]) + (v[2] + v[3]);  // (also true where infinities cancel: number_or then changes nothing)
    return s != s;
}
// v where it is a number, else the same element of w.  An infinite state, score or (fp16) C entry splits into hi = inf and
// inf - inf; the sum formed from the hi parts of both factors alone then has the value the single-number arithmetic gives.
__device__ __forceinline__ f32x4 number_or(f32x4 v, f32x4 w) {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = v[e] == v[e] ? v[e] : w[e];
    return v;
}

}  // namespace cott
