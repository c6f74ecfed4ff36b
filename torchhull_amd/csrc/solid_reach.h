// How far carving may trust a solid map (see "Solid maps" in vh_kernels.hip).  Plain constexpr code: the device calls
// it, and a host test checks the bound it rests on.

#pragma once

#include <cstdint>

namespace thull
{

// The box sum of a window of solid pixels has to stay within this of the window's area; carving's margin is 0.4, and
// the rest covers the rounding of area - margin and of the sum's last subtraction (below 0.001 for the windows that
// the maps can hold).
constexpr float kSolidError = 0.39f;

// Bounds of the rounding errors behind a box sum, for non-negative masks of H x W pixels whose integral image ends in
// `total`; all partial sums stay below 2^S = 2^24 ulps.
//  row:     2^(S - 24).  The row chains at the window's two ends each round once per column, by half an ulp of at most
//           this; the first two operations of the box sum round by 1.5 of it together.
//  columns: one more `row`, for all columns of the window together.  The additions of 1 along a column round only
//           where its sum crosses a power of two, by 2^-24 of the sum, and the columns' sums add up to less than 2^S.
//           A column that crosses several of them grows from below half its last power, all by the window's ones:
//  column:  H 2^-21 for each column of the window covers those.
// The chains' own errors, at most 2^-24 of the sum per addition, can carry a partial sum past the total: S belongs to
// the total widened by four times that.
struct SolidErrors
{
    float row, column;
};

constexpr SolidErrors
solid_errors(float total, int32_t H, int32_t W)
{
    const float bound = total * (1.0f + (float(H) + float(W)) * 0x1p-22f);
    // the power of two above the bound
    const float above = __builtin_bit_cast(float, (__builtin_bit_cast(uint32_t, bound) & 0x7f800000u) + 0x00800000u);
    return SolidErrors{ above * 0x1p-24f, float(H) * 0x1p-21f };
}

// How far (in pixels from a cell's centre) a window of solid pixels may reach so that its box sum is certain to
// classify as full; negative: no window is.  A window that reaches r from the centre has at most w = 2 r + 2 columns,
// and its error is at most (w + 3) row + w column.  Integral images of whole numbers below 2^23 are exact.
constexpr float
solid_reach(bool negative, bool fraction, float total, int32_t H, int32_t W)
{
    if (negative || !(total < 0x1p40f))
        return -1.0f;
    if (!fraction && total < 0x1p23f)
        return 1e9f;
    const SolidErrors e = solid_errors(total, H, W);
    return (kSolidError - 5.0f * e.row - 2.0f * e.column) / (2.0f * e.row + 2.0f * e.column);
}

} // namespace thull
