// The shape of a grid over a cloud (lds_grid.h): plain arithmetic, without a word of device code, so that it can be
// tried on the host for every cloud there can be.
#pragma once

// Extents outside this range get one cell, like an axis along which all coordinates are equal.  Below it the number of cells
// per unit overflows float32 (128 / 1e-37) and the squares of a cell's width vanish; beyond it the extent itself is no float32
// (coordinates of both signs above 1.7e38), and with it the share, a NaN.
constexpr float GRID_LEAST_EXTENT = 1e-16f;
constexpr float GRID_MOST_EXTENT = 3.402823466e38f;

constexpr float grid_extent(float low, float high)
{
    const float extent = high - low; // (NaN or -inf for a cloud without finite coordinates)
    return extent >= GRID_LEAST_EXTENT && extent <= GRID_MOST_EXTENT ? extent : 0.0f;
}

struct GridCounts
{
    int along[3];
    int all; // their product
};

// Cells per axis - between 1 and `axis` - for `along` cells on the longest one; share: extents over the longest extent.
constexpr GridCounts grid_fit(const float (&share)[3], float along, int axis)
{
    GridCounts counts = {{1, 1, 1}, 1};
    for (int a = 0; a < 3; ++a)
    {
        const float f = share[a] * along + 0.5f;
        counts.along[a] = f >= static_cast<float>(axis) ? axis : f >= 1.0f ? static_cast<int>(f) : 1;
        counts.all *= counts.along[a];
    }
    return counts;
}

// Cells per axis for about per_cell of m points per cell, as cubic as `axis` (at most 128) cells per axis and `most` in all
// allow.  fitting(f): for how many lane = 0 .. 63 f(lane) holds (a wavefront asks all at once).  The product grows with
// `along`: the largest of the sizes tried that stays within the cells wanted, in steps of 2 up to 128, then in steps of
// 1 / 32 inside the step found.
template <typename Fitting>
constexpr GridCounts grid_counts(const float (&extent)[3], int m, float per_cell, int axis, int most, Fitting fitting)
{
    float longest = 0.0f;
    for (int a = 0; a < 3; ++a)
        longest = extent[a] > longest ? extent[a] : longest;
    float share[3] = {0.0f, 0.0f, 0.0f};
    for (int a = 0; a < 3; ++a)
        share[a] = longest > 0.0f ? extent[a] / longest : 0.0f;
    const float cells = static_cast<float>(m) / per_cell;
    const int wanted = cells >= static_cast<float>(most) ? most : cells >= 1.0f ? static_cast<int>(cells) : 1;
    const int coarse = fitting([&](int lane) { return grid_fit(share, 2.0f * static_cast<float>(lane + 1), axis).all <= wanted; });
    const float from = 2.0f * static_cast<float>(coarse);
    const int fine = fitting([&](int lane) { return grid_fit(share, from + static_cast<float>(lane + 1) * (1.0f / 32.0f), axis).all <= wanted; });
    const GridCounts counts = grid_fit(share, from + static_cast<float>(fine) * (1.0f / 32.0f), axis);
    return counts.all <= most ? counts : GridCounts{{1, 1, 1}, 1}; // (what is behind the last cell belongs to others)
}
