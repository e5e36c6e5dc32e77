// Cells of the packed ball query's hash table (ball_table.hip): plain arithmetic, so that it can be tried on the host.
#pragma once

#include <cmath>
#include <cstdint>
#include <cstring>

#if defined(__HIPCC__) || defined(__HIP__)
#define BT_BOTH __host__ __device__
#else
#define BT_BOTH
#endif

// Half the side of a cube that holds every point the radius test accepts.  The test is d2 <= fl(r * r) with every product and sum
// rounded on its own, so an accepted difference along one axis exceeds r by a few units in its last place at most; squares that
// underflow are what the constant is for.
BT_BOTH inline float bt_reach(float radius)
{
    return std::fabs(radius) * 1.000001f + 2e-19f;
}

// Cell of a coordinate scaled by the cell's inverse width: the whole part, and from 2^23 on, where a float has no
// fraction left, one cell per float - a function that never falls as v rises, whatever the scale, and stays inside an int32.  (A
// point p that the test accepts lies in [q - reach, q + reach]; p is a float, so it is not below the rounded lower end either,
// and its cell lies between the cells of the two rounded ends.)
constexpr float BT_FAR = 8388608.0f; // 2^23
BT_BOTH inline int bt_scaled_cell(float t)
{
    if (std::fabs(t) < BT_FAR)
        return static_cast<int>(std::floor(t));
    int bits;
    std::memcpy(&bits, &t, sizeof(bits));
    const int far = (bits & 0x7fffffff) - 0x4b000000 + 0x800000;
    return bits < 0 ? -far : far;
}
BT_BOTH inline int bt_cell(float v, float inverse_width)
{
    return bt_scaled_cell(v * inverse_width);
}

// A row of cells (., iy, iz) of a cloud lies in one of BT_PARTS equal parts of the table: cell ix is bucket (place + ix) modulo the
// part's size.  Rows whose iy and iz differ by at most two lie in different parts, so that the runs of one query never overlap;
// the rows of a plane of constant iy or iz fill all parts evenly.
constexpr int BT_PARTS = 16;
struct BtRow
{
    uint32_t part, place;
};

BT_BOTH inline BtRow bt_row(int iy, int iz, int64_t cloud)
{
    const uint64_t id = static_cast<uint64_t>(cloud);
    uint32_t h = static_cast<uint32_t>(iy) * 0x9e3779b1u ^ (static_cast<uint32_t>(iz) * 0x85ebca77u + 0x165667b1u);
    h ^= (static_cast<uint32_t>(id) + static_cast<uint32_t>(id >> 32) * 0x2c1b3c6du) * 0x297a2d39u;
    h ^= h >> 15;
    h *= 0x2545f491u;
    h ^= h >> 13;
    return BtRow{(static_cast<uint32_t>(iy) + 3u * static_cast<uint32_t>(iz)) % BT_PARTS, h};
}

// part_mask: buckets of a part - 1 (a power of two less one).
BT_BOTH inline uint32_t bt_bucket(const BtRow& row, int ix, uint32_t part_mask)
{
    return row.part * (part_mask + 1u) + ((row.place + static_cast<uint32_t>(ix)) & part_mask);
}
