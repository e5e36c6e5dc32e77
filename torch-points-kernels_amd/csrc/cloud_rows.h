// Packed layouts: the rows of a cloud, found in the sorted cloud ids by a wavefront.
#pragma once

#include "tpk_device.h"

namespace {

// The equal range [first, last) of value v in sorted a[0..len), found by the whole wavefront: 64
// samples per round instead of one, and both ends in the same rounds, so that their loads
// travel together.
__device__ __forceinline__ void wave_equal_range(const int64_t* __restrict__ a, int len, int64_t v, int lane,
                                                 int& first, int& last)
{
    int lo0 = 0, hi0 = len, lo1 = 0, hi1 = len;
    while (hi0 > lo0 || hi1 > lo1)
    {
        const int step0 = (hi0 - lo0 + TPK_WAVE - 1) / TPK_WAVE, step1 = (hi1 - lo1 + TPK_WAVE - 1) / TPK_WAVE;
        const int pos0 = lo0 + lane * step0, pos1 = lo1 + lane * step1;
        const bool in0 = pos0 < hi0, in1 = pos1 < hi1;
        const int64_t sample0 = a[in0 ? pos0 : 0], sample1 = a[in1 ? pos1 : 0];
        const unsigned long long ge0 = __ballot(!in0 || sample0 >= v);
        const unsigned long long ge1 = __ballot(!in1 || sample1 > v);
        if (hi0 > lo0)
        {
            const int f = ge0 ? __builtin_ctzll(ge0) : TPK_WAVE;
            const int next_lo = f > 0 ? lo0 + (f - 1) * step0 + 1 : lo0;
            hi0 = f < TPK_WAVE ? min(lo0 + f * step0, hi0) : hi0;
            lo0 = next_lo;
        }
        if (hi1 > lo1)
        {
            const int f = ge1 ? __builtin_ctzll(ge1) : TPK_WAVE;
            const int next_lo = f > 0 ? lo1 + (f - 1) * step1 + 1 : lo1;
            hi1 = f < TPK_WAVE ? min(lo1 + f * step1, hi1) : hi1;
            lo1 = next_lo;
        }
    }
    first = lo0;
    last = lo1;
}

// Work that rides along with a launch that puts the support points in order, in workgroups of its own behind the others:
// for every query of a packed call, the rows [x, y) of the support points that carry
// the query's cloud id (both id arrays sorted).  A wavefront takes 64 consecutive queries and
// searches once per distinct id among them - nearly always one.
struct CloudRows
{
    const int64_t* batch_x;
    const int64_t* batch_y;
    int size_x;
    int64_t size_y;
    int2* rows;
};

__device__ __forceinline__ void cloud_rows_job(const CloudRows& job, int64_t wavefront, int lane)
{
    const int64_t q = wavefront * TPK_WAVE + lane;
    const bool has = q < job.size_y;
    const int64_t mine = has ? job.batch_y[q] : 0;
    unsigned long long todo = __ballot(has);
    while (todo != 0)
    {
        const int64_t id = __shfl(mine, __builtin_ctzll(todo));
        int first, last;
        wave_equal_range(job.batch_x, job.size_x, id, lane, first, last);
        const bool same = has && mine == id;
        if (same)
            job.rows[q] = make_int2(first, last);
        todo &= ~__ballot(same); // (the lane that gave the id is among them: the loop ends)
    }
}

} // namespace
