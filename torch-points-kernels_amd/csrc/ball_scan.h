// Ball query: one query answered by a wavefront that scans its cloud in index order.
#pragma once

#include "tpk_device.h"

namespace {

// The support rows s0 .. s1 of x against the query (qx, qy, qz); the query's row of the outputs at idx / dist.
// DENSE: the dense layout's rules (a hit has squared distance < radius2, indices count from s0, the slots behind the last
// hit repeat the first one), otherwise the packed layout's (<= radius2, rows of x, -1).
template <bool DENSE>
__device__ __forceinline__ void ball_scan_rows(const float* __restrict__ x, int s0, int s1, float qx, float qy, float qz, float radius2,
                                               int nsample, int lane, int64_t* __restrict__ idx, float* __restrict__ dist TPK_WORK_PARAM)
{
    // Serial semantics directly: lanes hold 64 consecutive support rows; ballot + prefix count
    // give the hits their slots in index order; stop after nsample hits.
    int cnt = 0;
    int first_hit = -1; // (dense layout: the row that fills the slots behind the last hit)
    constexpr int BATCH = 4; // loads of four steps in flight
    for (int base = s0; base < s1 && cnt < nsample; base += BATCH * TPK_WAVE)
    {
        float px[BATCH], py[BATCH], pz[BATCH];
#pragma unroll
        for (int u = 0; u < BATCH; ++u)
        {
            const int64_t pos = min(base + u * TPK_WAVE + lane, s1 - 1);
            px[u] = x[pos * 3 + 0];
            py[u] = x[pos * 3 + 1];
            pz[u] = x[pos * 3 + 2];
        }
#pragma unroll
        for (int u = 0; u < BATCH; ++u)
        {
            const int pos = base + u * TPK_WAVE + lane;
            const float d = tpk_dist2(qx, qy, qz, px[u], py[u], pz[u]);
            TPK_WORK_ADD(1);
            const bool hit = pos < s1 && (DENSE ? d < radius2 : d <= radius2);
            const unsigned long long mask = __ballot(hit);
            const int slot = cnt + static_cast<int>(tpk_prefix_count(mask));
            if (hit && slot < nsample)
            {
                idx[slot] = DENSE ? pos - s0 : pos;
                dist[slot] = d;
            }
            if (DENSE && first_hit < 0 && mask != 0)
                first_hit = base + u * TPK_WAVE + __builtin_ctzll(mask) - s0;
            cnt += __builtin_popcountll(mask);
        }
    }
    for (int s = cnt + lane; s < nsample; s += TPK_WAVE)
    {
        idx[s] = DENSE ? max(first_hit, 0) : -1;
        dist[s] = -1.0f;
    }
}

} // namespace
