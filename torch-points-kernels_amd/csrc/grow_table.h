// The table of the clusters a walk has found (cluster.hip gathers their members by it): plain arithmetic, tried on the host.
#pragma once

#include <cstdint>

#if defined(__HIPCC__) || defined(__HIP__)
#define GROW_BOTH __host__ __device__
#else
#define GROW_BOTH
#endif

constexpr int GROW_TABLE_ROW = 3; // words of a cluster: its first output, its first entry, the first place of its piece

// The cluster that output i belongs to, by halving.  word(w): word w of the table (up to 2^30 clusters, so w takes 64 bits); cluster
// 0's first output is 0.
template <typename Word>
GROW_BOTH inline int grow_cluster_of(Word word, int clusters, int64_t i)
{
    int low = 0, high = clusters - 1;
    while (low < high)
    {
        const int middle = low + (high - low + 1) / 2;
        if (word(GROW_TABLE_ROW * static_cast<int64_t>(middle)) <= i)
            low = middle;
        else
            high = middle - 1;
    }
    return low;
}
