// Ids of the clouds that region growing searches (cluster.hip): plain arithmetic, tried on the host.
#pragma once

#include <cstdint>

// Whether label * span + sample fits an int64 for every label below `labels` and every sample below `span` (0: 2^64 of them).
constexpr bool region_ids_fit(uint32_t labels, uint64_t span)
{
    return span != 0 && span <= static_cast<uint64_t>(INT64_MAX) / labels;
}
