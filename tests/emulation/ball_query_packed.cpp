// The packed ball query over the table of cells, its kernels' sources run on the host (hip/hip_runtime.h), every buffer and the LDS
// right in front of a page that cannot be touched: ball_query_packed <clouds> <points> <queries> <nsample> <radius> <sorted>.
// Even clouds of width 1 (the last one of half the others' points), the queries among them.  Prints what its test looks at.
#include "ball_table.cpp"

#include "guarded.h"

#include <algorithm>
#include <set>

int main(int argc, char** argv)
{
    if (argc != 7)
        return 1;
    const int b = atoi(argv[1]), n = atoi(argv[2]), m = atoi(argv[3]), nsample = atoi(argv[4]);
    const float radius = static_cast<float>(atof(argv[5])), radius2 = radius * radius;
    const bool sorted = atoi(argv[6]) != 0;
    report_accesses_out_of_bounds();

    const size_t points = static_cast<size_t>(b) * n - (b > 1 ? n / 2 : 0), queries = static_cast<size_t>(m);
    float* x = reinterpret_cast<float*>(guarded(points * 12, "the points"));
    float* y = reinterpret_cast<float*>(guarded(queries * 12, "the queries"));
    int64_t* bx = reinterpret_cast<int64_t*>(guarded(points * 8, "the points' clouds"));
    int64_t* by = reinterpret_cast<int64_t*>(guarded(queries * 8, "the queries' clouds"));
    int64_t* idx = reinterpret_cast<int64_t*>(guarded(queries * nsample * 8, "the indices"));
    float* dist = reinterpret_cast<float*>(guarded(queries * nsample * 4, "the distances"));
    std::mt19937 random(1);
    std::uniform_real_distribution<float> even(0.f, 1.f);
    for (size_t i = 0; i < points; ++i)
    {
        bx[i] = static_cast<int64_t>(i) / n * 3 - 1;
        for (int a = 0; a < 3; ++a)
            x[i * 3 + a] = even(random);
    }
    for (size_t q = 0; q < queries; ++q)
    {
        const size_t i = q * points / queries; // (ascending, so the cloud ids are)
        by[q] = bx[i];
        for (int a = 0; a < 3; ++a)
            y[q * 3 + a] = x[i * 3 + a] + (q % 3 == 0 ? 0.01f : 0.f);
    }
    const size_t bytes = tpk_table_ball_query_workspace_bytes(points, queries, nsample);
    if (bytes == 0 || bytes % 256 != 0)
        return 1;
    char* workspace = guarded((bytes + 4095) / 4096 * 4096, "the workspace");
    emulation::watched_begin = workspace;
    emulation::watched_end = workspace + bytes;
    if (tpk_table_ball_query_partial(points, queries, radius, radius2, nsample, sorted, x, y, bx, by, idx, dist, workspace, bytes, nullptr) != TPK_OK)
        return 1;

    long wrong = 0;
    std::vector<std::pair<float, int64_t>> hits;
    for (size_t q = 0; q < queries; q += queries / 300 + 1)
    {
        hits.clear();
        for (size_t j = 0; j < points; ++j)
        {
            const float d = tpk_dist2(y[q * 3], y[q * 3 + 1], y[q * 3 + 2], x[j * 3], x[j * 3 + 1], x[j * 3 + 2]);
            if (bx[j] == by[q] && (sorted ? d < radius2 : d <= radius2))
                hits.push_back({d, static_cast<int64_t>(j)});
        }
        if (sorted)
            std::sort(hits.begin(), hits.end());
        for (int s = 0; s < nsample; ++s)
            wrong += idx[q * nsample + s] != (s < static_cast<int>(hits.size()) ? hits[s].second : -1) ||
                     dist[q * nsample + s] != (s < static_cast<int>(hits.size()) ? hits[s].first : -1.f);
    }
    // Buckets that hold points, and those that the consecutive points of a counting workgroup lie in, added up.  A small array's workgroup may send an
    // atomic per point where less than 4 of a wavefront's share the buckets of four others - 6 would in 43 buckets, a sixth of 256 points.
    CellScale scale;
    scale.reach = bt_reach(radius);
    scale.inverse_x = 1.0f / (BT_WIDTH_X * scale.reach);
    scale.inverse_yz = 1.0f / (BT_WIDTH_YZ * scale.reach);
    const TableLayout l = table_layout(points, queries);
    std::set<uint32_t> all, near;
    const size_t together = points < BT_COUNT_MEDIUM ? 256 : points < BT_COUNT_LARGE ? 512 : 1024;
    long by_group = 0;
    for (size_t i = 0; i < points; ++i)
    {
        const uint32_t bucket = bt_point_bucket(x[i * 3], x[i * 3 + 1], x[i * 3 + 2], bx[i], scale, static_cast<uint32_t>(l.buckets / BT_PARTS - 1));
        all.insert(bucket);
        near.insert(bucket);
        if (i % together == together - 1 || i + 1 == points)
        {
            const size_t in_group = i % together + 1;
            by_group += static_cast<long>(together == 256 && (in_group < 64 || near.size() * 6 > in_group) ? in_group : near.size());
            near.clear();
        }
    }
    printf("%ld wrong, %ld atomics, %ld buckets, %ld by group, %ld chunks\n", wrong, emulation::watched, static_cast<long>(all.size()), by_group,
           static_cast<long>(l.buckets / BT_CHUNK));
    return wrong == 0 ? 0 : 5;
}
