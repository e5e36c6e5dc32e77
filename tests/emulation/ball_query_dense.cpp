// The dense ball query of clouds above 8192 points, its kernels' sources run on the host (hip/hip_runtime.h), every buffer and the
// LDS right in front of a page that cannot be touched: ball_query_dense <clouds> <points> <queries> <nsample> <radius> <own>.
// The queries are each cloud's first points (own: the support itself, same buffer).
#include "nn_grid.cpp"

#include "guarded.h"

int main(int argc, char** argv)
{
    if (argc != 7)
        return 1;
    const int b = atoi(argv[1]), n = atoi(argv[2]), m = atoi(argv[3]), nsample = atoi(argv[4]);
    const float radius = static_cast<float>(atof(argv[5]));
    const bool own = atoi(argv[6]) != 0;
    report_accesses_out_of_bounds();
    const size_t points = static_cast<size_t>(b) * n, queries = static_cast<size_t>(b) * m;
    float* xyz = reinterpret_cast<float*>(guarded(points * 12, "the points"));
    std::mt19937 random(1);
    std::uniform_real_distribution<float> even(0.f, 1.f);
    for (size_t i = 0; i < points * 3; ++i)
        xyz[i] = even(random);
    float* query = xyz;
    if (!own)
    {
        query = reinterpret_cast<float*>(guarded(queries * 12, "the queries"));
        for (int c = 0; c < b; ++c)
            memcpy(query + static_cast<size_t>(c) * m * 3, xyz + static_cast<size_t>(c) * n * 3, static_cast<size_t>(m) * 12);
    }
    int64_t* idx = reinterpret_cast<int64_t*>(guarded(queries * nsample * 8, "the indices"));
    float* dist = reinterpret_cast<float*>(guarded(queries * nsample * 4, "the distances"));
    const size_t bytes = tpk_grid_ball_query_dense_workspace_bytes(b, n, m, nsample);
    if (bytes == 0 || bytes % 256 != 0)
        return 1;
    char* workspace = guarded((bytes + 4095) / 4096 * 4096, "the workspace"); // (its size is a multiple of 256, its start of a page)
    const int status = tpk_grid_ball_query_dense(b, n, m, radius, radius * radius, nsample, query, xyz, idx, dist, workspace, bytes, nullptr);
    if (status != TPK_OK)
        return 1;

    long wrong = 0;
    std::vector<int64_t> hits;
    for (size_t q = 0; q < queries; q += queries / 400 + 1)
    {
        const float* at = query + q * 3;
        const float* cloud = xyz + q / m * n * 3;
        hits.clear();
        for (int j = 0; j < n && static_cast<int>(hits.size()) < nsample; ++j)
            if (tpk_dist2(at[0], at[1], at[2], cloud[j * 3], cloud[j * 3 + 1], cloud[j * 3 + 2]) < radius * radius)
                hits.push_back(j);
        for (int s = 0; s < nsample; ++s)
            wrong += idx[q * nsample + s] != (s < static_cast<int>(hits.size()) ? hits[s] : hits.empty() ? 0 : hits[0]);
    }
    printf("%ld wrong\n", wrong);
    return wrong == 0 ? 0 : 5;
}
