// Chamfer's search over cells, its kernels' sources run on the host (hip/hip_runtime.h), every buffer and the LDS right in front of a
// page that cannot be touched: chamfer <clouds> <n> <m> <kind> <seed>.  The matrix products are as far from the sums of their
// products as the sources assume at most.
#include "nn_grid.cpp"

#include "guarded.h"

int main(int argc, char** argv)
{
    if (argc != 6)
        return 1;
    const int b = atoi(argv[1]), n = atoi(argv[2]), m = atoi(argv[3]);
    const std::string kind = argv[4];
    report_accesses_out_of_bounds();
    emulation::product_error = 14 * 0x1p-24;
    std::mt19937 random(atoi(argv[5]));
    std::uniform_real_distribution<float> even(0.f, 1.f);
    std::normal_distribution<float> normal(0.f, 1.f);
    const int counts[2] = {n, m};
    float *xyz[2], *dist[2];
    int32_t* idx[2];
    for (int s = 0; s < 2; ++s)
    {
        const size_t points = static_cast<size_t>(b) * counts[s];
        xyz[s] = reinterpret_cast<float*>(guarded(points * 12, "the points"));
        dist[s] = reinterpret_cast<float*>(guarded(points * 4, "the distances"));
        idx[s] = reinterpret_cast<int32_t*>(guarded(points * 4, "the indices"));
        for (size_t i = 0; i < points; ++i)
        {
            float* const p = xyz[s] + i * 3;
            for (int a = 0; a < 3; ++a)
                p[a] = even(random);
            if (kind == "lattice")
                for (int a = 0; a < 3; ++a)
                    p[a] = floorf(p[a] * 6.f) / 6.f;
            else if (kind == "scan") // as a laser sees a floor
            {
                const float r = 1.5f * powf(50.f / 1.5f, p[0]), angle = 6.2832f * p[1];
                p[0] = r * cosf(angle), p[1] = r * sinf(angle), p[2] = 0.02f * p[2] - 1.7f;
            }
            else if (kind == "outliers" && even(random) < 0.05f)
                for (int a = 0; a < 3; ++a)
                    p[a] = 100.f * (p[a] - 0.5f);
            else if (kind == "scaled")
            {
                const float size = expf(-12.f * p[0]);
                for (int a = 0; a < 3; ++a)
                    p[a] = normal(random) * size;
            }
            else if (kind == "twins" && s == 1 && i % counts[1] >= static_cast<size_t>(counts[1] / 2)) // a few units in the last place from another point
                for (int a = 0; a < 3; ++a)
                    p[a] = p[a - 3 * (counts[1] / 2)] * (1.f + 0x1p-22f);
            else if (kind == "far" && s == 0)
                p[0] += 300.f;
            else if (kind == "not a number" && i % 15 == 3)
                p[1] = -__builtin_nanf("");
        }
    }
    const size_t bytes = tpk_grid_chamfer_workspace_bytes(b, n, m);
    if (bytes == 0 || bytes % 256 != 0)
        return 1;
    char* workspace = guarded((bytes + 4095) / 4096 * 4096, "the workspace"); // (its size is a multiple of 256, its start of a page)
    if (tpk_grid_chamfer_fwd(b, n, m, xyz[0], xyz[1], dist[0], dist[1], idx[0], idx[1], workspace, bytes, nullptr) != TPK_OK)
        return 1;

    long wrong = 0;
    for (int s = 0; s < 2; ++s)
        for (size_t q = 0; q < static_cast<size_t>(b) * counts[s]; ++q)
        {
            const float* const at = xyz[s] + q * 3;
            const float* const cloud = xyz[1 - s] + q / counts[s] * counts[1 - s] * 3;
            float best = INFINITY;
            int nearest = 0;
            for (int j = 0; j < counts[1 - s]; ++j)
            {
                const float d = tpk_dist2(cloud[j * 3], cloud[j * 3 + 1], cloud[j * 3 + 2], at[0], at[1], at[2]);
                if (d < best)
                    best = d, nearest = j;
            }
            wrong += dist[s][q] != best || idx[s][q] != nearest;
        }
    printf("%ld wrong\n", wrong);
    return wrong == 0 ? 0 : 5;
}
