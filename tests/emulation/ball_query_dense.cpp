// The dense ball query of clouds above 8192 points, its kernels' sources run on the host (hip/hip_runtime.h), every buffer and the
// LDS right in front of a page that cannot be touched: ball_query_dense <clouds> <points> <queries> <nsample> <radius> <own>.
// The queries are each cloud's first points (own: the support itself, same buffer).
#include "nn_grid.cpp"

#include <random>
#include <vector>

#include <signal.h>
#include <sys/mman.h>

namespace {

struct Region
{
    const char* name;
    char *begin, *end;
};
std::vector<Region> regions;

// `bytes` (of 4-byte words) whose end meets the page behind.
char* guarded(size_t bytes, const char* name)
{
    const size_t page = 4096, room = (bytes + page - 1) / page * page, guard = 64 * page;
    char* p = static_cast<char*>(mmap(nullptr, room + 2 * guard, PROT_NONE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0));
    if (p == MAP_FAILED || mprotect(p + guard, room, PROT_READ | PROT_WRITE) != 0)
        exit(4);
    char* begin = p + guard + room - bytes;
    regions.push_back({name, begin, begin + bytes});
    return begin;
}

void out_of_bounds(int, siginfo_t* info, void*)
{
    char* at = static_cast<char*>(info->si_addr);
    fprintf(stderr, "access out of bounds, workgroup %u, lane %d\n", emulation::block.x, emulation::now);
    for (const Region& r : regions)
        if (at >= r.begin - 65536 && at < r.end + 65536)
            fprintf(stderr, "  byte %ld of the %ld of %s\n", static_cast<long>(at - r.begin), static_cast<long>(r.end - r.begin), r.name);
    _exit(3);
}

} // namespace

namespace emulation {
char* dynamic_lds(size_t bytes)
{
    static char* const memory = guarded(TPK_LDS_BYTES, "the LDS");
    return memory + TPK_LDS_BYTES - (bytes + 15) / 16 * 16;
}
} // namespace emulation

int main(int argc, char** argv)
{
    if (argc != 7)
        return 1;
    const int b = atoi(argv[1]), n = atoi(argv[2]), m = atoi(argv[3]), nsample = atoi(argv[4]);
    const float radius = static_cast<float>(atof(argv[5]));
    const bool own = atoi(argv[6]) != 0;
    static char alternate[1 << 16];
    stack_t stack{};
    stack.ss_sp = alternate;
    stack.ss_size = sizeof alternate;
    sigaltstack(&stack, nullptr);
    struct sigaction action{};
    action.sa_sigaction = out_of_bounds;
    action.sa_flags = SA_SIGINFO | SA_ONSTACK;
    sigaction(SIGSEGV, &action, nullptr);
    sigaction(SIGBUS, &action, nullptr);

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
