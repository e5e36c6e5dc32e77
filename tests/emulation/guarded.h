// Buffers and an LDS that end right in front of a page that cannot be touched, for kernels' sources run on the host.
#pragma once

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

inline void report_accesses_out_of_bounds()
{
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

}
