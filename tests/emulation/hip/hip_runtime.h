// What the kernel sources need of the HIP runtime, on the host: a workgroup's lanes are fibres of one thread, a wavefront's
// exchanges (ballots, DPP, lane reads) and the barrier wait until all of its lanes have arrived.  One workgroup runs after the other.
// An exchange that only some of a wavefront's lanes reach, where the hardware would go on with those, ends the program here:
// the sources this is made for have none.
#pragma once

#include <climits>
#include <cmath>
#include <csetjmp>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>

#include <ucontext.h>

#define __device__
#define __host__
#define __global__
#define __forceinline__ inline
#define __launch_bounds__(...)
#define __shared__ static
#define __constant__
#define __align__(n) __attribute__((aligned(n)))

struct alignas(16) float4 { float x, y, z, w; };
struct alignas(16) int4 { int x, y, z, w; };
struct alignas(8) float2 { float x, y; };
struct alignas(8) int2 { int x, y; };
struct float3 { float x, y, z; };
struct dim3
{
    unsigned x, y, z;
    dim3(unsigned x_ = 1, unsigned y_ = 1, unsigned z_ = 1) : x(x_), y(y_), z(z_) {}
};
inline float4 make_float4(float x, float y, float z, float w) { return {x, y, z, w}; }
inline int4 make_int4(int x, int y, int z, int w) { return {x, y, z, w}; }
inline int2 make_int2(int x, int y) { return {x, y}; }

// ---- host side
typedef void* hipStream_t;
typedef int hipError_t;
enum { hipSuccess = 0 };
enum { hipFuncAttributeMaxDynamicSharedMemorySize };
enum { hipHostMallocDefault, hipMemcpyDeviceToHost };
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipGetDevice(int* device) { return *device = 0, hipSuccess; }
inline hipError_t hipFuncSetAttribute(const void*, int, int) { return hipSuccess; }
inline hipError_t hipHostMalloc(void** p, size_t bytes, int) { return *p = malloc(bytes), hipSuccess; }
inline hipError_t hipMemcpyAsync(void* to, const void* from, size_t bytes, int, hipStream_t) { return memcpy(to, from, bytes), hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }

// ---- fibres
namespace emulation {
constexpr int WAVE = 64, MOST_LANES = 1024;
struct Fibre
{
    jmp_buf where;
    ucontext_t start;
    char* stack;
    bool started, done;
};
struct Wave
{
    uint64_t offered[WAVE], seen[2][WAVE];
    int arrived, live;
    unsigned turn;
};
inline Fibre fibres[MOST_LANES];
inline Wave waves[MOST_LANES / WAVE];
inline jmp_buf scheduler;
inline dim3 block, grid;
inline int now, at_barrier, live;
inline unsigned barrier_turn;
inline long steps; // arrivals and ends: what tells a workgroup at work from one that waits for good
inline char* lds;  // the launch's dynamic LDS
inline std::function<void()> kernel;

[[noreturn]] inline void fail(const char* what)
{
    fprintf(stderr, "%s (workgroup %u, lane %d)\n", what, block.x, now);
    exit(2);
}
inline void yield()
{
    const int me = now;
    if (_setjmp(fibres[me].where) == 0)
        _longjmp(scheduler, 1);
    now = me;
}
inline void run_lane()
{
    kernel();
    Wave& wave = waves[now / WAVE];
    fibres[now].done = true;
    ++steps;
    --live;
    if (--wave.live > 0 && wave.arrived > 0)
        fail("a lane has ended while others of its wavefront exchange");
    _longjmp(scheduler, 1);
}
// Every lane's value (valid until the wavefront's next exchange but one).
inline const uint64_t* exchange(uint64_t value)
{
    Wave& wave = waves[now / WAVE];
    const unsigned turn = wave.turn;
    wave.offered[now % WAVE] = value;
    ++steps;
    if (++wave.arrived == wave.live)
    {
        for (int i = 0; i < WAVE; ++i) // (lanes that have ended by now offer nothing; others may end before all have looked)
            wave.seen[turn & 1][i] = fibres[now / WAVE * WAVE + i].done ? 0 : wave.offered[i];
        wave.arrived = 0;
        ++wave.turn;
    }
    else
        while (wave.turn == turn)
            yield();
    return wave.seen[turn & 1];
}
template <typename T>
inline T exchanged(T value, int from)
{
    uint64_t bits = 0;
    memcpy(&bits, &value, sizeof value);
    bits = exchange(bits)[from];
    memcpy(&value, &bits, sizeof value);
    return value;
}
inline int lane() { return now % WAVE; }
inline void launch(dim3 blocks, dim3 threads, size_t lds_bytes, std::function<void()> body)
{
    static char* stacks = static_cast<char*>(malloc(static_cast<size_t>(MOST_LANES) << 16));
    extern char* dynamic_lds(size_t bytes);
    grid = blocks;
    kernel = std::move(body);
    lds = dynamic_lds(lds_bytes);
    const int lanes = static_cast<int>(threads.x);
    static ucontext_t nowhere;
    for (unsigned b = 0; b < blocks.x; ++b)
    {
        block.x = b;
        live = lanes;
        at_barrier = 0;
        for (int w = 0; w < lanes / WAVE; ++w)
            waves[w].arrived = 0, waves[w].live = WAVE;
        for (int i = 0; i < lanes; ++i)
        {
            fibres[i].started = fibres[i].done = false;
            fibres[i].stack = stacks + (static_cast<size_t>(i) << 16);
        }
        while (live > 0)
        {
            const long before = steps;
            for (volatile int i = 0; i < lanes; ++i)
                if (!fibres[i].done && _setjmp(scheduler) == 0)
                {
                    now = i;
                    Fibre& f = fibres[i];
                    if (f.started)
                        _longjmp(f.where, 1);
                    f.started = true;
                    getcontext(&f.start);
                    f.start.uc_stack.ss_sp = f.stack;
                    f.start.uc_stack.ss_size = 1 << 16;
                    f.start.uc_link = &nowhere;
                    makecontext(&f.start, run_lane, 0);
                    setcontext(&f.start);
                }
            if (live > 0 && steps == before)
                fail("the workgroup waits for lanes that never arrive");
        }
    }
}
} // namespace emulation

struct EmulatedLane
{
    operator unsigned() const { return static_cast<unsigned>(emulation::now); }
};
struct EmulatedThread
{
    EmulatedLane x;
};
inline EmulatedThread threadIdx;
#define blockIdx emulation::block
#define gridDim emulation::grid
#define hipLaunchKernelGGL(k, blocks, threads, bytes, stream, ...) emulation::launch(blocks, threads, bytes, [=] { (k)(__VA_ARGS__); })

// ---- device side
inline int min(int a, int b) { return a < b ? a : b; }
inline int max(int a, int b) { return a > b ? a : b; }
inline unsigned min(unsigned a, unsigned b) { return a < b ? a : b; }
inline unsigned max(unsigned a, unsigned b) { return a > b ? a : b; }
inline float __int_as_float(int v) { return __builtin_bit_cast(float, v); }
inline int __float_as_int(float v) { return __builtin_bit_cast(int, v); }
inline void __syncthreads()
{
    const unsigned turn = emulation::barrier_turn;
    ++emulation::steps;
    if (++emulation::at_barrier == emulation::live)
    {
        emulation::at_barrier = 0;
        ++emulation::barrier_turn;
    }
    else
        while (emulation::barrier_turn == turn)
            emulation::yield();
}
inline int __syncthreads_or(int p)
{
    static int any;
    __syncthreads();
    any = 0;
    __syncthreads();
    any |= p;
    __syncthreads();
    return any;
}
inline unsigned long long __ballot(bool p)
{
    const uint64_t* all = emulation::exchange(p);
    unsigned long long mask = 0;
    for (int i = 0; i < emulation::WAVE; ++i)
        mask |= all[i] != 0 ? 1ull << i : 0ull;
    return mask;
}
template <typename T>
inline T __shfl(T v, int from, int = emulation::WAVE)
{
    return emulation::exchanged(v, from & 63);
}
template <typename T>
inline T __shfl_xor(T v, int mask, int = emulation::WAVE)
{
    return emulation::exchanged(v, emulation::lane() ^ mask);
}
template <typename T>
inline T __shfl_up(T v, unsigned by, int = emulation::WAVE)
{
    const int from = emulation::lane() - static_cast<int>(by);
    return emulation::exchanged(v, from < 0 ? emulation::lane() : from);
}
inline int __builtin_amdgcn_readlane(int v, int from)
{
    if (from < 0 || from > 63)
        emulation::fail("a lane that there is not is read");
    return emulation::exchanged(v, from);
}
inline int __builtin_amdgcn_readfirstlane(int v) { return emulation::exchanged(v, 0); }
inline int __builtin_amdgcn_ds_bpermute(int address, int v) { return emulation::exchanged(v, address >> 2 & 63); }
// (of the instruction's modes the one that masks the lane's number within its half of the wavefront)
#define __builtin_amdgcn_ds_swizzle(v, pattern) emulation::swizzled(v, pattern)
namespace emulation {
inline int swizzled(int v, int pattern)
{
    if (pattern & 0x8000)
        fail("a swizzle that is not emulated");
    const int in_half = lane() % 32;
    return exchanged(v, lane() - in_half + (((in_half & (pattern & 31)) | (pattern >> 5 & 31)) ^ (pattern >> 10 & 31)));
}
}
inline int __builtin_amdgcn_update_dpp(int old, int v, int control, int rows, int banks, bool zero)
{
    const int lane = emulation::lane(), row = lane / 16, in_row = lane % 16, by = control & 15;
    int from = -1;
    if (control < 0x100) // quad_perm
        from = (lane & ~3) + (control >> (lane & 3) * 2 & 3);
    else if (control >= 0x101 && control <= 0x10F) // row_shl
        from = in_row + by < 16 ? lane + by : -1;
    else if (control >= 0x111 && control <= 0x11F) // row_shr
        from = in_row - by >= 0 ? lane - by : -1;
    else if (control >= 0x121 && control <= 0x12F) // row_ror
        from = (lane & ~15) + (in_row + 16 - by) % 16;
    else if (control == 0x140) // row_mirror
        from = (lane & ~15) + 15 - in_row;
    else if (control == 0x141) // row_half_mirror
        from = (lane & ~7) + 7 - lane % 8;
    else if (control == 0x142) // row_bcast:15
        from = row > 0 ? row * 16 - 1 : -1;
    else if (control == 0x143) // row_bcast:31
        from = row >= 2 ? 31 : -1;
    else
        emulation::fail("a DPP control that is not emulated");
    const int got = emulation::exchanged(v, from < 0 ? lane : from);
    return (rows >> row & 1) == 0 || (banks >> in_row / 4 & 1) == 0 ? old : from >= 0 ? got : zero ? 0 : old;
}
// (a fence is where other lanes' accesses to LDS are waited for)
#define __builtin_amdgcn_fence(...) static_cast<void>(emulation::exchange(0))
#define __builtin_amdgcn_s_barrier() __syncthreads()
#define __builtin_amdgcn_sched_barrier(mask) static_cast<void>(0)
#define __builtin_amdgcn_s_waitcnt(x) static_cast<void>(0)
inline float __builtin_amdgcn_rcpf(float v) { return 1.0f / v; }
inline float __builtin_amdgcn_fmed3f(float a, float b, float c) { return fmaxf(fminf(a, b), fminf(fmaxf(a, b), c)); }
// A product of nought and infinity is a NaN of either sign, as the hardware likes: here of the one that orders above everything as an integer.
namespace emulation {
inline float fused(float a, float b, float c)
{
    const float v = fmaf(a, b, c);
    return v != v ? __builtin_nanf("") : v;
}
// Halves, rounded to nearest even, those below the normal range kept.  (The sources' vectors of them become these.)
struct Half
{
    uint16_t bits;
    Half() = default;
    Half(float v)
    {
        const double size = fabs(static_cast<double>(v));
        int exponent = -14;
        if (size >= 0x1p-14 && size < 65536.0)
            exponent = ilogb(size);
        const double unit = ldexp(1.0, exponent - 10), rounded = nearbyint(size / unit);
        int magnitude = 0x7C00;
        if (size < 65520.0)
            magnitude = static_cast<int>(rounded) + (exponent + 14) * 1024; // (a carry out of the mantissa is the next exponent)
        bits = static_cast<uint16_t>(v != v ? 0x7E00 : magnitude | (std::signbit(v) ? 0x8000 : 0));
    }
    operator float() const
    {
        const int exponent = bits >> 10 & 31, mantissa = bits & 1023;
        const double size = exponent == 31 ? (mantissa ? NAN : INFINITY)
                            : exponent == 0 ? mantissa * 0x1p-24 : ldexp(1024 + mantissa, exponent - 25);
        return static_cast<float>(bits >> 15 ? -size : size);
    }
};
template <int N>
struct Halves
{
    Half v[N];
    Half operator[](int i) const { return v[i]; }
};
// How far a matrix product may be from the sum of its products, in units of the sum of their magnitudes.
inline double product_error;
inline uint64_t product_noise = 1;
} // namespace emulation
#define __builtin_fmaf emulation::fused
#define _Float16 emulation::Half
// Lane l of the operands: row (column) l % 32, slots 8 (l / 32) .. 8 (l / 32) + 7; of the result: column l % 32, rows r % 4 + 8 (r / 4) + 4 (l / 32).
template <typename V, typename W>
inline W __builtin_amdgcn_mfma_f32_32x32x16_f16(const V& a, const V& b, W c, int, int, int)
{
    static float as_float[1 << 16];
    static bool made = false;
    for (int i = 0; i < (1 << 16) && !made; ++i)
    {
        const uint16_t bits = static_cast<uint16_t>(i);
        as_float[i] = __builtin_bit_cast(emulation::Half, bits);
    }
    made = true;
    uint16_t row[emulation::WAVE][8], own[16];
    for (int part = 0; part < 2; ++part)
    {
        uint64_t four;
        memcpy(&four, reinterpret_cast<const char*>(&a) + part * 8, 8);
        const uint64_t* all = emulation::exchange(four);
        for (int l = 0; l < emulation::WAVE; ++l)
            memcpy(&row[l][part * 4], &all[l], 8);
        memcpy(&four, reinterpret_cast<const char*>(&b) + part * 8, 8);
        all = emulation::exchange(four);
        for (int l = 0; l < 2; ++l)
            memcpy(&own[l * 8 + part * 4], &all[emulation::lane() % 32 + 32 * l], 8);
    }
    for (int r = 0; r < 16; ++r)
    {
        const int at = r % 4 + 8 * (r / 4) + 4 * (emulation::lane() / 32);
        double sum = c[r], magnitudes = 0.0;
        for (int k = 0; k < 16; ++k)
        {
            const double product = static_cast<double>(as_float[row[at + 32 * (k / 8)][k % 8]]) * as_float[own[k]];
            sum += product;
            magnitudes += fabs(product);
        }
        emulation::product_noise = emulation::product_noise * 6364136223846793005ull + 1442695040888963407ull;
        c[r] = static_cast<float>(sum + (emulation::product_noise >> 63 ? 1.0 : -1.0) * emulation::product_error * magnitudes);
    }
    return c;
}
struct EmulatedPair
{
    unsigned v[2];
    unsigned operator[](int i) const { return v[i]; }
};
// The lanes 32 .. 63 of the first and the lanes 0 .. 31 of the second change places.
inline EmulatedPair __builtin_amdgcn_permlane32_swap(unsigned first, unsigned second, bool, bool)
{
    const uint64_t* all = emulation::exchange(static_cast<uint64_t>(second) << 32 | first);
    const int lane = emulation::lane();
    return {{lane < 32 ? first : static_cast<unsigned>(all[lane - 32] >> 32), lane < 32 ? static_cast<unsigned>(all[lane + 32]) : second}};
}
inline unsigned __builtin_amdgcn_mbcnt_lo(unsigned mask, unsigned add)
{
    const int lane = emulation::lane();
    return add + __builtin_popcount(lane >= 32 ? mask : mask & ((1u << lane) - 1u));
}
inline unsigned __builtin_amdgcn_mbcnt_hi(unsigned mask, unsigned add)
{
    const int lane = emulation::lane() - 32;
    return add + __builtin_popcount(lane <= 0 ? 0u : mask & ((1u << lane) - 1u));
}
namespace emulation {
inline const char *watched_begin, *watched_end; // atomics in here are counted
inline long watched;
}
template <typename T, typename U>
inline T atomicAdd(T* p, U v)
{
    const char* const at = reinterpret_cast<const char*>(p);
    emulation::watched += at >= emulation::watched_begin && at < emulation::watched_end ? 1 : 0;
    const T old = *p;
    *p += v;
    return old;
}
inline unsigned atomicCAS(unsigned* p, unsigned compare, unsigned v)
{
    const unsigned old = *p;
    *p = old == compare ? v : old;
    return old;
}
inline int atomicMin(int* p, int v)
{
    const int old = *p;
    *p = min(old, v);
    return old;
}
inline int atomicMax(int* p, int v)
{
    const int old = *p;
    *p = max(old, v);
    return old;
}
