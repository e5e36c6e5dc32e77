// Inverted index ("lists"): for every target position of a cloud, the entries that refer to
// it.  The backward passes that would otherwise scatter with float atomics (three_interpolate,
// grouping) gather along these lists instead.
//
// Layout, made for the walk of gather.hip (one wavefront per span of targets, 64 lanes that
// each add up a run of consecutive entries):
//   * The index entries of one cloud - or of one column part of it - are sorted by target.
//     A target nobody refers to gets one empty entry, so every target owns at least one entry
//     and the last entry of every list is marked: a walker that counts these marks knows which
//     target a sum belongs to, and every output element gets written (no zero fill).
//   * The targets are cut into L_SPANS spans of equal size; span s is walked by wavefront s.
//     Its sorted entries, `len` of them, are dealt to the 64 lanes in runs of
//     c = ceil(len / 64) consecutive entries: the entry of rank q goes to lane q / c as its
//     step q % c, stored at  base + (q % c) * 64 + q / c  - one step of all lanes is one
//     contiguous row of 64 entries; the places behind rank len - 1 hold entries that refer to
//     nothing.  Runs are equally long whatever the lists look like; a list may cross from one
//     lane's run into the next, which the walker resolves with one scan over the lanes at the end.
//   * regions[cloud_part][span]              (base, len, c, 0)
//     first_target[cloud_part][span][lane]   target of the lane's first entry
//     entries[cloud_part][capacity]
#pragma once

#include "tpk_device.h"

namespace {

constexpr int G_THREADS = 1024;

template <typename Kernel>
int allow_lds(Kernel kernel, size_t bytes)
{
    return tpk_allow_lds(reinterpret_cast<const void*>(kernel), bytes);
}

// One entry of a target's list: the column that references it and the weight it carries.  The
// column is stored the way the walker uses it: as the byte offset of that column's value in a
// staged row, column * 4.  Bit 31 marks the last entry of a list.  An entry that refers to
// nothing (the entry of an empty list, the entries that fill a span's last row) carries
// L_NOTHING, an offset beyond the LDS: reads there return zero on gfx950, as on every GCN / CDNA
// part, and never fault.
template <bool WEIGHTED>
struct ListEntry;
template <>
struct ListEntry<true>
{
    int j;
    float w;
};
template <>
struct ListEntry<false>
{
    int j;
};
constexpr int L_LAST = static_cast<int>(0x80000000u);
constexpr int L_NOTHING = 0x7ffffffc - 3 * 0x40000; // (rows further down, at multiples of the row size, stay out of range too)
// The walker multiplies the offset by the number of rows it stages side by side (1, 2 or 4), in 32 bits: every
// product has to stay beyond the LDS.
static_assert(static_cast<uint32_t>(L_NOTHING) * 1u >= TPK_LDS_BYTES && static_cast<uint32_t>(L_NOTHING) * 2u >= TPK_LDS_BYTES &&
                  static_cast<uint32_t>(L_NOTHING) * 4u >= TPK_LDS_BYTES,
              "an entry that refers to nothing must read beyond the LDS whatever the number of staged rows");

constexpr int L_SPANS = G_THREADS / TPK_WAVE; // spans of targets per cloud: one per wavefront of the walker
constexpr int L_MAX_SPAN = 15360;             // targets of a span: their bookkeeping (2 ints each) fits in LDS
constexpr int L_REGION_GAP = 128;             // entry slots between the regions of consecutive spans
template <int K>
constexpr int L_MAX_PART = K * 32768; // index entries of a part: columns that the walker takes whole
constexpr int L_QUEUE = 512; // entries inside the span that a wavefront notes in LDS
constexpr int L_ENTRY_BITS = 17, L_TARGET_BITS = 14; // ... as the number of the entry and the target's place in the span
static_assert(L_MAX_PART<3> <= 1 << L_ENTRY_BITS && L_MAX_SPAN <= 1 << L_TARGET_BITS && L_ENTRY_BITS + L_TARGET_BITS <= 32, "a note's bits");

template <bool WEIGHTED>
struct Lists
{
    int4* regions;
    int* first_target;
    ListEntry<WEIGHTED>* entries;
    int64_t capacity; // entry slots per cloud part
};

inline size_t list_align(size_t v)
{
    return (v + 255) & ~static_cast<size_t>(255);
}
// Entry slots of one cloud part with m targets and `total` index entries: every entry, one
// empty entry per target at most, the rounding of every region to whole rows of 64 and the gaps.
inline int64_t list_capacity(int m, int64_t total)
{
    return ((total + m + 63) & ~static_cast<int64_t>(63)) + static_cast<int64_t>(L_REGION_GAP) * L_SPANS + 64;
}
// Workspace bytes of the lists of `clouds` cloud parts with m targets and `total` index entries each.
template <bool WEIGHTED>
size_t lists_bytes(int64_t clouds, int m, int64_t total)
{
    const size_t c = static_cast<size_t>(clouds);
    return list_align(c * L_SPANS * sizeof(int4)) + list_align(c * L_SPANS * TPK_WAVE * sizeof(int)) +
           list_align(c * static_cast<size_t>(list_capacity(m, total)) * sizeof(ListEntry<WEIGHTED>));
}
template <bool WEIGHTED>
Lists<WEIGHTED> lists_at(void* workspace, int64_t clouds, int m, int64_t total)
{
    const size_t c = static_cast<size_t>(clouds);
    char* p = static_cast<char*>(workspace);
    Lists<WEIGHTED> l;
    l.regions = reinterpret_cast<int4*>(p);
    p += list_align(c * L_SPANS * sizeof(int4));
    l.first_target = reinterpret_cast<int*>(p);
    p += list_align(c * L_SPANS * TPK_WAVE * sizeof(int));
    l.entries = reinterpret_cast<ListEntry<WEIGHTED>*>(p);
    l.capacity = list_capacity(m, total);
    return l;
}

// The job of inverting the index of `clouds` clouds: the `cloud_total` index entries of a cloud
// (K per column) are cut into `parts` runs of `part_total` entries (a multiple of K; the last may
// be shorter), and every (cloud, part) gets lists of its own, stored as cloud part number
// cloud * parts + part; the columns in its entries count from the first column of the part.
template <bool WEIGHTED, typename IdxT>
struct ListJob
{
    int m, cloud_total, parts, part_total, span, workgroups;
    const IdxT* idx;
    const float* weight;
    Lists<WEIGHTED> lists;
};

// A workgroup's share: workgroup `block` of clouds * parts * L_SPANS, (cloud part, s), builds the lists of the targets
// [s * span, (s + 1) * span).  It reads every index entry of its part and notes those inside its span in LDS, counts them
// with LDS integer atomics and those below the span - their number fixes where its region starts, so
// no workgroup waits for another -, prefix-sums the list lengths (empty lists count as one
// entry) and places its entries in a second pass over the notes.  Index values outside [0, m) are dropped.
// LDS (`counters`): list_lds_bytes().
//
// Where more entries of a wavefront crowd into the span than it can note, it counts the rest as it reads them and reads those once
// more to place them.  The index of a padded ball query is like that: every empty slot repeats the lowest row of its ball, and the
// first span of a cloud gets three to six times its share.  16 clouds, 32768 entries on 4096 targets, balls of 2, 4, 8, 16 points in
// 32 slots 13, 16, 20, 21 us (even 12; with the whole part read twice more 21, 25, 30, 31; with all values in registers 15, 18, 23,
// 24), 4 x 90000 weighted entries, Zipf exponent 0.7 and 1, 22 and 35 (42 and 45; 30 and 34).
//
// Bound by the instructions of the first pass, as all but one entry in L_SPANS are read in vain, and by the stores of single
// entries.  A part's workgroups run on one die, which reads its index once, where the parts are a multiple of eight, otherwise some
// on a second one (a single part: on all).  Keeping every index value in registers for a second pass over all of them took
// 12900 + 15300 clocks for the two passes at 16384 x 3 entries (124 registers; 16 clouds, 2048 targets 18.6 us), the notes take
// 13300 + 6800 (38 registers, 14.9 us); a bit per entry instead of a note, and the index read again, 11300 + 20100.
template <int K, bool WEIGHTED, typename IdxT>
__device__ __forceinline__ void build_lists(const ListJob<WEIGHTED, IdxT>& job, int block, int* counters)
{
    const int m = job.m, cloud_total = job.cloud_total, parts = job.parts, part_total = job.part_total, span = job.span;
    const IdxT* __restrict__ idx = job.idx;
    const float* __restrict__ weight = job.weight;

    // counters: [span] list lengths, in the second pass the places still free
    int* const ends = counters + span;          // [span] rank behind every list's last entry inside the span
    int* const scan = ends + span;              // [G_THREADS / 64], then below_total
    int* const below_total = scan + G_THREADS / TPK_WAVE;
    const int tid = threadIdx.x;
    const int lane = tid & (TPK_WAVE - 1);
    const int wave = tid / TPK_WAVE;
    block = static_cast<int>(xcd_local_block(static_cast<unsigned>(block), static_cast<unsigned>(job.workgroups)));
    const int cloud_part = block / L_SPANS;
    const int s = block - cloud_part * L_SPANS;
    const int part = cloud_part % parts;
    const int total = min(part_total, cloud_total - part * part_total);
    const int i0 = min(s * span, m);
    const int i1 = min(i0 + span, m);
    const int width = i1 - i0;
    const int64_t first_entry = static_cast<int64_t>(cloud_part / parts) * cloud_total + static_cast<int64_t>(part) * part_total;
    idx += first_entry;
    if (WEIGHTED)
        weight += first_entry;

    for (int t = tid; t < width; t += G_THREADS)
        counters[t] = 0;
    if (tid == 0)
        *below_total = 0;
    __syncthreads();

    // First pass.  Entry e of the part is read by thread e % G_THREADS in its round e / G_THREADS.  A wavefront notes those inside
    // the span in its queue, in order.
    // (a value that does not fit 32 bits is outside every cloud, like an entry behind the part's last)
    constexpr unsigned OUTSIDE = ~0u;
    auto index_value = [](IdxT v) {
        if constexpr (sizeof(IdxT) == 8)
            return (static_cast<unsigned long long>(v) >> 32) != 0 ? OUTSIDE : static_cast<unsigned>(v);
        else
            return static_cast<unsigned>(v);
    };
    constexpr int BATCH = 8; // rounds read together, while the batch before them is looked at
    auto read_batch = [&](int first, IdxT* v) {
        if (first + BATCH * G_THREADS <= total)
        {
#pragma unroll
            for (int u = 0; u < BATCH; ++u)
                v[u] = (idx + (first + u * G_THREADS))[static_cast<unsigned>(tid)];
        }
        else
        {
#pragma unroll
            for (int u = 0; u < BATCH; ++u)
            {
                const int e = first + u * G_THREADS + tid;
                v[u] = idx[min(e, total - 1)];
                v[u] = e < total ? v[u] : static_cast<IdxT>(-1);
            }
        }
    };
    auto read_entries = [&](int from, auto&& take) { // (first entry of the thread in the batch, the batch's values)
        IdxT v[BATCH], next[BATCH];
        if (from < total)
            read_batch(from, next);
        for (int first = from; first < total; first += BATCH * G_THREADS)
        {
#pragma unroll
            for (int u = 0; u < BATCH; ++u)
                v[u] = next[u];
            if (first + BATCH * G_THREADS < total)
                read_batch(first + BATCH * G_THREADS, next);
            take(first + tid, v);
        }
    };
    // (The values of a batch are counted per lane and their places in the queue follow from one prefix sum: with a ballot and
    // its prefix count per value the wavefronts spent their time between the vector and the scalar unit.)
    unsigned* const queue = reinterpret_cast<unsigned*>(below_total + 2) + wave * L_QUEUE;
    int below = 0, queued = 0; // of this thread: entries before the span; of its wavefront: entries noted
    int noted = total;         // the batches of the wavefront from this entry on are not noted, but counted at once
    read_entries(0, [&](int e, const IdxT* v) {
        unsigned t[BATCH];
        int own = 0;
#pragma unroll
        for (int u = 0; u < BATCH; ++u)
        {
            below += __builtin_sub_overflow(index_value(v[u]), static_cast<unsigned>(i0), &t[u]) ? 1 : 0;
            own += t[u] < static_cast<unsigned>(width) ? 1 : 0;
        }
        const int before = wave_exclusive_sum(own);
        const int all = __builtin_amdgcn_readlane(before + own, TPK_WAVE - 1);
        if (queued + all <= L_QUEUE && noted == total) // (wave-uniform)
        {
            unsigned* at = queue + queued + before;
#pragma unroll
            for (int u = 0; u < BATCH; ++u)
                if (t[u] < static_cast<unsigned>(width))
                    *at++ = t[u] << L_ENTRY_BITS | static_cast<unsigned>(e + u * G_THREADS);
            queued += all;
        }
        else
        {
            noted = min(noted, e - tid);
#pragma unroll
            for (int u = 0; u < BATCH; ++u)
                if (t[u] < static_cast<unsigned>(width))
                    atomicAdd(&counters[t[u]], 1);
        }
    });
    {
        const int below_before = wave_exclusive_sum(below);
        if (lane == TPK_WAVE - 1)
            atomicAdd(below_total, below_before + below);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); // (its own notes)
    for (int q = lane; q < queued; q += TPK_WAVE)
        atomicAdd(&counters[queue[q] >> L_ENTRY_BITS], 1);
    __syncthreads();

    // Prefix sum of the list lengths, an empty list counting as one entry (every thread owns a run of
    // `per` consecutive targets; sums inside a wavefront by DPP, across wavefronts through LDS).
    const int per = (width + G_THREADS - 1) / G_THREADS;
    const int lo = min(tid * per, width), hi = min(lo + per, width);
    int sum = 0;
    for (int t = lo; t < hi; ++t)
        sum += max(counters[t], 1);
    const int before_in_wave = wave_exclusive_sum(sum);
    if (lane == TPK_WAVE - 1)
        scan[wave] = before_in_wave + sum;
    __syncthreads();
    int run = before_in_wave, len = 0;
    for (int w = 0; w < G_THREADS / TPK_WAVE; ++w)
    {
        run += w < wave ? scan[w] : 0;
        len += scan[w];
    }
    // Where this span's region starts: behind all entries and all possible empty entries of the spans before it,
    // on a multiple of 64, with a gap that absorbs the rounding of the earlier regions to whole rows.
    const int base = ((*below_total + i0 + 63) & ~63) + L_REGION_GAP * s;
    const int c = (len + TPK_WAVE - 1) / TPK_WAVE; // steps of a lane; 0 for a span without targets
    ListEntry<WEIGHTED>* __restrict__ entries = job.lists.entries + static_cast<int64_t>(cloud_part) * job.lists.capacity;
    int* __restrict__ first_target = job.lists.first_target + (static_cast<int64_t>(cloud_part) * L_SPANS + s) * TPK_WAVE;
    if (tid == 0)
        job.lists.regions[static_cast<int64_t>(cloud_part) * L_SPANS + s] = make_int4(base, len, c, 0);
    // (rank -> lane and step: a division by c through the reciprocal in float, corrected; ranks stay below 2^24)
    const float per_c = c > 0 ? 1.0f / static_cast<float>(c) : 0.f;
    auto place = [&](int rank, int target, ListEntry<WEIGHTED> entry) {
        int ln = static_cast<int>(static_cast<float>(rank) * per_c);
        int step = rank - ln * c;
        if (step < 0)
        {
            --ln;
            step += c;
        }
        if (step >= c)
        {
            ++ln;
            step -= c;
        }
        entries[base + step * TPK_WAVE + ln] = entry;
        if (step == 0)
            first_target[ln] = target;
    };
    for (int t = lo; t < hi; ++t)
    {
        const int n = counters[t];
        run += max(n, 1);
        ends[t] = run;
        if (n == 0) // the empty list's entry: refers to nothing, ends the list
        {
            ListEntry<WEIGHTED> entry;
            entry.j = L_NOTHING | L_LAST;
            if constexpr (WEIGHTED)
                entry.w = 0.f;
            place(run - 1, i0 + t, entry);
        }
    }
    // the places behind the span's last entry, up to the end of the lanes' runs: entries that refer to nothing
    for (int rank = len + tid; rank < c * TPK_WAVE; rank += G_THREADS)
    {
        ListEntry<WEIGHTED> entry;
        entry.j = L_NOTHING;
        if constexpr (WEIGHTED)
            entry.w = 0.f;
        place(rank, 0, entry);
    }
    __syncthreads();

    // Second pass: an entry takes the next free place of its list, front to back.  `counters` holds the number of places
    // still free, so the entry that takes the last one knows that it ends the list.
    auto place_entry = [&](int e, unsigned t, [[maybe_unused]] float w) {
        const int free_places = atomicSub(&counters[t], 1);
        ListEntry<WEIGHTED> entry;
        entry.j = ((e / K) * 4) | (free_places == 1 ? L_LAST : 0);
        if constexpr (WEIGHTED)
            entry.w = w;
        place(ends[t] - free_places, i0 + static_cast<int>(t), entry);
    };
    {
        constexpr int AT_ONCE = 4;
        for (int first = lane; first < queued; first += AT_ONCE * TPK_WAVE)
        {
            unsigned note[AT_ONCE];
            [[maybe_unused]] float w[AT_ONCE];
#pragma unroll
            for (int u = 0; u < AT_ONCE; ++u)
            {
                note[u] = queue[min(first + u * TPK_WAVE, queued - 1)];
                if constexpr (WEIGHTED)
                    w[u] = weight[note[u] & ((1u << L_ENTRY_BITS) - 1)];
            }
#pragma unroll
            for (int u = 0; u < AT_ONCE; ++u)
                if (first + u * TPK_WAVE < queued)
                {
                    float own = 0.f;
                    if constexpr (WEIGHTED)
                        own = w[u];
                    place_entry(static_cast<int>(note[u] & ((1u << L_ENTRY_BITS) - 1)), note[u] >> L_ENTRY_BITS, own);
                }
        }
    }
    // (what was not noted is read once more)
    if (noted < total)
        read_entries(noted, [&](int e, const IdxT* v) {
#pragma unroll
            for (int u = 0; u < BATCH; ++u)
            {
                const unsigned t = index_value(v[u]) - static_cast<unsigned>(i0);
                if (t < static_cast<unsigned>(width))
                {
                    float own = 0.f;
                    if constexpr (WEIGHTED)
                        own = weight[e + u * G_THREADS];
                    place_entry(e + u * G_THREADS, t, own);
                }
            }
        });
}

template <int K, bool WEIGHTED, typename IdxT>
__global__ __launch_bounds__(G_THREADS, 8) void build_lists_kernel(ListJob<WEIGHTED, IdxT> job)
{
    extern __shared__ int list_memory[];
    build_lists<K, WEIGHTED, IdxT>(job, static_cast<int>(blockIdx.x), list_memory);
}

// Bytes of LDS a workgroup of the builder takes for spans of `span` targets.
inline size_t list_lds_bytes(int span)
{
    return (2 * static_cast<size_t>(span) + G_THREADS / TPK_WAVE + 2 + G_THREADS / TPK_WAVE * L_QUEUE) * sizeof(int);
}

// Describes the job of building the lists of `clouds` clouds of `m` targets and `cloud_total`
// index entries each, in parts of `part_total` entries (`lists` sized for clouds * parts cloud
// parts of part_total entries).  Returns TPK_ERR_UNSUPPORTED when a span of targets would not
// fit in LDS or entry positions would not fit an int.
template <int K, bool WEIGHTED, typename IdxT>
int make_list_job(int clouds, int m, int64_t cloud_total, int64_t part_total, const IdxT* idx, const float* weight,
                  const Lists<WEIGHTED>& lists, ListJob<WEIGHTED, IdxT>* job)
{
    *job = ListJob<WEIGHTED, IdxT>{};
    if (clouds <= 0 || m <= 0 || cloud_total <= 0)
        return TPK_OK; // nothing to build: no workgroups
    if (part_total <= 0 || part_total % K != 0)
        return TPK_ERR_INVALID_ARG;
    const int64_t parts = tpk_ceil_div(cloud_total, part_total);
    const int64_t span = tpk_ceil_div(m, L_SPANS);
    static_assert(L_MAX_PART<K> + L_MAX_SPAN < (1 << 24), "ranks inside a span: the builder divides them in float");
    if (span > L_MAX_SPAN || part_total > L_MAX_PART<K> || list_capacity(m, part_total) * 8 > 0x7fffffffLL ||
        cloud_total > 0x7fffffffLL || clouds * parts * L_SPANS > 0x7fffffffLL)
        return TPK_ERR_UNSUPPORTED;
    job->m = m;
    job->cloud_total = static_cast<int>(cloud_total);
    job->parts = static_cast<int>(parts);
    job->part_total = static_cast<int>(part_total);
    job->span = static_cast<int>(span);
    job->workgroups = static_cast<int>(clouds * parts * L_SPANS);
    job->idx = idx;
    job->weight = weight;
    job->lists = lists;
    return TPK_OK;
}

template <int K, bool WEIGHTED, typename IdxT>
int launch_build_lists(int clouds, int m, int64_t cloud_total, int64_t part_total, const IdxT* idx,
                       const float* weight, const Lists<WEIGHTED>& lists, hipStream_t s)
{
    ListJob<WEIGHTED, IdxT> job;
    const int st = make_list_job<K, WEIGHTED, IdxT>(clouds, m, cloud_total, part_total, idx, weight, lists, &job);
    if (st != TPK_OK || job.workgroups == 0)
        return st;
    const size_t lds = list_lds_bytes(job.span);
    auto build = build_lists_kernel<K, WEIGHTED, IdxT>;
    const int allowed = allow_lds(build, lds);
    if (allowed != TPK_OK)
        return allowed;
    hipLaunchKernelGGL(build, dim3(static_cast<unsigned>(job.workgroups)), dim3(G_THREADS), lds, s, job);
    return tpk_launch_status();
}

} // namespace
