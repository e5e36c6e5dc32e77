// The survivors of a k-nearest search by a wavefront (knn.hip).
#pragma once

#include "bracket.h"
#include "topk.h"

namespace {

// ---------------------------------------------------------------------------------------------
// Up to KNC_MAX_K neighbours, one wavefront per query.
//
// A wavefront offers itself 64 candidates at a time, one per lane, and keeps those that may belong to the answer - the
// survivors - as (squared distance, index) keys in its own stretch of LDS, in no order.  When the stretch would overflow
// it looks for a distance T with at least k and at most a few more survivors within it - a count of T is a comparison per
// slot and a population count, and one or two guesses suffice - and drops the rest; from then on candidates beyond T do
// not survive.  Only the 16 .. 40 survivors of the end are put in order: each lane counts the keys below its own, and the
// count is the key's place in the output.  Nothing is sorted and nothing is inserted into a list, which is what a lane
// that serves a query of its own spends its time on (a list of 32 in registers moves 64 of them per insertion, for the
// whole wavefront, and a wavefront of 64 queries leaves the chip idle where a call has few: k = 20 of 1646 points took
// 389 us).  The cost per query is 300 to 400 instructions whatever k.
// ---------------------------------------------------------------------------------------------
constexpr int KNC_MAX_K = 48;
constexpr int KNC_ROOM = 80;   // survivors held between two selections: one of 64, and some of the next step's
constexpr int KNC_MOST = 64;   // survivors of a selection at most: one per lane when they are ranked
constexpr int KNC_SPARE = 24;  // ... and beyond k at most

struct Survivors
{
    u64* keys; // [KNC_ROOM] in LDS, the wavefront's own
    int lane, k, count;
    float reach; // candidates beyond this squared distance do not matter
    float unit;  // about the squared distance within which one candidate lies, before reach is known

    __device__ __forceinline__ void clear()
    {
        count = 0;
        reach = __builtin_inff();
    }
    // Ratio of squared distances to a ratio of volumes.
    __device__ __forceinline__ float volume_ratio(float counts) const
    {
        return __builtin_amdgcn_exp2f(0.66667f * __builtin_amdgcn_logf(counts));
    }
    __device__ __forceinline__ int within(const float (&v)[3], float t) const
    {
        return __builtin_popcountll(__ballot(v[0] <= t)) + __builtin_popcountll(__ballot(v[1] <= t)) +
               __builtin_popcountll(__ballot(v[2] <= t));
    }
    // Reduces the survivors and this step's candidates (d; +inf for none) to between k and `most`, and `reach` with
    // them.  False when no distance separates so few (equal distances): the caller starts over another way.
    // The count within a distance grows about as the volume does: the first guess comes from `unit`, the later ones from
    // the last count.
    __device__ __forceinline__ bool select(float d, int i)
    {
        const float inf = __builtin_inff();
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        const u64 k0 = keys[lane], k1 = keys[min(lane + TPK_WAVE, KNC_ROOM - 1)];
        float v[3] = {lane < count ? __int_as_float(static_cast<int>(k0 >> 32)) : inf,
                      lane + TPK_WAVE < count ? __int_as_float(static_cast<int>(k1 >> 32)) : inf, d};
        const int most = min(k + KNC_SPARE, KNC_MOST);
        const float target = static_cast<float>(k + (most - k) / 2);
        Bracket bracket;
        float guess = reach; // (all of them, or +inf before the first selection)
        int in_guess = TPK_WAVE + count;
        if (reach == inf)
        {
            guess = tpk_read_lane(unit * volume_ratio(target), 0);
            in_guess = within(v, guess);
        }
        for (int tries = 0; in_guess < k || in_guess > most; ++tries)
        {
            if (tries >= BRACKET_TRIES)
                return false;
            const float estimate = guess * volume_ratio(target * __builtin_amdgcn_rcpf(fmaxf(static_cast<float>(in_guess), 0.5f)));
            guess = tpk_read_lane(bracket.next(guess, in_guess < k, estimate, tries), 0);
            in_guess = within(v, guess);
        }
        reach = guess;
        count = 0;
        put(v[0] <= reach, k0);
        put(v[1] <= reach, k1);
        put(v[2] <= reach, knn_key(d, i));
        return true;
    }
    __device__ __forceinline__ void put(bool in, u64 key)
    {
        const unsigned long long mask = __ballot(in);
        if (in)
            keys[count + static_cast<int>(tpk_prefix_count(mask))] = key;
        count += __builtin_popcountll(mask);
    }
    // One candidate per lane (in = false: none).
    __device__ __forceinline__ bool offer(bool in, float d, int i)
    {
        in = in && d <= reach && d < __builtin_inff();
        const int more = __builtin_popcountll(__ballot(in));
        if (more == 0)
            return true;
        if (count + more > KNC_ROOM)
            return select(in ? d : __builtin_inff(), i);
        put(in, knn_key(d, i));
        return true;
    }
    // Places of the lanes' survivors (at most KNC_MOST of them) among all; a lane without one: KNC_MOST or more.
    __device__ __forceinline__ int rank(u64& mine)
    {
        if (lane < 4) // (whole groups of four keys below)
            keys[min(count + lane, KNC_ROOM - 1)] = ~0ull;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        mine = lane < count ? keys[lane] : ~0ull;
        int place = 0;
        for (int j = 0; j < count; j += 4)
        {
#pragma unroll
            for (int u = 0; u < 4; ++u)
                place += keys[j + u] < mine ? 1 : 0;
        }
        return lane < count ? place : KNC_MOST;
    }
};

// The k nearest of all points by merging 64 sorted keys at a time: the queries no distance separates (many equal ones),
// or with fewer than k points at a finite distance.
template <typename Point>
__device__ __forceinline__ u64 nearest_by_merging(int m, int k, int lane, float qx, float qy, float qz, Point point TPK_WORK_PARAM)
{
    const u64 none = knn_key(__builtin_inff(), 0x7FFFFFFF); // (an entry left empty; a NaN distance is larger)
    u64 best = none, admit = none;
    for (int base = 0; base < m; base += TPK_WAVE)
    {
        const float4 p = point(min(base + lane, m - 1));
        TPK_WORK_ADD(1);
        u64 cand = knn_key(tpk_dist2(qx, qy, qz, p.x, p.y, p.z), __float_as_int(p.w));
        cand = base + lane < m && cand < admit ? cand : none;
        if (__ballot(cand != none) == 0)
            continue;
        cand = wave_sort_keys(cand, lane, true);
        best = wave_merge_ascending(best < cand ? best : cand, lane);
        admit = read_lane_key(best, k - 1);
    }
    return best;
}

} // namespace
