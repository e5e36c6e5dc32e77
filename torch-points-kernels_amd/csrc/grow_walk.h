// The reference's stack walk (torch_points_kernels/cluster.py:9-37) on host threads, over the compact pieces that
// tpk_grow_rows lays out: a piece is a block of rows whose entries are places inside the piece, so a core's cache holds
// what its walk touches, and pieces are independent of each other.
//
// A step takes a point off the stack and collects which of its row's entries are unseen in a bit mask, 16 entries at a
// time and without a branch; what is left to do per set bit happens once per point in all.  (Writing every entry to the
// stack and the cluster and moving their ends on only for unseen ones has no branch at all, but 48 stores a step:
// 14 ns per point against 7.)  The same step takes 0.8 us on the device.
#pragma once

#include <cstdint>
#include <cstring>
#include <vector>

namespace grow_walk {

// A cluster as the walk left it: the first place of its piece, its first point's place inside the piece, and where its members lie.
struct Cluster
{
    int64_t base, first, at, size;
};

struct Scratch
{
    std::vector<uint8_t> unseen;
    std::vector<uint32_t> stack, members;
};

// Bytes of pinned memory that hold rows at a time.  Such memory stays with the process (torch's pool of it gives nothing back), and
// the rows of millions of points are gigabytes.
constexpr int64_t MOST_STAGED = int64_t(256) << 20;
// The rows come in this many parts, so that the walk of the largest pieces, which lie first, begins when a fifth of them is there.
// Region growing of three rooms (9.4 MB of rows, 16 threads): 5 parts 752 - 782 us, 3 819, 8 787, 16 825 (an event costs the stream 6 us);
// all rows copied, then walked: 965; copied in 8 parts by the runtime, 32 us each: 938.
constexpr int64_t PARTS = 5, LEAST_PART = int64_t(1) << 20;

// Declared behind a host block that the device writes into by a kernel: whatever is thrown between begin() and end(), the wait for the
// device comes before the block goes.  (The pool that owns such blocks knows of copies into them, not of kernels.)
template <typename Wait>
class PendingWrites
{
public:
    explicit PendingWrites(const Wait& wait) : wait_(wait) {}
    PendingWrites(const PendingWrites&) = delete;
    PendingWrites& operator=(const PendingWrites&) = delete;
    ~PendingWrites()
    {
        if (!pending_)
            return;
        try
        {
            wait_();
        }
        catch (...) // (the device is gone, and with it whatever it was writing)
        {
        }
    }
    void begin() { pending_ = true; }
    void end() { pending_ = false; }

private:
    const Wait& wait_;
    bool pending_ = false;
};

// Walks one piece of `count` points.  Clusters of at least min_size members go to `found`, their members - as
// places inside the piece - to entries[at ...], which never takes more than the piece's own range (base and on).
template <typename E>
void walk_piece(const E* rows, int nsample, int64_t base, int64_t count, int64_t min_size,
                Scratch& scratch, E* entries, std::vector<Cluster>& found)
{
    // The rows have just arrived from the device and lie in no cache: read once in order they come at memory speed,
    // where the walk itself would wait for them one line at a time.
    const char* first_row = reinterpret_cast<const char*>(rows);
    uint64_t touched = 0;
    for (int64_t at = 0; at < count * nsample * static_cast<int64_t>(sizeof(E)); at += 64)
        touched += static_cast<unsigned char>(first_row[at]);
    asm volatile("" : : "r"(touched));
    scratch.unseen.assign(static_cast<size_t>(count), 1);
    if (scratch.stack.size() < static_cast<size_t>(count))
    {
        scratch.stack.resize(static_cast<size_t>(count));
        scratch.members.resize(static_cast<size_t>(count));
    }
    uint8_t* unseen = scratch.unseen.data();
    uint32_t* stack = scratch.stack.data();
    uint32_t* members = scratch.members.data();
    int64_t written = base;
    for (int64_t seed = 0; seed < count; ++seed)
    {
        if (!unseen[seed])
            continue;
        unseen[seed] = 0;
        members[0] = static_cast<uint32_t>(seed);
        stack[0] = static_cast<uint32_t>(seed);
        int64_t size = 1, top = 1;
        while (top > 0)
        {
            const E* row = rows + static_cast<int64_t>(stack[--top]) * nsample;
            for (int first = 0; first < nsample; first += 16)
            {
                uint32_t fresh = 0;
                if (first + 16 <= nsample)
                    for (int j = 0; j < 16; ++j)
                        fresh |= static_cast<uint32_t>(unseen[row[first + j]]) << j;
                else
                    for (int j = 0; first + j < nsample; ++j)
                        fresh |= static_cast<uint32_t>(unseen[row[first + j]]) << j;
                for (; fresh != 0; fresh &= fresh - 1)
                {
                    const uint32_t e = row[first + __builtin_ctz(fresh)];
                    if (!unseen[e])
                        continue; // (the row has named it twice)
                    unseen[e] = 0;
                    stack[top++] = e;
                    members[size++] = e;
                }
            }
        }
        if (size < min_size)
            continue;
        for (int64_t i = 0; i < size; ++i)
            entries[written + i] = static_cast<E>(members[i]);
        found.push_back(Cluster{base, seed, written, size});
        written += size;
    }
}

// Pieces begin .. end (returned) whose rows, row_bytes per point, take no more than `most` bytes together; at least one piece,
// whatever it takes.  starts: first place of every piece, then the total.
inline int64_t pieces_within(const int64_t* starts, int64_t pieces, int64_t begin, int64_t row_bytes, int64_t most)
{
    int64_t end = begin + 1;
    while (end < pieces && (starts[end + 1] - starts[begin]) <= most / row_bytes)
        ++end;
    return end;
}

} // namespace grow_walk
