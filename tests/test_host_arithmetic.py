"""Arithmetic the kernels share with the host (csrc headers without device code), compiled here with g++ and tried over
inputs a GPU test cannot afford to get wrong: what it returns sizes LDS and workspaces."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "torch-points-kernels_amd", "csrc")

SHIM = r"""
#include "arrivals.h"
#include "ball_table.h"
#include "bracket.h"
#include "cloud_ids.h"
#include "die_map.h"
#include "grid_shape.h"
#include "grow_table.h"
#include "grow_walk.h"
#include <cmath>
#include <atomic>
#include <chrono>
#include <ctime>
#include <stdexcept>
#include <thread>

// `threads` wait for parts that come `apart` seconds after each other; fails: the event that throws, -1 for none.  Returns the
// processor time the process took meanwhile; *right: how many threads got what they waited for, in time.
extern "C" double parts_waited_for(int threads, int parts, double apart, int fails, int* right)
{
    using Clock = std::chrono::steady_clock;
    struct Event
    {
        Clock::time_point at;
        bool throws;
        void synchronize()
        {
            std::this_thread::sleep_until(at);
            if (throws)
                throw std::runtime_error("event");
        }
    };
    const auto start = Clock::now();
    auto when = [&](int part) { return start + std::chrono::duration_cast<Clock::duration>(std::chrono::duration<double>(apart * (part + 1))); };
    Arrivals<Event> arrivals;
    for (int p = 0; p < parts; ++p)
        arrivals.part(10 * (p + 1), Event{when(p), p == fails});
    const std::clock_t before = std::clock();
    std::atomic<int> good{0};
    std::vector<std::thread> all;
    for (int t = 0; t < threads; ++t)
        all.emplace_back([&, t] {
            const int part = t % parts;
            const bool there = arrivals.wait(10 * part + 1 + t % 10);
            good += (there ? Clock::now() >= when(part) && (fails < 0 || part < fails) : fails >= 0 && part >= fails) ? 1 : 0;
        });
    for (auto& t : all)
        t.join();
    *right = good;
    try
    {
        arrivals.rethrow();
        *right = fails < 0 ? *right : -1;
    }
    catch (const std::runtime_error&)
    {
        *right = fails < 0 ? -1 : *right;
    }
    return static_cast<double>(std::clock() - before) / CLOCKS_PER_SEC;
}

// What happened to a block that the device was writing into when something was thrown, or not: 'w' the device was waited for, 'r' the
// block went.
extern "C" void block_given_up(int begun, int ended, int thrown, int wait_fails, char* log)
{
    struct Block
    {
        char*& log;
        ~Block() { *log++ = 'r'; }
    };
    try
    {
        Block block{log};
        auto wait = [&] {
            *log++ = 'w';
            if (wait_fails)
                throw std::runtime_error("wait");
        };
        grow_walk::PendingWrites<decltype(wait)> writes(wait);
        if (begun)
            writes.begin();
        if (thrown)
            throw std::runtime_error("between");
        if (ended)
            writes.end();
    }
    catch (const std::runtime_error&)
    {
    }
}

// The cluster of output i where cluster c's outputs begin at c * each; -1: a word outside the table was asked for.
extern "C" int cluster_of(int clusters, long long each, long long i)
{
    bool outside = false;
    const int c = grow_cluster_of(
        [&](int64_t word) {
            outside = outside || word < 0 || word >= int64_t(GROW_TABLE_ROW) * clusters || word % GROW_TABLE_ROW != 0;
            return word / GROW_TABLE_ROW * each;
        },
        clusters, i);
    return outside ? -1 : c;
}

extern "C" void grid_of(const float* low, const float* high, int m, float per_cell, int axis, int most, float* extent, int* along)
{
    float e[3];
    for (int a = 0; a < 3; ++a)
        extent[a] = e[a] = grid_extent(low[a], high[a]);
    const GridCounts counts = grid_counts(e, m, per_cell, axis, most, [](auto f) {
        int fitting = 0;
        for (int lane = 0; lane < 64; ++lane)
            fitting += f(lane) ? 1 : 0;
        return fitting;
    });
    for (int a = 0; a < 3; ++a)
        along[a] = counts.along[a];
}

extern "C" void table_cells(const float* v, int n, float inverse_width, int* cell)
{
    for (int i = 0; i < n; ++i)
        cell[i] = bt_cell(v[i], inverse_width);
}
extern "C" float table_reach(float radius) { return bt_reach(radius); }
extern "C" void table_bucket(int ix, int iy, int iz, int64_t cloud, uint32_t part_mask, uint32_t* part, uint32_t* bucket)
{
    const BtRow row = bt_row(iy, iz, cloud);
    *part = row.part;
    *bucket = bt_bucket(row, ix, part_mask);
}

// The guesses until between k and `most` of the distances lie within one; -1: none found.
extern "C" int guesses(const float* distance, int count, int k, int most, float first)
{
    auto within = [&](float t) {
        int in = 0;
        for (int i = 0; i < count; ++i)
            in += distance[i] <= t ? 1 : 0;
        return in;
    };
    Bracket bracket;
    float guess = first;
    int in = within(guess), tries = 0;
    for (; in < k || in > most; ++tries)
    {
        if (tries >= BRACKET_TRIES)
            return -1;
        const float estimate = guess * std::pow((k + (most - k) / 2) / std::fmax(static_cast<float>(in), 0.5f), 2.0f / 3.0f);
        guess = bracket.next(guess, in < k, estimate, tries);
        in = within(guess);
    }
    return tries;
}

extern "C" long long pieces_within(const int64_t* starts, long long pieces, long long begin, long long row_bytes, long long most)
{
    return grow_walk::pieces_within(starts, pieces, begin, row_bytes, most);
}

extern "C" long long most_staged()
{
    return grow_walk::MOST_STAGED;
}

// What each of the parts_grid() workgroups does; returns their number.
extern "C" unsigned tasks(unsigned items, unsigned parts, unsigned* item, unsigned* part)
{
    const unsigned blocks = parts_grid(items, parts);
    for (unsigned b = 0; b < blocks; ++b)
    {
        const PartTask task = part_task(b, items, parts);
        item[b] = task.item;
        part[b] = task.part;
    }
    return blocks;
}

extern "C" int ids_fit(unsigned labels, unsigned long long span)
{
    return region_ids_fit(labels, span) ? 1 : 0;
}
"""


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    folder = tmp_path_factory.mktemp("shim")
    source, library = str(folder / "shim.cpp"), str(folder / "shim.so")
    with open(source, "w") as f:
        f.write(SHIM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-ffp-contract=off", "-Wall", "-Werror", "-shared", "-fPIC", "-pthread", "-I" + CSRC, source, "-o", library],
                   check=True)
    return ctypes.CDLL(library)


def _grid(shim, low, high, m, per_cell, axis, most):
    low, high = (np.asarray(v, np.float32) for v in (low, high))
    extent, along = np.zeros(3, np.float32), np.zeros(3, np.int32)
    pointer = lambda a: a.ctypes.data_as(ctypes.c_void_p)
    shim.grid_of(pointer(low), pointer(high), m, ctypes.c_float(per_cell), axis, most, pointer(extent), pointer(along))
    return extent, along


# (the grid in LDS: 64 cells per axis, 4096 in all; the one in memory: 128 and 32768)
@pytest.mark.parametrize("axis,most", [(64, 4096), (128, 32768)])
@pytest.mark.parametrize("m,per_cell", [(1, 2.0), (7, 1.0), (8192, 1.0), (8192, 3.2), (16384, 9.6), (1 << 24, 1.0)])
def test_a_grid_has_no_more_cells_than_there_is_room(shim, axis, most, m, per_cell):
    inf = float("inf")
    sides = (0.0, 1e-45, 1e-38, 1e-20, 1e-7, 1.0, 2.0 ** 40, 1.7e38, 2e38, 3.4028235e38)
    spans = [(-a, b) for a in sides for b in (0.0, 1.0, 2e38, 3.4028235e38)] + [(a, a) for a in sides]
    # a cloud without a finite coordinate on an axis: the box of nothing
    spans += [(inf, -inf)]
    for x in spans:
        for y in spans[:: 3] + [x]:
            for z in (x, y, (0.0, 1.0), (-2e38, 2e38)):
                low, high = zip(x, y, z)
                extent, along = _grid(shim, low, high, m, per_cell, axis, most)
                assert (along >= 1).all() and (along <= axis).all(), (low, high, along)
                assert int(along.astype(np.int64).prod()) <= most, (low, high, along)
                assert np.isfinite(extent).all()
                assert np.isfinite(along[extent > 0] / extent[extent > 0]).all(), (low, high, along)
                assert (along[extent == 0] == 1).all()


def test_a_grid_follows_the_cloud(shim):
    """An even cloud gets about per_cell points per cell, a flat one a flat grid, a scaled one the same grid."""
    _, cube = _grid(shim, [0, 0, 0], [1, 1, 1], 8192, 2.0, 64, 4096)
    assert list(cube) == [16, 16, 16]
    for scale in (1e-12, 1e12, 1e37):
        _, along = _grid(shim, [0, 0, 0], [scale] * 3, 8192, 2.0, 64, 4096)
        assert list(along) == list(cube)
    _, flat = _grid(shim, [0, 0, 5], [1, 2, 5], 4096, 2.0, 64, 4096)
    assert flat[2] == 1 and flat[1] == 2 * flat[0] and 1800 <= flat.prod() <= 2048
    _, thin = _grid(shim, [0, 0, 0], [1, 1e-3, 1e-3], 8192, 2.0, 64, 4096)
    assert list(thin) == [64, 1, 1]


# (a first guess of 0 comes from a cloud without volume, one of +inf from a cell beyond float32; a query at 300 cloud sizes sees
# all points at about the same distance, far beyond the distance of neighbouring points)
@pytest.mark.parametrize("first", [0.0, 1e-30, 1e-3, 1.0, 1e20, float("inf")])
@pytest.mark.parametrize("offset,spread", [(0.0, 1.0), (0.0, 1e-30), (270000.0, 300.0), (3e37, 1e36), (0.0, 3e38)])
@pytest.mark.parametrize("k", [1, 16, 40, 48])
def test_a_selection_finds_a_distance(shim, first, offset, spread, k):
    rng = np.random.default_rng(k)
    for count in (65, 100, 144):
        distance = np.unique((offset + spread * rng.random(count)).astype(np.float32))
        rng.shuffle(distance)
        most = min(k + 24, 64)
        tries = shim.guesses(distance.ctypes.data_as(ctypes.c_void_p), len(distance), k, most, ctypes.c_float(first))
        assert 0 <= tries <= 6 + 31, (count, tries)


def test_a_selection_gives_up_on_equal_distances(shim):
    distance = np.full(100, 0.5, np.float32)
    assert shim.guesses(distance.ctypes.data_as(ctypes.c_void_p), 100, 16, 40, ctypes.c_float(1.0)) == -1


def test_cloud_ids_are_refused_before_they_overflow(shim):
    shim.ids_fit.argtypes = [ctypes.c_uint, ctypes.c_ulonglong]
    for labels in (1, 2, 3, 1000, 2 ** 31 - 1, 2 ** 31):
        for span in [1, 2, 1000] + [2 ** e + d for e in (31, 32, 33, 52, 61, 62, 63) for d in (-1, 0, 1)] + [2 ** 64 - 1]:
            largest = labels * span - 1  # label labels - 1, sample span - 1
            assert not shim.ids_fit(labels, span) or largest < 2 ** 63 - 1, (labels, span)
            assert shim.ids_fit(labels, span) or largest >= 2 ** 63 - 1 - labels, (labels, span)
        assert not shim.ids_fit(labels, 0)  # all 2^64 values


@pytest.mark.parametrize("parts", [1, 2, 3, 4])
@pytest.mark.parametrize("items", [1, 2, 3, 7, 8, 9, 16, 29, 63, 64, 65, 96, 257])
def test_the_parts_of_an_item_share_a_die(shim, items, parts):
    """Workgroups go to the eight dies in turn: every part of every item is somebody's, all parts of an item on one die, and no die
    has more items than an even share, rounded up."""
    item, part = np.zeros(4096, np.uint32), np.zeros(4096, np.uint32)
    blocks = shim.tasks(items, parts, *(a.ctypes.data_as(ctypes.c_void_p) for a in (item, part)))
    assert items * parts <= blocks < (items + 8) * parts
    die = np.arange(blocks) % 8
    item, part = item[:blocks], part[:blocks]
    done = item < items
    assert sorted(zip(item[done], part[done])) == [(i, p) for i in range(items) for p in range(parts)]
    for i in range(items):
        assert len(set(die[item == i])) == 1
    assert max(np.bincount(die[done], minlength=8)) == -(-items // 8) * parts
    assert (np.diff(die[done][np.argsort(item[done], kind="stable")]) >= 0).all()


@pytest.mark.parametrize("row_bytes,most", [(32, 1), (32, 3200), (6, 10 ** 4), (256, 10 ** 6), (4, 2 ** 62)])
def test_turns_of_pieces_stay_within_their_bytes(shim, row_bytes, most):
    """Every piece in one turn, no turn above the bytes unless it is a single piece, none that could have taken the next one too."""
    shim.pieces_within.restype = ctypes.c_longlong
    shim.pieces_within.argtypes = [ctypes.c_void_p] + [ctypes.c_longlong] * 4
    shim.most_staged.restype = ctypes.c_longlong
    assert 2 ** 24 <= shim.most_staged() <= 2 ** 28
    rng = np.random.default_rng(7)
    for pieces in (1, 2, 77):
        starts = np.concatenate([[0], np.cumsum(rng.integers(1, 200, pieces))]).astype(np.int64)
        begin = 0
        while begin < pieces:
            end = shim.pieces_within(starts.ctypes.data_as(ctypes.c_void_p), pieces, begin, row_bytes, most)
            assert begin < end <= pieces
            assert end == begin + 1 or (starts[end] - starts[begin]) * row_bytes <= most
            assert end == pieces or (starts[end + 1] - starts[begin]) * row_bytes > most
            begin = end


def test_a_block_goes_after_the_device_is_done_with_it(shim):
    """The host block that the rows kernel writes into: the wait for the device comes before it goes back to its pool, whatever is
    thrown behind the first launch that writes there."""
    for begun, ended, thrown, fails, want in ((1, 0, 1, 0, b"wr"), (1, 0, 1, 1, b"wr"), (1, 0, 0, 0, b"wr"), (1, 1, 0, 0, b"r"), (0, 0, 1, 0, b"r")):
        log = ctypes.create_string_buffer(8)
        shim.block_given_up(begun, ended, thrown, fails, log)
        assert log.value == want
    with open(os.path.join(CSRC, "points_cuda.cpp")) as f:
        body = f.read().split("at::Tensor grow_reference_order(")[1].split("\n}\n")[0]
    # the guard lives behind the block and is set before the first launch that is handed the block
    order = [body.index(s) for s in ("at::Tensor host =", "PendingWrites<decltype(wait)> writes(wait)", "writes.begin()", "tpk_grow_places(",
                                     "tpk_grow_rows_part(", "arrivals.wait(points + 1)", "writes.end()")]
    assert order == sorted(order)


def test_rows_in_one_part_need_no_events():
    """Calls whose rows come in one part wait for the stream: two events, their waits and threads cost 500 points 25 us of 170."""
    with open(os.path.join(CSRC, "points_cuda.cpp")) as f:
        body = f.read().split("at::Tensor grow_reference_order(")[1].split("\n}\n")[0]
    for made in body.split("event())")[:-1]:
        assert "if (part < points)" in made.splitlines()[-2] + made.splitlines()[-3]


@pytest.mark.parametrize("threads,parts,fails", [(1, 1, -1), (8, 5, -1), (16, 2, -1), (8, 5, 0), (8, 5, 3)])
def test_threads_sleep_until_their_part_is_there(shim, threads, parts, fails):
    """All threads get their part no sooner than it comes, or the error, and sleep while it is long in coming: a thread that asks for it
    again and again takes a processor for as long."""
    shim.parts_waited_for.restype = ctypes.c_double
    shim.parts_waited_for.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_double, ctypes.c_int, ctypes.c_void_p]
    right, apart = ctypes.c_int(), 0.1
    spent = shim.parts_waited_for(threads, parts, apart, fails, ctypes.addressof(right))
    assert right.value == threads
    assert spent < 0.5 * apart


@pytest.mark.parametrize("clusters", [1, 2, 3, 1000, 715827883, 715827884, 2 ** 30])
def test_an_outputs_cluster_is_found_in_a_table_of_any_size(shim, clusters):
    """(from 715827884 clusters on a word's number takes more than 31 bits)"""
    shim.cluster_of.argtypes = [ctypes.c_int, ctypes.c_longlong, ctypes.c_longlong]
    for each in (1, 7):
        for c in {0, 1, clusters // 3, clusters // 2, clusters - 2, clusters - 1}:
            for i in (c * each, c * each + each - 1):
                if 0 <= i < clusters * each:
                    assert shim.cluster_of(clusters, each, i) == c


@pytest.mark.parametrize("scale", [1e-30, 1e-3, 1.0, 5e3, 4e6, 3e30])
@pytest.mark.parametrize("radius", [0.0, 1e-25, 1e-12, 0.05, 3.0, 1e19])
def test_cells_of_the_ball_table_hold_every_accepted_point(shim, scale, radius):
    """A coordinate the radius test accepts lies between the cells of the query's two ends, at every scale and radius."""
    rng = np.random.default_rng(7)
    reach = np.float32(_table_reach(shim, radius))
    for width in (0.55, 2.2):
        inverse = np.float32(1.0) / (np.float32(width) * reach)
        q = ((rng.random(4000) - 0.5) * scale).astype(np.float32)
        with np.errstate(over="ignore", under="ignore", invalid="ignore"):
            step = np.concatenate([rng.uniform(-1.2, 1.2, 3000), np.repeat([-1.0, 1.0], 500)]) * radius
            p = (q.astype(np.float64) + step).astype(np.float32)
            d = p - q
            accepted = d * d <= np.float32(radius) * np.float32(radius)
            ends = [_table_cells(shim, v, inverse) for v in (q - reach, p, q + reach)]
        assert accepted.any()
        assert (ends[0] <= ends[1])[accepted].all() and (ends[1] <= ends[2])[accepted].all()


def test_rows_of_the_ball_table_near_each_other_never_share_a_part(shim):
    part, bucket = ctypes.c_uint32(), ctypes.c_uint32()
    rng = np.random.default_rng(3)
    for _ in range(50):
        ix, iy, iz = (int(v) for v in rng.integers(-2**30, 2**30, 3))
        cloud = int(rng.integers(-2**62, 2**62))
        parts = set()
        for dy in range(3):
            for dz in range(3):
                run = []
                for dx in range(5):
                    shim.table_bucket(ix + dx, iy + dy, iz + dz, ctypes.c_int64(cloud), 8191, ctypes.byref(part), ctypes.byref(bucket))
                    assert bucket.value // 8192 == part.value < 16
                    run.append(bucket.value % 8192)
                parts.add(part.value)
                assert all((b - a) % 8192 == 1 for a, b in zip(run, run[1:]))
        assert len(parts) == 9


def _table_reach(shim, radius):
    shim.table_reach.restype = ctypes.c_float
    return shim.table_reach(ctypes.c_float(radius))


def _table_cells(shim, v, inverse):
    v = np.ascontiguousarray(v, dtype=np.float32)
    cell = np.empty(v.shape[0], dtype=np.int32)
    shim.table_cells(v.ctypes.data_as(ctypes.c_void_p), v.shape[0], ctypes.c_float(inverse), cell.ctypes.data_as(ctypes.c_void_p))
    return cell
