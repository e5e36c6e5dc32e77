// torch_points_kernels.points_cuda for AMD MI355X: the pybind11 module the Python layer
// imports for tensors on the GPU.  It exports the names and signatures of the reference
// module (cuda/src/bindings.cpp:11-29) for the spatial-search operators, checks and
// allocates tensors the way the reference's host functions do, and hands raw pointers to
// the C ABI of libtpk_hip.so (include/tpk.h) on PyTorch's current HIP stream.  It contains
// no kernels and no CPU implementation: without a GPU tensor it raises.
#include <torch/extension.h>

#include <ATen/Parallel.h>
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/Event.h>

#include <algorithm>
#include <atomic>
#include <tuple>
#include <utility>
#include <vector>

#include "../../include/tpk.h"
#include "arrivals.h"
#include "grow_walk.h"

namespace {

void check_status(int status, const char* what)
{
    TORCH_CHECK(status == TPK_OK, what, " failed: ", tpk_status_string(status), " (status ",
                status, ")");
}

// The reference's checks (cuda/include/utils.h:5-27) made stricter where it would misread
// memory: exact dtypes instead of "some float" / "some int".
void check_gpu(const at::Tensor& t, const char* name)
{
    TORCH_CHECK(t.is_cuda(), name, " must be a CUDA tensor");
}
void check_contiguous(const at::Tensor& t, const char* name)
{
    TORCH_CHECK(t.is_contiguous(), name, " must be a contiguous tensor");
}
void check_f32(const at::Tensor& t, const char* name)
{
    TORCH_CHECK(t.scalar_type() == at::kFloat, name, " must be a float32 tensor");
}
void check_dtype(const at::Tensor& t, at::ScalarType st, const char* name)
{
    TORCH_CHECK(t.scalar_type() == st, name, " must be a ", c10::toString(st), " tensor");
}
void check_same_device(const at::Tensor& a, const at::Tensor& b, const char* names)
{
    TORCH_CHECK(a.device() == b.device(), names, " must be on the same device");
}
void check_points(const at::Tensor& t, int64_t dims, const char* name)
{
    TORCH_CHECK(t.dim() == dims && t.size(dims - 1) == 3, name, " must have shape (",
                dims == 3 ? "B, N, 3)" : "N, 3)");
}
int as_int(int64_t v, const char* name)
{
    TORCH_CHECK(v >= 0 && v <= INT32_MAX, name, " is out of range: ", v);
    return static_cast<int>(v);
}

void* current_stream(const at::Tensor& t)
{
    return static_cast<void*>(c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.get_device()).stream());
}

// cuda/src/sampling.cpp:8-25
at::Tensor furthest_point_sampling(at::Tensor points, const int nsamples)
{
    check_contiguous(points, "points");
    check_f32(points, "points");
    check_gpu(points, "points");
    check_points(points, 3, "points");
    TORCH_CHECK(nsamples >= 0, "nsamples must be non-negative");
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(points.device());

    at::Tensor output = torch::empty({points.size(0), nsamples},
                                     at::device(points.device()).dtype(at::ScalarType::Int));
    const int b = as_int(points.size(0), "batch size");
    const int n = as_int(points.size(1), "number of points");
    const size_t ws_bytes = tpk_fps_workspace_bytes(b, n);
    at::Tensor ws;
    if (ws_bytes)
        ws = torch::empty({static_cast<int64_t>(ws_bytes)},
                          at::device(points.device()).dtype(at::ScalarType::Byte));
    check_status(tpk_fps_f32(b, n, nsamples, points.data_ptr<float>(),
                             ws_bytes ? ws.data_ptr() : nullptr, ws_bytes,
                             output.data_ptr<int32_t>(), current_stream(points)),
                 "furthest_point_sampling");
    return output;
}

std::vector<at::Tensor> three_nearest(const at::Tensor& unknowns, const at::Tensor& knows, bool root)
{
    check_contiguous(unknowns, "unknowns");
    check_contiguous(knows, "knows");
    check_f32(unknowns, "unknowns");
    check_f32(knows, "knows");
    check_gpu(knows, "knows");
    check_gpu(unknowns, "unknowns");
    check_same_device(unknowns, knows, "unknowns and knows");
    check_points(unknowns, 3, "unknowns");
    check_points(knows, 3, "knows");
    TORCH_CHECK(unknowns.size(0) == knows.size(0), "unknowns and knows differ in batch size");
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(unknowns.device());

    at::Tensor idx = torch::empty({unknowns.size(0), unknowns.size(1), 3},
                                  at::device(unknowns.device()).dtype(at::ScalarType::Int));
    at::Tensor dist2 = torch::empty({unknowns.size(0), unknowns.size(1), 3},
                                    at::device(unknowns.device()).dtype(at::ScalarType::Float));
    const int b = as_int(unknowns.size(0), "batch size");
    const int n = as_int(unknowns.size(1), "number of unknown points");
    const int m = as_int(knows.size(1), "number of known points");
    const size_t ws_bytes = tpk_three_nn_workspace_bytes(b, n, m);
    at::Tensor ws;
    if (ws_bytes)
        ws = torch::empty({static_cast<int64_t>(ws_bytes)}, unknowns.options().dtype(torch::kUInt8));
    check_status((root ? tpk_three_nn_distance_f32 : tpk_three_nn_f32)(
                     b, n, m, unknowns.data_ptr<float>(), knows.data_ptr<float>(), dist2.data_ptr<float>(), idx.data_ptr<int32_t>(),
                     ws_bytes ? ws.data_ptr() : nullptr, ws_bytes, current_stream(unknowns)),
                 "three_nn");
    return {dist2, idx};
}

// cuda/src/interpolate.cpp:12-32
std::vector<at::Tensor> three_nn(at::Tensor unknowns, at::Tensor knows)
{
    return three_nearest(unknowns, knows, false);
}

// What the reference's torchpoints.py:64 makes of it: the distances, their square root taken as they are written.
std::vector<at::Tensor> three_nn_distance(at::Tensor unknowns, at::Tensor knows)
{
    return three_nearest(unknowns, knows, true);
}

// cpu/src/knn.cpp:43-62 (dense_knn; the reference has it for CPU tensors only)
std::pair<at::Tensor, at::Tensor> dense_knn(at::Tensor support, at::Tensor query, int64_t k)
{
    check_contiguous(support, "support");
    check_contiguous(query, "query");
    check_f32(support, "support");
    check_f32(query, "query");
    check_gpu(support, "support");
    check_gpu(query, "query");
    check_same_device(support, query, "support and query");
    check_points(support, 3, "support");
    check_points(query, 3, "query");
    TORCH_CHECK(support.size(0) == query.size(0), "support and query differ in batch size");
    TORCH_CHECK(k >= 0, "k must not be negative");
    // cpu/src/knn.cpp:12-14
    TORCH_CHECK(support.size(1) >= k, "Not enough points in support to find " + std::to_string(k) + " neighboors");
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(support.device());

    at::Tensor idx = torch::empty({query.size(0), query.size(1), k},
                                  at::device(query.device()).dtype(at::ScalarType::Long));
    at::Tensor dist2 = torch::empty({query.size(0), query.size(1), k},
                                    at::device(query.device()).dtype(at::ScalarType::Float));
    const int b = as_int(query.size(0), "batch size");
    const int n = as_int(support.size(1), "number of support points");
    const int m = as_int(query.size(1), "number of query points");
    const size_t ws_bytes = std::max(tpk_knn_workspace_bytes(b, n, m), tpk_knn_grid_workspace_bytes(b, n, m));
    at::Tensor ws;
    if (ws_bytes)
        ws = torch::empty({static_cast<int64_t>(ws_bytes)}, query.options().dtype(torch::kUInt8));
    check_status(tpk_knn_f32(b, n, m, as_int(k, "k"), support.data_ptr<float>(), query.data_ptr<float>(),
                             idx.data_ptr<int64_t>(), dist2.data_ptr<float>(),
                             ws_bytes ? ws.data_ptr() : nullptr, ws_bytes, current_stream(query)),
                 "dense_knn");
    return std::make_pair(idx, dist2);
}

// Host memory for copies to and from the device: pinned up to `most` bytes (torch's pool of such blocks, one given back is reused by
// the next call), pageable beyond, which the pool does not keep.
at::Tensor host_bytes(int64_t bytes, int64_t most)
{
    return at::empty({bytes}, at::TensorOptions().dtype(at::kByte).pinned_memory(bytes <= most));
}

// Walks the pieces begin .. end on host threads; rows: theirs, from the place starts[begin] on.  arrivals: the rows are still being
// written, in the order of places (nullptr: they are there).  Adds to `all`.
template <typename E>
void walk_pieces(const E* rows, int nsample, const int64_t* starts, int64_t begin, int64_t end, int64_t min_cluster_size, E* entries,
                 std::vector<grow_walk::Cluster>* all, Arrivals<c10::Event>* arrivals)
{
    const int64_t pieces = end - begin, points = starts[end] - starts[begin];
    std::vector<int64_t> turn(static_cast<size_t>(pieces));
    for (int64_t p = 0; p < pieces; ++p)
        turn[p] = begin + p;
    // The longest walks first: the end of the last one is what the caller waits for.  (Up to 1024 pieces lie in that order; more
    // do not, and where they arrive in parts a thread may have to wait for the last one.)
    std::stable_sort(turn.begin(), turn.end(), [&](int64_t a, int64_t b) { return starts[a + 1] - starts[a] > starts[b + 1] - starts[b]; });
    // (below 16384 points the walk takes less time than waking the other threads)
    const int64_t threads = points < 16384 ? 1 : std::min<int64_t>(at::get_num_threads(), pieces);
    std::vector<std::vector<grow_walk::Cluster>> found(static_cast<size_t>(threads));
    std::atomic<int64_t> next{0};
    auto work = [&](int64_t t) {
        grow_walk::Scratch scratch;
        for (int64_t i = next.fetch_add(1); i < pieces; i = next.fetch_add(1))
        {
            const int64_t base = starts[turn[i]], count = starts[turn[i] + 1] - base;
            if (arrivals && !arrivals->wait(base + count))
                return;
            grow_walk::walk_piece(rows + (base - starts[begin]) * nsample, nsample, base, count, min_cluster_size, scratch, entries, found[t]);
        }
    };
    if (threads == 1)
        work(0);
    else
        at::parallel_for(0, threads, 1, [&](int64_t first, int64_t last) {
            for (int64_t t = first; t < last; ++t)
                work(t);
        });
    if (arrivals)
        arrivals->rethrow();
    for (const auto& f : found)
        all->insert(all->end(), f.begin(), f.end());
}

// Clusters in the reference's member order: pieces from the device, walked on host threads.  members: one tensor on the
// device, clusters one after the other, as indices (order: what tpk_region_order put at every position; may be
// undefined); sizes: theirs.  most: bytes of pinned memory at a time; pieces that together take more are copied and walked in
// several turns.
at::Tensor grow_reference_order(const at::Tensor& neighbours, int64_t min_cluster_size, const at::Tensor& order,
                                std::vector<int64_t>* sizes, int64_t most = grow_walk::MOST_STAGED)
{
    const int64_t n = neighbours.size(0);
    const int nsample = as_int(neighbours.size(1), "nsample");
    auto bytes_on_device = at::device(neighbours.device()).dtype(at::kByte);
    auto longs = at::device(neighbours.device()).dtype(at::kLong);
    void* stream = current_stream(neighbours);
    auto wait = [&] { c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(neighbours.get_device()).synchronize(); };
    sizes->clear();
    const size_t ws_bytes = tpk_grow_components_workspace_bytes(n);
    TORCH_CHECK(ws_bytes > 0, "grow_proximity: too many points");
    at::Tensor ws = at::empty({static_cast<int64_t>(ws_bytes)}, bytes_on_device);
    int64_t found[3] = {0, 0, 0};
    check_status(tpk_grow_components_by_size(n, nsample, neighbours.data_ptr<int64_t>(), min_cluster_size, found, ws.data_ptr(), ws_bytes,
                                             stream),
                 "grow_proximity (components)");
    const int64_t pieces = found[0], points = found[1];
    if (pieces == 0)
        return at::empty({0}, longs);
    const int64_t entry = found[2] <= 65536 ? 2 : 4, row_bytes = nsample * entry;
    // One block of pinned memory for starts, positions and rows, the rows written there by the kernel that makes them; where they take
    // more than `most` they come by themselves.
    const int64_t at_positions = (pieces + 1) * 8, at_rows = (at_positions + points * 4 + 15) / 16 * 16;
    const bool at_once = at_rows + points * row_bytes <= most;
    at::Tensor host = host_bytes(at_once ? at_rows + points * row_bytes : at_rows, most);
    grow_walk::PendingWrites<decltype(wait)> writes(wait); // (gone before `host` is)
    uint8_t* h = host.data_ptr<uint8_t>();
    const int64_t* starts = reinterpret_cast<const int64_t*>(h);
    const int32_t* positions = reinterpret_cast<const int32_t*>(h + at_positions);
    at::Tensor staged = at::empty({at_rows + (at_once ? 0 : points * row_bytes)}, bytes_on_device);
    uint8_t* d = staged.data_ptr<uint8_t>();
    int32_t* positions_out = reinterpret_cast<int32_t*>(d + at_positions);
    if (at_once)
    {
        writes.begin();
        check_status(tpk_grow_places(n, found, positions_out, reinterpret_cast<int64_t*>(h), ws.data_ptr(), ws_bytes, stream),
                     "grow_proximity (places)");
    }
    else
        check_status(tpk_grow_rows(n, nsample, neighbours.data_ptr<int64_t>(), found, static_cast<int>(entry), d + at_rows, positions_out,
                                   reinterpret_cast<int64_t*>(d), ws.data_ptr(), ws_bytes, stream),
                     "grow_proximity (rows)");
    // What the walk leaves: the clusters' members as entries, then a table of the clusters.  (From the pool: fresh memory would cost a page fault
    // per 4 KiB.)
    const int64_t at_table = (points * entry + 7) / 8 * 8, most_clusters = points / std::max<int64_t>(min_cluster_size, 1);
    at::Tensor walked = host_bytes(at_table + most_clusters * 24, most);
    uint8_t* entries = walked.data_ptr<uint8_t>();
    std::vector<grow_walk::Cluster> all;
    auto walk = [&](const uint8_t* rows, int64_t begin, int64_t end, Arrivals<c10::Event>* arrivals) {
        if (entry == 2)
            walk_pieces(reinterpret_cast<const uint16_t*>(rows), nsample, starts, begin, end, min_cluster_size, reinterpret_cast<uint16_t*>(entries), &all,
                        arrivals);
        else
            walk_pieces(reinterpret_cast<const uint32_t*>(rows), nsample, starts, begin, end, min_cluster_size, reinterpret_cast<uint32_t*>(entries), &all,
                        arrivals);
    };
    if (at_once)
    {
        // The largest pieces lie first, so their walks, which end last, begin while the others' rows are being written.
        Arrivals<c10::Event> arrivals;
        auto event = [&] { // happens when the work enqueued so far is done
            c10::Event e(c10::DeviceType::CUDA);
            e.record(c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(neighbours.get_device()).unwrap());
            return e;
        };
        const int64_t part = std::max(grow_walk::LEAST_PART / row_bytes, points / grow_walk::PARTS) + 1;
        for (int64_t first = 0, count; first < points; first += count)
        {
            count = std::min(part, points - first);
            check_status(tpk_grow_rows_part(n, nsample, neighbours.data_ptr<int64_t>(), found, static_cast<int>(entry), first, count, h + at_rows,
                                            ws.data_ptr(), ws_bytes, stream),
                         "grow_proximity (rows)");
            if (part < points)
                arrivals.part(first + count, event());
        }
        const int64_t bytes = points * 4;
        host.narrow(0, at_positions, bytes).copy_(staged.narrow(0, at_positions, bytes), /*non_blocking=*/true);
        if (part < points)
        {
            arrivals.part(points + 1, event());
            if (arrivals.wait(1))
                walk(h + at_rows, 0, pieces, &arrivals);
            arrivals.wait(points + 1);
            arrivals.rethrow();
        }
        else
        {
            wait(); // (a single part: two events and two waits cost more than there is to overlap)
            walk(h + at_rows, 0, pieces, nullptr);
        }
        writes.end();
    }
    else
    {
        host.copy_(staged.narrow(0, 0, at_rows), /*non_blocking=*/true);
        wait();
        at::Tensor turn; // the rows of some pieces
        for (int64_t begin = 0, end = 0; begin < pieces; begin = end)
        {
            end = grow_walk::pieces_within(starts, pieces, begin, row_bytes, most);
            const int64_t bytes = (starts[end] - starts[begin]) * row_bytes;
            if (!turn.defined() || turn.numel() < bytes)
                turn = host_bytes(std::max(bytes, std::min(most, points * row_bytes)), most);
            at::Tensor rows = turn.narrow(0, 0, bytes);
            rows.copy_(staged.narrow(0, at_rows + starts[begin] * row_bytes, bytes), /*non_blocking=*/true);
            wait();
            walk(rows.data_ptr<uint8_t>(), begin, end, nullptr);
        }
    }
    std::sort(all.begin(), all.end(), [&](const grow_walk::Cluster& a, const grow_walk::Cluster& b) { return positions[a.base + a.first] < positions[b.base + b.first]; });
    int64_t* table = reinterpret_cast<int64_t*>(entries + at_table);
    int64_t total = 0;
    for (size_t c = 0; c < all.size(); ++c)
    {
        table[3 * c] = total;
        table[3 * c + 1] = all[c].at;
        table[3 * c + 2] = all[c].base;
        total += all[c].size;
        sizes->push_back(all[c].size);
    }
    at::Tensor members = at::empty({total}, longs);
    const int64_t clusters = static_cast<int64_t>(all.size()), bytes = at_table + clusters * 24;
    at::Tensor uploaded = at::empty({bytes}, bytes_on_device);
    uploaded.copy_(walked.narrow(0, 0, bytes), /*non_blocking=*/walked.numel() <= most); // (a pageable block goes with this call)
    const uint8_t* u = uploaded.data_ptr<uint8_t>();
    check_status(tpk_grow_members(total, clusters, reinterpret_cast<const int64_t*>(u + at_table), static_cast<int>(entry), u,
                                  reinterpret_cast<const int32_t*>(d + at_positions), order.defined() ? order.data_ptr<int32_t>() : nullptr,
                                  members.data_ptr<int64_t>(), stream),
                 "grow_proximity (members)");
    return members;
}

// torch_points_kernels/cluster.py:9-37 (_grow_proximity_core; host code in the reference)
// -> (members, starts): clusters one after the other and their offsets (one more than clusters).
// most_staged: see grow_reference_order.
std::pair<at::Tensor, at::Tensor> grow_proximity(at::Tensor neighbours, int64_t min_cluster_size, bool reference_order,
                                                 int64_t most_staged)
{
    check_contiguous(neighbours, "neighbours");
    check_dtype(neighbours, at::kLong, "neighbours");
    check_gpu(neighbours, "neighbours");
    TORCH_CHECK(neighbours.dim() == 2, "neighbours must have shape (N, nsample)");
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(neighbours.device());
    const int64_t n = neighbours.size(0);
    auto options = at::device(neighbours.device()).dtype(at::ScalarType::Long);
    at::Tensor members = torch::empty({n}, options);
    at::Tensor starts = torch::empty({n + 1}, options);
    int64_t found[2] = {0, 0};
    if (n > 0 && reference_order && neighbours.size(1) > 0)
    {
        std::vector<int64_t> sizes;
        members = grow_reference_order(neighbours, min_cluster_size, at::Tensor(), &sizes, most_staged);
        std::vector<int64_t> ends(1, 0);
        for (int64_t v : sizes)
            ends.push_back(ends.back() + v);
        return std::make_pair(members, at::tensor(ends, at::kLong).to(neighbours.device()));
    }
    if (n > 0)
    {
        const size_t ws_bytes = tpk_grow_proximity_workspace_bytes(n, as_int(neighbours.size(1), "nsample"));
        TORCH_CHECK(ws_bytes > 0, "grow_proximity: too many points");
        at::Tensor ws = torch::empty({static_cast<int64_t>(ws_bytes)}, options.dtype(torch::kUInt8));
        check_status(tpk_grow_proximity(n, as_int(neighbours.size(1), "nsample"), neighbours.data_ptr<int64_t>(),
                                        min_cluster_size,
                                        reference_order ? TPK_MEMBERS_AS_REFERENCE : TPK_MEMBERS_BY_INDEX,
                                        members.data_ptr<int64_t>(), starts.data_ptr<int64_t>(), found,
                                        ws.data_ptr(), ws_bytes, current_stream(neighbours)),
                     "grow_proximity");
    }
    if (found[0] == 0)
        return std::make_pair(members.narrow(0, 0, 0), torch::zeros({1}, options));
    return std::make_pair(members.narrow(0, 0, found[1]), starts.narrow(0, 0, found[0] + 1));
}

void check_interpolate(const at::Tensor& points, const at::Tensor& idx, const at::Tensor& weight)
{
    check_contiguous(points, "points");
    check_contiguous(idx, "idx");
    check_contiguous(weight, "weight");
    check_f32(points, "points");
    check_dtype(idx, at::kInt, "idx");
    check_f32(weight, "weight");
    check_gpu(points, "points");
    check_gpu(idx, "idx");
    check_gpu(weight, "weight");
    check_same_device(points, idx, "points and idx");
    check_same_device(points, weight, "points and weight");
    TORCH_CHECK(points.dim() == 3, "points must have shape (B, c, m)");
    TORCH_CHECK(idx.dim() == 3 && idx.size(2) == 3 && idx.size(0) == points.size(0),
                "idx must have shape (B, n, 3)");
    TORCH_CHECK(weight.sizes() == idx.sizes(), "weight must have the shape of idx");
}

// cuda/src/interpolate.cpp:34-54
at::Tensor three_interpolate(at::Tensor points, at::Tensor idx, at::Tensor weight)
{
    check_interpolate(points, idx, weight);
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(points.device());

    at::Tensor output = torch::empty({points.size(0), points.size(1), idx.size(1)},
                                     at::device(points.device()).dtype(at::ScalarType::Float));
    check_status(tpk_three_interpolate_f32(
                     as_int(points.size(0), "batch size"), as_int(points.size(1), "channels"),
                     as_int(points.size(2), "m"), as_int(idx.size(1), "n"),
                     points.data_ptr<float>(), idx.data_ptr<int32_t>(), weight.data_ptr<float>(),
                     output.data_ptr<float>(), current_stream(points)),
                 "three_interpolate");
    return output;
}

// cuda/src/interpolate.cpp:55-76
at::Tensor three_interpolate_grad(at::Tensor grad_out, at::Tensor idx, at::Tensor weight,
                                  const int m)
{
    check_contiguous(grad_out, "grad_out");
    check_contiguous(idx, "idx");
    check_contiguous(weight, "weight");
    check_f32(grad_out, "grad_out");
    check_dtype(idx, at::kInt, "idx");
    check_f32(weight, "weight");
    check_gpu(idx, "idx");
    check_gpu(weight, "weight");
    check_gpu(grad_out, "grad_out");
    check_same_device(grad_out, idx, "grad_out and idx");
    check_same_device(grad_out, weight, "grad_out and weight");
    TORCH_CHECK(grad_out.dim() == 3, "grad_out must have shape (B, c, n)");
    TORCH_CHECK(idx.dim() == 3 && idx.size(2) == 3 && idx.size(0) == grad_out.size(0) &&
                    idx.size(1) == grad_out.size(2),
                "idx must have shape (B, n, 3)");
    TORCH_CHECK(weight.sizes() == idx.sizes(), "weight must have the shape of idx");
    TORCH_CHECK(m >= 0, "m must be non-negative");
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(grad_out.device());

    at::Tensor output = torch::empty({grad_out.size(0), grad_out.size(1), m},
                                     at::device(grad_out.device()).dtype(at::ScalarType::Float));
    const int b = as_int(grad_out.size(0), "batch size");
    const int n = as_int(grad_out.size(2), "n");
    const size_t ws_bytes = tpk_three_interpolate_grad_workspace_bytes(b, n, m);
    at::Tensor ws = torch::empty({static_cast<int64_t>(ws_bytes)},
                                 at::device(grad_out.device()).dtype(at::ScalarType::Byte));
    check_status(tpk_three_interpolate_grad_f32(
                     b, as_int(grad_out.size(1), "channels"), n, m, grad_out.data_ptr<float>(),
                     idx.data_ptr<int32_t>(), weight.data_ptr<float>(), output.data_ptr<float>(),
                     ws_bytes ? ws.data_ptr() : nullptr, ws_bytes, current_stream(grad_out)),
                 "three_interpolate_grad");
    return output;
}

// three_interpolate for a caller that will ask for the gradient (autograd is recording): with the forward
// pass the index is inverted into the per-target lists that the backward pass walks (include/tpk.h,
// tpk_three_interpolate_lists_f32), so that the backward pass is the walk alone and several backward passes
// share one inversion.  Returns (output, lists); `lists` is empty where the list path does not serve the shape
// (then three_interpolate_grad is the backward pass).  No counterpart in the reference, whose backward scatters
// with atomics.  (Inverting on a second stream beside the gather was measured: the two event waits between the
// streams cost more than the 18 us they hide - 198 us per call against 52 us one after the other.)
std::pair<at::Tensor, at::Tensor> three_interpolate_recording(at::Tensor points, at::Tensor idx, at::Tensor weight)
{
    check_interpolate(points, idx, weight);
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(points.device());
    const int b = as_int(points.size(0), "batch size"), c = as_int(points.size(1), "channels"), m = as_int(points.size(2), "m");
    const int n = as_int(idx.size(1), "n");
    const size_t bytes = tpk_three_interpolate_grad_workspace_bytes(b, n, m);
    if (bytes == 0)
        return {three_interpolate(points, idx, weight), torch::empty({0}, at::device(points.device()).dtype(at::kByte))};
    at::Tensor lists = torch::empty({static_cast<int64_t>(bytes)}, at::device(points.device()).dtype(at::kByte));
    at::Tensor output = torch::empty({points.size(0), points.size(1), idx.size(1)}, at::device(points.device()).dtype(at::kFloat));
    check_status(tpk_three_interpolate_recording_f32(b, c, m, n, points.data_ptr<float>(), idx.data_ptr<int32_t>(),
                                                     weight.data_ptr<float>(), output.data_ptr<float>(), lists.data_ptr(), bytes,
                                                     current_stream(points)),
                 "three_interpolate (with the lists for the backward pass)");
    return {output, lists};
}

// The backward pass over the lists three_interpolate_recording() returned.
at::Tensor three_interpolate_grad_lists(at::Tensor grad_out, at::Tensor lists, const int m)
{
    check_contiguous(grad_out, "grad_out");
    check_f32(grad_out, "grad_out");
    check_gpu(grad_out, "grad_out");
    check_gpu(lists, "lists");
    check_same_device(grad_out, lists, "grad_out and lists");
    TORCH_CHECK(grad_out.dim() == 3, "grad_out must have shape (B, c, n)");
    TORCH_CHECK(lists.scalar_type() == at::kByte && lists.is_contiguous() && m >= 0, "lists as three_interpolate_recording returned them");
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(grad_out.device());
    at::Tensor output = torch::empty({grad_out.size(0), grad_out.size(1), m}, at::device(grad_out.device()).dtype(at::kFloat));
    check_status(tpk_three_interpolate_grad_lists_f32(as_int(grad_out.size(0), "batch size"), as_int(grad_out.size(1), "channels"),
                                                      as_int(grad_out.size(2), "n"), m, grad_out.data_ptr<float>(),
                                                      lists.data_ptr(), static_cast<size_t>(lists.numel()),
                                                      output.data_ptr<float>(), current_stream(grad_out)),
                 "three_interpolate_grad (from lists)");
    return output;
}

// cuda/src/ball_query.cpp:15-36.  Query centres first, as in the reference.
// sorted: the nsample nearest neighbours within the radius, nearest first (what the reference
// computes for CPU tensors with sort=True, cpu/src/ball_query.cpp:127-146).
std::pair<at::Tensor, at::Tensor> ball_query_dense(at::Tensor new_xyz, at::Tensor xyz,
                                                   const float radius, const int nsample, const bool sorted)
{
    check_contiguous(new_xyz, "new_xyz");
    check_contiguous(xyz, "xyz");
    check_f32(new_xyz, "new_xyz");
    check_f32(xyz, "xyz");
    check_gpu(xyz, "xyz");
    check_gpu(new_xyz, "new_xyz");
    check_same_device(xyz, new_xyz, "xyz and new_xyz");
    check_points(new_xyz, 3, "new_xyz");
    check_points(xyz, 3, "xyz");
    TORCH_CHECK(xyz.size(0) == new_xyz.size(0), "xyz and new_xyz differ in batch size");
    TORCH_CHECK(nsample >= 0, "nsample must be non-negative");
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(new_xyz.device());

    at::Tensor idx = torch::empty({new_xyz.size(0), new_xyz.size(1), nsample},
                                  at::device(new_xyz.device()).dtype(at::ScalarType::Long));
    at::Tensor dist = torch::empty({new_xyz.size(0), new_xyz.size(1), nsample},
                                   at::device(new_xyz.device()).dtype(at::ScalarType::Float));
    if (sorted)
    {
        const int b = as_int(xyz.size(0), "batch size"), n = as_int(xyz.size(1), "support points");
        const int m = as_int(new_xyz.size(1), "query points");
        const size_t ws_bytes = tpk_ball_query_sorted_dense_workspace_bytes(b, n, m);
        at::Tensor ws;
        if (ws_bytes)
            ws = torch::empty({static_cast<int64_t>(ws_bytes)}, new_xyz.options().dtype(torch::kUInt8));
        check_status(tpk_ball_query_sorted_dense_f32(b, n, m, radius, nsample, new_xyz.data_ptr<float>(),
                                                     xyz.data_ptr<float>(), idx.data_ptr<int64_t>(),
                                                     dist.data_ptr<float>(), ws_bytes ? ws.data_ptr() : nullptr,
                                                     ws_bytes, current_stream(new_xyz)),
                     "ball_query_dense (sorted)");
        return std::make_pair(idx, dist);
    }
    {
        const int b = as_int(xyz.size(0), "batch size"), n = as_int(xyz.size(1), "support points");
        const int m = as_int(new_xyz.size(1), "query points");
        const size_t ws_bytes = tpk_ball_query_dense_workspace_bytes(b, n, m, nsample);
        at::Tensor ws;
        if (ws_bytes)
            ws = torch::empty({static_cast<int64_t>(ws_bytes)}, new_xyz.options().dtype(torch::kUInt8));
        check_status(tpk_ball_query_dense_ws_f32(b, n, m, radius, nsample, new_xyz.data_ptr<float>(), xyz.data_ptr<float>(),
                                                 idx.data_ptr<int64_t>(), dist.data_ptr<float>(),
                                                 ws_bytes ? ws.data_ptr() : nullptr, ws_bytes, current_stream(new_xyz)),
                     "ball_query_dense");
    }
    return std::make_pair(idx, dist);
}

// cuda/src/ball_query.cpp:45-81.  Support first, as in the reference.  The cloud ranges
// are found on the device from the sorted batch vectors; nothing is copied to the host.
std::pair<at::Tensor, at::Tensor> ball_query_partial_dense(at::Tensor x, at::Tensor y,
                                                           at::Tensor batch_x, at::Tensor batch_y,
                                                           const float radius, const int nsample, const bool sorted)
{
    check_contiguous(x, "x");
    check_contiguous(y, "y");
    check_f32(x, "x");
    check_f32(y, "y");
    check_gpu(x, "x");
    check_gpu(y, "y");
    check_gpu(batch_x, "batch_x");
    check_gpu(batch_y, "batch_y");
    check_same_device(x, y, "x and y");
    check_same_device(x, batch_x, "x and batch_x");
    check_same_device(x, batch_y, "x and batch_y");
    check_points(x, 2, "x");
    check_points(y, 2, "y");
    check_dtype(batch_x, at::kLong, "batch_x");
    check_dtype(batch_y, at::kLong, "batch_y");
    TORCH_CHECK(batch_x.dim() == 1 && batch_x.size(0) == x.size(0),
                "batch_x must have one entry per point of x");
    TORCH_CHECK(batch_y.dim() == 1 && batch_y.size(0) == y.size(0),
                "batch_y must have one entry per point of y");
    TORCH_CHECK(nsample >= 0, "nsample must be non-negative");
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
    batch_x = batch_x.contiguous();
    batch_y = batch_y.contiguous();

    at::Tensor idx =
        torch::empty({y.size(0), nsample}, at::device(y.device()).dtype(at::ScalarType::Long));
    at::Tensor dist =
        torch::empty({y.size(0), nsample}, at::device(y.device()).dtype(at::ScalarType::Float));
    if (sorted)
    {
        // cpu/src/ball_query.cpp:65-124 with sorted = true
        const size_t sorted_ws_bytes = tpk_ball_query_sorted_partial_workspace_bytes(x.size(0), y.size(0));
        at::Tensor sorted_ws;
        if (sorted_ws_bytes)
            sorted_ws = torch::empty({static_cast<int64_t>(sorted_ws_bytes)}, x.options().dtype(torch::kUInt8));
        check_status(tpk_ball_query_sorted_partial_f32(x.size(0), y.size(0), radius, nsample, x.data_ptr<float>(),
                                                       y.data_ptr<float>(), batch_x.data_ptr<int64_t>(),
                                                       batch_y.data_ptr<int64_t>(), idx.data_ptr<int64_t>(),
                                                       dist.data_ptr<float>(),
                                                       sorted_ws_bytes ? sorted_ws.data_ptr() : nullptr, sorted_ws_bytes,
                                                       current_stream(x)),
                     "ball_query_partial_dense (sorted)");
        return std::make_pair(idx, dist);
    }
    const size_t ws_bytes = tpk_ball_query_partial_table_workspace_bytes(x.size(0), y.size(0), nsample);
    at::Tensor ws;
    if (ws_bytes)
        ws = torch::empty({static_cast<int64_t>(ws_bytes)}, x.options().dtype(torch::kUInt8));
    check_status(tpk_ball_query_partial_f32(x.size(0), y.size(0), radius, nsample,
                                            x.data_ptr<float>(), y.data_ptr<float>(),
                                            batch_x.data_ptr<int64_t>(),
                                            batch_y.data_ptr<int64_t>(), idx.data_ptr<int64_t>(),
                                            dist.data_ptr<float>(), ws_bytes ? ws.data_ptr() : nullptr,
                                            ws_bytes, current_stream(x)),
                 "ball_query_partial_dense");
    return std::make_pair(idx, dist);
}

// torch_points_kernels/cluster.py:48-109 for all labels at once: the points label by label, every (label, sample) a cloud
// of one packed self query, one growth.  Returns the clusters label after label, ordered by first point inside a label.
std::vector<at::Tensor> region_grow(at::Tensor pos, at::Tensor labels, at::Tensor batch, std::vector<int64_t> ignore_labels,
                                    int64_t nsample, double radius, int64_t min_cluster_size, bool reference_order)
{
    check_gpu(pos, "pos");
    check_f32(pos, "pos");
    check_points(pos, 2, "pos");
    check_same_device(pos, labels, "pos and labels");
    check_same_device(pos, batch, "pos and batch");
    check_dtype(labels, at::kLong, "labels");
    check_dtype(batch, at::kLong, "batch");
    const int64_t n = pos.size(0);
    TORCH_CHECK(labels.dim() == 1 && labels.size(0) == n && batch.dim() == 1 && batch.size(0) == n,
                "pos, labels and batch differ in length");
    TORCH_CHECK(ignore_labels.size() <= TPK_REGION_IGNORED, "region_grow: too many labels to ignore");
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(pos.device());
    if (n == 0)
        return {};
    pos = pos.contiguous();
    labels = labels.contiguous();
    batch = batch.contiguous();
    void* stream = current_stream(pos);
    at::Tensor order = at::empty({n}, pos.options().dtype(at::kInt));
    at::Tensor sorted = at::empty({n, 3}, pos.options());
    at::Tensor ids = at::empty({n}, batch.options());
    int64_t found[2] = {0, 0};
    {
        const size_t ws_bytes = tpk_region_order_workspace_bytes(n);
        TORCH_CHECK(ws_bytes > 0, "region_grow: too many points");
        at::Tensor ws = at::empty({static_cast<int64_t>(ws_bytes)}, pos.options().dtype(at::kByte));
        const int status = tpk_region_order(n, labels.data_ptr<int64_t>(), batch.data_ptr<int64_t>(), pos.data_ptr<float>(),
                                            static_cast<int>(ignore_labels.size()), ignore_labels.data(), found,
                                            order.data_ptr<int32_t>(), sorted.data_ptr<float>(), ids.data_ptr<int64_t>(),
                                            ws.data_ptr(), ws_bytes, stream);
        if (status == TPK_ERR_UNSUPPORTED)
        {
            // labels far apart, or sample ids too far apart for as many labels: the ranks of both instead
            at::Tensor values, ranks;
            batch = std::get<1>(at::unique_consecutive(batch, /*return_inverse=*/true));
            std::tie(values, ranks) = at::_unique(labels, /*sorted=*/true, /*return_inverse=*/true);
            values = values.cpu();
            std::vector<int64_t> ignored_ranks;
            for (int64_t i = 0; i < values.numel(); ++i)
                if (std::count(ignore_labels.begin(), ignore_labels.end(), values.data_ptr<int64_t>()[i]))
                    ignored_ranks.push_back(i);
            return region_grow(pos, ranks, batch, ignored_ranks, nsample, radius, min_cluster_size, reference_order);
        }
        check_status(status, "region_grow (order)");
    }
    const int64_t kept = found[0];
    if (kept == 0)
        return {};
    if (found[1])
    {
        sorted = sorted.narrow(0, 0, kept);
        ids = ids.narrow(0, 0, kept);
    }
    else
    {
        sorted = pos;
        ids = batch;
        order = at::Tensor();
    }
    at::Tensor neighbours =
        ball_query_partial_dense(sorted, sorted, ids, ids, static_cast<float>(radius), as_int(nsample, "nsample"), false).first;
    std::vector<int64_t> sizes;
    at::Tensor members;
    if (reference_order && nsample > 0)
        members = grow_reference_order(neighbours, min_cluster_size, order, &sizes);
    else
    {
        at::Tensor starts;
        std::tie(members, starts) = grow_proximity(neighbours, min_cluster_size, false, grow_walk::MOST_STAGED);
        if (order.defined())
            check_status(tpk_region_members(members.numel(), order.data_ptr<int32_t>(), 8, members.data_ptr<int64_t>(),
                                            members.data_ptr<int64_t>(), stream),
                         "region_grow (members)");
        const at::Tensor ends = starts.cpu();
        const int64_t* e = ends.data_ptr<int64_t>();
        for (int64_t c = 0; c + 1 < ends.numel(); ++c)
            sizes.push_back(e[c + 1] - e[c]);
    }
    return members.split_with_sizes(sizes);
}

// cuda/src/metrics.cpp:12-52
at::Tensor instance_iou_cuda(at::Tensor instance_idx, at::Tensor instance_offsets, at::Tensor gt_instances,
                             at::Tensor gt_instance_sizes, at::Tensor num_gt_instances, at::Tensor batch)
{
    const at::Tensor* all[] = {&instance_idx, &instance_offsets, &gt_instances, &gt_instance_sizes, &num_gt_instances, &batch};
    const char* names[] = {"instance_idx", "instance_offsets", "gt_instances", "gt_instance_sizes", "num_gt_instances", "batch"};
    for (int i = 0; i < 6; ++i)
    {
        check_contiguous(*all[i], names[i]);
        check_gpu(*all[i], names[i]);
        check_dtype(*all[i], at::kLong, names[i]);
        check_same_device(*all[i], gt_instances, names[i]);
        TORCH_CHECK(all[i]->dim() == 1, names[i], " must have one dimension");
    }
    TORCH_CHECK(instance_offsets.size(0) >= 1, "instance_offsets must hold at least one entry");
    TORCH_CHECK(batch.size(0) == gt_instances.size(0), "batch and gt_instances differ in length");
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(gt_instances.device());
    const int64_t num_proposed_instances = instance_offsets.size(0) - 1;
    // as the reference: the total is read back to size the output
    const int64_t total_gt_instances = num_gt_instances.numel() ? num_gt_instances.sum().item<int64_t>() : 0;
    TORCH_CHECK(gt_instance_sizes.size(0) == total_gt_instances, "gt_instance_sizes must hold one entry per ground-truth instance");
    at::Tensor output = torch::empty({num_proposed_instances, total_gt_instances},
                                     at::device(gt_instances.device()).dtype(at::ScalarType::Float));
    at::Tensor offset_num_gt_instances = at::cat({at::zeros(1, num_gt_instances.options()), num_gt_instances.cumsum(0)}, 0);
    check_status(tpk_instance_iou(total_gt_instances, num_proposed_instances, gt_instances.size(0), num_gt_instances.size(0),
                                  num_gt_instances.data_ptr<int64_t>(), instance_idx.data_ptr<int64_t>(),
                                  instance_offsets.data_ptr<int64_t>(), gt_instances.data_ptr<int64_t>(),
                                  offset_num_gt_instances.data_ptr<int64_t>(), batch.data_ptr<int64_t>(),
                                  gt_instance_sizes.data_ptr<int64_t>(), output.data_ptr<float>(),
                                  current_stream(gt_instances)),
                 "instance_iou_cuda");
    return output;
}

// torch_points_kernels/metrics.py:37-104 for index tensors on the device: None where a proposal is not a contiguous
// int64 vector there, or the samples are more than the kernels count (the general path serves those).  The table of the
// proposals is made while the device counts the instances; the host waits once, for the width of the output.
pybind11::object instance_iou_lists(const pybind11::list& proposals, const at::Tensor& gt_instances, const at::Tensor& batch)
{
    const at::Tensor* all[] = {&gt_instances, &batch};
    const char* names[] = {"gt_instances", "batch"};
    for (int i = 0; i < 2; ++i)
    {
        check_contiguous(*all[i], names[i]);
        check_gpu(*all[i], names[i]);
        check_dtype(*all[i], at::kLong, names[i]);
        TORCH_CHECK(all[i]->dim() == 1, names[i], " must have one dimension");
    }
    check_same_device(gt_instances, batch, "gt_instances and batch");
    TORCH_CHECK(batch.size(0) == gt_instances.size(0), "batch and gt_instances differ in length");
    const int64_t n = gt_instances.size(0), rows = static_cast<int64_t>(pybind11::len(proposals));
    if (n == 0 || rows == 0)
        return pybind11::none();
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(gt_instances.device());
    void* stream = current_stream(gt_instances);
    at::Tensor counts = at::empty({1 + TPK_IOU_SAMPLES}, gt_instances.options());
    check_status(tpk_instance_counts(n, gt_instances.data_ptr<int64_t>(), batch.data_ptr<int64_t>(), counts.data_ptr<int64_t>(), stream),
                 "instance_iou (counts)");
    at::Tensor table = at::empty({rows, 2}, at::TensorOptions().dtype(at::kLong).pinned_memory(true));
    int64_t* entry = table.data_ptr<int64_t>();
    for (int64_t p = 0; p < rows; ++p, entry += 2)
    {
        PyObject* o = PyList_GET_ITEM(proposals.ptr(), p);
        if (!THPVariable_Check(o))
            return pybind11::none();
        const at::Tensor& t = THPVariable_Unpack(o);
        if (t.dim() != 1 || t.scalar_type() != at::kLong || t.device() != gt_instances.device() || (t.size(0) > 1 && t.stride(0) != 1))
            return pybind11::none();
        entry[0] = reinterpret_cast<int64_t>(t.const_data_ptr());
        entry[1] = t.size(0);
    }
    const at::Tensor on_device = table.to(gt_instances.device(), /*non_blocking=*/true);
    int64_t found[1 + TPK_IOU_SAMPLES];
    {
        pybind11::gil_scoped_release waiting;
        check_status(tpk_instance_counts_read(counts.data_ptr<int64_t>(), found, stream), "instance_iou (counts)");
    }
    const int64_t samples = std::max<int64_t>(found[0], 0);
    if (samples > TPK_IOU_SAMPLES)
        return pybind11::none();
    int64_t total = 0;
    for (int64_t s = 0; s < samples; ++s)
        total += found[1 + s];
    at::Tensor sizes = at::empty({total}, gt_instances.options().dtype(at::kInt));
    at::Tensor iou = at::empty({rows, total}, gt_instances.options().dtype(at::kFloat));
    check_status(tpk_instance_iou_lists(total, rows, n, samples, on_device.data_ptr<int64_t>(), gt_instances.data_ptr<int64_t>(),
                                        batch.data_ptr<int64_t>(), counts.data_ptr<int64_t>(), sizes.data_ptr<int32_t>(),
                                        iou.data_ptr<float>(), stream),
                 "instance_iou");
    return pybind11::cast(iou);
}

// cuda/src/gridding.cpp:4-12 -> {grid_weights, grid_pt_weights, grid_pt_indexes}
std::vector<at::Tensor> gridding(float min_x, float max_x, float min_y, float max_y, float min_z, float max_z,
                                 at::Tensor ptcloud)
{
    check_gpu(ptcloud, "ptcloud");
    check_contiguous(ptcloud, "ptcloud");
    TORCH_CHECK(ptcloud.scalar_type() == at::kFloat || ptcloud.scalar_type() == at::kDouble,
                "ptcloud must be float32 or float64");
    TORCH_CHECK(ptcloud.dim() == 3 && ptcloud.size(2) == 3, "ptcloud must have shape (B, n_pts, 3)");
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(ptcloud.device());
    const int b = as_int(ptcloud.size(0), "batch size"), n = as_int(ptcloud.size(1), "number of points");
    const int64_t len_x = static_cast<int>(max_x - min_x + 1), len_y = static_cast<int>(max_y - min_y + 1);
    const int64_t len_z = static_cast<int>(max_z - min_z + 1);
    TORCH_CHECK(len_x > 0 && len_y > 0 && len_z > 0, "gridding: empty grid");
    at::Tensor grid = torch::empty({b, len_x * len_y * len_z}, ptcloud.options());
    at::Tensor weights = torch::empty({b, n, 8, 3}, ptcloud.options());
    at::Tensor indexes = torch::empty({b, n, 8}, ptcloud.options().dtype(at::kInt));
    if (ptcloud.scalar_type() == at::kFloat)
        check_status(tpk_gridding_f32(b, n, min_x, max_x, min_y, max_y, min_z, max_z, ptcloud.data_ptr<float>(),
                                      grid.data_ptr<float>(), weights.data_ptr<float>(), indexes.data_ptr<int32_t>(),
                                      current_stream(ptcloud)),
                     "gridding");
    else
        check_status(tpk_gridding_f64(b, n, min_x, max_x, min_y, max_y, min_z, max_z, ptcloud.data_ptr<double>(),
                                      grid.data_ptr<double>(), weights.data_ptr<double>(), indexes.data_ptr<int32_t>(),
                                      current_stream(ptcloud)),
                     "gridding");
    return {grid, weights, indexes};
}

// cuda/src/gridding.cpp:14-26
at::Tensor gridding_grad(at::Tensor grid_pt_weights, at::Tensor grid_pt_indexes, at::Tensor grad_grid)
{
    check_gpu(grid_pt_weights, "grid_pt_weights");
    check_gpu(grid_pt_indexes, "grid_pt_indexes");
    check_gpu(grad_grid, "grad_grid");
    check_contiguous(grid_pt_weights, "grid_pt_weights");
    check_contiguous(grid_pt_indexes, "grid_pt_indexes");
    check_contiguous(grad_grid, "grad_grid");
    check_dtype(grid_pt_indexes, at::kInt, "grid_pt_indexes");
    TORCH_CHECK(grid_pt_weights.scalar_type() == at::kFloat || grid_pt_weights.scalar_type() == at::kDouble,
                "grid_pt_weights must be float32 or float64");
    TORCH_CHECK(grad_grid.scalar_type() == grid_pt_weights.scalar_type(), "grad_grid and grid_pt_weights differ in dtype");
    TORCH_CHECK(grid_pt_indexes.dim() == 3 && grid_pt_indexes.size(2) == 8, "grid_pt_indexes must have shape (B, n_pts, 8)");
    TORCH_CHECK(grid_pt_weights.dim() == 4 && grid_pt_weights.size(0) == grid_pt_indexes.size(0) &&
                    grid_pt_weights.size(1) == grid_pt_indexes.size(1) && grid_pt_weights.size(2) == 8 &&
                    grid_pt_weights.size(3) == 3,
                "grid_pt_weights must have shape (B, n_pts, 8, 3)");
    TORCH_CHECK(grad_grid.dim() == 2 && grad_grid.size(0) == grid_pt_indexes.size(0), "grad_grid must have shape (B, n_grid_vertices)");
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(grad_grid.device());
    const int b = as_int(grad_grid.size(0), "batch size"), n = as_int(grid_pt_indexes.size(1), "number of points");
    const int vertices = as_int(grad_grid.size(1), "grid vertices");
    at::Tensor grad = torch::empty({b, n, 3}, grid_pt_weights.options());
    if (grid_pt_weights.scalar_type() == at::kFloat)
        check_status(tpk_gridding_grad_f32(b, n, vertices, grid_pt_weights.data_ptr<float>(),
                                           grid_pt_indexes.data_ptr<int32_t>(), grad_grid.data_ptr<float>(),
                                           grad.data_ptr<float>(), current_stream(grad_grid)),
                     "gridding_grad");
    else
        check_status(tpk_gridding_grad_f64(b, n, vertices, grid_pt_weights.data_ptr<double>(),
                                           grid_pt_indexes.data_ptr<int32_t>(), grad_grid.data_ptr<double>(),
                                           grad.data_ptr<double>(), current_stream(grad_grid)),
                     "gridding_grad");
    return grad;
}

// torch_points_kernels/gridding.py:34-60 (the reference's front end, a loop over the clouds there) for the whole
// batch: one launch forward, one backward (tpk_gridding_batch_f32).  kept: receives a copy of the points, or nullptr.
at::Tensor gridding_batch_forward(const at::Tensor& ptcloud, double scale, at::Tensor* kept = nullptr)
{
    check_gpu(ptcloud, "ptcloud");
    TORCH_CHECK(ptcloud.scalar_type() == at::kFloat || ptcloud.scalar_type() == at::kDouble,
                "ptcloud must be float32 or float64");
    TORCH_CHECK(ptcloud.dim() == 3 && ptcloud.size(2) == 3, "ptcloud must have shape (B, n_pts, 3)");
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(ptcloud.device());
    const int b = as_int(ptcloud.size(0), "batch size"), n = as_int(ptcloud.size(1), "number of points");
    const int64_t side = static_cast<int>(static_cast<float>(scale - 1) - static_cast<float>(-scale) + 1);
    TORCH_CHECK(side > 0, "gridding: empty grid");
    at::Tensor grid = at::empty({b, side * side * side}, ptcloud.options());
    if (kept)
        *kept = at::empty(ptcloud.sizes(), ptcloud.options()); // (contiguous, as ptcloud is)
    if (ptcloud.scalar_type() == at::kFloat)
        check_status(kept ? tpk_gridding_batch_keep_f32(b, n, scale, ptcloud.data_ptr<float>(), grid.data_ptr<float>(),
                                                        kept->data_ptr<float>(), current_stream(ptcloud))
                          : tpk_gridding_batch_f32(b, n, scale, ptcloud.data_ptr<float>(), grid.data_ptr<float>(),
                                                   current_stream(ptcloud)),
                     "gridding");
    else
        check_status(kept ? tpk_gridding_batch_keep_f64(b, n, scale, ptcloud.data_ptr<double>(), grid.data_ptr<double>(),
                                                        kept->data_ptr<double>(), current_stream(ptcloud))
                          : tpk_gridding_batch_f64(b, n, scale, ptcloud.data_ptr<double>(), grid.data_ptr<double>(),
                                                   current_stream(ptcloud)),
                     "gridding");
    return grid;
}

at::Tensor gridding_batch_backward(const at::Tensor& ptcloud, double scale, const at::Tensor& grad_grid)
{
    check_gpu(grad_grid, "grad_grid");
    check_same_device(ptcloud, grad_grid, "ptcloud and grad_grid");
    TORCH_CHECK(grad_grid.scalar_type() == ptcloud.scalar_type(), "grad_grid and ptcloud differ in dtype");
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(ptcloud.device());
    const int b = as_int(ptcloud.size(0), "batch size"), n = as_int(ptcloud.size(1), "number of points");
    at::Tensor grad = at::empty(ptcloud.sizes(), ptcloud.options());
    if (ptcloud.scalar_type() == at::kFloat)
        check_status(tpk_gridding_batch_grad_f32(b, n, scale, ptcloud.data_ptr<float>(), grad_grid.data_ptr<float>(),
                                                 grad.data_ptr<float>(), current_stream(ptcloud)),
                     "gridding_grad");
    else
        check_status(tpk_gridding_batch_grad_f64(b, n, scale, ptcloud.data_ptr<double>(), grad_grid.data_ptr<double>(),
                                                 grad.data_ptr<double>(), current_stream(ptcloud)),
                     "gridding_grad");
    return grad;
}

// cuda/src/cubic_feature_sampling.cpp:4-16 -> {point_features, grid_pt_indexes}
// mapped: ptcloud in [-1, 1), as the front end takes it.
std::vector<at::Tensor> sample_cubes(int scale, int neighborhood_size, const at::Tensor& ptcloud, const at::Tensor& cubic_features,
                                     bool mapped)
{
    check_gpu(ptcloud, "ptcloud");
    check_gpu(cubic_features, "cubic_features");
    check_contiguous(ptcloud, "ptcloud");
    check_contiguous(cubic_features, "cubic_features");
    check_same_device(ptcloud, cubic_features, "ptcloud and cubic_features");
    TORCH_CHECK(ptcloud.scalar_type() == at::kFloat || ptcloud.scalar_type() == at::kDouble,
                "ptcloud must be float32 or float64");
    TORCH_CHECK(cubic_features.scalar_type() == ptcloud.scalar_type(), "ptcloud and cubic_features differ in dtype");
    TORCH_CHECK(ptcloud.dim() == 3 && ptcloud.size(2) == 3, "ptcloud must have shape (B, n_pts, 3)");
    TORCH_CHECK(cubic_features.dim() == 5 && cubic_features.size(0) == ptcloud.size(0) && cubic_features.size(2) == scale &&
                    cubic_features.size(3) == scale && cubic_features.size(4) == scale,
                "cubic_features must have shape (B, c, scale, scale, scale)");
    TORCH_CHECK(neighborhood_size >= 1 && neighborhood_size <= 64, "neighborhood_size out of range");
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(ptcloud.device());
    const int b = as_int(ptcloud.size(0), "batch size"), n = as_int(ptcloud.size(1), "number of points");
    const int channels = as_int(cubic_features.size(1), "channels");
    const int64_t side = 2 * static_cast<int64_t>(neighborhood_size), vertices = side * side * side;
    at::Tensor features = torch::empty({b, n, vertices, channels}, ptcloud.options());
    at::Tensor indexes = torch::empty({b, n, vertices}, ptcloud.options().dtype(at::kInt));
    const bool single = ptcloud.scalar_type() == at::kFloat;
    const size_t ws_bytes = tpk_cubic_feature_sampling_workspace_bytes(b, n, channels, scale, neighborhood_size, single ? 4 : 8);
    at::Tensor ws;
    if (ws_bytes)
        ws = at::empty({static_cast<int64_t>(ws_bytes)}, ptcloud.options().dtype(at::kByte));
    void* wsp = ws_bytes ? ws.data_ptr() : nullptr;
    if (single)
        check_status(tpk_cubic_feature_sampling_ws_f32(b, n, channels, scale, neighborhood_size, mapped, ptcloud.data_ptr<float>(),
                                                       cubic_features.data_ptr<float>(), features.data_ptr<float>(),
                                                       indexes.data_ptr<int32_t>(), wsp, ws_bytes, current_stream(ptcloud)),
                     "cubic_feature_sampling");
    else
        check_status(tpk_cubic_feature_sampling_ws_f64(b, n, channels, scale, neighborhood_size, mapped, ptcloud.data_ptr<double>(),
                                                       cubic_features.data_ptr<double>(), features.data_ptr<double>(),
                                                       indexes.data_ptr<int32_t>(), wsp, ws_bytes, current_stream(ptcloud)),
                     "cubic_feature_sampling");
    return {features, indexes};
}

std::vector<at::Tensor> cubic_feature_sampling(int scale, int neighborhood_size, at::Tensor ptcloud,
                                               at::Tensor cubic_features)
{
    return sample_cubes(scale, neighborhood_size, ptcloud, cubic_features, false);
}

// cuda/src/cubic_feature_sampling.cpp:18-30 -> {grad_ptcloud, grad_cubic_features}
std::vector<at::Tensor> sample_cubes_grad(int scale, int neighborhood_size, const at::Tensor& grad_point_features,
                                          const at::Tensor& grid_pt_indexes, bool points_too)
{
    check_gpu(grad_point_features, "grad_point_features");
    check_gpu(grid_pt_indexes, "grid_pt_indexes");
    check_contiguous(grad_point_features, "grad_point_features");
    check_contiguous(grid_pt_indexes, "grid_pt_indexes");
    check_dtype(grid_pt_indexes, at::kInt, "grid_pt_indexes");
    TORCH_CHECK(grad_point_features.scalar_type() == at::kFloat || grad_point_features.scalar_type() == at::kDouble,
                "grad_point_features must be float32 or float64");
    TORCH_CHECK(neighborhood_size >= 1 && neighborhood_size <= 64, "neighborhood_size out of range");
    TORCH_CHECK(scale > 0, "scale must be positive");
    const int64_t side = 2 * static_cast<int64_t>(neighborhood_size), vertices = side * side * side;
    TORCH_CHECK(grid_pt_indexes.dim() == 3 && grid_pt_indexes.size(2) == vertices, "grid_pt_indexes must have shape (B, n_pts, n_vertices)");
    TORCH_CHECK(grad_point_features.dim() == 4 && grad_point_features.size(0) == grid_pt_indexes.size(0) &&
                    grad_point_features.size(1) == grid_pt_indexes.size(1) && grad_point_features.size(2) == vertices,
                "grad_point_features must have shape (B, n_pts, n_vertices, c)");
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(grad_point_features.device());
    const int b = as_int(grad_point_features.size(0), "batch size"), n = as_int(grid_pt_indexes.size(1), "number of points");
    const int channels = as_int(grad_point_features.size(3), "channels");
    at::Tensor grad_ptcloud;
    if (points_too)
        grad_ptcloud = torch::empty({b, n, 3}, grad_point_features.options());
    at::Tensor grad_cubic = torch::empty({b, channels, scale, scale, scale}, grad_point_features.options());
    if (grad_point_features.scalar_type() == at::kFloat)
        check_status(tpk_cubic_feature_sampling_grad_f32(b, n, channels, scale, neighborhood_size,
                                                         grad_point_features.data_ptr<float>(),
                                                         grid_pt_indexes.data_ptr<int32_t>(), points_too ? grad_ptcloud.data_ptr<float>() : nullptr,
                                                         grad_cubic.data_ptr<float>(), current_stream(grad_point_features)),
                     "cubic_feature_sampling_grad");
    else
        check_status(tpk_cubic_feature_sampling_grad_f64(b, n, channels, scale, neighborhood_size,
                                                         grad_point_features.data_ptr<double>(),
                                                         grid_pt_indexes.data_ptr<int32_t>(), points_too ? grad_ptcloud.data_ptr<double>() : nullptr,
                                                         grad_cubic.data_ptr<double>(), current_stream(grad_point_features)),
                     "cubic_feature_sampling_grad");
    return {grad_ptcloud, grad_cubic};
}

std::vector<at::Tensor> cubic_feature_sampling_grad(int scale, int neighborhood_size, at::Tensor grad_point_features,
                                                    at::Tensor grid_pt_indexes)
{
    return sample_cubes_grad(scale, neighborhood_size, grad_point_features, grid_pt_indexes, true);
}

void check_group(const at::Tensor& features, const at::Tensor& idx)
{
    check_contiguous(features, "features");
    check_contiguous(idx, "idx");
    check_f32(features, "features");
    check_dtype(idx, at::kLong, "idx");
    check_gpu(features, "features");
    check_gpu(idx, "idx");
    check_same_device(features, idx, "features and idx");
    TORCH_CHECK(features.dim() == 3, "features must have shape (B, C, N)");
    TORCH_CHECK(idx.dim() == 3 && idx.size(0) == features.size(0),
                "idx must have shape (B, npoint, nsample)");
}

// No counterpart in the reference's native module: its grouping_operation is
// torch.gather on a repeated index (torch_points_kernels/torchpoints.py:129-146).
at::Tensor grouping_operation(at::Tensor features, at::Tensor idx)
{
    check_group(features, idx);
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(features.device());

    at::Tensor out = torch::empty({features.size(0), features.size(1), idx.size(1), idx.size(2)},
                                  at::device(features.device()).dtype(at::ScalarType::Float));
    check_status(tpk_group_f32(as_int(features.size(0), "batch size"),
                               as_int(features.size(1), "channels"), as_int(features.size(2), "N"),
                               as_int(idx.size(1), "npoint"), as_int(idx.size(2), "nsample"),
                               features.data_ptr<float>(), idx.data_ptr<int64_t>(),
                               out.data_ptr<float>(), current_stream(features)),
                 "grouping_operation");
    return out;
}

at::Tensor grouping_operation_grad(at::Tensor grad_out, at::Tensor idx, const int n)
{
    check_contiguous(grad_out, "grad_out");
    check_contiguous(idx, "idx");
    check_f32(grad_out, "grad_out");
    check_dtype(idx, at::kLong, "idx");
    check_gpu(grad_out, "grad_out");
    check_gpu(idx, "idx");
    check_same_device(grad_out, idx, "grad_out and idx");
    TORCH_CHECK(grad_out.dim() == 4, "grad_out must have shape (B, C, npoint, nsample)");
    TORCH_CHECK(idx.dim() == 3 && idx.size(0) == grad_out.size(0) &&
                    idx.size(1) == grad_out.size(2) && idx.size(2) == grad_out.size(3),
                "idx must have shape (B, npoint, nsample)");
    TORCH_CHECK(n >= 0, "n must be non-negative");
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(grad_out.device());

    at::Tensor out = torch::empty({grad_out.size(0), grad_out.size(1), n},
                                  at::device(grad_out.device()).dtype(at::ScalarType::Float));
    const int b = as_int(grad_out.size(0), "batch size");
    const int npoint = as_int(idx.size(1), "npoint");
    const int nsample = as_int(idx.size(2), "nsample");
    const size_t ws_bytes = tpk_group_grad_workspace_bytes(b, n, npoint, nsample);
    at::Tensor ws = torch::empty({static_cast<int64_t>(ws_bytes)},
                                 at::device(grad_out.device()).dtype(at::ScalarType::Byte));
    check_status(tpk_group_grad_f32(b, as_int(grad_out.size(1), "channels"), n, npoint, nsample,
                                    grad_out.data_ptr<float>(), idx.data_ptr<int64_t>(),
                                    out.data_ptr<float>(), ws_bytes ? ws.data_ptr() : nullptr,
                                    ws_bytes, current_stream(grad_out)),
                 "grouping_operation_grad");
    return out;
}

// grouping_operation for a caller that will ask for the gradient: as three_interpolate_recording.
std::pair<at::Tensor, at::Tensor> grouping_operation_recording(at::Tensor features, at::Tensor idx)
{
    check_group(features, idx);
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(features.device());
    const int b = as_int(features.size(0), "batch size"), c = as_int(features.size(1), "channels"), n = as_int(features.size(2), "N");
    const int npoint = as_int(idx.size(1), "npoint"), nsample = as_int(idx.size(2), "nsample");
    const size_t bytes = tpk_group_grad_workspace_bytes(b, n, npoint, nsample);
    if (bytes == 0)
        return {grouping_operation(features, idx), torch::empty({0}, at::device(features.device()).dtype(at::kByte))};
    at::Tensor lists = torch::empty({static_cast<int64_t>(bytes)}, at::device(features.device()).dtype(at::kByte));
    at::Tensor output =
        torch::empty({features.size(0), features.size(1), idx.size(1), idx.size(2)}, at::device(features.device()).dtype(at::kFloat));
    check_status(tpk_group_recording_f32(b, c, n, npoint, nsample, features.data_ptr<float>(), idx.data_ptr<int64_t>(),
                                         output.data_ptr<float>(), lists.data_ptr(), bytes, current_stream(features)),
                 "grouping_operation (with the lists for the backward pass)");
    return {output, lists};
}

at::Tensor grouping_operation_grad_lists(at::Tensor grad_out, at::Tensor lists, const int n)
{
    check_contiguous(grad_out, "grad_out");
    check_f32(grad_out, "grad_out");
    check_gpu(grad_out, "grad_out");
    check_gpu(lists, "lists");
    check_same_device(grad_out, lists, "grad_out and lists");
    TORCH_CHECK(grad_out.dim() == 4, "grad_out must have shape (B, C, npoint, nsample)");
    TORCH_CHECK(lists.scalar_type() == at::kByte && lists.is_contiguous() && n >= 0, "lists as grouping_operation_recording returned them");
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(grad_out.device());
    at::Tensor out = torch::empty({grad_out.size(0), grad_out.size(1), n}, at::device(grad_out.device()).dtype(at::kFloat));
    check_status(tpk_group_grad_lists_f32(as_int(grad_out.size(0), "batch size"), as_int(grad_out.size(1), "channels"), n,
                                          as_int(grad_out.size(2), "npoint"), as_int(grad_out.size(3), "nsample"),
                                          grad_out.data_ptr<float>(), lists.data_ptr(), static_cast<size_t>(lists.numel()),
                                          out.data_ptr<float>(), current_stream(grad_out)),
                 "grouping_operation_grad (from lists)");
    return out;
}

// cuda/src/chamfer_dist.cpp:3-6 -> cuda/src/chamfer_dist_gpu.cu:157-184
std::vector<torch::Tensor> chamfer_dist(torch::Tensor xyz1, torch::Tensor xyz2)
{
    check_gpu(xyz1, "xyz1");
    check_gpu(xyz2, "xyz2");
    check_same_device(xyz1, xyz2, "xyz1 and xyz2");
    check_points(xyz1, 3, "xyz1");
    check_points(xyz2, 3, "xyz2");
    TORCH_CHECK(xyz1.size(0) == xyz2.size(0), "xyz1 and xyz2 differ in batch size");
    TORCH_CHECK(xyz1.scalar_type() == xyz2.scalar_type(), "xyz1 and xyz2 differ in dtype");
    TORCH_CHECK(xyz1.scalar_type() == at::kFloat || xyz1.scalar_type() == at::kDouble,
                "chamfer_dist supports float32 and float64");
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(xyz1.device());
    xyz1 = xyz1.contiguous();
    xyz2 = xyz2.contiguous();

    const int b = as_int(xyz1.size(0), "batch size");
    const int n = as_int(xyz1.size(1), "points of xyz1");
    const int m = as_int(xyz2.size(1), "points of xyz2");
    auto fopt = xyz1.options();
    auto iopt = xyz1.options().dtype(torch::kInt);
    torch::Tensor dist1 = torch::empty({b, n}, fopt);
    torch::Tensor dist2 = torch::empty({b, m}, fopt);
    torch::Tensor idx1 = torch::empty({b, n}, iopt);
    torch::Tensor idx2 = torch::empty({b, m}, iopt);
    void* s = current_stream(xyz1);
    if (xyz1.scalar_type() == at::kFloat)
    {
        const size_t ws_bytes = tpk_chamfer_fwd_workspace_bytes(b, n, m);
        torch::Tensor ws;
        if (ws_bytes)
            ws = torch::empty({static_cast<int64_t>(ws_bytes)}, xyz1.options().dtype(torch::kUInt8));
        check_status(tpk_chamfer_fwd_f32(b, n, m, xyz1.data_ptr<float>(), xyz2.data_ptr<float>(),
                                         dist1.data_ptr<float>(), dist2.data_ptr<float>(),
                                         idx1.data_ptr<int32_t>(), idx2.data_ptr<int32_t>(),
                                         ws_bytes ? ws.data_ptr() : nullptr, ws_bytes, s),
                     "chamfer_dist");
    }
    else
        check_status(tpk_chamfer_fwd_f64(b, n, m, xyz1.data_ptr<double>(),
                                         xyz2.data_ptr<double>(), dist1.data_ptr<double>(),
                                         dist2.data_ptr<double>(), idx1.data_ptr<int32_t>(),
                                         idx2.data_ptr<int32_t>(), s),
                     "chamfer_dist");
    return {dist1, dist2, idx1, idx2};
}

// cuda/src/chamfer_dist.cpp:8-13 -> cuda/src/chamfer_dist_gpu.cu:215-245
std::vector<torch::Tensor> chamfer_dist_grad(torch::Tensor xyz1, torch::Tensor xyz2,
                                             torch::Tensor idx1, torch::Tensor idx2,
                                             torch::Tensor grad_dist1, torch::Tensor grad_dist2)
{
    check_gpu(xyz1, "xyz1");
    check_gpu(xyz2, "xyz2");
    check_gpu(idx1, "idx1");
    check_gpu(idx2, "idx2");
    check_gpu(grad_dist1, "grad_dist1");
    check_gpu(grad_dist2, "grad_dist2");
    check_points(xyz1, 3, "xyz1");
    check_points(xyz2, 3, "xyz2");
    check_dtype(idx1, at::kInt, "idx1");
    check_dtype(idx2, at::kInt, "idx2");
    TORCH_CHECK(xyz1.scalar_type() == xyz2.scalar_type() &&
                    xyz1.scalar_type() == grad_dist1.scalar_type() &&
                    xyz1.scalar_type() == grad_dist2.scalar_type(),
                "clouds and gradients differ in dtype");
    TORCH_CHECK(xyz1.scalar_type() == at::kFloat || xyz1.scalar_type() == at::kDouble,
                "chamfer_dist_grad supports float32 and float64");
    const int b = as_int(xyz1.size(0), "batch size");
    const int n = as_int(xyz1.size(1), "points of xyz1");
    const int m = as_int(xyz2.size(1), "points of xyz2");
    TORCH_CHECK(xyz2.size(0) == b && idx1.numel() == static_cast<int64_t>(b) * n &&
                    idx2.numel() == static_cast<int64_t>(b) * m &&
                    grad_dist1.numel() == idx1.numel() && grad_dist2.numel() == idx2.numel(),
                "shapes of clouds, indices and gradients do not match");
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(xyz1.device());
    xyz1 = xyz1.contiguous();
    xyz2 = xyz2.contiguous();
    idx1 = idx1.contiguous();
    idx2 = idx2.contiguous();
    grad_dist1 = grad_dist1.contiguous();
    grad_dist2 = grad_dist2.contiguous();

    torch::Tensor grad_xyz1 = torch::empty_like(xyz1);
    torch::Tensor grad_xyz2 = torch::empty_like(xyz2);
    const size_t ws_bytes = tpk_chamfer_bwd_workspace_bytes(b, n, m);
    torch::Tensor ws = torch::empty({static_cast<int64_t>(ws_bytes)}, xyz1.options().dtype(torch::kByte));
    void* wsp = ws_bytes ? ws.data_ptr() : nullptr;
    void* s = current_stream(xyz1);
    if (xyz1.scalar_type() == at::kFloat)
        check_status(tpk_chamfer_bwd_f32(b, n, m, xyz1.data_ptr<float>(), xyz2.data_ptr<float>(),
                                         idx1.data_ptr<int32_t>(), idx2.data_ptr<int32_t>(),
                                         grad_dist1.data_ptr<float>(),
                                         grad_dist2.data_ptr<float>(),
                                         grad_xyz1.data_ptr<float>(),
                                         grad_xyz2.data_ptr<float>(), wsp, ws_bytes, s),
                     "chamfer_dist_grad");
    else
        check_status(tpk_chamfer_bwd_f64(b, n, m, xyz1.data_ptr<double>(),
                                         xyz2.data_ptr<double>(), idx1.data_ptr<int32_t>(),
                                         idx2.data_ptr<int32_t>(), grad_dist1.data_ptr<double>(),
                                         grad_dist2.data_ptr<double>(),
                                         grad_xyz1.data_ptr<double>(),
                                         grad_xyz2.data_ptr<double>(), wsp, ws_bytes, s),
                     "chamfer_dist_grad");
    return {grad_xyz1, grad_xyz2};
}

// mean(dist1) + mean(dist2) over the whole batch, what the reference's chamfer_dist.py:25-54 makes of the distances, and
// the nearest neighbours its gradient needs: {loss, idx1 (b, n) then idx2 (b, m) in one array}.
std::vector<at::Tensor> chamfer_loss_forward(const at::Tensor& xyz1, const at::Tensor& xyz2)
{
    check_gpu(xyz1, "xyz1");
    check_gpu(xyz2, "xyz2");
    check_same_device(xyz1, xyz2, "xyz1 and xyz2");
    check_points(xyz1, 3, "xyz1");
    check_points(xyz2, 3, "xyz2");
    TORCH_CHECK(xyz1.size(0) == xyz2.size(0), "xyz1 and xyz2 differ in batch size");
    TORCH_CHECK(xyz1.scalar_type() == xyz2.scalar_type(), "xyz1 and xyz2 differ in dtype");
    TORCH_CHECK(xyz1.scalar_type() == at::kFloat || xyz1.scalar_type() == at::kDouble, "chamfer_dist supports float32 and float64");
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(xyz1.device());
    const int b = as_int(xyz1.size(0), "batch size"), n = as_int(xyz1.size(1), "points of xyz1"), m = as_int(xyz2.size(1), "points of xyz2");
    const bool narrow = xyz1.scalar_type() == at::kFloat;
    const size_t total1 = static_cast<size_t>(b) * n, total2 = static_cast<size_t>(b) * m;
    at::Tensor idx = torch::empty({static_cast<int64_t>(total1 + total2)}, xyz1.options().dtype(at::kInt));
    at::Tensor loss = torch::empty({}, xyz1.options());
    int32_t* const idx1 = idx.data_ptr<int32_t>();
    void* const s = current_stream(xyz1);
    // one scratch: the search's workspace, the sums' workspace, the distances
    const size_t ws_bytes = narrow ? tpk_chamfer_fwd_workspace_bytes(b, n, m) : 0, sum_bytes = tpk_chamfer_loss_workspace_bytes(b, n, m);
    const size_t sums_at = (ws_bytes + 255) & ~static_cast<size_t>(255), dist_at = (sums_at + sum_bytes + 255) & ~static_cast<size_t>(255);
    at::Tensor scratch = torch::empty({static_cast<int64_t>(dist_at + (total1 + total2) * xyz1.element_size())}, xyz1.options().dtype(at::kByte));
    char* const bytes = static_cast<char*>(scratch.data_ptr());
    void* const ws = ws_bytes ? bytes : nullptr;
    void* const sums = sum_bytes ? bytes + sums_at : nullptr;
    if (narrow)
    {
        float* const dist1 = reinterpret_cast<float*>(bytes + dist_at);
        check_status(tpk_chamfer_fwd_f32(b, n, m, xyz1.data_ptr<float>(), xyz2.data_ptr<float>(), dist1, dist1 + total1, idx1, idx1 + total1,
                                         ws, ws_bytes, s),
                     "chamfer_dist");
        check_status(tpk_chamfer_loss_f32(b, n, m, dist1, dist1 + total1, loss.data_ptr<float>(), sums, sum_bytes, s), "chamfer_dist");
    }
    else
    {
        double* const dist1 = reinterpret_cast<double*>(bytes + dist_at);
        check_status(tpk_chamfer_fwd_f64(b, n, m, xyz1.data_ptr<double>(), xyz2.data_ptr<double>(), dist1, dist1 + total1, idx1,
                                         idx1 + total1, s),
                     "chamfer_dist");
        check_status(tpk_chamfer_loss_f64(b, n, m, dist1, dist1 + total1, loss.data_ptr<double>(), sums, sum_bytes, s), "chamfer_dist");
    }
    return {loss, idx};
}

std::vector<at::Tensor> chamfer_loss_backward(const at::Tensor& xyz1, const at::Tensor& xyz2, const at::Tensor& idx, const at::Tensor& grad_loss)
{
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(xyz1.device());
    check_gpu(grad_loss, "the gradient of the loss");
    TORCH_CHECK(grad_loss.scalar_type() == xyz1.scalar_type() && grad_loss.numel() == 1, "the gradient of the loss is one number of its type");
    const int b = as_int(xyz1.size(0), "batch size"), n = as_int(xyz1.size(1), "points of xyz1"), m = as_int(xyz2.size(1), "points of xyz2");
    at::Tensor grad_xyz1 = torch::empty_like(xyz1), grad_xyz2 = torch::empty_like(xyz2);
    const int32_t* const idx1 = idx.data_ptr<int32_t>();
    const int32_t* const idx2 = idx1 + static_cast<int64_t>(b) * n;
    void* const s = current_stream(xyz1);
    if (xyz1.scalar_type() == at::kFloat)
        check_status(tpk_chamfer_loss_bwd_f32(b, n, m, xyz1.data_ptr<float>(), xyz2.data_ptr<float>(), idx1, idx2, grad_loss.data_ptr<float>(),
                                              grad_xyz1.data_ptr<float>(), grad_xyz2.data_ptr<float>(), s),
                     "chamfer_dist_grad");
    else
        check_status(tpk_chamfer_loss_bwd_f64(b, n, m, xyz1.data_ptr<double>(), xyz2.data_ptr<double>(), idx1, idx2,
                                              grad_loss.data_ptr<double>(), grad_xyz1.data_ptr<double>(), grad_xyz2.data_ptr<double>(), s),
                     "chamfer_dist_grad");
    return {grad_xyz1, grad_xyz2};
}

#include "differentiable.h"

} // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m)
{
    m.def("furthest_point_sampling", &furthest_point_sampling);
    m.def("three_nn", &three_nn);
    m.def("three_nn_distance", &three_nn_distance);
    m.def("dense_knn", &dense_knn);
    m.def("grow_proximity", &grow_proximity, pybind11::arg("neighbours"), pybind11::arg("min_cluster_size"), pybind11::arg("reference_order"),
          pybind11::arg("most_staged") = grow_walk::MOST_STAGED, pybind11::call_guard<pybind11::gil_scoped_release>());
    m.def("region_grow", &region_grow, pybind11::call_guard<pybind11::gil_scoped_release>());
    m.def("instance_iou_cuda", &instance_iou_cuda);
    m.def("instance_iou_lists", &instance_iou_lists);
    m.def("gridding", &gridding);
    m.def("gridding_grad", &gridding_grad);
    m.def("gridding_batch", &gridding_batch);
    m.def("cubic_sampling", &cubic_sampling);
    m.def("cubic_feature_sampling", &cubic_feature_sampling);
    m.def("cubic_feature_sampling_grad", &cubic_feature_sampling_grad);
    m.def("three_interpolate", &three_interpolate);
    m.def("three_interpolate_grad", &three_interpolate_grad);
    m.def("three_interpolate_recording", &three_interpolate_recording);
    m.def("three_interpolate_grad_lists", &three_interpolate_grad_lists);
    m.def("ball_query_dense", &ball_query_dense, pybind11::arg("new_xyz"), pybind11::arg("xyz"), pybind11::arg("radius"),
          pybind11::arg("nsample"), pybind11::arg("sorted") = false);
    m.def("ball_query_partial_dense", &ball_query_partial_dense, pybind11::arg("x"), pybind11::arg("y"),
          pybind11::arg("batch_x"), pybind11::arg("batch_y"), pybind11::arg("radius"), pybind11::arg("nsample"),
          pybind11::arg("sorted") = false);
    m.def("grouping_operation", &grouping_operation);
    m.def("grouping_operation_grad", &grouping_operation_grad);
    m.def("grouping_operation_recording", &grouping_operation_recording);
    m.def("grouping_operation_grad_lists", &grouping_operation_grad_lists);
    m.def("chamfer_dist", &chamfer_dist);
    m.def("chamfer_dist_grad", &chamfer_dist_grad);
    m.def("interpolate_features", &interpolate_features);
    m.def("group_features", &group_features);
    m.def("chamfer_loss", &chamfer_loss);
    m.def("tpk_version", &tpk_version);
}
