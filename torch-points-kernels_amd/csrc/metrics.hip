// IoU between proposed instances and ground-truth instances (PointGroup's scoring step).
// Reference: cuda/src/metrics_gpu.cu:9-61 - one block per proposal, one thread per ground-truth
// instance, each thread walking the whole proposal: |proposal| x instances label look-ups.
// Here a workgroup owns a proposal and counts its points per ground-truth instance once, in an
// LDS histogram (integer LDS atomics); the quotients are then formed from the counts:
// |proposal| + instances steps.  Samples with more instances than the histogram holds fall back
// to the reference's walk.  Every element of the output row is written (zeros outside the columns
// of the proposal's sample; the reference pre-zeroes the tensor, cuda/src/metrics.cpp:37-39).
#include "tpk_device.h"

namespace {

constexpr int IOU_THREADS = 256;
constexpr int IOU_BINS = 8192; // ground-truth instances of one sample counted in LDS (32 KiB)

// The kernel's expression, with its types: float operands, the 1e-5 a double, stored as float.
__device__ __forceinline__ float iou_value(int intersection, int proposal_total, int instance_total)
{
    return static_cast<float>(static_cast<float>(intersection) /
                              (static_cast<float>(proposal_total + instance_total - intersection) + 1e-5));
}

// One proposal: its points' labels counted per ground-truth instance of its sample (columns first ..
// first + count of the row), then the quotients.  Called by a whole workgroup.
template <typename Size>
__device__ __forceinline__ void proposal_row(int* bins, const int64_t* __restrict__ points, int64_t length, int64_t n_points,
                                             const int64_t* __restrict__ labels, int64_t total_instances, int64_t first, int64_t count,
                                             const Size* __restrict__ instance_pointnum, float* __restrict__ row)
{
    const int tid = threadIdx.x;
    if (first < 0 || count < 0 || first + count > total_instances)
        count = 0; // inconsistent description: the row stays zero
    for (int64_t c = tid; c < total_instances; c += IOU_THREADS)
        if (c < first || c >= first + count)
            row[c] = 0.0f;
    const int proposal_total = static_cast<int>(length);
    if (count <= IOU_BINS)
    {
        for (int k = tid; k < count; k += IOU_THREADS)
            bins[k] = 0;
        __syncthreads();
        for (int64_t i = tid; i < length; i += IOU_THREADS)
        {
            const int64_t point = points[i];
            if (point < 0 || point >= n_points)
                continue;
            const int label = static_cast<int>(labels[point]); // label k + 1 = instance k; 0: none
            if (label >= 1 && label <= count)
                atomicAdd(&bins[label - 1], 1);
        }
        __syncthreads();
        for (int k = tid; k < count; k += IOU_THREADS)
            row[first + k] = iou_value(bins[k], proposal_total, static_cast<int>(instance_pointnum[first + k]));
        __syncthreads(); // the histogram is reused by the next proposal
    }
    else
    {
        for (int64_t k = tid; k < count; k += IOU_THREADS)
        {
            int intersection = 0;
            for (int64_t i = 0; i < length; ++i)
            {
                const int64_t point = points[i];
                if (point >= 0 && point < n_points && static_cast<int>(labels[point]) == k + 1)
                    ++intersection;
            }
            row[first + k] = iou_value(intersection, proposal_total, static_cast<int>(instance_pointnum[first + k]));
        }
    }
}

// The sample a proposal is compared with: that of its first point; -1 if there is none.
__device__ __forceinline__ int64_t proposal_sample(const int64_t* points, int64_t length, int64_t n_points, int64_t n_samples,
                                                   const int64_t* __restrict__ batch)
{
    if (length <= 0)
        return -1;
    const int64_t point = points[0];
    const int64_t sample = point >= 0 && point < n_points ? batch[point] : -1;
    return sample >= 0 && sample < n_samples ? sample : -1;
}

__global__ __launch_bounds__(IOU_THREADS) void instance_iou_kernel(
    int64_t total_instances, int64_t n_proposals, int64_t n_points, int64_t n_samples,
    const int64_t* __restrict__ n_instances, const int64_t* __restrict__ proposals_idx,
    const int64_t* __restrict__ proposals_offset, const int64_t* __restrict__ labels,
    const int64_t* __restrict__ instance_offset, const int64_t* __restrict__ batch,
    const int64_t* __restrict__ instance_pointnum, float* __restrict__ iou)
{
    __shared__ int bins[IOU_BINS];
    for (int64_t p = blockIdx.x; p < n_proposals; p += gridDim.x)
    {
        const int64_t start = proposals_offset[p], length = proposals_offset[p + 1] - start;
        const int64_t sample = proposal_sample(proposals_idx + start, length, n_points, n_samples, batch);
        proposal_row(bins, proposals_idx + start, length, n_points, labels, total_instances,
                     sample < 0 ? 0 : instance_offset[sample], sample < 0 ? 0 : n_instances[sample], instance_pointnum,
                     iou + p * total_instances);
    }
}

// ---- proposals as they stand: a list of index arrays, ground truth described on the device ------

// counts[0]: samples (the last point's sample + 1); counts[1 + s]: instances of sample s = its largest
// label, at least 0.  Samples beyond TPK_IOU_SAMPLES are not counted (the host sees that from counts[0]).
__global__ __launch_bounds__(IOU_THREADS) void instance_counts_clear_kernel(int64_t n_points, const int64_t* __restrict__ batch,
                                                                            int64_t* __restrict__ counts)
{
    for (int i = threadIdx.x; i < TPK_IOU_SAMPLES; i += IOU_THREADS)
        counts[1 + i] = 0;
    if (threadIdx.x == 0)
        counts[0] = batch[n_points - 1] + 1;
}

// Points per workgroup: 4 per thread, so that their loads are in flight together.  The histogram's workgroups are large,
// because each adds all its columns to the one array at its end.
constexpr int IOU_COUNT_POINTS = 4 * IOU_THREADS;
constexpr int IOU_SIZE_THREADS = 1024;
constexpr int IOU_SIZE_POINTS = 4 * IOU_SIZE_THREADS;

__global__ __launch_bounds__(IOU_THREADS) void instance_counts_kernel(int64_t n_points, const int64_t* __restrict__ labels,
                                                                      const int64_t* __restrict__ batch, int64_t* counts)
{
    __shared__ unsigned long long largest[2]; // of the sample of the workgroup's first point, and of the one after it
    if (threadIdx.x < 2)
        largest[threadIdx.x] = 0;
    __syncthreads();
    const int64_t begin = static_cast<int64_t>(blockIdx.x) * IOU_COUNT_POINTS;
    const int64_t here = batch[begin];
    int64_t best[2] = {0, 0};
#pragma unroll 4
    for (int64_t i = begin + threadIdx.x; i < n_points && i < begin + IOU_COUNT_POINTS; i += IOU_THREADS)
    {
        const int64_t sample = batch[i], label = labels[i];
        if (sample == here)
            best[0] = max(best[0], label);
        else if (sample == here + 1)
            best[1] = max(best[1], label);
        else if (sample >= 0 && sample < TPK_IOU_SAMPLES && label > 0)
            atomicMax(reinterpret_cast<unsigned long long*>(&counts[1 + sample]), static_cast<unsigned long long>(label));
    }
    for (int k = 0; k < 2; ++k)
        if (best[k] > 0)
            atomicMax(&largest[k], static_cast<unsigned long long>(best[k]));
    __syncthreads();
    if (threadIdx.x < 2)
    {
        const int64_t sample = here + threadIdx.x;
        if (largest[threadIdx.x] > 0 && sample >= 0 && sample < TPK_IOU_SAMPLES)
            atomicMax(reinterpret_cast<unsigned long long*>(&counts[1 + sample]), largest[threadIdx.x]);
    }
}

// Columns before sample s, for all samples: every workgroup forms them for itself (there are few).
__device__ __forceinline__ void first_columns(int n_samples, const int64_t* __restrict__ counts, int* firsts)
{
    if (threadIdx.x == 0)
    {
        int at = 0;
        for (int s = 0; s < n_samples; ++s)
        {
            firsts[s] = at;
            at += static_cast<int>(counts[1 + s]);
        }
    }
    __syncthreads();
}

__global__ __launch_bounds__(IOU_THREADS) void instance_sizes_clear_kernel(int total_instances, int* __restrict__ sizes)
{
    const int i = blockIdx.x * IOU_THREADS + threadIdx.x;
    if (i < total_instances)
        sizes[i] = 0;
}

// Points per ground-truth instance: a histogram in LDS where the columns fit, added to `sizes` once per workgroup.
__global__ __launch_bounds__(IOU_SIZE_THREADS) void instance_sizes_kernel(int64_t n_points, int n_samples, int total_instances,
                                                                     const int64_t* __restrict__ labels,
                                                                     const int64_t* __restrict__ batch,
                                                                     const int64_t* __restrict__ counts, int* sizes)
{
    __shared__ int firsts[TPK_IOU_SAMPLES];
    __shared__ int bins[IOU_BINS];
    const bool in_lds = total_instances <= IOU_BINS;
    if (in_lds)
        for (int i = threadIdx.x; i < total_instances; i += IOU_SIZE_THREADS)
            bins[i] = 0;
    first_columns(n_samples, counts, firsts);
    const int64_t begin = static_cast<int64_t>(blockIdx.x) * IOU_SIZE_POINTS;
    for (int64_t i = begin + threadIdx.x; i < n_points && i < begin + IOU_SIZE_POINTS; i += IOU_SIZE_THREADS)
    {
        const int64_t sample = batch[i], label = labels[i];
        if (sample < 0 || sample >= n_samples || label <= 0)
            continue;
        const int column = firsts[sample] + static_cast<int>(label) - 1;
        atomicAdd(in_lds ? &bins[column] : &sizes[column], 1);
    }
    __syncthreads();
    if (in_lds)
        for (int i = threadIdx.x; i < total_instances; i += IOU_SIZE_THREADS)
            if (bins[i] > 0)
                atomicAdd(&sizes[i], bins[i]);
}

// table[2 p], table[2 p + 1]: address and length of proposal p's indices.
__global__ __launch_bounds__(IOU_THREADS) void instance_iou_lists_kernel(
    int total_instances, int64_t n_proposals, int64_t n_points, int n_samples, const int64_t* __restrict__ table,
    const int64_t* __restrict__ labels, const int64_t* __restrict__ batch, const int64_t* __restrict__ counts,
    const int* __restrict__ sizes, float* __restrict__ iou)
{
    __shared__ int firsts[TPK_IOU_SAMPLES];
    __shared__ int bins[IOU_BINS];
    first_columns(n_samples, counts, firsts);
    for (int64_t p = blockIdx.x; p < n_proposals; p += gridDim.x)
    {
        const int64_t* points = reinterpret_cast<const int64_t*>(table[2 * p]);
        const int64_t length = table[2 * p + 1];
        const int64_t sample = proposal_sample(points, length, n_points, n_samples, batch);
        proposal_row(bins, points, length, n_points, labels, total_instances, sample < 0 ? 0 : firsts[sample],
                     sample < 0 ? 0 : counts[1 + sample], sizes, iou + p * total_instances);
    }
}

} // namespace

extern "C" int tpk_instance_iou(int64_t total_gt_instances, int64_t n_proposals, int64_t n_points, int64_t n_samples,
                                const int64_t* num_gt_instances, const int64_t* proposals_idx,
                                const int64_t* proposals_offset, const int64_t* instance_labels,
                                const int64_t* offset_num_gt_instances, const int64_t* batch,
                                const int64_t* instance_pointnum, float* proposals_iou, void* stream)
{
    if (total_gt_instances < 0 || n_proposals < 0 || n_points < 0 || n_samples < 0)
        return TPK_ERR_INVALID_ARG;
    if (n_proposals == 0 || total_gt_instances == 0)
        return TPK_OK;
    if (!proposals_offset || !proposals_iou || !num_gt_instances || !offset_num_gt_instances || !instance_pointnum ||
        (n_points > 0 && (!instance_labels || !batch)))
        return TPK_ERR_INVALID_ARG;
    const int64_t blocks = n_proposals < 262144 ? n_proposals : 262144;
    hipLaunchKernelGGL(instance_iou_kernel, dim3(static_cast<unsigned>(blocks)), dim3(IOU_THREADS), 0,
                       tpk_stream(stream), total_gt_instances, n_proposals, n_points, n_samples, num_gt_instances,
                       proposals_idx, proposals_offset, instance_labels, offset_num_gt_instances, batch,
                       instance_pointnum, proposals_iou);
    return tpk_launch_status();
}

extern "C" int tpk_instance_counts(int64_t n_points, const int64_t* labels, const int64_t* batch, int64_t* counts, void* stream)
{
    if (n_points <= 0 || !labels || !batch || !counts)
        return TPK_ERR_INVALID_ARG;
    const int64_t blocks = tpk_ceil_div(n_points, IOU_COUNT_POINTS);
    if (blocks > 0x7fffffffLL)
        return TPK_ERR_UNSUPPORTED;
    hipStream_t s = tpk_stream(stream);
    hipLaunchKernelGGL(instance_counts_clear_kernel, dim3(1), dim3(IOU_THREADS), 0, s, n_points, batch, counts);
    hipLaunchKernelGGL(instance_counts_kernel, dim3(static_cast<unsigned>(blocks)), dim3(IOU_THREADS), 0, s, n_points, labels, batch, counts);
    return tpk_launch_status();
}

extern "C" int tpk_instance_counts_read(const int64_t* counts, int64_t* host_counts, void* stream)
{
    if (!counts || !host_counts)
        return TPK_ERR_INVALID_ARG;
    return tpk_read_back(host_counts, counts, (1 + TPK_IOU_SAMPLES) * sizeof(int64_t), tpk_stream(stream));
}

extern "C" int tpk_instance_iou_lists(int64_t total_gt_instances, int64_t n_proposals, int64_t n_points, int64_t n_samples,
                                      const int64_t* table, const int64_t* labels, const int64_t* batch, const int64_t* counts,
                                      int32_t* sizes, float* proposals_iou, void* stream)
{
    if (total_gt_instances < 0 || n_proposals < 0 || n_points <= 0 || n_samples < 0 || n_samples > TPK_IOU_SAMPLES)
        return TPK_ERR_INVALID_ARG;
    if (n_proposals == 0 || total_gt_instances == 0)
        return TPK_OK;
    if (!table || !labels || !batch || !counts || !sizes || !proposals_iou)
        return TPK_ERR_INVALID_ARG;
    const int64_t blocks = tpk_ceil_div(n_points, IOU_SIZE_POINTS);
    if (total_gt_instances > 0x7fffffffLL || blocks > 0x7fffffffLL)
        return TPK_ERR_UNSUPPORTED;
    hipStream_t s = tpk_stream(stream);
    const int total = static_cast<int>(total_gt_instances), samples = static_cast<int>(n_samples);
    hipLaunchKernelGGL(instance_sizes_clear_kernel, dim3(static_cast<unsigned>(tpk_ceil_div(total, IOU_THREADS))), dim3(IOU_THREADS), 0,
                       s, total, sizes);
    hipLaunchKernelGGL(instance_sizes_kernel, dim3(static_cast<unsigned>(blocks)), dim3(IOU_SIZE_THREADS), 0, s, n_points, samples, total,
                       labels, batch, counts, sizes);
    const int64_t rows = n_proposals < 262144 ? n_proposals : 262144;
    hipLaunchKernelGGL(instance_iou_lists_kernel, dim3(static_cast<unsigned>(rows)), dim3(IOU_THREADS), 0, s, total, n_proposals,
                       n_points, samples, table, labels, batch, counts, sizes, proposals_iou);
    return tpk_launch_status();
}
