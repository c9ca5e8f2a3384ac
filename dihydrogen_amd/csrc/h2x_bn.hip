// Channel-wise batch-normalisation kernels for gfx950 and their C entry points.
//
// Two layouts (and, for tensors whose (sample, channel) segments have at most
// 256 elements, a third family of kernels that gives a workgroup a window of
// neighbouring whole channels: see "short segments" below).  Dense: element
// (n, c, i) of a tensor lives at
// base[(n*C + c)*real + i], i < spatial -- the geometry of the reference's
// optimised kernels (legacy/src/dnn_backend/batchnorm.cu:134-190).  Strided:
// the interior of a tensor with halos on any spatial dimension, addressed
// through the tensor's strides like the reference's generic kernels
// (batchnorm.cu:39-90,369-418,899-980,1303-1369); rows are padded to whole
// vectors, an index is split into (row, vector of the row) with multiply-high
// divisions, and every vector is one unaligned 16-byte access (see TensorMap).
// Every kernel is a pure HBM stream: 16-byte
// accesses when the geometry allows, several loads in flight per lane,
// per-channel parameters fetched once per workgroup.
//
// Float tensors that lie alike and whose channels fit the registers of one or
// several workgroups are read once (h2x_bn_once.hpp, h2x_bn_team.hpp); what
// follows is about the kernels that read them twice.
//
// Cache policy.  The layer reads x four times (sums, apply, backprop1,
// backprop2) and dy twice, while y and dx are written once.  x of the headline
// shapes is about the size of the 256 MB memory-side cache, so what must not
// happen is that the outputs or dy push it out: y and dx are written with
// nontemporal stores and dy is read with nontemporal loads; x uses plain
// loads.  Measured on NCDHW 4x64x64^3: forward+backward 381 us -> 285 us.
//
// Reductions (forward sums, backward sums) cut every channel into contiguous
// chunks, one workgroup per chunk.  A thread accumulates in fp64, the
// workgroup combines lanes with DPP permutes and waves through LDS, and writes
// one fp64 partial per sum into the workspace.  A second, tiny kernel adds the
// partials of each channel in index order and writes the channel's result
// (a kernel boundary is the cheapest device-wide ordering on this GPU: an
// in-kernel "last workgroup finishes" scheme needs a device-scope fence per
// workgroup, which costs an L2 write-back/invalidate each and was measured
// 10x slower than the whole stream).  All orders are fixed, so results are
// deterministic; the reference's float atomics are not
// (batchnorm.cu:127-131,1047-1053).
#include "h2x_bn_maps.hpp"
#include "h2x_bn_plan.hpp"
#include "h2x_device.hpp"

#include <algorithm>
#include <atomic>
#include <cmath>
#include <limits>
#include <mutex>
#include <type_traits>

// Partial sums of h2x_bn_channel_sums_and_sqsums_static, the entry point for
// callers that can neither allocate nor bring a workspace.  Every device the
// library runs on holds its own copy of this array, at its own address, until
// the process ends.  In host code the name is only a handle for
// hipGetSymbolAddress; kernels receive the address that call returned.
static constexpr size_t kStaticScratchBytes = size_t(1) << 20;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

namespace h2x
{
namespace
{

using namespace bn;

// The log the calling thread has installed (h2x_bn_plan.hpp): launches are then
// described instead of issued.
thread_local LaunchLog* t_launch_log = nullptr;

// Appends a planned launch to the installed log; false: no log, issue it.
bool logged(const LaunchRecord& r)
{
    if (!t_launch_log)
        return false;
    if (t_launch_log->keep)
        t_launch_log->records.push_back(r);
    return true;
}

// Status of the launches just issued (none while a log is installed).
int issued()
{
    return t_launch_log ? static_cast<int>(H2X_SUCCESS) : launch_status();
}

// A launch of a kernel whose threads hold `vectors` vectors of their channel each.
template <typename... P, typename... A>
void launch_whole(Kernel kernel, int vectors, void (*f)(P...), uint32_t blocks, int threads, hipStream_t st, A&&... args)
{
    if (!t_launch_log)
        return launch(f, blocks, threads, st, std::forward<A>(args)...);
    LaunchRecord r;
    r.kernel = kernel;
    r.grid_x = blocks;
    r.threads = threads;
    r.vectors = vectors;
    logged(r);
}

// Installs a log for the lifetime of the object and puts the previous one back.
struct ScopedLaunchLog
{
    explicit ScopedLaunchLog(LaunchLog* log) : before(t_launch_log) { t_launch_log = log; }
    ~ScopedLaunchLog() { t_launch_log = before; }
    void restore() { t_launch_log = before; }
    ScopedLaunchLog(const ScopedLaunchLog&) = delete;
    ScopedLaunchLog& operator=(const ScopedLaunchLog&) = delete;
    LaunchLog* before;
};

// Device address of `scratch` on the current device, looked up once per device.
std::mutex static_scratch_mutex;
void* static_scratch_address[kMaxDevices] = {};

int static_scratch(void** out)
{
    int device = -1;
    hipError_t err = hipGetDevice(&device);
    if (err != hipSuccess)
        return static_cast<int>(err);
    if (device < 0 || device >= kMaxDevices)
        return H2X_ERR_UNSUPPORTED;
    std::lock_guard<std::mutex> lock(static_scratch_mutex);
    if (static_scratch_address[device] == nullptr)
    {
        void* p = nullptr;
        err = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (err != hipSuccess)
            return static_cast<int>(err);
        if (p == nullptr)
            return static_cast<int>(hipErrorInvalidSymbol);
        static_scratch_address[device] = p;
    }
    *out = static_scratch_address[device];
    return H2X_SUCCESS;
}

constexpr int kUnroll = 4;
// Workgroups a reduction aims at over all channels, from sweeps on MI355X: 4096
// on dense tensors, 16384 on haloed ones (the haloed C3 shard: two-launch
// forward 141 -> 134 us, backward 217 -> 211 us; dense shapes are the same or
// up to 4 % slower with more).  The workspace holds partial sums for the larger
// number.
constexpr int kTargetGroups = 16384;
constexpr int kDenseTargetGroups = 4096;
// Elementwise passes aim at 16384 workgroups (from a sweep on MI355X at the
// headline shapes) - except on haloed tensors and on tensors beyond the
// memory-side cache, where a workgroup gets two passes of its 256 lanes (8 KB
// of fp32 per tensor) however large the tensor is.  Measured against the
// budget of 16384: normalise on the haloed C3 shard 158 -> 145 us, input
// gradient 240 -> 222 us; dense tensors of 1 GB 571 -> 529 us and 896 -> 836
// us, of 537 MB 279 -> 267 us and 443 -> 423 us.  Dense tensors that the cache
// holds lose with the small chunks (268 MB: input gradient 191 -> 194 us, the
// benchmark step 676 -> 680 us; N 64 x 256 x 56 x 56: 150 -> 161 us) and keep
// the budget.
constexpr int kElementwiseBlocks = 16384;
constexpr int kUnboundedBlocks = 1 << 30;
constexpr size_t kBeyondCacheBytes = size_t(384) << 20;
constexpr int kMinGroupsPerChannel = 8;
constexpr int kMaxGroupsPerChannel = 2048;
constexpr int kMaxSums = 4;

int groups_per_channel(int num_channels, int target)
{
    const int g = (target + num_channels - 1) / std::max(num_channels, 1);
    return std::min(std::max(g, kMinGroupsPerChannel), kMaxGroupsPerChannel);
}

// Partial sums the workspace holds per channel and sum: the stride of the
// partials of a channel, and the most groups any launch uses.
int max_groups_per_channel(int num_channels)
{
    return groups_per_channel(num_channels, kTargetGroups);
}

// Groups a long-segment reduction cuts a channel into.
int reduction_groups_per_channel(int num_channels, bool strided)
{
    return strided ? max_groups_per_channel(num_channels)
                   : groups_per_channel(num_channels, kDenseTargetGroups);
}

size_t partials_bytes(int num_channels)
{
    return static_cast<size_t>(num_channels) * max_groups_per_channel(num_channels) * kMaxSums
           * sizeof(double);
}

// How one (sample, channel) segment of `spatial` elements is cut into chunks.
// With vectors, `spatial` is a whole number of them (dense: a condition of the
// aligned path; strided: rows are padded), and so is every chunk.
struct Chunking
{
    size_t chunk;        // elements per workgroup, multiple of the tile
    int chunks_per_seg;  // workgroups per (sample, channel) segment
};

// `segments`: segments that contribute workgroups to one scheduling unit
// (num_samples for a per-channel reduction, N*C for an elementwise pass);
// `budget`: workgroups wanted (reduction: cap per channel; elementwise: total).
Chunking make_chunking(size_t spatial, size_t segments, size_t budget, size_t tile, size_t min_chunk)
{
    Chunking c;
    size_t per_seg = std::max<size_t>(budget / std::max<size_t>(segments, 1), 1);
    size_t chunk = (spatial + per_seg - 1) / per_seg;
    chunk = std::max(chunk, min_chunk);
    chunk = (chunk + tile - 1) / tile * tile;
    c.chunk = chunk;
    c.chunks_per_seg = static_cast<int>((spatial + chunk - 1) / chunk);
    if (c.chunks_per_seg < 1)
        c.chunks_per_seg = 1;
    return c;
}

// ALIGNED: the address is a multiple of the vector size (dense layout); rows
// of a strided tensor may start on any element.
// STREAM: the data is not read again soon; a nontemporal load keeps it from
// displacing what should stay in the memory-side cache.
template <typename T, int VEC, bool ALIGNED = true, bool STREAM = false>
__device__ __forceinline__ void load_vec(const T* p, T (&r)[VEC])
{
    if constexpr (VEC == 1)
    {
        r[0] = STREAM ? __builtin_nontemporal_load(p) : *p;
    }
    else
    {
        typedef T V __attribute__((ext_vector_type(VEC), aligned(ALIGNED ? sizeof(T) * VEC : sizeof(T))));
        const V t = STREAM ? __builtin_nontemporal_load(reinterpret_cast<const V*>(p))
                           : *reinterpret_cast<const V*>(p);
#pragma unroll
        for (int j = 0; j < VEC; ++j)
            r[j] = t[j];
    }
}

template <typename T, int VEC, bool ALIGNED = true, bool STREAM = true>
__device__ __forceinline__ void store_vec(T* p, const T (&r)[VEC])
{
    // Outputs are written once and not read by the next kernel of the layer;
    // nontemporal stores keep them from evicting x (and dy), which the next
    // kernel reads again, from the 256 MB memory-side cache.
    if constexpr (VEC == 1)
    {
        if constexpr (STREAM)
            __builtin_nontemporal_store(r[0], p);
        else
            *p = r[0];
    }
    else
    {
        typedef T V __attribute__((ext_vector_type(VEC), aligned(ALIGNED ? sizeof(T) * VEC : sizeof(T))));
        V t;
#pragma unroll
        for (int j = 0; j < VEC; ++j)
            t[j] = r[j];
        if constexpr (STREAM)
            __builtin_nontemporal_store(t, reinterpret_cast<V*>(p));
        else
            *reinterpret_cast<V*>(p) = t;
    }
}

// How a kernel walks a tensor: as it lies (dense) or row by row in vectors
// that start on any element (rows; see Place in h2x_bn_maps.hpp).
enum Layout : int
{
    kLayoutDense = 0,
    kLayoutRows = 1
};

// Where the vector at index i lies.  Worked out once per vector, from the map
// of one tensor of the launch, and shared by all of them (index splitting costs
// two multiply-high divisions; done per tensor it was a third of the
// instructions of the strided kernels).  Without vectors or index splitting
// the place is not used.
template <typename T, int VEC, int LAYOUT>
__device__ __forceinline__ Place place_at(const TensorMap& m, size_t i)
{
    Place pl{0, 0, 0, 0};
    if constexpr (VEC > 1 && LAYOUT == kLayoutRows)
        place_vector<VEC>(m, row_split<VEC>(m, i, &pl), &pl);
    return pl;
}

// The VEC elements of tensor p at index i / place pl.
template <typename T, int VEC, int LAYOUT, bool STREAM = false>
__device__ __forceinline__ void load_in(const T* p, const TensorMap& m, size_t i, const Place& pl,
                                        T (&r)[VEC])
{
    if constexpr (VEC == 1 || LAYOUT == kLayoutDense)
    {
        load_vec<T, VEC, LAYOUT == kLayoutDense, STREAM>(
            p + seg_offset<LAYOUT != kLayoutDense>(m, i), r);
    }
    else
    {
        load_vec<T, VEC, false, STREAM>(p + (row_offset(m, pl) + pl.first), r);
    }
}

// rewrite (rows layout): the elements a vector shares with the one before it
// may be stored by both (the output shares no memory with the inputs they were
// made from).
template <typename T, int VEC, int LAYOUT, bool STREAM = true>
__device__ __forceinline__ void store_out(T* p, const TensorMap& m, size_t i, const Place& pl,
                                          const T (&r)[VEC], bool rewrite)
{
    if constexpr (VEC == 1 || LAYOUT == kLayoutDense)
    {
        store_vec<T, VEC, LAYOUT == kLayoutDense, STREAM>(p + seg_offset<LAYOUT != kLayoutDense>(m, i), r);
    }
    else
    {
        T* q = p + (row_offset(m, pl) + pl.first);
        if (pl.skip == 0 || rewrite)
        {
            store_vec<T, VEC, false, STREAM>(q, r);
        }
        else
        {
#pragma unroll
            for (int j = 1; j < VEC; ++j)
                if (j >= static_cast<int>(pl.skip))
                    store_vec<T, 1, true, STREAM>(q + j, {r[j]});
        }
    }
}

__device__ __forceinline__ float fma_t(float a, float b, float c)
{
    return __builtin_fmaf(a, b, c);
}
__device__ __forceinline__ double fma_t(double a, double b, double c)
{
    return __builtin_fma(a, b, c);
}
__device__ __forceinline__ float inv_sqrt_t(float v)
{
    return 1.0f / __builtin_sqrtf(v);
}
__device__ __forceinline__ double inv_sqrt_t(double v)
{
    return 1.0 / __builtin_sqrt(v);
}

// Combines the K per-thread sums of a workgroup.  With a single workgroup per
// channel returns true (totals in acc[], to be written by the caller);
// otherwise stores this workgroup's partials for the finishing kernel.
template <int K>
__device__ __forceinline__ bool finish_workgroup(double (&acc)[K], double* partials, int channel,
                                                 int groups_per_channel_max, bool always_partials)
{
    __shared__ double lds[K * kWavesPerBlock];
    block_sum<K>(acc, lds);
    if (gridDim.x == 1 && !always_partials)
        return true;
    if (threadIdx.x == 0)
    {
        double* mine = partials
                       + (static_cast<size_t>(channel) * groups_per_channel_max + blockIdx.x) * K;
#pragma unroll
        for (int k = 0; k < K; ++k)
            mine[k] = acc[k];
    }
    return false;
}

// Adds the `groups` partials of every channel in index order: thread t takes
// partials t, t + 256, ...; the workgroup then combines its threads in the
// fixed order of block_sum.  out_k[c] receives sum k of channel c.
template <typename T, int K>
__global__ __launch_bounds__(kBlockSize) void bn_finish_kernel(
    const double* __restrict__ partials, int groups, int groups_per_channel_max, T* out0, T* out1,
    T* out2, T* out3)
{
    __shared__ double lds[K * kWavesPerBlock];
    const int c = blockIdx.x;
    const double* mine = partials + static_cast<size_t>(c) * groups_per_channel_max * K;
    double t[K];
#pragma unroll
    for (int k = 0; k < K; ++k)
        t[k] = 0.0;
    for (int g = threadIdx.x; g < groups; g += kBlockSize)
    {
#pragma unroll
        for (int k = 0; k < K; ++k)
            t[k] += mine[static_cast<size_t>(g) * K + k];
    }
    block_sum<K>(t, lds);
    if (threadIdx.x == 0)
    {
        T* outs[4] = {out0, out1, out2, out3};
#pragma unroll
        for (int k = 0; k < K; ++k)
            outs[k][c] = static_cast<T>(t[k]);
    }
}

// The K sums of channel c from its `groups` partials, in the order of
// bn_finish_kernel (so a consumer that adds them itself gets the same bits).
template <int K>
__device__ __forceinline__ void channel_totals(const double* __restrict__ partials, int groups,
                                               int groups_per_channel_max, int c, double (&t)[K],
                                               double* lds)
{
    const double* mine = partials + static_cast<size_t>(c) * groups_per_channel_max * K;
#pragma unroll
    for (int k = 0; k < K; ++k)
        t[k] = 0.0;
    for (int g = threadIdx.x; g < groups; g += kBlockSize)
    {
#pragma unroll
        for (int k = 0; k < K; ++k)
            t[k] += mine[static_cast<size_t>(g) * K + k];
    }
    block_sum<K>(t, lds);
}

// What the statistics kernel below makes of a channel's sum and sum of squares.
template <typename T>
__device__ __forceinline__ void sums_to_mean_var(T sum, T sqsum, T n, T* mean, T* var)
{
    const T m = sum / n;
    const T sqmean = sqsum / n;
    T v = fma_t(-m, m, sqmean);
    v = v > T(0) ? v : T(0);
    v *= n / (n - T(1));
    *mean = m;
    *var = v;
}

// ---- forward: sums and sums of squares --------------------------------------
// Replaces channel_sums_and_sqsums_opt_kernel, batchnorm.cu:92-132.
template <typename T, int VEC, bool STRIDED>
__global__ __launch_bounds__(kBlockSize) void bn_sums_kernel(
    const T* __restrict__ x, T* __restrict__ sums, T* __restrict__ sqsums, double* partials,
    const TensorMap mx, size_t spatial, size_t chunk, int chunks_per_seg, unsigned int num_units,
    int groups_per_channel_max, bool always_partials)
{
    const int c = blockIdx.y;
    constexpr int LAYOUT = STRIDED ? kLayoutRows : kLayoutDense;
    constexpr size_t kStride = static_cast<size_t>(kBlockSize) * VEC;
    constexpr size_t kTile = kStride * kUnroll;
    double acc[2] = {0.0, 0.0};

    auto accumulate = [&](T v) {
        const double d = static_cast<double>(v);
        acc[0] += d;
        if constexpr (sizeof(T) == 4)
            acc[1] = __builtin_fma(d, d, acc[1]); // the product of two floats is exact in fp64
        else
            acc[1] += d * d;
    };

    // unit = (sample, chunk); a workgroup takes units blockIdx.x, blockIdx.x + gridDim.x, ...
    for (unsigned int unit = blockIdx.x; unit < num_units; unit += gridDim.x)
    {
        const int n = unit / chunks_per_seg;
        const int k = unit - n * chunks_per_seg;
        const size_t begin = static_cast<size_t>(k) * chunk;
        const size_t end = begin + chunk < spatial ? begin + chunk : spatial;
        const T* p = x + n * mx.stride_n + c * mx.stride_c;
        size_t tile = begin;
        for (; tile + kTile <= end; tile += kTile)
        {
            T v[kUnroll][VEC];
            uint32_t skip[kUnroll];
#pragma unroll
            for (int u = 0; u < kUnroll; ++u)
            {
                const size_t i = tile + u * kStride + threadIdx.x * VEC;
                const Place pl = place_at<T, VEC, LAYOUT>(mx, i);
                load_in<T, VEC, LAYOUT>(p, mx, i, pl, v[u]);
                skip[u] = pl.skip;
            }
#pragma unroll
            for (int u = 0; u < kUnroll; ++u)
#pragma unroll
                for (int j = 0; j < VEC; ++j)
                    if (j >= static_cast<int>(skip[u]))
                        accumulate(v[u][j]);
        }
        for (size_t i = tile + threadIdx.x * VEC; i + VEC <= end; i += kStride)
        {
            T v[VEC];
            const Place pl = place_at<T, VEC, LAYOUT>(mx, i);
            load_in<T, VEC, LAYOUT>(p, mx, i, pl, v);
#pragma unroll
            for (int j = 0; j < VEC; ++j)
                if (j >= static_cast<int>(pl.skip))
                    accumulate(v[j]);
        }
    }
    if (finish_workgroup<2>(acc, partials, c, groups_per_channel_max, always_partials)
        && threadIdx.x == 0)
    {
        sums[c] = static_cast<T>(acc[0]);
        sqsums[c] = static_cast<T>(acc[1]);
    }
}

template <typename T>
__global__ void fill_kernel(T* p, size_t n, T value)
{
    for (size_t i = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x; i < n;
         i += static_cast<size_t>(gridDim.x) * blockDim.x)
        p[i] = value;
}

// ---- forward: sums -> mean / unbiased variance / running statistics ---------
// Replaces sums_to_statistics_functor, batchnorm.cu:288-346.
template <typename T>
__global__ void bn_statistics_kernel(int num_channels, size_t num_per_sum, T decay, T* mean,
                                     T* var, T* running_mean, T* running_var)
{
    const T n = static_cast<T>(num_per_sum);
    for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < num_channels;
         c += gridDim.x * blockDim.x)
    {
        if (num_per_sum == 0)
        {
            var[c] = T(1);
            continue;
        }
        T m, v;
        sums_to_mean_var(mean[c], var[c], n, &m, &v);
        mean[c] = m;
        var[c] = v;
        running_mean[c] = fma_t(decay, running_mean[c], (T(1) - decay) * m);
        running_var[c] = fma_t(decay, running_var[c], (T(1) - decay) * v);
    }
}

// What a consumer kernel needs to finish a reduction itself: the partial sums
// the reduction kernel left in the workspace, and where the channel results go.
// Every workgroup of a channel adds that channel's partials in the order of
// bn_finish_kernel and so arrives at the same bits; the channel's first
// workgroup stores them.  Saves the finishing launch (and, forward, the
// statistics launch) when no all-reduce sits between the two stages.
template <typename T>
struct FusedStats
{
    const double* partials;
    int groups;
    int groups_per_channel_max;
    size_t num_per_sum;
    T decay;
    T* out[4];          // forward: mean, var, running_mean, running_var; backward: dscale, dbias, dmean, dvar
    bool sequential;    // the partials come from a short-segment kernel and are added one after the other
};

// How a normalising kernel works: with statistics that it reads, past the caches; with those that it makes of partial
// sums; as the first, with normal stores (see kNormalStores).
enum ApplyMode : int
{
    kPlainApply = 0,
    kFusedApply = 1,
    kNormalApply = 2
};

// ---- forward: normalise ------------------------------------------------------
// Replaces batch_normalization_opt_kernel, batchnorm.cu:420-455.  FUSED: mean
// and variance are not read but made from the partial sums of bn_sums_kernel
// (bn_finish_kernel + bn_statistics_kernel folded in).
template <typename T, int VEC, int LAYOUT, int MODE>
__global__ __launch_bounds__(kBlockSize) void bn_apply_kernel(
    const T* __restrict__ x, const T* __restrict__ mean, const T* __restrict__ var,
    const T* __restrict__ scale, const T* __restrict__ bias, T* __restrict__ y, T epsilon,
    int num_channels, size_t spatial, const TensorMap mx, const TensorMap my, size_t chunk,
    int chunks_per_seg, const FusedStats<T> fused = FusedStats<T>())
{
    constexpr bool FUSED = MODE == kFusedApply, STREAM = MODE != kNormalApply;
    const size_t seg = blockIdx.x / chunks_per_seg;
    const int k = blockIdx.x - seg * chunks_per_seg;
    const int c = seg % num_channels;
    T m, variance;
    if constexpr (FUSED)
    {
        __shared__ double lds[2 * kWavesPerBlock];
        double t[2];
        channel_totals<2>(fused.partials, fused.groups, fused.groups_per_channel_max, c, t, lds);
        sums_to_mean_var(static_cast<T>(t[0]), static_cast<T>(t[1]),
                         static_cast<T>(fused.num_per_sum), &m, &variance);
        if (seg < static_cast<size_t>(num_channels) && k == 0 && threadIdx.x == 0) // sample 0, chunk 0
        {
            fused.out[0][c] = m;
            fused.out[1][c] = variance;
            fused.out[2][c] = fma_t(fused.decay, fused.out[2][c], (T(1) - fused.decay) * m);
            fused.out[3][c] = fma_t(fused.decay, fused.out[3][c], (T(1) - fused.decay) * variance);
        }
    }
    else
    {
        m = mean[c];
        variance = var[c];
    }
    const T inv_stdev = inv_sqrt_t(variance + epsilon);
    const T sc = scale[c];
    const T bi = bias[c];
    const size_t begin = static_cast<size_t>(k) * chunk;
    const size_t end = begin + chunk < spatial ? begin + chunk : spatial;
    const size_t n = seg / num_channels;
    const T* xp = x + n * mx.stride_n + c * mx.stride_c;
    T* yp = y + n * my.stride_n + c * my.stride_c;

    constexpr size_t kStride = static_cast<size_t>(kBlockSize) * VEC;
    constexpr size_t kTile = kStride * kUnroll;
    size_t tile = begin;
    for (; tile + kTile <= end; tile += kTile)
    {
        T v[kUnroll][VEC];
        Place pl[kUnroll];
#pragma unroll
        for (int u = 0; u < kUnroll; ++u)
        {
            const size_t i = tile + u * kStride + threadIdx.x * VEC;
            pl[u] = place_at<T, VEC, LAYOUT>(my, i);
            load_in<T, VEC, LAYOUT>(xp, mx, i, pl[u], v[u]);
        }
#pragma unroll
        for (int u = 0; u < kUnroll; ++u)
        {
#pragma unroll
            for (int j = 0; j < VEC; ++j)
                v[u][j] = fma_t((v[u][j] - m) * inv_stdev, sc, bi);
            store_out<T, VEC, LAYOUT, STREAM>(yp, my, tile + u * kStride + threadIdx.x * VEC, pl[u], v[u], true);
        }
    }
    for (size_t i = tile + threadIdx.x * VEC; i + VEC <= end; i += kStride)
    {
        T v[VEC];
        const Place pl = place_at<T, VEC, LAYOUT>(my, i);
        load_in<T, VEC, LAYOUT>(xp, mx, i, pl, v);
#pragma unroll
        for (int j = 0; j < VEC; ++j)
            v[j] = fma_t((v[j] - m) * inv_stdev, sc, bi);
        store_out<T, VEC, LAYOUT, STREAM>(yp, my, i, pl, v, true);
    }
}

// ---- backward: per-channel sums ----------------------------------------------
// Replaces backprop1_opt_kernel, batchnorm.cu:982-1054.
template <typename T, int VEC, bool STRIDED>
__global__ __launch_bounds__(kBlockSize) void bn_backprop1_kernel(
    const T* __restrict__ x, const T* __restrict__ dy, const T* __restrict__ mean,
    const T* __restrict__ var, const T* __restrict__ scale, T* __restrict__ dscale,
    T* __restrict__ dbias, T* __restrict__ dmean, T* __restrict__ dvar, T epsilon,
    double* partials, size_t spatial, const TensorMap mx, const TensorMap md, size_t chunk,
    int chunks_per_seg, unsigned int num_units, int groups_per_channel_max, bool always_partials)
{
    const int c = blockIdx.y;
    const T m = mean[c];
    const T sc = scale[c];
    const T inv_stdev = inv_sqrt_t(var[c] + epsilon);
    const T dvar_factor = inv_stdev * inv_stdev * inv_stdev / T(2);
    const double neg_inv = -static_cast<double>(inv_stdev);
    const double neg_fac = -static_cast<double>(dvar_factor);

    constexpr int LAYOUT = STRIDED ? kLayoutRows : kLayoutDense;
    constexpr size_t kStride = static_cast<size_t>(kBlockSize) * VEC;
    constexpr int kUnroll2 = kUnroll / 2; // two streams: same bytes in flight
    constexpr size_t kTile = kStride * kUnroll2;
    double acc[4] = {0.0, 0.0, 0.0, 0.0};

    auto accumulate = [&](T xv, T dv) {
        const T xm = xv - m;
        const T xhat = xm * inv_stdev;
        const T dxhat = dv * sc;
        const T t = dxhat * xm;
        const double dd = static_cast<double>(dv);
        acc[0] = __builtin_fma(dd, static_cast<double>(xhat), acc[0]);
        acc[1] += dd;
        acc[2] = __builtin_fma(static_cast<double>(dxhat), neg_inv, acc[2]);
        acc[3] = __builtin_fma(static_cast<double>(t), neg_fac, acc[3]);
    };

    for (unsigned int unit = blockIdx.x; unit < num_units; unit += gridDim.x)
    {
        const int n = unit / chunks_per_seg;
        const int k = unit - n * chunks_per_seg;
        const size_t begin = static_cast<size_t>(k) * chunk;
        const size_t end = begin + chunk < spatial ? begin + chunk : spatial;
        const T* xp = x + n * mx.stride_n + c * mx.stride_c;
        const T* dp = dy + n * md.stride_n + c * md.stride_c;
        size_t tile = begin;
        for (; tile + kTile <= end; tile += kTile)
        {
            T xv[kUnroll2][VEC], dv[kUnroll2][VEC];
            uint32_t skip[kUnroll2];
#pragma unroll
            for (int u = 0; u < kUnroll2; ++u)
            {
                const size_t i = tile + u * kStride + threadIdx.x * VEC;
                const Place pl = place_at<T, VEC, LAYOUT>(mx, i);
                load_in<T, VEC, LAYOUT>(xp, mx, i, pl, xv[u]);
                load_in<T, VEC, LAYOUT, true>(dp, md, i, pl, dv[u]);
                skip[u] = pl.skip;
            }
#pragma unroll
            for (int u = 0; u < kUnroll2; ++u)
#pragma unroll
                for (int j = 0; j < VEC; ++j)
                    if (j >= static_cast<int>(skip[u]))
                        accumulate(xv[u][j], dv[u][j]);
        }
        for (size_t i = tile + threadIdx.x * VEC; i + VEC <= end; i += kStride)
        {
            T xv[VEC], dv[VEC];
            const Place pl = place_at<T, VEC, LAYOUT>(mx, i);
            load_in<T, VEC, LAYOUT>(xp, mx, i, pl, xv);
            load_in<T, VEC, LAYOUT, true>(dp, md, i, pl, dv);
#pragma unroll
            for (int j = 0; j < VEC; ++j)
                if (j >= static_cast<int>(pl.skip))
                    accumulate(xv[j], dv[j]);
        }
    }
    if (finish_workgroup<4>(acc, partials, c, groups_per_channel_max, always_partials)
        && threadIdx.x == 0)
    {
        dscale[c] = static_cast<T>(acc[0]);
        dbias[c] = static_cast<T>(acc[1]);
        dmean[c] = static_cast<T>(acc[2]);
        dvar[c] = static_cast<T>(acc[3]);
    }
}

// ---- backward: input gradient ------------------------------------------------
// Replaces backprop2_opt_kernel, batchnorm.cu:1371-1418.  x and dx may alias:
// each thread reads its elements before it writes them, so neither is
// restrict-qualified (`disjoint`: they share no memory).
template <typename T, int VEC, int LAYOUT, bool FUSED = false>
__global__ __launch_bounds__(kBlockSize) void bn_backprop2_kernel(
    const T* x, const T* __restrict__ dy, const T* __restrict__ mean,
    const T* __restrict__ var, const T* __restrict__ scale, const T* __restrict__ dmean,
    const T* __restrict__ dvar, T* dx, T epsilon, size_t num_per_sum, int num_channels,
    size_t spatial, const TensorMap mx, const TensorMap md, const TensorMap mo, size_t chunk,
    int chunks_per_seg, bool disjoint, const FusedStats<T> fused = FusedStats<T>())
{
    const size_t seg = blockIdx.x / chunks_per_seg;
    const int k = blockIdx.x - seg * chunks_per_seg;
    const int c = seg % num_channels;
    const T m = mean[c];
    const T sc = scale[c];
    const T inv_stdev = inv_sqrt_t(var[c] + epsilon);
    T dmean_c, dvar_c;
    if constexpr (FUSED)
    {
        // the four sums of bn_backprop1_kernel, finished here (bn_finish_kernel folded in)
        __shared__ double lds[4 * kWavesPerBlock];
        double t[4];
        channel_totals<4>(fused.partials, fused.groups, fused.groups_per_channel_max, c, t, lds);
        dmean_c = static_cast<T>(t[2]);
        dvar_c = static_cast<T>(t[3]);
        if (seg < static_cast<size_t>(num_channels) && k == 0 && threadIdx.x == 0)
        {
            fused.out[0][c] = static_cast<T>(t[0]);
            fused.out[1][c] = static_cast<T>(t[1]);
            fused.out[2][c] = dmean_c;
            fused.out[3][c] = dvar_c;
        }
    }
    else
    {
        dmean_c = dmean[c];
        dvar_c = dvar[c];
    }
    const T dmean_term = dmean_c / static_cast<T>(num_per_sum);
    const T dvar_term = dvar_c * T(2) / static_cast<T>(num_per_sum - 1);
    const size_t begin = static_cast<size_t>(k) * chunk;
    const size_t end = begin + chunk < spatial ? begin + chunk : spatial;
    const size_t n = seg / num_channels;
    const T* xp = x + n * mx.stride_n + c * mx.stride_c;
    const T* dp = dy + n * md.stride_n + c * md.stride_c;
    T* op = dx + n * mo.stride_n + c * mo.stride_c;

    constexpr size_t kStride = static_cast<size_t>(kBlockSize) * VEC;
    constexpr int kUnroll2 = kUnroll / 2;
    constexpr size_t kTile = kStride * kUnroll2;
    size_t tile = begin;
    for (; tile + kTile <= end; tile += kTile)
    {
        T xv[kUnroll2][VEC], dv[kUnroll2][VEC];
        Place pl[kUnroll2];
#pragma unroll
        for (int u = 0; u < kUnroll2; ++u)
        {
            const size_t i = tile + u * kStride + threadIdx.x * VEC;
            pl[u] = place_at<T, VEC, LAYOUT>(mo, i);
            load_in<T, VEC, LAYOUT>(xp, mx, i, pl[u], xv[u]);
            load_in<T, VEC, LAYOUT, true>(dp, md, i, pl[u], dv[u]);
        }
#pragma unroll
        for (int u = 0; u < kUnroll2; ++u)
        {
#pragma unroll
            for (int j = 0; j < VEC; ++j)
            {
                T r = fma_t(dv[u][j] * sc, inv_stdev, dmean_term);
                xv[u][j] = fma_t(xv[u][j] - m, dvar_term, r);
            }
            store_out<T, VEC, LAYOUT>(op, mo, tile + u * kStride + threadIdx.x * VEC, pl[u], xv[u], disjoint);
        }
    }
    for (size_t i = tile + threadIdx.x * VEC; i + VEC <= end; i += kStride)
    {
        T xv[VEC], dv[VEC];
        const Place pl = place_at<T, VEC, LAYOUT>(mo, i);
        load_in<T, VEC, LAYOUT>(xp, mx, i, pl, xv);
        load_in<T, VEC, LAYOUT, true>(dp, md, i, pl, dv);
#pragma unroll
        for (int j = 0; j < VEC; ++j)
        {
            T r = fma_t(dv[j] * sc, inv_stdev, dmean_term);
            xv[j] = fma_t(xv[j] - m, dvar_term, r);
        }
        store_out<T, VEC, LAYOUT>(op, mo, i, pl, xv, disjoint);
    }
}

// ---- normalise / input gradient that leave the halo of their output cleared ----
// For tensors that share one haloed geometry.  The kernel walks the REAL local
// tensor of every (sample, channel) segment - interior and halo cells alike - in
// aligned 16-byte vectors, computes the interior elements and stores zeros into
// the halo cells: what the reference's kernel followed by Tensor::clear_halo on
// every spatial dimension leaves (legacy/src/tensor/tensor_mpi_cuda.cu:14-84;
// Convolution::forward clears the halos of its input before every exchange,
// legacy/include/distconv/dnn_backend/convolution.hpp:400-411), in one pass and
// without the partly written sectors that the gaps between interior rows cost
// the kernels above.  Halo cells of the inputs are loaded and ignored.
// BACKWARD: the input gradient (x, dy -> dx); else normalise (x -> y).  Segments
// are `real` elements long and follow one another (channel stride = real).
template <typename T, int VEC, bool BACKWARD>
__global__ __launch_bounds__(kBlockSize) void bn_clearing_kernel(
    const T* x, const T* __restrict__ dy, const T* __restrict__ mean, const T* __restrict__ var,
    const T* __restrict__ scale, const T* __restrict__ bias, const T* __restrict__ dmean,
    const T* __restrict__ dvar, T* out, T epsilon, size_t num_per_sum, int num_channels, size_t real,
    const RealBox box, size_t chunk, int chunks_per_seg)
{
    const size_t seg = blockIdx.x / chunks_per_seg;
    const int k = blockIdx.x - seg * chunks_per_seg;
    const int c = seg % num_channels;
    const T m = mean[c];
    const T sc = scale[c];
    const T inv_stdev = inv_sqrt_t(var[c] + epsilon);
    T bi = T(0), dmean_term = T(0), dvar_term = T(0);
    if constexpr (BACKWARD)
    {
        dmean_term = dmean[c] / static_cast<T>(num_per_sum);
        dvar_term = dvar[c] * T(2) / static_cast<T>(num_per_sum - 1);
    }
    else
    {
        bi = bias[c];
    }
    const size_t begin = static_cast<size_t>(k) * chunk;
    const size_t end = begin + chunk < real ? begin + chunk : real;
    const T* xp = x + seg * real;
    const T* dp = BACKWARD ? dy + seg * real : nullptr;
    T* op = out + seg * real;

    auto result = [&](T xv, T dv) {
        if constexpr (BACKWARD)
            return fma_t(xv - m, dvar_term, fma_t(dv * sc, inv_stdev, dmean_term));
        else
            return fma_t((xv - m) * inv_stdev, sc, bi);
    };
    constexpr size_t kStride = static_cast<size_t>(kBlockSize) * VEC;
    constexpr int kInFlight = BACKWARD ? kUnroll / 2 : kUnroll;
    constexpr size_t kTile = kStride * kInFlight;
    size_t tile = begin;
    for (; tile + kTile <= end; tile += kTile)
    {
        T xv[kInFlight][VEC], dv[kInFlight][VEC];
#pragma unroll
        for (int u = 0; u < kInFlight; ++u)
        {
            const size_t i = tile + u * kStride + threadIdx.x * VEC;
            load_vec<T, VEC, true>(xp + i, xv[u]);
            if constexpr (BACKWARD)
                load_vec<T, VEC, true, true>(dp + i, dv[u]);
        }
#pragma unroll
        for (int u = 0; u < kInFlight; ++u)
        {
            const size_t i = tile + u * kStride + threadIdx.x * VEC;
            const uint32_t inside = interior_bits<VEC>(box, static_cast<uint32_t>(i));
#pragma unroll
            for (int j = 0; j < VEC; ++j)
                xv[u][j] = inside >> j & 1 ? result(xv[u][j], BACKWARD ? dv[u][j] : T(0)) : T(0);
            store_vec<T, VEC, true>(op + i, xv[u]);
        }
    }
    for (size_t i = tile + threadIdx.x * VEC; i + VEC <= end; i += kStride)
    {
        T xv[VEC], dv[VEC];
        load_vec<T, VEC, true>(xp + i, xv);
        if constexpr (BACKWARD)
            load_vec<T, VEC, true, true>(dp + i, dv);
        const uint32_t inside = interior_bits<VEC>(box, static_cast<uint32_t>(i));
#pragma unroll
        for (int j = 0; j < VEC; ++j)
            xv[j] = inside >> j & 1 ? result(xv[j], BACKWARD ? dv[j] : T(0)) : T(0);
        store_vec<T, VEC, true>(op + i, xv);
    }
}

// ---- short segments: whole channels side by side in one workgroup ------------
// A (sample, channel) segment of a few hundred bytes (7 x 7 or 14 x 14
// activations, 1 x 1 after a fully connected layer) shares its first and last
// cache line with the neighbouring channels.  A workgroup per channel that walks
// from sample to sample then fetches 2-3 lines for 196 bytes and leaves its
// output as partial lines (N 256, C 2048, 7 x 7: 169 MB read and 637 k partial
// writes for a 103 MB tensor; 106 MB read here, forward 102 us -> 52 us,
// backward 170 us -> 91 us; N 512, C 4096, 1 x 1: 100 -> 12 us, 138 -> 25 us).
// These kernels give a workgroup a window of
// neighbouring whole channels instead -- one contiguous piece of memory per
// sample -- and walk through a range of samples.  A segment is padded to
// `slots` vectors; lane t serves slot t mod slots of channel t div slots for
// every sample, so its channel and that channel's parameters are fixed for the
// whole kernel.  The last slot of a segment whose length is no multiple of the
// vector owns fewer elements: its vector starts that much earlier, so that it
// is still loaded whole, overlaps the slot before it, and only the elements it
// owns are added up or stored (kTailOverlap; in place of x, dx may be written
// by the neighbouring lane before this lane reads the overlap, which it does
// not use).  Segments shorter than a vector move element by element
// (kTailScalar).  When a tensor of the launch has halos inside its segments
// the slots follow the rows of the segment instead (each row padded to whole
// vectors, the last vector of a row overlapping the one before it), so that a
// slot is contiguous in every tensor; where it starts in each tensor is worked
// out once, as the lane's place in the segment never changes (N 32, C 512,
// 14 x 14 with a halo of 1: forward 34 -> 14 us, backward 46 -> 20 us against
// the strided kernels, which give such a segment a workgroup of its own).
// Where few
// channels and many samples would leave a reduction with too few workgroups,
// the lanes of a workgroup form `rows` rows that take every rows-th sample of
// a narrower window.
template <typename T, int VEC, int TAIL, bool STREAM = false>
__device__ __forceinline__ void load_slot(const T* p, const ShortLane& l, T (&r)[VEC])
{
    if constexpr (TAIL != kTailScalar)
    {
        load_vec<T, VEC, false, STREAM>(p, r);
    }
    else
    {
#pragma unroll
        for (int j = 0; j < VEC; ++j)
            r[j] = T(0);
#pragma unroll
        for (int j = 0; j < VEC - 1; ++j)
            if (j < l.valid)
                r[j] = STREAM ? __builtin_nontemporal_load(p + j) : p[j];
    }
}

// rewrite: the output does not alias an input, so the elements in which the
// last vector of a row overlaps its neighbour may be stored by both lanes (each
// made the same values from the same inputs) and every lane stores a whole vector.
template <typename T, int VEC, int TAIL, bool STREAM = true>
__device__ __forceinline__ void store_slot(T* p, const ShortLane& l, const T (&r)[VEC],
                                           bool rewrite)
{
    if (TAIL == kTailNone || (TAIL == kTailOverlap && (rewrite || l.skip == 0)))
    {
        store_vec<T, VEC, false, STREAM>(p, r);
    }
    else
    {
#pragma unroll
        for (int j = 0; j < VEC; ++j)
            if (slot_owns<VEC, TAIL>(l, j))
                store_vec<T, 1, true, STREAM>(p + j, {r[j]});
    }
}

// The K sums of channel c from its `groups` partials, one after the other.  The
// finishing kernel and the consumers (window_totals) that finish a reduction themselves both
// add in this order and so arrive at the same bits.  The short-segment kernels
// keep their partials group by group, partials[(group * C + c) * K + k]:
// neighbouring lanes, which serve neighbouring channels, then read neighbouring
// memory (at most groups_per_channel_max * C * K values, like the other layout).
template <int K>
__device__ __forceinline__ void sequential_totals(const double* __restrict__ partials, int groups,
                                                  int num_channels, int c, double (&t)[K])
{
    const double* mine = partials + static_cast<size_t>(c) * K;
    const size_t pitch = static_cast<size_t>(num_channels) * K;
#pragma unroll
    for (int k = 0; k < K; ++k)
        t[k] = mine[k];
    // four groups' loads are issued together: the additions wait for one memory
    // latency per batch instead of one per group
    for (int g0 = 1; g0 < groups; g0 += 4)
    {
        double p[4][K];
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int k = 0; k < K; ++k)
                p[u][k] = g0 + u < groups ? mine[(g0 + u) * pitch + k] : 0.0;
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int k = 0; k < K; ++k)
                if (g0 + u < groups)
                    t[k] += p[u][k];
    }
}

// The K sums of the channels of a workgroup's window, added as sequential_totals does, a sum by a thread: totals[k][q]
// of channel q, and the outputs where the workgroup is the window's first. Ends with a barrier. The passes that finish
// a reduction so are bound by what they wait for before their first store: their first batch of elements is loaded
// ahead of the sums. One lane a channel adding all K sums, elements loaded behind them -> this, doubles, forward,
// backward in us of the two launches, going round three sets of tensors: N 135, C 455, 5 x 7 14.9, 26.3 -> 13.4, 21.4;
// N 228, C 69, 10 x 9 12.6, 20.7 -> 12.1, 17.5; N 173, C 143, 13 x 10 19.2, 35.4 -> 18.1, 28.2; N 200, C 600, 7 x 7
// 27.4, 53.6 -> 26.4, 41.9; N 40, C 2000, 14 x 14 with a halo 97, 136 -> 94, 134. (The elements alone ahead: backward
// 26.3, 20.1, 35.9, 55.3. Batches of four samples backward 21.2, 17.1, 29.3, 42.3, and 59 against 58 for N 243, C 306,
// 4 x 6 x 5; of all four sums in a lane 98 registers instead of 80.)
template <typename T, int K>
__device__ __forceinline__ void window_totals(const FusedStats<T>& f, const ShortGeometry& g, T (&totals)[K][kBlockSize], bool store)
{
    const int first = static_cast<int>(blockIdx.x) * g.channels_per_group;
    const size_t pitch = static_cast<size_t>(g.num_channels) * K;
    const double* const window = f.partials + static_cast<size_t>(first) * K;
    for (int i = threadIdx.x; i < g.channels_per_group * K; i += kBlockSize)
    {
        const int q = i / K, k = i % K, c = first + q;
        if (c >= g.num_channels)
            break;
        const uint32_t at = static_cast<uint32_t>(i) * 8u; // in bytes, behind the window's first sum, which is in scalars: of many
                                                           // channels the place among all of a range's needs more bits
        const auto of_group = [&](int group) {
            return *reinterpret_cast<const double*>(reinterpret_cast<const char*>(window + group * pitch) + at);
        };
        double t = of_group(0);
        constexpr int kBatch = 7; // with the first as many as kShortMaxGroups
        for (int g0 = 1; g0 < f.groups; g0 += kBatch)
        {
            double p[kBatch];
#pragma unroll
            for (int u = 0; u < kBatch; ++u)
                if (g0 + u < f.groups)
                    p[u] = of_group(g0 + u);
#pragma unroll
            for (int u = 0; u < kBatch; ++u)
                if (g0 + u < f.groups)
                    t += p[u];
        }
        totals[k][q] = static_cast<T>(t);
        if (store)
            f.out[k][c] = totals[k][q];
    }
    __syncthreads();
}

// Adds what the lanes of each channel hold and stores the
// channel's partial sums of this range of samples, or, when the launch has a
// single range and nobody else finishes the reduction, the results themselves.
template <typename T, int K>
__device__ __forceinline__ void finish_short(const ShortGeometry& g, const ShortLane& l,
                                             const double (&acc)[K], double* partials,
                                             bool always_partials, T* const (&out)[K])
{
    __shared__ double lds[K][kBlockSize];
#pragma unroll
    for (int k = 0; k < K; ++k)
        lds[k][threadIdx.x] = acc[k];
    __syncthreads();
    // The slots of a channel in one row are added as a tree (lane v takes what
    // lane v + step holds, step = 2^k downwards), then the channel's first lane
    // adds the rows one after the other: a fixed order, a handful of steps.
    double t[K];
#pragma unroll
    for (int k = 0; k < K; ++k)
        t[k] = acc[k];
    int width = 1;
    while (width < g.slots)
        width <<= 1;
    for (int step = width >> 1; step >= 1; step >>= 1)
    {
        // lanes below `step` read lanes from `step` on and write their own: one barrier a step
        if (l.valid > 0 && l.slot < step && l.slot + step < g.slots)
        {
#pragma unroll
            for (int k = 0; k < K; ++k)
            {
                t[k] += lds[k][threadIdx.x + step];
                lds[k][threadIdx.x] = t[k];
            }
        }
        __syncthreads();
    }
    if (l.leads)
    {
        const int lanes_per_row = kBlockSize / g.rows;
        for (int r = 1; r < g.rows; ++r)
        {
#pragma unroll
            for (int k = 0; k < K; ++k)
                t[k] += lds[k][threadIdx.x + r * lanes_per_row];
        }
    }
    if (!l.leads)
        return;
    if (gridDim.y == 1 && !always_partials)
    {
#pragma unroll
        for (int k = 0; k < K; ++k)
            out[k][l.c] = static_cast<T>(t[k]);
    }
    else
    {
        double* mine =
            partials + (static_cast<size_t>(blockIdx.y) * g.num_channels + l.c) * K;
#pragma unroll
        for (int k = 0; k < K; ++k)
            mine[k] = t[k];
    }
}

template <typename T, int K>
__global__ void bn_finish_short_kernel(const double* __restrict__ partials, int groups,
                                       int num_channels, T* out0, T* out1, T* out2, T* out3)
{
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= num_channels)
        return;
    double t[K];
    sequential_totals<K>(partials, groups, num_channels, c, t);
    T* outs[4] = {out0, out1, out2, out3};
#pragma unroll
    for (int k = 0; k < K; ++k)
        outs[k][c] = static_cast<T>(t[k]);
}

template <typename T, int VEC, int TAIL>
__global__ __launch_bounds__(kBlockSize) void bn_sums_short_kernel(
    const T* __restrict__ x, T* __restrict__ sums, T* __restrict__ sqsums, double* partials,
    const ShortTensor tx, const ShortGeometry g, bool always_partials)
{
    const ShortLane l = short_lane<VEC, TAIL>(g, static_cast<int>(threadIdx.x), static_cast<int>(blockIdx.x));
    double acc[2] = {0.0, 0.0};
    if (l.valid > 0)
    {
        auto accumulate = [&](const T (&v)[VEC]) {
#pragma unroll
            for (int j = 0; j < VEC; ++j)
            {
                if (!slot_owns<VEC, TAIL>(l, j))
                    continue;
                const double d = static_cast<double>(v[j]);
                acc[0] += d;
                if constexpr (sizeof(T) == 4)
                    acc[1] = __builtin_fma(d, d, acc[1]); // the product of two floats is exact in fp64
                else
                    acc[1] += d * d;
            }
        };
        const T* p = x + l.c * tx.stride_c + slot_offset(l, tx);
        const int64_t stride_n = tx.stride_n;
        int n = blockIdx.y * g.samples_per_group;
        const int end = n + g.samples_per_group < g.num_samples ? n + g.samples_per_group
                                                                : g.num_samples;
        const int step = g.rows;
        n += l.row;
        for (; n + (kUnroll - 1) * step < end; n += kUnroll * step)
        {
            T v[kUnroll][VEC];
#pragma unroll
            for (int u = 0; u < kUnroll; ++u)
                load_slot<T, VEC, TAIL>(p + (n + u * step) * stride_n, l, v[u]);
#pragma unroll
            for (int u = 0; u < kUnroll; ++u)
                accumulate(v[u]);
        }
        for (; n < end; n += step)
        {
            T v[VEC];
            load_slot<T, VEC, TAIL>(p + n * stride_n, l, v);
            accumulate(v);
        }
    }
    T* const out[2] = {sums, sqsums};
    finish_short<T, 2>(g, l, acc, partials, always_partials, out);
}

template <typename T, int VEC, int TAIL, int MODE>
__global__ __launch_bounds__(kBlockSize) void bn_apply_short_kernel(
    const T* __restrict__ x, const T* __restrict__ mean, const T* __restrict__ var,
    const T* __restrict__ scale, const T* __restrict__ bias, T* __restrict__ y, T epsilon,
    const ShortTensor tx, const ShortTensor ty, const ShortGeometry g, const FusedStats<T> fused)
{
    constexpr bool FUSED = MODE == kFusedApply, STREAM = MODE != kNormalApply;
    const ShortLane l = short_lane<VEC, TAIL>(g, static_cast<int>(threadIdx.x), static_cast<int>(blockIdx.x));
    const T* const xp = x + l.c * tx.stride_c + slot_offset(l, tx);
    const int64_t x_stride_n = tx.stride_n, y_stride_n = ty.stride_n;
    int n = blockIdx.y * g.samples_per_group;
    const int end =
        n + g.samples_per_group < g.num_samples ? n + g.samples_per_group : g.num_samples;
    T v[kUnroll][VEC];
    const auto load = [&] {
#pragma unroll
        for (int u = 0; u < kUnroll; ++u)
            if (n + u < end)
                load_slot<T, VEC, TAIL>(xp + (n + u) * x_stride_n, l, v[u]);
    };
    T sc = T(0), bi = T(0);
    if (l.valid > 0)
    {
        load();
        sc = scale[l.c];
        bi = bias[l.c];
    }
    T m = T(0), variance = T(0);
    if constexpr (FUSED)
    {
        __shared__ T totals[2][kBlockSize];
        window_totals<T, 2>(fused, g, totals, false);
        if (l.valid > 0)
            sums_to_mean_var(totals[0][l.q], totals[1][l.q], static_cast<T>(fused.num_per_sum), &m, &variance);
        if (l.leads && blockIdx.y == 0)
        {
            fused.out[0][l.c] = m;
            fused.out[1][l.c] = variance;
            fused.out[2][l.c] = fma_t(fused.decay, fused.out[2][l.c], (T(1) - fused.decay) * m);
            fused.out[3][l.c] = fma_t(fused.decay, fused.out[3][l.c], (T(1) - fused.decay) * variance);
        }
    }
    else if (l.valid > 0)
    {
        m = mean[l.c];
        variance = var[l.c];
    }
    if (l.valid == 0)
        return;
    const T inv_stdev = inv_sqrt_t(variance + epsilon);
    T* const yp = y + l.c * ty.stride_c + slot_offset(l, ty);
    for (;;)
    {
#pragma unroll
        for (int u = 0; u < kUnroll; ++u)
            if (n + u < end)
            {
#pragma unroll
                for (int j = 0; j < VEC; ++j)
                    v[u][j] = fma_t((v[u][j] - m) * inv_stdev, sc, bi);
                store_slot<T, VEC, TAIL, STREAM>(yp + (n + u) * y_stride_n, l, v[u], true);
            }
        n += kUnroll;
        if (n >= end) // uniform
            break;
        load();
    }
}

template <typename T, int VEC, int TAIL>
__global__ __launch_bounds__(kBlockSize) void bn_backprop1_short_kernel(
    const T* __restrict__ x, const T* __restrict__ dy, const T* __restrict__ mean,
    const T* __restrict__ var, const T* __restrict__ scale, T* __restrict__ dscale,
    T* __restrict__ dbias, T* __restrict__ dmean, T* __restrict__ dvar, T epsilon,
    double* partials, const ShortTensor tx, const ShortTensor td, const ShortGeometry g,
    bool always_partials)
{
    const ShortLane l = short_lane<VEC, TAIL>(g, static_cast<int>(threadIdx.x), static_cast<int>(blockIdx.x));
    double acc[4] = {0.0, 0.0, 0.0, 0.0};
    if (l.valid > 0)
    {
        const T m = mean[l.c];
        const T sc = scale[l.c];
        const T inv_stdev = inv_sqrt_t(var[l.c] + epsilon);
        const T dvar_factor = inv_stdev * inv_stdev * inv_stdev / T(2);
        const double neg_inv = -static_cast<double>(inv_stdev);
        const double neg_fac = -static_cast<double>(dvar_factor);
        auto accumulate = [&](const T (&xv)[VEC], const T (&dv)[VEC]) {
#pragma unroll
            for (int j = 0; j < VEC; ++j)
            {
                if (!slot_owns<VEC, TAIL>(l, j))
                    continue;
                const T xm = xv[j] - m;
                const T xhat = xm * inv_stdev;
                const T dxhat = dv[j] * sc;
                const T t = dxhat * xm;
                const double dd = static_cast<double>(dv[j]);
                acc[0] = __builtin_fma(dd, static_cast<double>(xhat), acc[0]);
                acc[1] += dd;
                acc[2] = __builtin_fma(static_cast<double>(dxhat), neg_inv, acc[2]);
                acc[3] = __builtin_fma(static_cast<double>(t), neg_fac, acc[3]);
            }
        };
        constexpr int kUnroll2 = kUnroll / 2; // two streams: same bytes in flight
        const T* xp = x + l.c * tx.stride_c + slot_offset(l, tx);
        const T* dp = dy + l.c * td.stride_c + slot_offset(l, td);
        const int64_t x_stride_n = tx.stride_n, d_stride_n = td.stride_n;
        int n = blockIdx.y * g.samples_per_group;
        const int end = n + g.samples_per_group < g.num_samples ? n + g.samples_per_group
                                                                : g.num_samples;
        const int step = g.rows;
        n += l.row;
        for (; n + (kUnroll2 - 1) * step < end; n += kUnroll2 * step)
        {
            T xv[kUnroll2][VEC], dv[kUnroll2][VEC];
#pragma unroll
            for (int u = 0; u < kUnroll2; ++u)
            {
                load_slot<T, VEC, TAIL>(xp + (n + u * step) * x_stride_n, l, xv[u]);
                load_slot<T, VEC, TAIL, true>(dp + (n + u * step) * d_stride_n, l, dv[u]);
            }
#pragma unroll
            for (int u = 0; u < kUnroll2; ++u)
                accumulate(xv[u], dv[u]);
        }
        for (; n < end; n += step)
        {
            T xv[VEC], dv[VEC];
            load_slot<T, VEC, TAIL>(xp + n * x_stride_n, l, xv);
            load_slot<T, VEC, TAIL, true>(dp + n * d_stride_n, l, dv);
            accumulate(xv, dv);
        }
    }
    T* const out[4] = {dscale, dbias, dmean, dvar};
    finish_short<T, 4>(g, l, acc, partials, always_partials, out);
}

// x and dx may alias: each lane reads its elements before it writes them
// (`disjoint`: they share no memory).
template <typename T, int VEC, int TAIL, bool FUSED>
__global__ __launch_bounds__(kBlockSize) void bn_backprop2_short_kernel(
    const T* x, const T* __restrict__ dy, const T* __restrict__ mean, const T* __restrict__ var,
    const T* __restrict__ scale, const T* __restrict__ dmean, const T* __restrict__ dvar, T* dx,
    T epsilon, size_t num_per_sum, const ShortTensor tx, const ShortTensor td,
    const ShortTensor to, const ShortGeometry g, bool disjoint, const FusedStats<T> fused)
{
    const ShortLane l = short_lane<VEC, TAIL>(g, static_cast<int>(threadIdx.x), static_cast<int>(blockIdx.x));
    constexpr int kBatch = kUnroll / 2; // two streams: same bytes in flight
    const T* const xp = x + l.c * tx.stride_c + slot_offset(l, tx);
    const T* const dp = dy + l.c * td.stride_c + slot_offset(l, td);
    const int64_t x_stride_n = tx.stride_n, d_stride_n = td.stride_n, o_stride_n = to.stride_n;
    int n = blockIdx.y * g.samples_per_group;
    const int end =
        n + g.samples_per_group < g.num_samples ? n + g.samples_per_group : g.num_samples;
    T xv[kBatch][VEC], dv[kBatch][VEC];
    const auto load = [&] {
#pragma unroll
        for (int u = 0; u < kBatch; ++u)
            if (n + u < end)
            {
                load_slot<T, VEC, TAIL>(xp + (n + u) * x_stride_n, l, xv[u]);
                load_slot<T, VEC, TAIL, true>(dp + (n + u) * d_stride_n, l, dv[u]);
            }
    };
    T m = T(0), sc = T(0), variance = T(0);
    if (l.valid > 0)
    {
        load();
        m = mean[l.c];
        sc = scale[l.c];
        variance = var[l.c];
    }
    T dmean_c = T(0), dvar_c = T(0);
    if constexpr (FUSED)
    {
        __shared__ T totals[4][kBlockSize];
        window_totals<T, 4>(fused, g, totals, blockIdx.y == 0);
        if (l.valid > 0)
        {
            dmean_c = totals[2][l.q];
            dvar_c = totals[3][l.q];
        }
    }
    else if (l.valid > 0)
    {
        dmean_c = dmean[l.c];
        dvar_c = dvar[l.c];
    }
    if (l.valid == 0)
        return;
    const T inv_stdev = inv_sqrt_t(variance + epsilon);
    const T dmean_term = dmean_c / static_cast<T>(num_per_sum);
    const T dvar_term = dvar_c * T(2) / static_cast<T>(num_per_sum - 1);
    T* const op = dx + l.c * to.stride_c + slot_offset(l, to);
    for (;;)
    {
#pragma unroll
        for (int u = 0; u < kBatch; ++u)
            if (n + u < end)
            {
#pragma unroll
                for (int j = 0; j < VEC; ++j)
                {
                    const T r = fma_t(dv[u][j] * sc, inv_stdev, dmean_term);
                    xv[u][j] = fma_t(xv[u][j] - m, dvar_term, r);
                }
                store_slot<T, VEC, TAIL>(op + (n + u) * o_stride_n, l, xv[u], disjoint);
            }
        n += kBatch;
        if (n >= end) // uniform
            break;
        load();
    }
}

// ---- whole channels in one workgroup: one launch ------------------------------
#include "h2x_bn_once.hpp"

#include "h2x_bn_window.hpp"
// ---- whole channels in several workgroups: one launch ---------------------------
#include "h2x_bn_team.hpp"

#include "h2x_bn_ordered.hpp"

#include "h2x_bn_short.hpp"

// ---- host side ---------------------------------------------------------------

template <typename T>
constexpr int full_vec()
{
    return 16 / sizeof(T);
}

bool grid_ok(size_t blocks)
{
    return blocks <= 0x7fffffffull;
}

// One tensor as the kernels see it, plus what decides the vector width.
struct HostTensor
{
    TensorMap map;
    bool strided = false; // needs index splitting
    size_t row = 0;       // contiguous interior elements per row (strided) or `spatial` (dense)
    bool aligned = false; // dense: every segment starts on a 16-byte boundary
};

// Index splitting that is the identity (x = i, y = z = 0), for a dense tensor
// that takes part in a launch of the strided kernels: every index is below the
// divisor 2^31 - 1.
void set_dense_map(TensorMap* m)
{
    m->w = make_fastdiv(0x7fffffffu);
    m->h = make_fastdiv(1);
    m->sy = m->sz = 0;
    m->spr = make_fastdiv(1);
    m->width = 0;
}

template <typename T>
HostTensor dense_tensor(const void* p, int num_channels, size_t spatial, size_t real)
{
    HostTensor t;
    t.map.stride_c = static_cast<int64_t>(real);
    t.map.stride_n = static_cast<int64_t>(real) * num_channels;
    set_dense_map(&t.map);
    t.row = spatial;
    t.aligned = aligned16(p) && real % full_vec<T>() == 0;
    return t;
}

// A tensor given by local shape and strides (innermost first; channel and
// sample are the last two dimensions).  Falls back to the dense description
// when the inner spatial dimensions carry no halo.
template <typename T>
int strided_tensor(const h2x_tensor_geometry* g, const void* p, int num_samples, HostTensor* out,
                   int* num_channels, size_t* spatial)
{
    if (!g || g->num_dims < 3 || g->num_dims > 5)
        return H2X_ERR_INVALID_ARGUMENT;
    const int nd = g->num_dims, ns = nd - 2;
    size_t sp = 1;
    for (int i = 0; i < nd; ++i)
        if (g->local_shape[i] < 0 || g->strides[i] < 0)
            return H2X_ERR_INVALID_ARGUMENT;
    if (g->strides[0] != 1 && g->local_shape[0] > 1)
        return H2X_ERR_UNSUPPORTED;
    for (int i = 0; i < ns; ++i)
        sp *= static_cast<size_t>(g->local_shape[i]);
    if (g->local_shape[nd - 1] != num_samples && num_samples != 0)
        return H2X_ERR_INVALID_ARGUMENT;
    *num_channels = static_cast<int>(g->local_shape[nd - 2]);
    *spatial = sp;
    HostTensor t;
    t.map.stride_c = g->strides[nd - 2];
    t.map.stride_n = g->strides[nd - 1];
    // dense inside a segment?  (stride of each spatial dimension = product of the extents below it)
    bool dense = true;
    int64_t expect = 1;
    for (int i = 0; i < ns; ++i)
    {
        if (g->local_shape[i] > 1 && g->strides[i] != expect)
            dense = false;
        expect *= g->local_shape[i];
    }
    if (dense)
    {
        set_dense_map(&t.map);
        t.row = sp;
        t.aligned = aligned16(p) && t.map.stride_c % full_vec<T>() == 0
                    && t.map.stride_n % full_vec<T>() == 0;
    }
    else
    {
        if (sp >= (1ull << 31))
            return H2X_ERR_TOO_LARGE;
        t.strided = true;
        t.row = static_cast<size_t>(g->local_shape[0]);
        t.map.w = make_fastdiv(static_cast<uint32_t>(g->local_shape[0]));
        t.map.h = make_fastdiv(ns > 1 ? static_cast<uint32_t>(g->local_shape[1]) : 1u);
        if ((ns > 1 && g->strides[1] > 0xffffffffll) || (ns > 2 && g->strides[2] > 0xffffffffll))
            return H2X_ERR_TOO_LARGE; // strides inside a segment are kept as 32-bit integers
        t.map.sy = ns > 1 ? static_cast<uint32_t>(g->strides[1]) : 0;
        t.map.sz = ns > 2 ? static_cast<uint32_t>(g->strides[2]) : 0;
        t.map.spr = make_fastdiv(1);
        t.map.width = 0;
        t.aligned = false;
    }
    *out = t;
    return H2X_SUCCESS;
}

// Vector width all tensors of a launch allow, and whether the strided kernels are needed.
// Dense tensors whose segments are no multiple of the vector long, or start off a
// 16-byte boundary, are handed to the strided kernels too, as tensors with one row
// per segment: vectors aligned to one element, the last one of a segment overlapping
// the one before it (N 16, C 64, 57 x 57: forward 23 -> 15 us against element by element).
constexpr size_t kMinUnalignedSegment = 256;

template <typename T, typename H> // H: HostTensor or const HostTensor
int common_vector(std::initializer_list<H*> ts, bool* strided)
{
    const int full = full_vec<T>();
    *strided = false;
    for (const HostTensor* t : ts)
        *strided = *strided || t->strided;
    if (!*strided)
    {
        bool aligned_vectors = true, unaligned_vectors = true;
        for (const HostTensor* t : ts)
        {
            if (t->row % full != 0 || !t->aligned)
                aligned_vectors = false;
            if (t->row < kMinUnalignedSegment || t->row >= (1ull << 31))
                unaligned_vectors = false;
        }
        if (aligned_vectors)
            return full;
        if (!unaligned_vectors)
            return 1;
        *strided = true;
        return full;
    }
    // a row of a strided tensor must hold a vector
    for (const HostTensor* t : ts)
        if (t->strided && t->row < static_cast<size_t>(full))
            return 1;
    return full;
}

// Sets the tensors of a strided launch with vectors up for padded rows (see
// TensorMap) and returns the padded length of a segment.  The rows are those of
// the tensors with halos or folded samples; a launch of dense tensors only has
// one row per segment.  Dense tensors in a launch with rows are addressed row by
// row like the others.
template <typename T>
size_t pad_rows(std::initializer_list<HostTensor*> ts, size_t spatial)
{
    const uint32_t vec = full_vec<T>();
    size_t width = spatial;
    uint32_t rows_per_plane = 1;
    for (const HostTensor* t : ts)
        if (t->strided)
        {
            width = t->row;
            rows_per_plane = t->map.h.divisor;
        }
    const size_t spr = (width + vec - 1) / vec;
    for (HostTensor* t : ts)
    {
        if (!t->strided)
        {
            t->map.h = make_fastdiv(rows_per_plane);
            t->map.sy = static_cast<uint32_t>(width);
            t->map.sz = static_cast<uint32_t>(width * rows_per_plane); // below 2^31: a segment's elements
        }
        t->map.spr = make_fastdiv(static_cast<uint32_t>(spr));
        t->map.width = static_cast<uint32_t>(width);
    }
    return spatial / width * spr * vec;
}

// Segments of 257 to 1023 elements (19 x 19, 27 x 27, 28 x 28 activations; shorter
// ones go to the short-segment kernels).  A (sample, channel) segment shorter than
// what a workgroup moves leaves lanes idle in the dense kernels.  The samples of a
// channel are then folded
// into the spatial index: the tensor is addressed as ONE sample whose segments
// are N rows of `spatial` elements, `stride_n` apart, through the index
// splitting of the strided kernels (x = i mod spatial, y = i / spatial), so
// that a workgroup streams through many samples of its channel.  (Measured on
// segments of 49 elements before those had kernels of their own: normalise
// 387 us -> 75 us, backprop2 520 us -> 110 us at N 256, C 2048.)
constexpr size_t kFoldBelow = 1024;

bool fold_samples(int* num_samples, size_t* spatial, std::initializer_list<HostTensor*> ts)
{
    if (*num_samples <= 1 || *spatial >= kFoldBelow)
        return false;
    for (const HostTensor* t : ts)
        if (t->strided || t->map.stride_n > 0xffffffffll)
            return false; // rows are already split, or lie further apart than a 32-bit stride
    for (HostTensor* t : ts)
    {
        t->strided = true;
        t->row = *spatial;
        t->map.w = make_fastdiv(static_cast<uint32_t>(*spatial));
        t->map.h = make_fastdiv(static_cast<uint32_t>(*num_samples));
        t->map.sy = static_cast<uint32_t>(t->map.stride_n);
        t->map.sz = 0;
        t->aligned = false;
    }
    *spatial *= static_cast<size_t>(*num_samples); // < 1024 * 2^31: the callers' grid checks apply
    *num_samples = 1;
    return true;
}

// Segments of at most this many elements go to the short-segment kernels: up
// to here a segment's share of the cache lines at its two ends is 11 % or more.
constexpr size_t kShortSegment = 256;
// Workgroups an elementwise short-segment pass aims at.  The input gradient
// (three tensors a sample) does better with half of what normalise takes: N 64,
// C 1024, 14 x 14 backward 55 -> 48 us, N 256, C 2048, 7 x 7 91 -> 86 us with
// 4096 (2048: 48 / 88 us); forward is the same from 2048 to 32768.
constexpr int kShortElementwiseBlocks = 8192;
constexpr int kShortGradientBlocks = 4096;

// Elements from the first to the last interior element of a segment.
size_t short_span(const HostTensor& t, size_t spatial)
{
    if (!t.strided)
        return spatial;
    const size_t w = t.map.w.divisor, h = t.map.h.divisor;
    const size_t d = spatial / (w * h);
    return (w - 1) + (h - 1) * static_cast<size_t>(t.map.sy) + (d - 1) * static_cast<size_t>(t.map.sz)
           + 1;
}

// A tensor as a short-segment launch addresses it.  When the launch goes row by
// row (some tensor has halos inside its segments), a dense tensor's rows follow
// one another: strides row and row * h.
ShortTensor short_tensor(const HostTensor& t, const ShortGeometry& g)
{
    ShortTensor r;
    r.stride_n = t.map.stride_n;
    r.stride_c = t.map.stride_c;
    r.h = g.rows_per_plane;
    r.sy = t.strided ? t.map.sy : g.row;
    r.sz = t.strided ? t.map.sz : static_cast<int64_t>(g.row) * g.rows_per_plane;
    return r;
}

// Whether a launch over these tensors takes the short-segment kernels, and the
// window of channels a workgroup serves then.
template <typename T>
bool short_segments(int num_samples, int num_channels, size_t spatial,
                    std::initializer_list<const HostTensor*> ts, ShortGeometry* g)
{
    if (spatial == 0 || spatial > kShortSegment || num_samples < 1 || num_channels < 1)
        return false;
    for (const HostTensor* t : ts)
        if (t->strided && short_span(*t, spatial) > 0x7fffffffull)
            return false; // offsets within a segment are kept as 32-bit integers
    const int vec = full_vec<T>();
    g->num_samples = num_samples;
    g->num_channels = num_channels;
    g->spatial = static_cast<int>(spatial);
    // dense tensors only: the segment is one row; else every tensor goes row by row
    g->row = g->spatial;
    g->rows_per_plane = 1;
    for (const HostTensor* t : ts)
        if (t->strided)
        {
            g->row = static_cast<int>(t->map.w.divisor);
            g->rows_per_plane = static_cast<int>(t->map.h.divisor);
        }
    g->slots_per_row = (g->row + vec - 1) / vec;
    g->slots = g->spatial / g->row * g->slots_per_row;
    if (g->slots > kBlockSize)
        return false;
    g->rows = 1;
    g->channels_per_group = kBlockSize / g->slots;
    g->samples_per_group = num_samples;
    return true;
}

int short_windows(const ShortGeometry& g)
{
    return (g.num_channels + g.channels_per_group - 1) / g.channels_per_group;
}

// How a short-segment reduction is spread over the GPU.  The lanes of a
// workgroup may split into `rows` that take every rows-th sample of a narrower
// window (never narrower than kShortMinRowBytes per sample, so that a row still
// reads whole cache lines), and the samples may be cut into ranges whose partial
// sums a later kernel adds (at most kShortMaxGroups: that kernel adds them one
// after the other).  A tensor small enough for every lane to get by with two
// batches of loads takes rows only and a single range: no partial sums, no
// finishing work.  Otherwise ranges first, up to kShortWantGroups workgroups,
// and rows only if that leaves fewer than kShortMinGroups.
constexpr int kShortWantGroups = 2048;
constexpr int kShortMinGroups = 512;
constexpr int kShortMaxGroups = 8;
constexpr size_t kShortMinRowBytes = 256;

bool short_split_rows(ShortGeometry* g, size_t elem_bytes)
{
    const int narrower = kBlockSize / (g->rows * 2) / g->slots;
    if (static_cast<size_t>(narrower) * g->spatial * elem_bytes < kShortMinRowBytes)
        return false;
    g->rows *= 2;
    g->channels_per_group = narrower;
    return true;
}

int short_reduction_groups(ShortGeometry* g, int gmax, int unroll, size_t elem_bytes)
{
    const ShortGeometry whole = *g;
    while (g->num_samples / g->rows > unroll && short_split_rows(g, elem_bytes))
    {
    }
    if ((g->num_samples + g->rows * unroll - 1) / (g->rows * unroll) <= 2)
    {
        g->samples_per_group = g->num_samples;
        return 1;
    }
    *g = whole;
    const int want = (kShortWantGroups + short_windows(*g) - 1) / short_windows(*g);
    const int groups = std::max(1, std::min({g->num_samples / unroll, gmax, kShortMaxGroups, want}));
    const int per = (g->num_samples + groups - 1) / groups;
    while (static_cast<long long>(short_windows(*g)) * groups < kShortMinGroups
           && per >= 2 * unroll * g->rows && short_split_rows(g, elem_bytes))
    {
    }
    g->samples_per_group = per;
    return (g->num_samples + per - 1) / per;
}

// Ranges of samples of a short-segment elementwise pass: whole batches of
// `unroll` samples (what a lane keeps in flight) where there are that many.  A
// pass that finishes a reduction first (`prologue_bytes` of partial sums per
// channel) takes ranges long enough to move at least as many bytes of tensors
// (`sample_bytes` per channel and sample).
int short_elementwise_groups(ShortGeometry* g, int unroll, int budget, size_t prologue_bytes = 0,
                             size_t sample_bytes = 1)
{
    const long long units = static_cast<long long>(g->num_samples) * short_windows(*g);
    long long per = std::max<long long>(unroll, units / budget);
    per = std::max<long long>(per, (prologue_bytes + sample_bytes - 1) / sample_bytes);
    per = (per + unroll - 1) / unroll * unroll;
    per = std::max<long long>(per, (g->num_samples + 65534) / 65535); // grid.y
    g->samples_per_group = static_cast<int>(std::min<long long>(per, g->num_samples));
    return (g->num_samples + g->samples_per_group - 1) / g->samples_per_group;
}

// Launches kernel<T, V, TAIL> of the short-segment family (`sg`: the geometry).
#define H2X_DISPATCH_SHORT(KERNEL, GRID, ...)                                                      \
    do                                                                                             \
    {                                                                                              \
        if (sg.row % full_vec<T>() == 0)                                                           \
            launch(KERNEL<T, full_vec<T>(), kTailNone>, GRID, kBlockSize, stream, __VA_ARGS__);    \
        else if (sg.row > full_vec<T>())                                                           \
            launch(KERNEL<T, full_vec<T>(), kTailOverlap>, GRID, kBlockSize, stream, __VA_ARGS__); \
        else                                                                                       \
            launch(KERNEL<T, full_vec<T>(), kTailScalar>, GRID, kBlockSize, stream, __VA_ARGS__);  \
    } while (0)

#define H2X_DISPATCH_SHORT_FUSED(KERNEL, FUSED, GRID, ...)                                         \
    do                                                                                             \
    {                                                                                              \
        if (sg.row % full_vec<T>() == 0)                                                           \
            launch(KERNEL<T, full_vec<T>(), kTailNone, FUSED>, GRID, kBlockSize, stream, __VA_ARGS__);\
        else if (sg.row > full_vec<T>())                                                           \
            launch(KERNEL<T, full_vec<T>(), kTailOverlap, FUSED>, GRID, kBlockSize, stream, __VA_ARGS__);\
        else                                                                                       \
            launch(KERNEL<T, full_vec<T>(), kTailScalar, FUSED>, GRID, kBlockSize, stream, __VA_ARGS__);\
    } while (0)

// Launches kernel<T, V, STRIDED> for the width and layout chosen at run time.
#define H2X_DISPATCH(KERNEL, GRID, ...)                                                            \
    do                                                                                             \
    {                                                                                              \
        if (strided)                                                                               \
        {                                                                                          \
            if (vw > 1)                                                                            \
                launch(KERNEL<T, full_vec<T>(), true>, GRID, kBlockSize, stream, __VA_ARGS__);     \
            else                                                                                   \
                launch(KERNEL<T, 1, true>, GRID, kBlockSize, stream, __VA_ARGS__);                 \
        }                                                                                          \
        else                                                                                       \
        {                                                                                          \
            if (vw > 1)                                                                            \
                launch(KERNEL<T, full_vec<T>(), false>, GRID, kBlockSize, stream, __VA_ARGS__);    \
            else                                                                                   \
                launch(KERNEL<T, 1, false>, GRID, kBlockSize, stream, __VA_ARGS__);                \
        }                                                                                          \
    } while (0)

// Launches an elementwise kernel<T, V, LAYOUT, FUSED>.
#define H2X_DISPATCH_ELEMENTWISE(KERNEL, FUSED, GRID, ...)                                         \
    do                                                                                             \
    {                                                                                              \
        if (vw > 1 && strided)                                                                     \
            launch(KERNEL<T, full_vec<T>(), kLayoutRows, FUSED>, GRID, kBlockSize, stream, __VA_ARGS__);\
        else if (vw > 1)                                                                           \
            launch(KERNEL<T, full_vec<T>(), kLayoutDense, FUSED>, GRID, kBlockSize, stream, __VA_ARGS__);\
        else if (strided)                                                                          \
            launch(KERNEL<T, 1, kLayoutRows, FUSED>, GRID, kBlockSize, stream, __VA_ARGS__);       \
        else                                                                                       \
            launch(KERNEL<T, 1, kLayoutDense, FUSED>, GRID, kBlockSize, stream, __VA_ARGS__);      \
    } while (0)

// ---- what a launch looks like to the log ----------------------------------------

LaunchRecord short_record(int kernel, const ShortGeometry& sg, dim3 grid, int vec,
                          std::initializer_list<const HostTensor*> ts, bool last_is_output)
{
    LaunchRecord r;
    r.kernel = kernel;
    r.family = kFamilyShort;
    r.vec = vec;
    r.tail = sg.row % vec == 0 ? kTailNone : sg.row > vec ? kTailOverlap : kTailScalar;
    r.grid_x = grid.x;
    r.grid_y = grid.y;
    r.num_samples = sg.num_samples;
    r.num_channels = sg.num_channels;
    r.spatial = static_cast<size_t>(sg.spatial);
    r.geometry = sg;
    r.last_is_output = last_is_output;
    for (const HostTensor* t : ts)
        r.tensor[r.num_tensors++] = short_tensor(*t, sg);
    return r;
}

LaunchRecord long_record(int kernel, bool strided, int vw, dim3 grid, int num_samples,
                         int num_channels, size_t spatial, const Chunking& ch,
                         std::initializer_list<const HostTensor*> ts, bool last_is_output)
{
    LaunchRecord r;
    r.kernel = kernel;
    r.family = strided ? kFamilyStrided : kFamilyDense;
    r.vec = vw;
    r.grid_x = grid.x;
    r.grid_y = grid.y;
    r.num_samples = num_samples;
    r.num_channels = num_channels;
    r.spatial = spatial;
    r.chunk = ch.chunk;
    r.chunks_per_seg = ch.chunks_per_seg;
    r.last_is_output = last_is_output;
    for (const HostTensor* t : ts)
        r.map[r.num_tensors++] = t->map;
    return r;
}

LaunchRecord small_record(int kernel, unsigned int grid_x, int num_channels, int num_sums = 0)
{
    LaunchRecord r;
    r.kernel = kernel;
    r.grid_x = grid_x;
    r.num_channels = num_channels;
    r.num_sums = num_sums;
    return r;
}

template <typename T>
int zero_outputs(std::initializer_list<void*> outs, int num_channels, hipStream_t stream)
{
    const int blocks = (num_channels + kBlockSize - 1) / kBlockSize;
    for (void* p : outs)
        if (!logged(small_record(kKernelFill, blocks, num_channels)))
            launch(fill_kernel<T>, blocks, kBlockSize, stream, static_cast<T*>(p), num_channels, T(0));
    return issued();
}

// How a long-segment reduction over tensors `ts` (which it sets up for the launch) is cut: into
// units of whole tiles, which `groups` workgroups a channel take in turn.
struct ReductionPlan
{
    bool folded, strided;
    int vw;
    int num_samples;
    size_t spatial;
    Chunking ch;
    size_t units, groups;
    int groups_max;
};

// Doubles of a channel that a team holds backward: 64 members of 512 threads with eight vectors.
constexpr size_t kMostOrdered = 64 * 512 * 8 * 2;

// unroll: vectors of a tile a thread.  Units of doubles are tiles of kUnroll vectors in both directions, which
// the kernels that read once keep in registers (h2x_bn_ordered.hpp); not those of channels beyond the largest team,
// where shorter units fill the chip better (backward, N 8, C 2, 64 x 64 x 32 18.8 and 19.8 us).
template <typename T>
int plan_reduction(int num_samples, int num_channels, size_t spatial, std::initializer_list<HostTensor*> ts, int unroll,
                   ReductionPlan* p)
{
    p->folded = fold_samples(&num_samples, &spatial, ts);
    bool any = false;
    for (const HostTensor* t : ts)
        any = any || t->strided;
    if (spatial >= (1ull << 31) && any)
        return H2X_ERR_TOO_LARGE;
    p->vw = common_vector<T>(ts, &p->strided);
    if (p->strided && p->vw > 1)
        spatial = pad_rows<T>(ts, spatial);
    if (spatial >= (1ull << 31) && p->strided)
        return H2X_ERR_TOO_LARGE;
    p->num_samples = num_samples;
    p->spatial = spatial;
    p->groups_max = max_groups_per_channel(num_channels);
    const int budget = reduction_groups_per_channel(num_channels, p->strided);
    const bool held = sizeof(T) == 8 && num_samples * spatial <= kMostOrdered;
    const size_t tile = static_cast<size_t>(kBlockSize) * p->vw * (held ? kUnroll : unroll);
    p->ch = make_chunking(spatial, num_samples, budget, tile, tile);
    p->units = static_cast<size_t>(p->ch.chunks_per_seg) * num_samples;
    if (p->units > 0xffffffffull || num_channels > 65535)
        return H2X_ERR_TOO_LARGE;
    p->groups = std::min<size_t>(p->units, budget);
    if (held && p->units > p->groups)
    {
        // As many units a group as the busiest one plays anyway, and as fill the batches of a thread: 70 units in 69 groups leave
        // every other place of a team empty (N 70, C 60, 38 x 38, forward, backward 30.2, 46.2 us, in 35 groups 21.7, 35.7; N 96
        // 34.8, 55.5 and 26.9, 41.1; N 184, C 91, 23 x 26, halo of 1 106, 162 and 62, 104; two launches are the same either way).
        const size_t batches = p->ch.chunk / tile;
        size_t rounds = (p->units + budget - 1) / budget;
        if (batches * rounds == 3)
            rounds = 4;
        p->groups = (p->units + rounds - 1) / rounds;
    }
    return H2X_SUCCESS;
}

// `fused_out` non-null: the caller finishes the reduction itself (a fused
// consumer kernel): every workgroup stores partials, no finishing launch.
template <typename T>
int sums_impl(int num_samples, int num_channels, size_t spatial, const HostTensor& tx_in,
              const void* x, void* sums, void* sqsums, void* workspace, hipStream_t stream,
              FusedStats<T>* fused_out = nullptr)
{
    if (num_channels == 0)
        return H2X_SUCCESS;
    if (num_samples == 0 || spatial == 0)
        return zero_outputs<T>({sums, sqsums}, num_channels, stream);
    if (fused_out)
        fused_out->sequential = false;
    ShortGeometry sg;
    if (short_segments<T>(num_samples, num_channels, spatial, {&tx_in}, &sg))
    {
        const int gmax = max_groups_per_channel(num_channels);
        const int groups = short_reduction_groups(&sg, gmax, kUnroll, sizeof(T));
        double* partials = static_cast<double*>(workspace);
        const dim3 grid(short_windows(sg), groups);
        LaunchRecord rec = short_record(kKernelSums, sg, grid, full_vec<T>(), {&tx_in}, false);
        rec.num_sums = 2;
        rec.groups_max = gmax;
        rec.partials = groups > 1 || fused_out != nullptr;
        if (!logged(rec))
            H2X_DISPATCH_SHORT(bn_sums_short_kernel, grid, static_cast<const T*>(x),
                               static_cast<T*>(sums), static_cast<T*>(sqsums), partials,
                               short_tensor(tx_in, sg), sg, fused_out != nullptr);
        if (fused_out)
        {
            fused_out->groups = groups;
            fused_out->sequential = true;
            return issued();
        }
        const unsigned int blocks = (num_channels + kBlockSize - 1) / kBlockSize;
        if (groups > 1 && !logged(small_record(kKernelFinish, blocks, num_channels, 2)))
            launch(bn_finish_short_kernel<T, 2>, blocks, kBlockSize, stream, partials, groups, num_channels,
                   static_cast<T*>(sums), static_cast<T*>(sqsums), nullptr, nullptr);
        return issued();
    }
    HostTensor tx = tx_in;
    ReductionPlan plan;
    const int err = plan_reduction<T>(num_samples, num_channels, spatial, {&tx}, kUnroll, &plan);
    if (err)
        return err;
    const bool strided = plan.strided;
    const int vw = plan.vw, gmax = plan.groups_max;
    const size_t units = plan.units, groups = plan.groups;
    const Chunking& ch = plan.ch;
    num_samples = plan.num_samples;
    spatial = plan.spatial;
    double* partials = static_cast<double*>(workspace);
    const dim3 grid(static_cast<unsigned int>(groups), num_channels);
    LaunchRecord rec = long_record(kKernelSums, strided, vw, grid, num_samples, num_channels,
                                   spatial, ch, {&tx}, false);
    rec.folded = plan.folded;
    rec.num_units = static_cast<unsigned int>(units);
    rec.num_sums = 2;
    rec.groups_max = gmax;
    rec.partials = groups > 1 || fused_out != nullptr;
    if (!logged(rec))
        H2X_DISPATCH(bn_sums_kernel, grid, static_cast<const T*>(x), static_cast<T*>(sums),
                     static_cast<T*>(sqsums), partials, tx.map, spatial, ch.chunk,
                     ch.chunks_per_seg, static_cast<unsigned int>(units), gmax,
                     fused_out != nullptr);
    if (fused_out != nullptr)
    {
        fused_out->groups = static_cast<int>(groups);
        return issued();
    }
    if (groups > 1 && !logged(small_record(kKernelFinish, num_channels, num_channels, 2)))
        launch(bn_finish_kernel<T, 2>, num_channels, kBlockSize, stream, partials, static_cast<int>(groups), gmax,
               static_cast<T*>(sums), static_cast<T*>(sqsums), nullptr, nullptr);
    return issued();
}

template <typename T>
int statistics_impl(int num_channels, size_t num_per_sum, double decay, void* mean, void* var,
                    void* running_mean, void* running_var, hipStream_t stream)
{
    if (num_channels == 0)
        return H2X_SUCCESS;
    const int blocks = std::min((num_channels + kBlockSize - 1) / kBlockSize, 1024);
    if (!logged(small_record(kKernelStatistics, blocks, num_channels)))
        launch(bn_statistics_kernel<T>, blocks, kBlockSize, stream, num_channels, num_per_sum,
               static_cast<T>(decay), static_cast<T*>(mean), static_cast<T*>(var), static_cast<T*>(running_mean),
               static_cast<T*>(running_var));
    return issued();
}

// Chunking of an elementwise pass over N*C segments: at least one full vector
// per thread, about kElementwiseBlocks workgroups.
Chunking elementwise_chunking(size_t spatial, size_t segments, int vw, int unroll,
                              int budget = kElementwiseBlocks)
{
    const size_t tile = static_cast<size_t>(kBlockSize) * vw * unroll;
    const size_t one_pass = static_cast<size_t>(kBlockSize) * vw;
    Chunking c = make_chunking(spatial, segments, budget, one_pass,
                               one_pass * 2 > tile ? one_pass : one_pass * 2);
    // A chunk of more than a tile is cut down to whole tiles: the passes beyond the
    // last whole tile run with one load in flight per lane instead of `unroll`
    // (5 passes as 4 + 1 took a quarter longer than 4 on the haloed C3 shard).
    if (c.chunk > tile && c.chunk % tile != 0)
    {
        c.chunk = c.chunk / tile * tile;
        c.chunks_per_seg = static_cast<int>((spatial + c.chunk - 1) / c.chunk);
    }
    return c;
}

// Haloed outputs that lie within this many bytes are stored normally by a pass that reads its statistics, inference or
// the staged one: the ends of their rows are partial lines, which the caches merge with the neighbours'; larger ones
// push the inputs out of the memory-side cache. Inference, past the caches and normally, us going round three sets of
// tensors: N 106, C 257, 13 x 12, halo of 2, 28 MiB 14.1 and 10.4; N 27, C 57, 14 x 11 x 10, halo of 2, 22 MiB 9.1 and
// 7.1; doubles N 125, C 346, 7 x 8, 30 MiB 14.9 and 11.3; below 5 MiB level; larger N 5, C 7, 63 x 67 x 61, 38 MiB 14.0
// and 13.2, N 152, C 5, 29 x 21 x 21, 47 MiB 19.4 and 20.4, N 25, C 245, 41 x 60, 62 MiB 23.8 and 33.1. The line lies
// below where inference alone would have it for the training that runs in stages, and reads x again: forward + backward
// there 5 % less with 29 to 32 MiB.
// (With normal stores of dx, and of passes that finish their sums, training in stages loses up to 10 %: N 8, C 60, 129
// x 142, 35 MiB 60.7 and 66.1.)
constexpr size_t kNormalStores = size_t(32) << 20;

// Of tensors with one plane a channel and segments beyond the short ones, whose partial lines are few or many to a
// workgroup, these lose (inference, us, past the caches and normally, of 190 calls): from 5 to 10 MiB, where three sets
// of inputs stay in the L2 if nothing else goes there, N 15, C 16, 65 x 99, halo of 2 4.78 and 5.13, doubles N 3, C 11,
// 183 x 151, halo of 2 4.53 and 5.00 (below 5 MiB 0.98 of the time on average); and segments of up to 700 floats or 470
// doubles, N 68, C 61, 17 x 27, halo of 2, 10 MiB 6.86 and 7.58, N 36, C 310, 19 x 23, 22 MiB 12.5 and 13.4, doubles N
// 13, C 195, 20 x 23, halo of 2 6.23 and 6.68. The others from 10 MiB N 29, C 15, 94 x 75 7.15 and 6.77, N 62, C 35, 38
// x 37, halo of 3 8.50 and 7.50, doubles N 58, C 88, 23 x 30 13.4 and 12.2; several planes of any size 0.78 to 1.04 of
// the time, 0.92 on average.
constexpr size_t kPlaneInL2 = size_t(5) << 20, kPlaneBeyondL2 = size_t(10) << 20, kPlaneFloats = 700, kPlaneDoubles = 470;

bool stored_normally(const HostTensor& output, int num_samples, int num_channels, size_t spatial, size_t elem_bytes, bool is_short)
{
    if (!output.strided)
        return false;
    const size_t bytes = (static_cast<size_t>(num_channels - 1) * output.map.stride_c
                          + static_cast<size_t>(num_samples - 1) * output.map.stride_n + short_span(output, spatial)) * elem_bytes;
    if (bytes > kNormalStores)
        return false;
    const bool one_plane = spatial == static_cast<size_t>(output.map.w.divisor) * output.map.h.divisor;
    return is_short || !one_plane || bytes < kPlaneInL2
           || (bytes >= kPlaneBeyondL2 && spatial > (elem_bytes == sizeof(float) ? kPlaneFloats : kPlaneDoubles));
}

template <typename T>
int apply_impl(int num_samples, int num_channels, size_t spatial, const HostTensor& tx_in,
               const HostTensor& ty_in, const void* x, const void* mean, const void* var,
               const void* scale, const void* bias, void* y, double epsilon, hipStream_t stream,
               const FusedStats<T>* fused = nullptr)
{
    if (static_cast<size_t>(num_samples) * num_channels == 0 || spatial == 0)
        return H2X_SUCCESS;
    ShortGeometry sg;
    const bool is_short = short_segments<T>(num_samples, num_channels, spatial, {&tx_in, &ty_in}, &sg);
    const bool normally = stored_normally(ty_in, num_samples, num_channels, spatial, sizeof(T), is_short);
    if (fused && fused->sequential != is_short)
        return H2X_ERR_UNSUPPORTED; // the partials are laid out for the other family of kernels
    if (is_short)
    {
        const dim3 grid(short_windows(sg),
                        short_elementwise_groups(&sg, kUnroll, kShortElementwiseBlocks,
                                                 fused ? fused->groups * 2 * sizeof(double) : 0,
                                                 spatial * sizeof(T) * 2));
        LaunchRecord rec =
            short_record(kKernelApply, sg, grid, full_vec<T>(), {&tx_in, &ty_in}, true);
        rec.fused = fused != nullptr;
        if (logged(rec))
            return H2X_SUCCESS;
        if (fused)
            H2X_DISPATCH_SHORT_FUSED(bn_apply_short_kernel, kFusedApply, grid, static_cast<const T*>(x),
                                     nullptr, nullptr, static_cast<const T*>(scale),
                                     static_cast<const T*>(bias), static_cast<T*>(y),
                                     static_cast<T>(epsilon), short_tensor(tx_in, sg),
                                     short_tensor(ty_in, sg), sg, *fused);
        else if (normally)
            H2X_DISPATCH_SHORT_FUSED(bn_apply_short_kernel, kNormalApply, grid, static_cast<const T*>(x),
                                     static_cast<const T*>(mean), static_cast<const T*>(var),
                                     static_cast<const T*>(scale), static_cast<const T*>(bias),
                                     static_cast<T*>(y), static_cast<T>(epsilon),
                                     short_tensor(tx_in, sg), short_tensor(ty_in, sg), sg, FusedStats<T>());
        else
            H2X_DISPATCH_SHORT_FUSED(bn_apply_short_kernel, kPlainApply, grid, static_cast<const T*>(x),
                                     static_cast<const T*>(mean), static_cast<const T*>(var),
                                     static_cast<const T*>(scale), static_cast<const T*>(bias),
                                     static_cast<T*>(y), static_cast<T>(epsilon),
                                     short_tensor(tx_in, sg), short_tensor(ty_in, sg), sg, FusedStats<T>());
        return issued();
    }
    HostTensor tx = tx_in, ty = ty_in;
    const bool folded = fold_samples(&num_samples, &spatial, {&tx, &ty});
    if (spatial >= (1ull << 31) && (tx.strided || ty.strided))
        return H2X_ERR_TOO_LARGE;
    const size_t segments = static_cast<size_t>(num_samples) * num_channels;
    bool strided;
    const int vw = common_vector<T>({&tx, &ty}, &strided);
    if (strided && vw > 1)
        spatial = pad_rows<T>({&tx, &ty}, spatial);
    if (spatial >= (1ull << 31) && strided)
        return H2X_ERR_TOO_LARGE;
    const bool beyond_cache = segments * spatial * sizeof(T) > kBeyondCacheBytes;
    const Chunking ch = elementwise_chunking(spatial, segments, vw, kUnroll,
                                             strided || beyond_cache ? kUnboundedBlocks : kElementwiseBlocks);
    const size_t workgroups = segments * ch.chunks_per_seg;
    if (!grid_ok(workgroups))
        return H2X_ERR_TOO_LARGE;
    const unsigned int grid = static_cast<unsigned int>(workgroups);
    LaunchRecord rec = long_record(kKernelApply, strided, vw, dim3(grid), num_samples, num_channels,
                                   spatial, ch, {&tx, &ty}, true);
    rec.folded = folded;
    rec.fused = fused != nullptr;
    if (logged(rec))
        return H2X_SUCCESS;
    if (fused)
        H2X_DISPATCH_ELEMENTWISE(bn_apply_kernel, kFusedApply, grid, static_cast<const T*>(x), nullptr,
                                 nullptr, static_cast<const T*>(scale), static_cast<const T*>(bias),
                                 static_cast<T*>(y), static_cast<T>(epsilon), num_channels, spatial,
                                 tx.map, ty.map, ch.chunk, ch.chunks_per_seg, *fused);
    else if (normally && vw > 1) // (such a launch goes row by row)
        launch(bn_apply_kernel<T, full_vec<T>(), kLayoutRows, kNormalApply>, grid, kBlockSize, stream,
               static_cast<const T*>(x),
               static_cast<const T*>(mean), static_cast<const T*>(var),
               static_cast<const T*>(scale), static_cast<const T*>(bias),
               static_cast<T*>(y), static_cast<T>(epsilon), num_channels, spatial,
               tx.map, ty.map, ch.chunk, ch.chunks_per_seg, FusedStats<T>());
    else
        H2X_DISPATCH_ELEMENTWISE(bn_apply_kernel, kPlainApply, grid, static_cast<const T*>(x),
                                 static_cast<const T*>(mean), static_cast<const T*>(var),
                                 static_cast<const T*>(scale), static_cast<const T*>(bias),
                                 static_cast<T*>(y), static_cast<T>(epsilon), num_channels, spatial,
                                 tx.map, ty.map, ch.chunk, ch.chunks_per_seg, FusedStats<T>());
    return issued();
}

template <typename T>
int backprop1_impl(int num_samples, int num_channels, size_t spatial, const HostTensor& tx_in,
                   const HostTensor& td_in, const void* x, const void* dy, const void* mean,
                   const void* var, const void* scale, void* dscale, void* dbias, void* dmean,
                   void* dvar, double epsilon, void* workspace, hipStream_t stream,
                   FusedStats<T>* fused_out = nullptr)
{
    if (num_channels == 0)
        return H2X_SUCCESS;
    if (num_samples == 0 || spatial == 0)
        return zero_outputs<T>({dscale, dbias, dmean, dvar}, num_channels, stream);
    if (fused_out)
        fused_out->sequential = false;
    ShortGeometry sg;
    if (short_segments<T>(num_samples, num_channels, spatial, {&tx_in, &td_in}, &sg))
    {
        const int gmax = max_groups_per_channel(num_channels);
        const int groups = short_reduction_groups(&sg, gmax, kUnroll / 2, sizeof(T));
        double* partials = static_cast<double*>(workspace);
        const dim3 grid(short_windows(sg), groups);
        LaunchRecord rec =
            short_record(kKernelBackprop1, sg, grid, full_vec<T>(), {&tx_in, &td_in}, false);
        rec.num_sums = 4;
        rec.groups_max = gmax;
        rec.partials = groups > 1 || fused_out != nullptr;
        if (!logged(rec))
            H2X_DISPATCH_SHORT(bn_backprop1_short_kernel, grid, static_cast<const T*>(x),
                               static_cast<const T*>(dy), static_cast<const T*>(mean),
                               static_cast<const T*>(var), static_cast<const T*>(scale),
                               static_cast<T*>(dscale), static_cast<T*>(dbias),
                               static_cast<T*>(dmean), static_cast<T*>(dvar),
                               static_cast<T>(epsilon), partials, short_tensor(tx_in, sg),
                               short_tensor(td_in, sg), sg, fused_out != nullptr);
        if (fused_out)
        {
            fused_out->groups = groups;
            fused_out->sequential = true;
            return issued();
        }
        const unsigned int blocks = (num_channels + kBlockSize - 1) / kBlockSize;
        if (groups > 1 && !logged(small_record(kKernelFinish, blocks, num_channels, 4)))
            launch(bn_finish_short_kernel<T, 4>, blocks, kBlockSize, stream, partials, groups, num_channels,
                   static_cast<T*>(dscale), static_cast<T*>(dbias), static_cast<T*>(dmean), static_cast<T*>(dvar));
        return issued();
    }
    HostTensor tx = tx_in, td = td_in;
    ReductionPlan plan;
    const int err = plan_reduction<T>(num_samples, num_channels, spatial, {&tx, &td}, kUnroll / 2, &plan);
    if (err)
        return err;
    const bool strided = plan.strided;
    const int vw = plan.vw, gmax = plan.groups_max;
    const size_t units = plan.units, groups = plan.groups;
    const Chunking& ch = plan.ch;
    num_samples = plan.num_samples;
    spatial = plan.spatial;
    double* partials = static_cast<double*>(workspace);
    const dim3 grid(static_cast<unsigned int>(groups), num_channels);
    LaunchRecord rec = long_record(kKernelBackprop1, strided, vw, grid, num_samples, num_channels,
                                   spatial, ch, {&tx, &td}, false);
    rec.folded = plan.folded;
    rec.num_units = static_cast<unsigned int>(units);
    rec.num_sums = 4;
    rec.groups_max = gmax;
    rec.partials = groups > 1 || fused_out != nullptr;
    if (!logged(rec))
        H2X_DISPATCH(bn_backprop1_kernel, grid, static_cast<const T*>(x),
                     static_cast<const T*>(dy), static_cast<const T*>(mean),
                     static_cast<const T*>(var), static_cast<const T*>(scale),
                     static_cast<T*>(dscale), static_cast<T*>(dbias), static_cast<T*>(dmean),
                     static_cast<T*>(dvar), static_cast<T>(epsilon), partials, spatial, tx.map,
                     td.map, ch.chunk, ch.chunks_per_seg, static_cast<unsigned int>(units), gmax,
                     fused_out != nullptr);
    if (fused_out != nullptr)
    {
        fused_out->groups = static_cast<int>(groups);
        return issued();
    }
    if (groups > 1 && !logged(small_record(kKernelFinish, num_channels, num_channels, 4)))
        launch(bn_finish_kernel<T, 4>, num_channels, kBlockSize, stream, partials, static_cast<int>(groups), gmax,
               static_cast<T*>(dscale), static_cast<T*>(dbias), static_cast<T*>(dmean), static_cast<T*>(dvar));
    return issued();
}

template <typename T>
int backprop2_impl(int num_samples, int num_channels, size_t spatial, size_t num_per_sum,
                   const HostTensor& tx_in, const HostTensor& td_in, const HostTensor& to_in,
                   const void* x, const void* dy, const void* mean, const void* var,
                   const void* scale, const void* dmean, const void* dvar, void* dx,
                   double epsilon, hipStream_t stream, const FusedStats<T>* fused = nullptr)
{
    if (static_cast<size_t>(num_samples) * num_channels == 0 || spatial == 0)
        return H2X_SUCCESS;
    ShortGeometry sg;
    const bool is_short =
        short_segments<T>(num_samples, num_channels, spatial, {&tx_in, &td_in, &to_in}, &sg);
    if (fused && fused->sequential != is_short)
        return H2X_ERR_UNSUPPORTED; // the partials are laid out for the other family of kernels
    // whether x and dx share memory (the reference allows dx to be x itself)
    const auto span = [&](const HostTensor& t) {
        return (static_cast<size_t>(num_samples - 1) * t.map.stride_n
                + static_cast<size_t>(num_channels - 1) * t.map.stride_c + short_span(t, spatial))
               * sizeof(T);
    };
    const char* xb = static_cast<const char*>(x);
    const char* ob = static_cast<const char*>(dx);
    const bool disjoint = xb + span(tx_in) <= ob || ob + span(to_in) <= xb;
    if (is_short)
    {
        const dim3 grid(short_windows(sg),
                        short_elementwise_groups(&sg, kUnroll / 2, kShortGradientBlocks,
                                                 fused ? fused->groups * 4 * sizeof(double) : 0,
                                                 spatial * sizeof(T) * 3));
        LaunchRecord rec = short_record(kKernelBackprop2, sg, grid, full_vec<T>(),
                                        {&tx_in, &td_in, &to_in}, true);
        rec.fused = fused != nullptr;
        rec.rewrite = disjoint;
        if (logged(rec))
            return H2X_SUCCESS;
        if (fused)
            H2X_DISPATCH_SHORT_FUSED(bn_backprop2_short_kernel, true, grid,
                                     static_cast<const T*>(x), static_cast<const T*>(dy),
                                     static_cast<const T*>(mean), static_cast<const T*>(var),
                                     static_cast<const T*>(scale), nullptr, nullptr,
                                     static_cast<T*>(dx), static_cast<T>(epsilon), num_per_sum,
                                     short_tensor(tx_in, sg), short_tensor(td_in, sg), short_tensor(to_in, sg),
                                     sg, disjoint, *fused);
        else
            H2X_DISPATCH_SHORT_FUSED(bn_backprop2_short_kernel, false, grid,
                                     static_cast<const T*>(x), static_cast<const T*>(dy),
                                     static_cast<const T*>(mean), static_cast<const T*>(var),
                                     static_cast<const T*>(scale), static_cast<const T*>(dmean),
                                     static_cast<const T*>(dvar), static_cast<T*>(dx),
                                     static_cast<T>(epsilon), num_per_sum, short_tensor(tx_in, sg),
                                     short_tensor(td_in, sg), short_tensor(to_in, sg), sg, disjoint,
                                     FusedStats<T>());
        return issued();
    }
    HostTensor tx = tx_in, td = td_in, to = to_in;
    const bool folded = fold_samples(&num_samples, &spatial, {&tx, &td, &to});
    if (spatial >= (1ull << 31) && (tx.strided || td.strided || to.strided))
        return H2X_ERR_TOO_LARGE;
    const size_t segments = static_cast<size_t>(num_samples) * num_channels;
    bool strided;
    const int vw = common_vector<T>({&tx, &td, &to}, &strided);
    if (strided && vw > 1)
        spatial = pad_rows<T>({&tx, &td, &to}, spatial);
    if (spatial >= (1ull << 31) && strided)
        return H2X_ERR_TOO_LARGE;
    const bool beyond_cache = segments * spatial * sizeof(T) > kBeyondCacheBytes;
    const Chunking ch = elementwise_chunking(spatial, segments, vw, kUnroll / 2,
                                             strided || beyond_cache ? kUnboundedBlocks : kElementwiseBlocks);
    const size_t workgroups = segments * ch.chunks_per_seg;
    if (!grid_ok(workgroups))
        return H2X_ERR_TOO_LARGE;
    const unsigned int grid = static_cast<unsigned int>(workgroups);
    LaunchRecord rec = long_record(kKernelBackprop2, strided, vw, dim3(grid), num_samples,
                                   num_channels, spatial, ch, {&tx, &td, &to}, true);
    rec.folded = folded;
    rec.fused = fused != nullptr;
    rec.rewrite = disjoint;
    if (logged(rec))
        return H2X_SUCCESS;
    if (fused)
        H2X_DISPATCH_ELEMENTWISE(bn_backprop2_kernel, true, grid, static_cast<const T*>(x),
                                 static_cast<const T*>(dy), static_cast<const T*>(mean),
                                 static_cast<const T*>(var), static_cast<const T*>(scale), nullptr,
                                 nullptr, static_cast<T*>(dx), static_cast<T>(epsilon), num_per_sum,
                                 num_channels, spatial, tx.map, td.map, to.map, ch.chunk,
                                 ch.chunks_per_seg, disjoint, *fused);
    else
        H2X_DISPATCH_ELEMENTWISE(bn_backprop2_kernel, false, grid, static_cast<const T*>(x),
                                 static_cast<const T*>(dy), static_cast<const T*>(mean),
                                 static_cast<const T*>(var), static_cast<const T*>(scale),
                                 static_cast<const T*>(dmean), static_cast<const T*>(dvar),
                                 static_cast<T*>(dx), static_cast<T>(epsilon), num_per_sum,
                                 num_channels, spatial, tx.map, td.map, to.map, ch.chunk,
                                 ch.chunks_per_seg, disjoint, FusedStats<T>());
    return issued();
}

// The allocation of a (sample, channel) segment: its interior, and its elements.
int real_box(const h2x_haloed_geometry* g, RealBox* out, size_t* elements)
{
    if (!g || g->num_dims < 3 || g->num_dims > 5)
        return H2X_ERR_INVALID_ARGUMENT;
    const int nd = g->num_dims, ns = nd - 2;
    RealBox box;
    size_t real = 1, extent[3] = {1, 1, 1};
    for (int d = 0; d < 3; ++d)
    {
        box.lo[d] = 0;
        box.hi[d] = 1;
    }
    for (int d = 0; d < nd; ++d)
    {
        if (g->local_shape[d] < 0 || g->lower_halo[d] < 0
            || g->lower_halo[d] + g->local_shape[d] > g->real_shape[d])
            return H2X_ERR_INVALID_ARGUMENT;
        if (d >= ns && (g->lower_halo[d] != 0 || g->real_shape[d] != g->local_shape[d]))
            return H2X_ERR_UNSUPPORTED; // no halo on the channel and sample dimensions
    }
    for (int d = 0; d < ns; ++d)
    {
        extent[d] = static_cast<size_t>(g->real_shape[d]);
        real *= extent[d];
        if (real >= (1ull << 31))
            return H2X_ERR_TOO_LARGE;
        box.lo[d] = static_cast<uint32_t>(g->lower_halo[d]);
        box.hi[d] = static_cast<uint32_t>(g->lower_halo[d] + g->local_shape[d]);
    }
    box.wr = make_fastdiv(static_cast<uint32_t>(extent[0]));
    box.hr = make_fastdiv(static_cast<uint32_t>(extent[1]));
    *out = box;
    *elements = real;
    return H2X_SUCCESS;
}

// Normalise / input gradient over tensors of one haloed geometry, the halo of
// the output cleared (bn_clearing_kernel).
template <typename T>
int clearing_impl(bool backward, size_t num_per_sum, const h2x_haloed_geometry* g, const void* x,
                  const void* dy, const void* mean, const void* var, const void* scale,
                  const void* bias, const void* dmean, const void* dvar, void* out, double epsilon,
                  hipStream_t stream)
{
    RealBox box;
    size_t real;
    const int err = real_box(g, &box, &real);
    if (err)
        return err;
    const int nd = g->num_dims;
    const int num_channels = static_cast<int>(g->local_shape[nd - 2]);
    const size_t segments = static_cast<size_t>(g->local_shape[nd - 1]) * num_channels;
    if (segments == 0 || real == 0)
        return H2X_SUCCESS;
    if (!x || !out || (backward && !dy))
        return H2X_ERR_INVALID_ARGUMENT;
    const bool vectors = real % full_vec<T>() == 0 && aligned16(x) && aligned16(out)
                         && (!backward || aligned16(dy));
    const int vw = vectors ? full_vec<T>() : 1;
    const Chunking ch = elementwise_chunking(real, segments, vw, backward ? kUnroll / 2 : kUnroll);
    const size_t workgroups = segments * ch.chunks_per_seg;
    if (!grid_ok(workgroups))
        return H2X_ERR_TOO_LARGE;
    const unsigned int grid = static_cast<unsigned int>(workgroups);
    {
        LaunchRecord rec;
        rec.kernel = kKernelClearing;
        rec.family = kFamilyDense;
        rec.vec = vw;
        rec.grid_x = grid;
        rec.num_samples = static_cast<int>(g->local_shape[nd - 1]);
        rec.num_channels = num_channels;
        rec.spatial = real;
        rec.real = real;
        rec.chunk = ch.chunk;
        rec.chunks_per_seg = ch.chunks_per_seg;
        rec.num_tensors = backward ? 3 : 2;
        rec.last_is_output = true;
        rec.box = box;
        if (logged(rec))
            return H2X_SUCCESS;
    }
#define H2X_LAUNCH_CLEARING(VEC, BACKWARD)                                                         \
    launch(bn_clearing_kernel<T, VEC, BACKWARD>, grid, kBlockSize, stream,                         \
        static_cast<const T*>(x), static_cast<const T*>(dy), static_cast<const T*>(mean),          \
        static_cast<const T*>(var), static_cast<const T*>(scale), static_cast<const T*>(bias),     \
        static_cast<const T*>(dmean), static_cast<const T*>(dvar), static_cast<T*>(out),           \
        static_cast<T>(epsilon), num_per_sum, num_channels, real, box, ch.chunk, ch.chunks_per_seg)
    if (backward)
    {
        if (vectors)
            H2X_LAUNCH_CLEARING(full_vec<T>(), true);
        else
            H2X_LAUNCH_CLEARING(1, true);
    }
    else
    {
        if (vectors)
            H2X_LAUNCH_CLEARING(full_vec<T>(), false);
        else
            H2X_LAUNCH_CLEARING(1, false);
    }
#undef H2X_LAUNCH_CLEARING
    return launch_status();
}

bool bad_geometry(int num_samples, int num_channels, size_t spatial, size_t real)
{
    return num_samples < 0 || num_channels < 0 || real < spatial;
}

// ---- typed bodies of the C entry points ----------------------------------------

template <typename T>
int sums_dense(int n, int c, size_t s, size_t sr, const void* x, void* sums, void* sqsums, void* ws,
               hipStream_t st)
{
    return sums_impl<T>(n, c, s, dense_tensor<T>(x, c, s, sr), x, sums, sqsums, ws, st);
}

template <typename T>
int sums_strided(int n, const h2x_tensor_geometry* g, const void* x, void* sums, void* sqsums,
                 void* ws, hipStream_t st)
{
    HostTensor tx;
    int c;
    size_t s;
    const int err = strided_tensor<T>(g, x, n, &tx, &c, &s);
    return err ? err : sums_impl<T>(n, c, s, tx, x, sums, sqsums, ws, st);
}

// Two geometries describe the same elements only if every local extent agrees:
// equal products are not enough (8 x 4 against 4 x 8 would pair other elements).
bool same_local_shape(const h2x_tensor_geometry* a, const h2x_tensor_geometry* b)
{
    if (a->num_dims != b->num_dims)
        return false;
    for (int i = 0; i < a->num_dims; ++i)
        if (a->local_shape[i] != b->local_shape[i])
            return false;
    return true;
}

template <typename T>
int apply_strided(int n, const h2x_tensor_geometry* gx, const h2x_tensor_geometry* gy, const void* x,
                  const void* mean, const void* var, const void* scale, const void* bias, void* y,
                  double eps, hipStream_t st)
{
    HostTensor tx, ty;
    int c, c2;
    size_t s, s2;
    int err = strided_tensor<T>(gx, x, n, &tx, &c, &s);
    if (!err)
        err = strided_tensor<T>(gy, y, n, &ty, &c2, &s2);
    if (!err && (c != c2 || s != s2 || !same_local_shape(gx, gy)))
        err = H2X_ERR_INVALID_ARGUMENT;
    return err ? err : apply_impl<T>(n, c, s, tx, ty, x, mean, var, scale, bias, y, eps, st);
}

template <typename T>
int backprop1_strided(int n, const h2x_tensor_geometry* gx, const h2x_tensor_geometry* gd,
                      const void* x, const void* dy, const void* mean, const void* var,
                      const void* scale, void* dscale, void* dbias, void* dmean, void* dvar,
                      double eps, void* ws, hipStream_t st)
{
    HostTensor tx, td;
    int c, c2;
    size_t s, s2;
    int err = strided_tensor<T>(gx, x, n, &tx, &c, &s);
    if (!err)
        err = strided_tensor<T>(gd, dy, n, &td, &c2, &s2);
    if (!err && (c != c2 || s != s2 || !same_local_shape(gx, gd)))
        err = H2X_ERR_INVALID_ARGUMENT;
    return err ? err
               : backprop1_impl<T>(n, c, s, tx, td, x, dy, mean, var, scale, dscale, dbias, dmean,
                                   dvar, eps, ws, st);
}

template <typename T>
int backprop2_strided(int n, size_t num_per_sum, const h2x_tensor_geometry* gx,
                      const h2x_tensor_geometry* gd, const h2x_tensor_geometry* go, const void* x,
                      const void* dy, const void* mean, const void* var, const void* scale,
                      const void* dmean, const void* dvar, void* dx, double eps, hipStream_t st)
{
    HostTensor tx, td, to;
    int c, c2, c3;
    size_t s, s2, s3;
    int err = strided_tensor<T>(gx, x, n, &tx, &c, &s);
    if (!err)
        err = strided_tensor<T>(gd, dy, n, &td, &c2, &s2);
    if (!err)
        err = strided_tensor<T>(go, dx, n, &to, &c3, &s3);
    if (!err
        && (c != c2 || s != s2 || c != c3 || s != s3 || !same_local_shape(gx, gd)
            || !same_local_shape(gx, go)))
        err = H2X_ERR_INVALID_ARGUMENT;
    return err ? err
               : backprop2_impl<T>(n, c, s, num_per_sum, tx, td, to, x, dy, mean, var, scale, dmean,
                                   dvar, dx, eps, st);
}

// Forward pass of a rank that shares its statistics with no one: sums, then a
// normalising kernel that finishes them itself (2 launches instead of 4).
template <typename T>
int forward_local(int n, int c, size_t s, const HostTensor& tx, const HostTensor& ty, const void* x,
                  const void* scale, const void* bias, size_t num_per_sum, double decay, double eps,
                  void* mean, void* var, void* running_mean, void* running_var, void* y, void* ws,
                  hipStream_t st)
{
    if (c == 0)
        return H2X_SUCCESS;
    if (n == 0 || s == 0 || num_per_sum == 0)
    {
        // nothing to normalise or nothing counted: the staged calls define the result
        int err = sums_impl<T>(n, c, s, tx, x, mean, var, ws, st);
        if (!err)
            err = statistics_impl<T>(c, num_per_sum, decay, mean, var, running_mean, running_var, st);
        return err ? err : apply_impl<T>(n, c, s, tx, ty, x, mean, var, scale, bias, y, eps, st);
    }
    FusedStats<T> f;
    f.sequential = false;
    f.partials = static_cast<const double*>(ws);
    f.groups_per_channel_max = max_groups_per_channel(c);
    f.num_per_sum = num_per_sum;
    f.decay = static_cast<T>(decay);
    f.out[0] = static_cast<T*>(mean);
    f.out[1] = static_cast<T*>(var);
    f.out[2] = static_cast<T*>(running_mean);
    f.out[3] = static_cast<T*>(running_var);
    {
        // both launches are planned before the first is issued: a call that is rejected writes nothing
        LaunchLog plan;
        plan.keep = false;
        ScopedLaunchLog scope(&plan);
        FusedStats<T> g = f;
        int err = sums_impl<T>(n, c, s, tx, x, nullptr, nullptr, ws, st, &g);
        if (!err)
            err = apply_impl<T>(n, c, s, tx, ty, x, nullptr, nullptr, scale, bias, y, eps, st, &g);
        if (err == H2X_ERR_UNSUPPORTED)
        {
            // the two tensors take different families of kernels (one of them with halos inside
            // short segments, say): the staged calls
            scope.restore();
            err = sums_impl<T>(n, c, s, tx, x, mean, var, ws, st);
            if (!err)
                err = statistics_impl<T>(c, num_per_sum, decay, mean, var, running_mean, running_var, st);
            return err ? err : apply_impl<T>(n, c, s, tx, ty, x, mean, var, scale, bias, y, eps, st);
        }
        if (err)
            return err;
    }
    const int err = sums_impl<T>(n, c, s, tx, x, nullptr, nullptr, ws, st, &f);
    return err ? err : apply_impl<T>(n, c, s, tx, ty, x, nullptr, nullptr, scale, bias, y, eps, st, &f);
}

// Backward pass likewise: the four sums, then an input-gradient kernel that
// finishes them itself (2 launches instead of 3).
template <typename T>
int backward_local(int n, int c, size_t s, const HostTensor& tx, const HostTensor& td,
                   const HostTensor& to, size_t num_per_sum, const void* x, const void* dy,
                   const void* mean, const void* var, const void* scale, void* dscale, void* dbias,
                   void* dmean, void* dvar, void* dx, double eps, void* ws, hipStream_t st)
{
    if (c == 0)
        return H2X_SUCCESS;
    if (n == 0 || s == 0)
        return backprop1_impl<T>(n, c, s, tx, td, x, dy, mean, var, scale, dscale, dbias, dmean,
                                 dvar, eps, ws, st); // zeroes the four outputs; no dx to write
    FusedStats<T> f;
    f.sequential = false;
    f.partials = static_cast<const double*>(ws);
    f.groups_per_channel_max = max_groups_per_channel(c);
    f.num_per_sum = num_per_sum;
    f.decay = T(0);
    f.out[0] = static_cast<T*>(dscale);
    f.out[1] = static_cast<T*>(dbias);
    f.out[2] = static_cast<T*>(dmean);
    f.out[3] = static_cast<T*>(dvar);
    {
        // both launches are planned before the first is issued: a call that is rejected writes nothing
        LaunchLog plan;
        plan.keep = false;
        ScopedLaunchLog scope(&plan);
        FusedStats<T> g = f;
        int err = backprop1_impl<T>(n, c, s, tx, td, x, dy, mean, var, scale, nullptr, nullptr,
                                    nullptr, nullptr, eps, ws, st, &g);
        if (!err)
            err = backprop2_impl<T>(n, c, s, num_per_sum, tx, td, to, x, dy, mean, var, scale,
                                    nullptr, nullptr, dx, eps, st, &g);
        if (err == H2X_ERR_UNSUPPORTED)
        {
            // the tensors take different families of kernels: the staged calls
            scope.restore();
            err = backprop1_impl<T>(n, c, s, tx, td, x, dy, mean, var, scale, dscale, dbias, dmean,
                                    dvar, eps, ws, st);
            return err ? err
                       : backprop2_impl<T>(n, c, s, num_per_sum, tx, td, to, x, dy, mean, var, scale,
                                           dmean, dvar, dx, eps, st);
        }
        if (err)
            return err;
    }
    const int err = backprop1_impl<T>(n, c, s, tx, td, x, dy, mean, var, scale, nullptr, nullptr,
                                      nullptr, nullptr, eps, ws, st, &f);
    return err ? err
               : backprop2_impl<T>(n, c, s, num_per_sum, tx, td, to, x, dy, mean, var, scale,
                                   nullptr, nullptr, dx, eps, st, &f);
}

// The tensors of a call given by local shapes and strides, which must be equal in shape.
template <typename T>
int two_tensors(int n, const h2x_tensor_geometry* gx, const h2x_tensor_geometry* gy, const void* x, const void* y,
                HostTensor* tx, HostTensor* ty, int* c, size_t* s)
{
    int c2;
    size_t s2;
    int err = strided_tensor<T>(gx, x, n, tx, c, s);
    if (!err)
        err = strided_tensor<T>(gy, y, n, ty, &c2, &s2);
    if (!err && (*c != c2 || *s != s2 || !same_local_shape(gx, gy)))
        err = H2X_ERR_INVALID_ARGUMENT;
    return err;
}

template <typename T>
int three_tensors(int n, const h2x_tensor_geometry* gx, const h2x_tensor_geometry* gd, const h2x_tensor_geometry* go,
                  const void* x, const void* dy, const void* dx, HostTensor* tx, HostTensor* td, HostTensor* to,
                  int* c, size_t* s)
{
    int err = two_tensors<T>(n, gx, gd, x, dy, tx, td, c, s);
    return err ? err : two_tensors<T>(n, gx, go, x, dx, tx, to, c, s);
}

template <typename T>
int forward_local_strided(int n, const h2x_tensor_geometry* gx, const h2x_tensor_geometry* gy,
                          const void* x, const void* scale, const void* bias, size_t num_per_sum,
                          double decay, double eps, void* mean, void* var, void* running_mean,
                          void* running_var, void* y, void* ws, hipStream_t st)
{
    HostTensor tx, ty;
    int c;
    size_t s;
    const int err = two_tensors<T>(n, gx, gy, x, y, &tx, &ty, &c, &s);
    return err ? err
               : forward_local<T>(n, c, s, tx, ty, x, scale, bias, num_per_sum, decay, eps, mean, var,
                                  running_mean, running_var, y, ws, st);
}

template <typename T>
int backward_local_strided(int n, size_t num_per_sum, const h2x_tensor_geometry* gx,
                           const h2x_tensor_geometry* gd, const h2x_tensor_geometry* go,
                           const void* x, const void* dy, const void* mean, const void* var,
                           const void* scale, void* dscale, void* dbias, void* dmean, void* dvar,
                           void* dx, double eps, void* ws, hipStream_t st)
{
    HostTensor tx, td, to;
    int c;
    size_t s;
    const int err = three_tensors<T>(n, gx, gd, go, x, dy, dx, &tx, &td, &to, &c, &s);
    return err ? err
               : backward_local<T>(n, c, s, tx, td, to, num_per_sum, x, dy, mean, var, scale, dscale,
                                   dbias, dmean, dvar, dx, eps, ws, st);
}

// ---- whole channels in one workgroup: which calls, which team -------------------
// float only: the staged calls of double tensors are promised bit for bit, and here
// the fp64 sums are added in another order (ordered_geometry below keeps it).  All tensors of the call lie
// alike, a row holds a vector, and offsets within a channel fit 30 bits.
bool lie_alike(std::initializer_list<const HostTensor*> ts)
{
    const HostTensor& a = **ts.begin();
    for (const HostTensor* t : ts)
        if (t->strided != a.strided || t->map.stride_n != a.map.stride_n || t->map.stride_c != a.map.stride_c
            || t->map.sy != a.map.sy || t->map.sz != a.map.sz || t->map.w.divisor != a.map.w.divisor
            || t->map.h.divisor != a.map.h.divisor)
            return false;
    return true;
}

bool once_geometry(int num_samples, int num_channels, size_t spatial, std::initializer_list<const HostTensor*> ts,
                   OnceGeometry* g)
{
    constexpr size_t vec = full_vec<float>();
    const HostTensor& a = **ts.begin();
    if (!lie_alike(ts))
        return false;
    const size_t w = a.row, h = a.strided ? a.map.h.divisor : 1, d = a.strided ? spatial / (w * h) : 1;
    if (w < vec || a.map.stride_n >= (1ll << 30))
        return false;
    const size_t spr = (w + vec - 1) / vec;
    const size_t end = (num_samples - 1) * static_cast<size_t>(a.map.stride_n)
                       + (d - 1) * static_cast<size_t>(a.map.sz) + (h - 1) * static_cast<size_t>(a.map.sy) + w;
    const size_t vectors = num_samples * d * h * spr;
    if (end >= (1ull << 30) || vectors >= (1ull << 30))
        return false;
    g->vectors = static_cast<uint32_t>(vectors);
    g->width = static_cast<uint32_t>(w);
    g->spr = make_fastdiv(static_cast<uint32_t>(spr));
    g->h = make_fastdiv(static_cast<uint32_t>(h));
    g->d = make_fastdiv(static_cast<uint32_t>(d));
    g->sy = a.map.sy;
    g->sz = a.map.sz;
    g->stride_n = static_cast<uint32_t>(a.map.stride_n);
    g->stride_c = a.map.stride_c;
    g->num_channels = static_cast<uint32_t>(num_channels);
    return true;
}

template <int TEAM, typename G>
unsigned int once_grid(const G& g)
{
    constexpr unsigned int teams = once_block<TEAM>() / TEAM;
    return ((g.num_channels + teams - 1) / teams + kNumXcd - 1) / kNumXcd * kNumXcd;
}

// Dense rows of at least this many bytes are stored past the caches; shorter ones end in
// partial lines, which the L2 merges with the neighbours' (N 1024, C 1024, 7 x 7, 206 MB: 324 us,
// past the caches 406).
constexpr size_t kStreamRow = 512;
// Haloed rows, whose ends are partial lines as well, are stored normally up to this size of a
// tensor; larger outputs push the inputs out of the memory-side cache.  Forward + backward going
// round three sets of tensors, stored normally and past the caches: N 1, C 256, 28^3, 28 MB, 29 and
// 37 us; N 4, C 64, 30^3, 34 MB, 46.8 and 44.9 (one set over and over 38.8 and 44.7); N 8, C 64, 30^3,
// 67 MB, 91 and 80; N 2, C 512, 28^3, 111 MB, 158 and 147.
constexpr size_t kHaloedNormalStores = size_t(48) << 20;
// Channels from which a variant that fills a CU with one channel pays: below, the two-launch
// kernels spread a channel of this size over the idle CUs (N 4, C 64, 128 x 128 forward 11.7 us,
// in one launch 12.3; C 64, 28^3 x 2 9.6 and 9.1).
constexpr unsigned int kOnceManyChannels = 96;

template <int TEAM, int K, bool STREAM, typename G>
void issue_once(const G& g, const OnceForward<float>& a, hipStream_t st)
{
    launch_whole(kKernelOnce, K, bn_once_forward_kernel<float, TEAM, K, STREAM, G>, once_grid<TEAM>(g), once_block<TEAM>(), st, g, a);
}
template <int TEAM, int K, bool STREAM, typename G>
void issue_once(const G& g, const OnceBackward<float>& a, hipStream_t st)
{
    // 144 of the 160 KB.  With 16 vectors a thread and nine of dy parked there the kernel has registers for the rest only if
    // it works the places of the vectors out again in each step (kept, 16 registers and a 16-byte spill that waits for the first
    // load: backward, N 40, C 128, 38 x 38 22.3 -> 20.9 us, N 1, C 361, 35 x 46 x 38 69 -> 61, N 2, C 512, 30^3 with a halo 100
    // -> 90). Where the halo is cleared a place is long to work out (N 32, C 116, 13 x 9 x 9 25.2 -> 31.6): it is kept,
    // 16 registers are spilled (9 words of scratch a lane), and the kernel remains faster than two launches: N 4, C
    // 256, 112 x 112 47.5 -> 38.7, N 2, C 512, 30^3 97 -> 90, N 16, C 1024, 54 x 54 154 -> 142 (going round three sets
    // of tensors).
    constexpr int kInLds = TEAM * K > 8192 ? 9 : 0;
    launch_whole(kKernelOnce, K, bn_once_backward_kernel<float, TEAM, K, STREAM, kInLds, G>, once_grid<TEAM>(g), once_block<TEAM>(),
                 st, g, a);
}

// A channel fits the registers of one workgroup, in a variant that pays.
template <typename A, typename G>
bool once_holds(const G& g)
{
    constexpr uint32_t kMost = 1024 * (std::is_same<A, OnceForward<float>>::value ? 20 : 16);
    return g.vectors <= (g.num_channels >= kOnceManyChannels ? kMost : 1024 * 8);
}

// The smallest team whose K vectors a thread hold the channel: four where that is enough
// workgroups (more threads wait for memory together), more only beyond 1024 threads.
// False: no variant holds it.
template <bool STREAM, typename G, typename A>
bool once_launch(const G& g, const A& a, hipStream_t st)
{
    constexpr bool kForward = std::is_same<A, OnceForward<float>>::value;
    if (!once_holds<A>(g))
        return false;
    if (g.vectors <= 64 * 2)
        issue_once<64, 2, STREAM>(g, a, st);
    else if (g.vectors <= 256 * 4)
        issue_once<256, 4, STREAM>(g, a, st);
    else if (g.vectors <= 512 * 4)
        issue_once<512, 4, STREAM>(g, a, st);
    else if (g.vectors <= 1024 * 4)
        issue_once<1024, 4, STREAM>(g, a, st);
    else if (g.vectors <= 1024 * 8)
        issue_once<1024, 8, STREAM>(g, a, st);
    else if (g.vectors <= 1024 * 16)
        issue_once<1024, 16, STREAM>(g, a, st);
    else
        issue_once<1024, kForward ? 20 : 16, STREAM>(g, a, st);
    return true;
}

// Bytes from the first to behind the last element of a tensor of the call.
size_t reach_bytes(const OnceGeometry& g, int n)
{
    const size_t last = static_cast<size_t>(g.num_channels - 1) * g.stride_c
                        + static_cast<size_t>(n - 1) * g.stride_n + static_cast<size_t>(g.d.divisor - 1) * g.sz
                        + static_cast<size_t>(g.h.divisor - 1) * g.sy + g.width;
    return last * sizeof(float);
}

bool dense_rows(const OnceGeometry& g)
{
    return g.h.divisor * g.d.divisor == 1;
}

bool streamed(const OnceGeometry& g, int n)
{
    return dense_rows(g) ? g.width * sizeof(float) >= kStreamRow : reach_bytes(g, n) > kHaloedNormalStores;
}

// ---- windows of neighbouring channels: which calls ---------------------------------
// Short dense segments (those that are stored normally) of tensors from 21 MiB, whose sets of x, y, dy and dx the memory-side
// cache does not hold from pass to pass.  Backward a CU holds two workgroups of up to four samples a thread; of seven or
// eight it holds one, of five and six too, with registers idle.  Where the windows are one round of the chip, or fill the last
// round, or segments are of up to 40 elements.  Forward + backward in us, by a workgroup a channel and by windows, going round
// three sets of tensors:
//   one round: N 128, C 1024, 7 x 7 32.1 and 26.5; N 72, C 1983, 6 x 7 28.4 and 24.8 (four channels); N 104, C 830, 8 x
//   9 28.5 and 26.3; N 85, C 593, 11 x 11 28.8 and 26.9; N 256, C 512, 7 x 7, seven samples, 32.4 and 28.0; five
//   samples N 170, C 759, 7 x 8 31.5 and 34.6; rounds filled: N 128, C 2048, 7 x 7 64.1 and 56.3; N 256, C 1024, 7 x 7
//   67.1 and 58.0; not: N 80, C 1039, 8 x 10 28.6 and 30.4, N 143, C 1122, 8 x 7 41.7 and 43.3, seven or eight samples
//   N 135, C 669, 10 x 11 44.3 and 49.8, N 125, C 1204, 11 x 9 66.4 and 71.6;
//   short: N 151, C 1394, 5 x 7 37.6 and 33.9; N 238, C 1325, 5 x 4 33.7 and 29.6; N 141, C 1629, 5 x 6 34.7 and 34.1;
//   eight samples of whole 64-byte pieces, which share no line halves: N 238, C 1514, 8 x 8 91.3 and 101.0;
//   smaller tensors: N 128, C 1024, 6 x 6, 19 MB, 18.7 and 19.5; N 64, C 1024, 7 x 7, 13 MB, 15.6 both; N 41, C 1661, 8
//   x 10, 21.8 MB, 22.1 and 23.8.  Segments of 128 to 160 elements lose up to a third.
constexpr int kWindowBlock = 1024;
constexpr size_t kWindowBytes = size_t(21) << 20;

template <int K>
void issue_window(const WindowGeometry& g, const OnceForward<float>& a, uint32_t blocks, hipStream_t st)
{
    launch_whole(kKernelWindow, K, bn_window_forward_kernel<float, kWindowBlock, K>, blocks, kWindowBlock, st, g, a);
}
template <int K>
void issue_window(const WindowGeometry& g, const OnceBackward<float>& a, uint32_t blocks, hipStream_t st)
{
    launch_whole(kKernelWindow, K, bn_window_backward_kernel<float, kWindowBlock, K>, blocks, kWindowBlock, st, g, a);
}

// False: the call is not for windows.
template <typename A>
bool window_launch(const OnceGeometry& o, const A& a, int n, hipStream_t st)
{
    // (channels that lie side by side: a window is one run of memory in each sample)
    if (!dense_rows(o) || streamed(o, n) || o.stride_c < o.width || o.stride_c > 2 * static_cast<int64_t>(o.width)
        || static_cast<size_t>(o.width) * n * o.num_channels * sizeof(float) < kWindowBytes)
        return false;
    WindowGeometry g;
    g.width = o.width;
    g.num_channels = o.num_channels;
    g.samples = static_cast<uint32_t>(n);
    g.spr = o.spr;
    g.stride_n = o.stride_n;
    g.stride_c = o.stride_c;
    const uint32_t cus = chip_units();
    for (const uint32_t channels : {4u, 2u})
    {
        const uint32_t windows = (o.num_channels + channels - 1) / channels;
        g.channels = channels;
        g.slots = make_fastdiv(channels * o.spr.divisor); // up to 128: a segment that is stored normally has 32 vectors
        g.rows = kWindowBlock / g.slots.divisor;
        const uint32_t turns = (g.samples + g.rows - 1) / g.rows, blocks = (windows + kNumXcd - 1) / kNumXcd * kNumXcd;
        const bool few = turns <= 4;
        const uint32_t round = few ? 2 * cus : cus, rounds = (windows + round - 1) / round;
        const bool fills = rounds == 1 ? windows >= cus : windows * 16 >= rounds * round * 15;
        if (few && (fills || (o.width <= 40 && windows >= cus)))
            issue_window<4>(g, a, blocks, st);
        else if (channels == 2 && (turns == 7 || turns == 8) && fills && o.width % 16 != 0)
            issue_window<8>(g, a, blocks, st);
        else
            continue;
        return true;
    }
    return false;
}

template <typename A>
bool once_launch(const OnceGeometry& g, const A& a, int n, hipStream_t st)
{
    return window_launch(g, a, n, st) || (streamed(g, n) ? once_launch<true>(g, a, st) : once_launch<false>(g, a, st));
}

// ---- whole channels in several workgroups: which calls, which team ---------------
// Whether a backward pass reads dy, for the last time, past the caches, so that x, which the forward pass has left in
// the memory-side cache, stays there.  In dense tensors, and whole allocations where the halo is cleared, of `vectors` of 16
// bytes a channel: from 48 MiB. Smaller ones the cache holds all together. Backward in us, dy by the caches, past them
// (going round three sets of tensors): N 4, C 40, 40^3, 41 MB, 26.0, 27.5; N 96, C 60, 38 x 38, 33 MB, 23.6, 27.2; N
// 134, C 60, 38 x 38, 46 MB, 29.6, 29.7; N 64, C 64, 56 x 56, 51 MB, 34.0, 32.9; N 32, C 256, 56 x 56, 103 MB, 68, 63;
// doubles, N 4, C 32, 33^3, 37 MB, 28.9, 31.5; N 32, C 64, 56 x 56, 51 MB, 32.8, 31.7; N 8, C 32, 33^3, 74 MB, 58, 53.
// Forward + backward N 4, C 64, 64^3 269, 257, with x past the caches too 10 more. Cleared: of 28 to 44 MB 4 % more
// past the caches, of 60 to 95 MB 6 % less (235 calls). Rows with a halo between them at all sizes: below 28 MB equal,
// beyond 2 to 8 % less (664 calls; N 4, C 64, 30^3, halo of 1, forward + backward 45, 39).
constexpr size_t kStreamedGradient = size_t(48) << 20;

bool streams_gradient(size_t vectors, uint32_t num_channels)
{
    return vectors * num_channels * 16 >= kStreamedGradient;
}

template <typename G>
bool streams_gradient(const G& g)
{
    if constexpr (!G::kClears)
        if (!dense_rows(g))
            return true;
    return streams_gradient(g.vectors, g.num_channels);
}

template <typename T, int TEAM, int K, bool STREAM, typename G>
void issue_team(const TeamGeometry<G>& g, const OnceForward<T>& a, unsigned long long* states, hipStream_t st)
{
    launch_whole(kKernelTeam, K, bn_team_forward_kernel<T, TEAM, K, STREAM, G>, g.once.num_channels * g.members.divisor, TEAM, st,
                 g, a, states);
}
template <typename T, int TEAM, int K, bool STREAM, typename G>
void issue_team(const TeamGeometry<G>& g, const OnceBackward<T>& a, unsigned long long* states, hipStream_t st)
{
    const uint32_t blocks = g.once.num_channels * g.members.divisor;
    if constexpr (K >= 8) // the smallest members are those of small tensors
        if (streams_gradient(g.once))
        {
            launch_whole(kKernelTeam, K, bn_team_backward_kernel<T, TEAM, K, STREAM, true, G>, blocks, TEAM, st, g, a, states);
            return;
        }
    launch_whole(kKernelTeam, K, bn_team_backward_kernel<T, TEAM, K, STREAM, false, G>, blocks, TEAM, st, g, a, states);
}

template <int TEAM, int K, typename G, template <typename> class A, typename T>
void team_launch(const G& once, const A<T>& a, bool stream, uint32_t members, uint32_t max_polls, void* team_state,
                 hipStream_t st)
{
    TeamGeometry<G> g;
    g.once = once;
    g.members = make_fastdiv(members);
    g.span = ((once.vectors + members - 1) / members + TEAM - 1) / TEAM * TEAM;
    g.max_polls = max_polls;
    unsigned long long* const states = static_cast<unsigned long long*>(team_state);
    if (stream || G::kClears)
        issue_team<T, TEAM, K, true>(g, a, states, st);
    else
        issue_team<T, TEAM, K, G::kClears>(g, a, states, st);
}

// Looks of about a microsecond, or of two in launches of more than kCrowd workgroups, which sleep longer between them: a team
// that other streams keep off the chip for 2 ms, or for 5, works its sums out (a launch takes tens to hundreds of us).
constexpr uint32_t kTeamPolls = 2048;
// Workgroups from which teams are taken, of the smallest members and of larger ones (forward + backward, N 1, C 1, 64^3, 32
// workgroups of 32 KB, 17.0 us in two launches, 13.2 by them; backward N 2, C 1, 96^3 11.6 in two launches, 14.6 in 54 of 128 KB;
// doubles, forward + backward, N 2, C 3, 50 x 52 x 55 with a halo of 1 21.8 in two launches, 24.2 in 108 of 64 KB).
constexpr uint32_t kFewestMembers = 16, kFewestLarger = 128;

// What a pass takes beyond what all ways to run it share, in us: the bytes it moves, at the rate that members of
// its size reach, and for every round of workgroups that the chip holds at once what a member needs between its first
// load and its last store, the longer the larger its team.  Members that are mostly padding cost what full ones do;
// beyond the first round one that is not full costs less, by a part of what it lacks.  In two launches x (backward: x and dy)
// is read twice.  Haloed outputs of floats that are stored normally (kHaloedNormalStores) push out what members have read
// from some 30 MiB on.  Fitted to calls of 4 to 300 MB a tensor, each timed in all the ways that hold it, forward with
// backward, going round three sets of tensors; where only differences between the ways count.  The way these name makes both
// together 0.2 % longer than the fastest one on average (2053 dense tensors of floats; also in the half not fitted to), with
// halos 1.2 % (2402; doubles 0.3 and 1.2).  Rules on the number of workgroups alone made it 0.9 % longer, with
// halos 2.5, and more where the last round is nearly empty or members are mostly padding (forward, N 4, C 16, 96 x 63 x 84,
// 2000 members of 64 KB, 66 us, as now 53; doubles, forward, backward, N 184, C 91, 23 x 26 with a halo of 1 64, 105 and 57, 85;
// N 160, C 133, 23 x 19 with a halo of 1 67, 112 and 58, 81).  That was with four barriers between a member's last load and its
// first store; with the two of now the rounds and waits of teams cost less than these constants say, and two launches are named
// where teams are level (N 4, C 64, 64^3 with a halo of 1, forward in two launches, as named, 317, by teams 319; going over one
// set 295 both; N 8, C 64, 30^3, by teams, as named, 74.5, forward in two launches 78.5).
struct PassCost
{
    float wait; // of a round, for a team of 64
    struct
    {
        float per_mb, per_round;
    } members[3]; // of 512 threads with 4 and 8 vectors; then 512 with 16 (forward), 1024 with 8 (backward, floats)
    float launches, launches_per_mb;
    float displaced_per_mb; // of members
    float saved; // of what the last round of several lacks
};
// Floats and doubles, each of dense (or whole) tensors, and of rows with a halo between them.
constexpr PassCost kForwardCost[2][2] = {{{1.71f, {{0.336f, 2.85f}, {0.329f, 3.8f}, {0.24f, 9.21f}}, 4.2f, 0.57f, 0.0f, 0.3f},
                                          {2.25f, {{0.345f, 2.69f}, {0.358f, 3.66f}, {0.397f, 4.12f}}, 4.73f, 0.438f, 0.48f, 0.5f}},
                                         {{2.2f, {{0.31f, 2.5f}, {0.30f, 3.9f}, {0.28f, 6.8f}}, 4.2f, 0.57f, 0.0f, 0.5f},
                                          {3.65f, {{0.246f, 2.53f}, {0.309f, 3.54f}, {0.272f, 8.04f}}, 4.23f, 0.526f, 0.0f, 0.25f}}};
constexpr PassCost kBackwardCost[2][2] = {{{0.18f, {{0.522f, 4.28f}, {0.524f, 4.45f}, {0.263f, 13.6f}}, 9.3f, 0.78f, 0.0f, 0.3f},
                                           {0.01f, {{0.553f, 4.15f}, {0.404f, 7.21f}, {0.615f, 6.6f}}, 5.25f, 0.798f, 0.0f, 0.5f}},
                                          {{1.7f, {{0.49f, 2.8f}, {0.38f, 5.4f}, {}}, 9.3f, 0.78f, 0.0f, 0.5f},
                                           {4.03f, {{0.415f, 3.9f}, {0.492f, 5.06f}, {}}, 4.84f, 0.891f, 0.0f, 0.25f}}};
// Workgroups of each size of member that a CU holds (measured: the time of a call steps up where there is one more).
constexpr uint32_t kForwardOnCu[3] = {3, 3, 2}, kBackwardOnCu[3] = {3, 2, 1}, kBackwardDoublesOnCu[3] = {2, 2, 1};

struct PassShape
{
    size_t bytes;        // of a tensor, and of the lines at the ends of haloed rows
    uint32_t channels;
    bool rows;           // haloed
    size_t displaced;    // bytes of haloed rows stored normally, beyond the first 30 MiB
};

size_t displaced_bytes(size_t bytes, bool stream)
{
    constexpr size_t kBeside = size_t(30) << 20;
    return stream || bytes < kBeside ? 0 : bytes - kBeside;
}

// Rows that do not follow one another bring up to a line of what is between them along.
size_t moved_bytes(size_t rows, size_t width, size_t pitch, size_t item)
{
    return rows * item * (width + std::min(pitch - width, size_t(128) / item));
}

// The cheapest of three sizes of members, teams of members[i] each (0: none), or -1: two launches.
template <typename T, bool FORWARD>
int cheapest_pass(const PassShape& p, const uint32_t (&members)[3], bool forced)
{
    const PassCost& cost = (FORWARD ? kForwardCost : kBackwardCost)[sizeof(T) == 8][p.rows];
    const auto& on_cu = FORWARD ? kForwardOnCu : sizeof(T) == 4 ? kBackwardOnCu : kBackwardDoublesOnCu;
    const uint32_t cus = chip_units();
    const float mb = p.bytes * 1e-6f;
    float least = forced ? std::numeric_limits<float>::max() : cost.launches + cost.launches_per_mb * mb;
    int best = -1;
    for (int i = 0; i < 3; ++i)
    {
        if (members[i] == 0)
            continue;
        const float full = static_cast<float>(static_cast<uint64_t>(members[i]) * p.channels) / (cus * on_cu[i]);
        const float rounds = full <= 1 ? 1 : cost.saved * full + (1 - cost.saved) * std::ceil(full);
        const float us = cost.members[i].per_mb * mb + rounds * (cost.members[i].per_round + cost.wait * members[i] / 64)
                         + cost.displaced_per_mb * p.displaced * 1e-6f;
        if (us < least)
        {
            least = us;
            best = i;
        }
    }
    return best;
}

// `members`, or 0 where they are more than `most`, exchange more sums than a channel's state has, or are fewer than `least`
// workgroups.
uint32_t fit_team(size_t members, uint32_t channels, size_t sums, uint32_t most, uint32_t least)
{
    const size_t blocks = members * channels;
    return members > most || sums > most_team_sums(channels) || blocks < least || blocks >= (1u << 30)
               ? 0
               : static_cast<uint32_t>(members);
}

PassShape pass_shape(const OnceGeometry& g, bool stream)
{
    const size_t rows = g.vectors / g.spr.divisor * g.num_channels;
    const size_t pitch = std::max<size_t>(g.h.divisor > 1 ? g.sy : g.d.divisor > 1 ? g.sz : g.width, g.width);
    return {moved_bytes(rows, g.width, pitch, sizeof(float)), g.num_channels, !dense_rows(g),
            displaced_bytes(rows * pitch * sizeof(float), stream)};
}
PassShape pass_shape(const ClearGeometry& g, bool)
{
    return {static_cast<size_t>(g.vectors) * g.num_channels * 16, g.num_channels, false, 0};
}

// Backward, teams of 65 to 128 members of 128 KB only in tensors that the memory-side cache nearly holds.  Dense ones below
// 240 MiB: 7 % less than two launches on average (N 16, C 10, 64^3, 168 MB, 117 us and 131; N 2, C 6, 110 x 120 x 130 55 and
// 69; N 8, C 13, 73 x 85 x 84, 217 MB, 162 and 170; 17 % more at worst; N 16, C 16, 64^3, 268 MB, 231 and 202). With a
// halo below 104 MiB, where x, dy and dx take half of it: 7 % less (N 100, C 8, 200 x 160, 102 MB, 87 and 101), beyond
// 9 % more (N 158, C 13, 25 x 23 x 21 128 and 112; N 14, C 11, 65 x 66 x 48, halo of 2, 150 and 133) unless rows are
// long, which leaves few partial lines: from 80 elements 1 % less, up to 10 (N 4, C 8, 96^3, forward + backward 154 and
// 171; N 118, C 15, 124 x 152, halo of 2, 183 and 195). Where the halo is cleared never (4 % more; N 50, C 16, 33 x 36
// x 45 with a halo of 2 206 and 171).
constexpr size_t kHeldTensor = size_t(240) << 20, kHeldRows = size_t(104) << 20;
constexpr uint32_t kLongRow = 80;

bool for_large_teams(const OnceGeometry& g)
{
    return static_cast<size_t>(g.vectors) * g.num_channels * 16
           < (dense_rows(g) || g.width >= kLongRow ? kHeldTensor : kHeldRows);
}
bool for_large_teams(const ClearGeometry&)
{
    return false;
}

// By teams, or false.  Without a: whether.  `forced`: however few workgroups that is, and however long it takes.
template <typename G, typename T>
bool team_variant(const G& g, const OnceForward<T>* a, bool stream, bool forced, uint32_t most, uint32_t polls,
                  void* team_state, hipStream_t st)
{
    const auto fit = [&](uint32_t held, uint32_t least) {
        const size_t m = (g.vectors + held - 1) / held;
        return fit_team(m, g.num_channels, 2 * m, most, forced ? 1 : least);
    };
    const uint32_t members[3] = {fit(512 * 4, kFewestMembers), fit(512 * 8, kFewestLarger), fit(512 * 16, kFewestLarger)};
    const int best = cheapest_pass<T, true>(pass_shape(g, stream), members, forced);
    if (best < 0 || !a)
        return best >= 0;
    if (best == 0)
        team_launch<512, 4>(g, *a, stream, members[0], polls, team_state, st);
    else if (best == 1)
        team_launch<512, 8>(g, *a, stream, members[1], polls, team_state, st);
    else
        team_launch<512, 16>(g, *a, stream, members[2], polls, team_state, st);
    return true;
}

template <typename G, typename T>
bool team_variant(const G& g, const OnceBackward<T>* a, bool stream, bool forced, uint32_t most, uint32_t polls,
                  void* team_state, hipStream_t st)
{
    const auto fit = [&](uint32_t held, uint32_t least, uint32_t at_most) {
        const size_t m = (g.vectors + held - 1) / held;
        return fit_team(m, g.num_channels, 4 * m, at_most, forced ? 1 : least);
    };
    const uint32_t members[3] = {fit(512 * 4, kFewestMembers, most / 2), fit(512 * 8, kFewestLarger, most / 2),
                                 fit(1024 * 8, kFewestLarger, for_large_teams(g) ? most : most / 2)};
    const int best = cheapest_pass<T, false>(pass_shape(g, stream), members, forced);
    if (best < 0 || !a)
        return best >= 0;
    if (best == 0)
        team_launch<512, 4>(g, *a, stream, members[0], polls, team_state, st);
    else if (best == 1)
        team_launch<512, 8>(g, *a, stream, members[1], polls, team_state, st);
    else
        team_launch<1024, 8>(g, *a, stream, members[2], polls, team_state, st);
    return true;
}

// Channels that one workgroup of 1024 threads would hold, for teams first: where such workgroups leave much of the chip idle, or
// a CU holds one of them, which loads, adds and stores with nothing beside it.  Forward + backward in us, by workgroups and by
// teams, going round three sets of tensors (330 calls):
//   few channels (N 8, C 64, 56 x 56 14.4 and 11.8; C 16 13.5 and 10.9; with 4096 vectors or fewer equal);
//   more than 8192 vectors, with 16 or 20 a thread: 15 % less on average, 2 % more at worst, but for channels that fill one round
//   of the chip (C 128, N 16 27.9 and 23.2; N 6, C 283, 90 x 99 77.7 and 54.9; N 1, C 682, 203 x 188, cleared 118 and
//   96; N 6, C 174, 5 % more);
//   up to 8192, whose backward workgroups a CU holds one of: with a halo, or dense, where channels leave half of a second round
//   empty, or an eighth of more rounds (N 53, C 1185, 21 x 22 with a halo 173 and 158; C 622, 6800 vectors 4 % less; C
//   401 and 506, 3 and 9 % more, C 1022 7); cleared, unless they nearly fill the rounds (N 7, C 328, 15 x 15 x 12 49
//   and 37; C 202 and 993, 6 % more).
// The state of more than 2048 channels would be as large as many a tensor.
template <typename G>
bool teams_first(const G& g)
{
    constexpr uint32_t kMostChannels = 2048;
    if (g.vectors <= 4096 || g.num_channels > kMostChannels)
        return false;
    if (g.num_channels <= kOnceManyChannels || g.vectors > 8192)
        return true;
    const uint32_t cus = chip_units();
    const uint32_t rounds = (g.num_channels + cus - 1) / cus;
    const uint32_t filled = g.num_channels * 16 / (rounds * cus); // sixteenths of the rounds
    if constexpr (G::kClears)
        return rounds == 1 ? filled <= 10 : filled < 15;
    return rounds > 1 && filled < (rounds == 2 ? 12 : 14);
}

// A team keeps within half of the chip.
uint32_t most_members()
{
    const uint32_t cus = compute_units();
    return cus ? std::min(cus / 2, kMaxMembers) : kMaxMembers;
}

// Bytes of the state for calls on tensors like this, apart from one another: 0 if none is for teams.
template <typename G>
size_t team_state_needed(const G& g)
{
    const uint32_t most = most_members();
    const OnceForward<float>* const forward = nullptr;
    const OnceBackward<float>* const backward = nullptr;
    const bool teams = ((teams_first(g) || !once_holds<OnceForward<float>>(g))
                        && team_variant(g, forward, true, false, most, 0, nullptr, nullptr))
                       || ((teams_first(g) || !once_holds<OnceBackward<float>>(g))
                           && team_variant(g, backward, true, false, most, 0, nullptr, nullptr));
    return teams ? team_state_at(g.num_channels) * sizeof(unsigned long long) : 0;
}

// Short segments have kernels of their own (N 2048, C 256, 7 x 7: 141 us, by teams 172).
bool for_teams(const OnceGeometry& g, int n)
{
    return !dense_rows(g) || streamed(g, n);
}

// False: the call is not for teams.  bytes: from the first to behind the last element of a tensor.
template <typename G, typename A>
bool launch_by_teams(const G& g, const A& a, size_t bytes, bool stream, std::initializer_list<const void*> inputs,
                     const void* output, bool forced, uint32_t polls, void* team_state, hipStream_t st)
{
    if (!team_state)
        return false;
    for (const void* p : inputs)
        if (!apart(p, output, bytes))
            return false;
    return team_variant(g, &a, stream, forced, most_members(), polls, team_state, st);
}

template <typename A>
bool launch_by_teams(const OnceGeometry& g, const A& a, int n, std::initializer_list<const void*> inputs,
                     const void* output, bool forced, uint32_t polls, void* team_state, hipStream_t st)
{
    return for_teams(g, n)
           && launch_by_teams(g, a, reach_bytes(g, n), streamed(g, n), inputs, output, forced, polls, team_state, st);
}

// ---- whole channels of doubles, in the order of the staged calls ------------------
// Tensors that lie alike (`ts`: the inputs, x first), whose staged reduction is one of the long-segment kernels in
// vectors, with no more groups a channel than the staged kernels add in one go.
bool ordered_geometry(int num_samples, int num_channels, size_t spatial, std::initializer_list<const HostTensor*> ts,
                      const HostTensor& output, OrderedGeometry* g, bool* rows)
{
    HostTensor t[2];
    size_t inputs = 0;
    for (const HostTensor* i : ts)
    {
        if (!lie_alike({i, &output}))
            return false;
        t[inputs++] = *i;
    }
    ShortGeometry sg;
    const bool one = inputs == 1;
    if (one ? short_segments<double>(num_samples, num_channels, spatial, {&t[0]}, &sg)
            : short_segments<double>(num_samples, num_channels, spatial, {&t[0], &t[1]}, &sg))
        return false;
    const size_t last = (num_samples - 1) * static_cast<size_t>(t[0].map.stride_n) + short_span(t[0], spatial);
    ReductionPlan plan;
    if (last >= (1ull << 30) || t[0].map.stride_n >= (1ll << 30)
        || (one ? plan_reduction<double>(num_samples, num_channels, spatial, {&t[0]}, kUnroll, &plan)
                : plan_reduction<double>(num_samples, num_channels, spatial, {&t[0], &t[1]}, kUnroll / 2, &plan)))
        return false;
    // (outputs are stored in the same vectors, so they have to be aligned where those are)
    if (plan.vw != full_vec<double>() || (!plan.strided && !output.aligned) || plan.groups > kBlockSize
        || plan.spatial >= (1ull << 31) || plan.units >= (1ull << 31))
        return false;
    constexpr size_t kBatch = kBlockSize * 2 * kOrderedBatch; // elements
    if (plan.ch.chunk % kBatch != 0)
        return false;
    const uint32_t batches = static_cast<uint32_t>(plan.ch.chunk / kBatch);
    const uint32_t rounds = static_cast<uint32_t>((plan.units + plan.groups - 1) / plan.groups);
    *rows = plan.strided;
    g->map = t[0].map;
    g->spatial = static_cast<uint32_t>(plan.spatial);
    g->chunk = static_cast<uint32_t>(plan.ch.chunk);
    g->per_segment = make_fastdiv(static_cast<uint32_t>(plan.ch.chunks_per_seg));
    g->unit_batches = make_fastdiv(batches);
    g->group_batches = make_fastdiv(batches * rounds);
    g->units = static_cast<uint32_t>(plan.units);
    g->groups = static_cast<uint32_t>(plan.groups);
    g->num_channels = static_cast<uint32_t>(num_channels);
    g->max_polls = kTeamPolls;
    return true;
}

template <int TEAM, int K, bool TEAMS, bool ROWS, bool STREAM, typename G>
void issue_ordered(const G& g, const OnceForward<double>& a, unsigned long long* states, uint32_t blocks,
                   hipStream_t st)
{
    constexpr Kernel kOrdered = TEAMS ? kKernelOrderedTeam : kKernelOrdered;
    launch_whole(kOrdered, K, bn_ordered_forward_kernel<TEAM, K, TEAMS, ROWS, STREAM, G>, blocks, TEAM, st, g, a, states);
}
template <int TEAM, int K, bool TEAMS, bool ROWS, bool STREAM, typename G>
void issue_ordered(const G& g, const OnceBackward<double>& a, unsigned long long* states, uint32_t blocks,
                   hipStream_t st)
{
    constexpr Kernel kOrdered = TEAMS ? kKernelOrderedTeam : kKernelOrdered;
    if constexpr (K >= 8)
        if (g.streams_gradient)
        {
            launch_whole(kOrdered, K, bn_ordered_backward_kernel<TEAM, K, TEAMS, ROWS, STREAM, true, G>, blocks, TEAM, st, g, a, states);
            return;
        }
    launch_whole(kOrdered, K, bn_ordered_backward_kernel<TEAM, K, TEAMS, ROWS, STREAM, false, G>, blocks, TEAM, st, g, a, states);
}

// Groups that a workgroup of TEAM threads with K vectors each holds.
template <int TEAM, int K>
uint32_t ordered_holds(const OrderedGeometry& g)
{
    return TEAM / kBlockSize * (K / kOrderedBatch / g.group_batches.divisor);
}

template <int TEAM, int K, bool TEAMS, typename G, typename A>
void ordered_issue(const G& g, const A& a, bool rows, bool stream, void* state, hipStream_t st)
{
    unsigned long long* const states = static_cast<unsigned long long*>(state);
    const uint32_t blocks = TEAMS ? g.num_channels * g.members.divisor : (g.num_channels + kNumXcd - 1) / kNumXcd * kNumXcd;
    if constexpr (std::is_same<G, OrderedClearing>::value) // (rows: see ordered_launch)
        return issue_ordered<TEAM, K, TEAMS, true, false>(g, a, states, blocks, st);
    else if (!rows)
        issue_ordered<TEAM, K, TEAMS, false, true>(g, a, states, blocks, st);
    else if (stream)
        issue_ordered<TEAM, K, TEAMS, true, true>(g, a, states, blocks, st);
    else
        issue_ordered<TEAM, K, TEAMS, true, false>(g, a, states, blocks, st);
}

// One workgroup a channel.  Without a: whether.
template <int TEAM, int K, typename G, typename A>
bool ordered_once(G g, const A* a, bool rows, bool stream, hipStream_t st)
{
    if (g.groups > ordered_holds<TEAM, K>(g))
        return false;
    g.passes = K / kOrderedBatch / g.group_batches.divisor;
    g.members = make_fastdiv(1);
    if (a)
        ordered_issue<TEAM, K, false>(g, *a, rows, stream, nullptr, st);
    return true;
}

// Members of a team of workgroups of TEAM threads with K vectors each, or 0.
template <int TEAM, int K, int SUMS>
uint32_t ordered_members(const OrderedGeometry& g, uint32_t most, uint32_t least)
{
    const uint32_t own = ordered_holds<TEAM, K>(g);
    if (own < 2)
        return 0;
    const uint32_t width = own % 4 == 0 ? 4 : 2;
    return fit_team((g.groups + own - 1) / own, g.num_channels, (g.groups + width - 1) / width * SUMS, most, least);
}

template <int TEAM, int K, typename G, typename A>
void ordered_team(G g, const A& a, bool rows, bool stream, uint32_t members, void* state, hipStream_t st)
{
    g.passes = K / kOrderedBatch / g.group_batches.divisor;
    g.members = make_fastdiv(members);
    ordered_issue<TEAM, K, true>(g, a, rows, stream, state, st);
}

// By teams, as for floats (team_variant).
template <typename G, typename A>
bool ordered_by_teams(const G& g, const A* a, size_t bytes, bool rows, bool stream, uint32_t most, bool forced,
                      void* state, hipStream_t st)
{
    constexpr bool kForward = std::is_same<A, OnceForward<double>>::value;
    constexpr int kSums = kForward ? 2 : 4;
    const uint32_t larger = forced ? 1 : kFewestLarger;
    uint32_t members[3] = {ordered_members<512, 4, kSums>(g, most / 2, forced ? 1 : kFewestMembers),
                           ordered_members<512, 8, kSums>(g, kForward ? most : most / 2, larger), 0};
    if constexpr (kForward)
        members[2] = ordered_members<512, 16, kSums>(g, most, larger);
    const int best = cheapest_pass<double, kForward>({bytes, g.num_channels, rows, 0}, members, forced);
    if (best < 0 || !a)
        return best >= 0;
    if (best == 0)
        ordered_team<512, 4>(g, *a, rows, stream, members[0], state, st);
    else if (best == 1)
        ordered_team<512, 8>(g, *a, rows, stream, members[1], state, st);
    else if constexpr (kForward)
        ordered_team<512, 16>(g, *a, rows, stream, members[2], state, st);
    return true;
}

// Which of them, as for floats (once_launch, team_variant).  most_members 0: no teams, where the outputs
// overlap the inputs or there is no state.  bytes: see PassShape.  *team: whether it is one.
template <typename G, typename A>
bool ordered_variant(const G& g, const A* a, size_t bytes, bool rows, bool stream, uint32_t most, bool forced,
                     void* state, hipStream_t st, bool* team)
{
    constexpr bool kForward = std::is_same<A, OnceForward<double>>::value;
    const size_t vectors = static_cast<size_t>(g.groups) * g.group_batches.divisor * kOrderedBatch * kBlockSize;
    const bool few = g.num_channels <= kOnceManyChannels;
    const auto by_teams = [&] {
        *team = true;
        return ordered_by_teams(g, a, bytes, rows, stream, most, forced, state, st);
    };
    if ((forced || (few && vectors > 4096)) && by_teams())
        return true;
    *team = false;
    if (forced)
        return false;
    if (ordered_once<256, 4>(g, a, rows, stream, st) || ordered_once<512, 4>(g, a, rows, stream, st)
        || ordered_once<1024, 4>(g, a, rows, stream, st) || ordered_once<1024, 8>(g, a, rows, stream, st))
        return true;
    if constexpr (kForward)
        if (!few && ordered_once<1024, 16>(g, a, rows, stream, st))
            return true;
    return by_teams();
}

// ---- short segments of doubles, in the order of the staged calls -------------------
// Dense or haloed tensors that lie alike (`ts`: the inputs, x first), cut as the staged reduction cuts them; g->turns is the
// samples of a lane in a range.
bool short_once_geometry(int num_samples, int num_channels, size_t spatial, std::initializer_list<const HostTensor*> ts,
                         const HostTensor& output, ShortOnceGeometry* g)
{
    const HostTensor& x = **ts.begin();
    for (const HostTensor* t : ts)
        if (!lie_alike({t, &output}))
            return false;
    ShortGeometry sg;
    if (!short_segments<double>(num_samples, num_channels, spatial, {&x}, &sg))
        return false;
    const size_t last = (num_samples - 1) * static_cast<size_t>(x.map.stride_n)
                        + (std::min(num_channels, kBlockSize * 4) - 1) * static_cast<size_t>(x.map.stride_c)
                        + short_span(x, spatial);
    if (last >= (1ull << 30))
        return false;
    const int unroll = ts.size() == 1 ? kUnroll : kUnroll / 2;
    const int groups = short_reduction_groups(&sg, max_groups_per_channel(num_channels), unroll, sizeof(double));
    const ShortTensor t = short_tensor(x, sg);
    g->row = static_cast<uint32_t>(sg.row);
    g->slots_per_row = make_fastdiv(static_cast<uint32_t>(sg.slots_per_row));
    g->slots = make_fastdiv(static_cast<uint32_t>(sg.slots));
    g->h = make_fastdiv(static_cast<uint32_t>(t.h));
    g->sy = t.sy;
    g->sz = t.sz;
    g->stride_n = static_cast<uint32_t>(t.stride_n);
    g->stride_c = t.stride_c;
    g->rows = make_fastdiv(static_cast<uint32_t>(sg.rows));
    g->turns = make_fastdiv(static_cast<uint32_t>((sg.samples_per_group + sg.rows - 1) / sg.rows));
    g->per = static_cast<uint32_t>(sg.samples_per_group);
    g->ranges = static_cast<uint32_t>(groups);
    g->num_samples = static_cast<uint32_t>(num_samples);
    g->num_channels = static_cast<uint32_t>(num_channels);
    return true;
}

// Fewer windows than this that play ranges one after another (g.passes) leave the chip idle longer than a second launch takes:
// forward, or backward, N 255, C 34, 4 x 7 x 4 5.8 us more than in two launches, N 231, C 20, 6 x 7 3.9, N 85, C 22, 4
// x 7 x 5 level. So do the largest workgroups with many samples, whose rows one thread adds up: forward in us, in two
// launches and so, N 112, C 10, 5 x 4 x 6 8.3 and 10.2, N 145, C 13, 7 x 8 8.2 and 9.5, N 83, C 27, 10 x 11 with a halo
// 8.9 and 10.0; N 56, C 21, 5 x 6 x 5 with a halo 9.0 and 8.5, N 34, C 12, 17 x 15 with a halo 8.4 and 8.2.
constexpr uint32_t kShortWindows = 64, kShortManySamples = 64;

template <int VEC, int TEAM, int K, typename G>
void issue_short_once(const G& g, const OnceForward<double>& a, uint32_t blocks, hipStream_t st)
{
    launch_whole(kKernelShortOnce, K, bn_short_once_forward_kernel<VEC, TEAM, K, G>, blocks, TEAM, st, g, a);
}
template <int VEC, int TEAM, int K, typename G>
void issue_short_once(const G& g, const OnceBackward<double>& a, uint32_t blocks, hipStream_t st)
{
    launch_whole(kKernelShortOnce, K, bn_short_once_backward_kernel<VEC, TEAM, K, G>, blocks, TEAM, st, g, a);
}

// Windows of workgroups of `threads` with `vectors` each that play up to most_passes ranges a thread; 0: such a workgroup does
// not hold a channel.
uint32_t short_once_windows(ShortOnceGeometry* g, uint32_t threads, uint32_t vectors, uint32_t most_passes)
{
    const uint32_t passes = std::min(vectors / g->turns.divisor, most_passes);
    if (passes == 0)
        return 0;
    g->together = (g->ranges + passes - 1) / passes;
    g->passes = (g->ranges + g->together - 1) / g->together;
    const uint32_t lanes = g->slots.divisor * g->rows.divisor * g->together; // of a channel
    if (lanes > threads)
        return 0;
    const uint32_t channels = std::min(threads / lanes, g->num_channels);
    g->channels = make_fastdiv(channels);
    return (g->num_channels + channels - 1) / channels;
}

// Outputs whose halo is cleared, larger than this, are left to the staged calls, which store whole lines past the
// caches, unless a few long segments, or one workgroup a channel with little halo, leave few parts of lines to store.
// Forward + backward in us, staged and by these: N 8, C 64, 30^3, 128 MiB 168 and 199; N 63, C 65, 29 x 39, 40 MiB 67.0
// and 72.1; N 48, C 242, 9 x 8 x 7, 88 MiB 120 and 136; rows of 80 elements and more: N 1, C 744, 149 x 140, 122 MiB
// 168 and 140; N 12, C 61, 85 x 84, 42 MiB 69 and 56; one workgroup: N 4, C 1963, 63 x 52, halo of 2, 225 MiB 298 and
// 258; N 3, C 1290, 35 x 48, halo of 2, 60 MiB 88 and 69; smaller: N 12, C 77, 11 x 15 x 15, halo of 2, 38 MiB 58 and
// 42; N 5, C 16, 38 x 65 30.4 and 13.7.
constexpr size_t kClearedByOrder = size_t(39) << 20;

// Whether short segments whose output's halo is cleared are for `windows` workgroups that hold so many vectors. The
// staged calls take a time for each segment, and those of up to 200 cells, allocated, are always for one launch (N 193,
// C 941, 4 x 5 301 and 100 us, N 176, C 910, 3 x 2 255 and 38); beyond they run at memory's rate, and a workgroup with
// all of a channel's cells to itself needs neighbours that keep memory busy. Forward + backward in us, staged and in
// one launch each way, of 220 calls:
//   few workgroups of much: N 106, C 26, 4^3, halo of 3 36 and 62; N 119, C 88, 4 x 5 x 6, halo of 2 65 and 89; N 92, C
//   71, 4^3, halo of 2 38 and 41; more of them N 43, C 107, 5 x 5 x 4, halo of 3 62 and 52; of little N 29, C 72, 7 x 6
//   x 6, halo of 2 41 and 34;
//   the largest, one a CU, in more than one round: N 57, C 454, 18 x 9, halo of 3 95 and 115; N 36, C 359, 16 x 13,
//   halo of 3 65 and 75; in one N 83, C 183, 9 x 13, halo of 3 61 and 49; N 53, C 120, 11 x 16, halo of 2 37 and 31;
//   large outputs in a little more than one round: N 53, C 284, 4 x 4 x 5, halo of 2 73 and 95 (C 350 106 and 100);
//   and with less halo than three times the interior, segments of more than 350 cells: N 22, C 1078, 20 x 12, halo of 3
//   115 and 123; N 18, C 896, 18 x 12, halo of 2 67 and 72; up to 350 N 41, C 556, 9 x 16, halo of 2 80 and 70; with
//   more N 9, C 412, 7 x 5 x 4, halo of 3 55 and 40.
bool clearing_pays(const ShortOnceClearing& g, uint32_t windows, uint32_t vectors)
{
    constexpr size_t kMuch = 260000;
    const size_t segment = g.stride_c, allocated = segment * g.num_channels * g.num_samples * sizeof(double);
    const size_t inside = static_cast<size_t>(g.halo.width) * g.halo.h.divisor * g.halo.d.divisor;
    if (segment <= 200)
        return true;
    const uint32_t cus = chip_units();
    const bool much = allocated > kMuch * windows;
    if (much && windows * 8 < cus * 3)
        return false;
    if (vectors >= 1024 * 8 && windows > cus)
        return false;
    if (allocated <= kClearedByOrder)
        return true;
    return !(g.num_channels > cus && g.num_channels * 20 < cus * 23) && (segment <= 350 || segment >= 4 * inside);
}
bool clearing_pays(const ShortOnceGeometry&, uint32_t, uint32_t)
{
    return true; // nothing is cleared
}

// False: workgroups of TEAM threads with K vectors each do not hold a channel, or are not for this call.
template <int TEAM, int K, typename G, typename A>
bool short_once(G g, const A& a, hipStream_t st)
{
    constexpr bool kForward = std::is_same<A, OnceForward<double>>::value;
    const uint32_t windows = short_once_windows(&g, TEAM, K, short_once_passes(K, kForward));
    const bool idles = g.passes > 1 || (TEAM * K >= 1024 * 8 && g.num_samples > kShortManySamples);
    if (windows == 0 || (idles && windows < kShortWindows) || !clearing_pays(g, windows, TEAM * K))
        return false;
    // The largest workgroups have to have more than ten of sixteen lanes play something (forward in us, by them less in
    // two launches: 1024 threads N 29, C 911, 12 x 20, nine, +5.0, N 38, C 489, 14 x 11 with a halo, 10.5, -4.6; 512
    // threads N 71, C 291, 8 x 10, ten, +3.6, N 129, C 319, 8 x 5 with a halo, 12, -3.3); those of 16 vectors in one
    // pass (N 70, C 135, 12 x 11, three, +1.1), and in more than a round of the chip nearly all of them (N 83, C 1398,
    // 12 x 8 with a halo, 12, +9, N 46, C 832, 16 x 12, 15, -3.4).
    const uint32_t playing = g.channels.divisor * g.slots.divisor * g.rows.divisor * g.together;
    if (TEAM * K >= 1024 * 8 && playing * 16 <= TEAM * 10)
        return false;
    if (TEAM * K >= 1024 * 8 && K == 16 && (g.passes > 1 || (windows > 2 * chip_units() && playing * 16 < TEAM * 14)))
        return false;
    // (the smallest workgroup of so many vectors, backward: N 71, C 291, 8 x 10 3.4 us more than in two launches, N
    // 109, C 1893, 5 x 6, 947 of them, 18.2 less)
    if (TEAM == 256 && K == 16 && windows <= 2 * chip_units())
        return false;
    const uint32_t blocks = (windows + kNumXcd - 1) / kNumXcd * kNumXcd;
    if (g.row == 1)
        issue_short_once<1, TEAM, K>(g, a, blocks, st);
    else
        issue_short_once<2, TEAM, K>(g, a, blocks, st);
    return true;
}

template <int THREADS, int VECTORS>
struct ShortWorkgroup
{
    static constexpr int threads = THREADS, vectors = VECTORS;
};

// f of the workgroups that there are, until one is true: the smallest first, more threads before more vectors a thread.
template <bool FORWARD, typename F>
bool any_short_workgroup(const F& f)
{
    if (f(ShortWorkgroup<256, 4>()) || f(ShortWorkgroup<512, 4>()))
        return true;
    if constexpr (FORWARD)
        return f(ShortWorkgroup<256, 8>()) || f(ShortWorkgroup<512, 8>()) || f(ShortWorkgroup<1024, 8>()) || f(ShortWorkgroup<512, 16>());
    else
        return f(ShortWorkgroup<1024, 4>()) || f(ShortWorkgroup<256, 8>()) || f(ShortWorkgroup<512, 8>())
               || f(ShortWorkgroup<1024, 8>()) || f(ShortWorkgroup<256, 16>());
}

// The smallest workgroup that holds a channel.
template <typename G, typename A>
bool short_once_launch(const G& g, const A& a, hipStream_t st)
{
    return any_short_workgroup<std::is_same<A, OnceForward<double>>::value>(
        [&](auto w) { return short_once<decltype(w)::threads, decltype(w)::vectors>(g, a, st); });
}

size_t moved_bytes(const HostTensor& t, int n, int c, size_t s)
{
    const size_t all = static_cast<size_t>(n) * c * s;
    if (!t.strided)
        return all * sizeof(double);
    const size_t w = t.row, h = t.map.h.divisor, pitch = h > 1 ? t.map.sy : s > w * h ? t.map.sz : w;
    return moved_bytes(all / w, w, std::max(pitch, w), sizeof(double));
}

// False: the staged kernels.  halo: the output's is cleared.
template <typename A>
bool ordered_launch(int n, int c, size_t s, std::initializer_list<const HostTensor*> ts, const HostTensor& output,
                    std::initializer_list<const void*> inputs, const void* out, const A& a, void* state,
                    const uint32_t* team_polls, hipStream_t st, const HaloCells* halo = nullptr)
{
    ShortOnceClearing sg;
    if (!team_polls && short_once_geometry(n, c, s, ts, output, &sg))
    {
        if (!halo)
        {
            if (short_once_launch<ShortOnceGeometry>(sg, a, st))
                return true;
        }
        else
        {
            sg.halo = *halo;
            if (short_once_launch(sg, a, st))
                return true;
        }
    }
    OrderedClearing g;
    bool rows, team;
    // (a halo on the outermost spatial dimension alone leaves dense segments, which the kernels that clear are not
    // built for: staged)
    if (!ordered_geometry(n, c, s, ts, output, &g, &rows) || (halo && !rows))
        return false;
    const size_t bytes = (static_cast<size_t>(c - 1) * output.map.stride_c + static_cast<size_t>(n - 1) * output.map.stride_n
                          + short_span(output, s)) * sizeof(double);
    bool teams = state != nullptr;
    for (const void* p : inputs)
        teams = teams && apart(p, out, bytes);
    if (team_polls)
        g.max_polls = *team_polls;
    g.streams_gradient = output.strided || streams_gradient(n * s / 2, c);
    const bool stream = !output.strided || bytes > kHaloedNormalStores;
    const size_t moved = moved_bytes(output, n, c, s);
    uint32_t most = teams ? most_members() : 0;
    const size_t allocated = static_cast<size_t>(n) * output.map.stride_n * sizeof(double), inside = size_t(n) * c * s * sizeof(double);
    // (units that segments fill a quarter of, in more than a round of workgroups: N 11, C 333, 8 x 6 x 7 40.0 and 42.6
    // us, C 165 32.9 and 24.1)
    if (halo && c > static_cast<int>(chip_units())
        && static_cast<size_t>(g.groups) * g.group_batches.divisor * kOrderedBatch * kBlockSize > 2 * size_t(n) * s)
        return false;
    if (halo && allocated > kClearedByOrder && output.row < kLongRow)
    {
        if (allocated * 10 > inside * 13)
            return false;
        most = 0; // no teams
    }
    if (!halo)
        return ordered_variant<OrderedGeometry>(g, &a, moved, rows, stream, most, team_polls != nullptr, state, st, &team);
    g.halo = *halo;
    return ordered_variant(g, &a, moved, rows, stream, most, false, state, st, &team);
}

// team_polls: by teams or not at all, however few workgroups that is, with this many looks.
template <typename T>
int forward_once(int n, const h2x_tensor_geometry* gx, const h2x_tensor_geometry* gy, const void* x,
                 const void* scale, const void* bias, size_t num_per_sum, double decay, double eps, void* mean,
                 void* var, void* running_mean, void* running_var, void* y, void* ws, void* team_state, hipStream_t st,
                  const uint32_t* team_polls = nullptr)
{
    HostTensor tx, ty;
    int c;
    size_t s;
    const int err = two_tensors<T>(n, gx, gy, x, y, &tx, &ty, &c, &s);
    if (err)
        return err;
    if constexpr (sizeof(T) == 4) // see once_geometry
    {
        OnceGeometry g;
        if (x && y && n > 0 && c > 0 && s > 0 && num_per_sum > 0 && once_geometry(n, c, s, {&tx, &ty}, &g))
        {
            const OnceForward<T> a{static_cast<const T*>(x), static_cast<const T*>(scale), static_cast<const T*>(bias),
                                   static_cast<T*>(mean), static_cast<T*>(var), static_cast<T*>(running_mean),
                                   static_cast<T*>(running_var), static_cast<T*>(y), static_cast<T>(num_per_sum),
                                   static_cast<T>(decay), static_cast<T>(eps)};
            if (team_polls)
                return launch_by_teams(g, a, n, {x}, y, true, *team_polls, team_state, st) ? issued()
                                                                                           : H2X_ERR_UNSUPPORTED;
            const auto by_teams = [&] { return launch_by_teams(g, a, n, {x}, y, false, kTeamPolls, team_state, st); };
            const bool teams = teams_first(g);
            if ((teams && by_teams()) || once_launch(g, a, n, st) || (!teams && by_teams()))
                return issued();
        }
    }
    else if (x && y && n > 0 && c > 0 && s > 0 && num_per_sum > 0)
    {
        const OnceForward<T> a{static_cast<const T*>(x), static_cast<const T*>(scale), static_cast<const T*>(bias),
                               static_cast<T*>(mean), static_cast<T*>(var), static_cast<T*>(running_mean),
                               static_cast<T*>(running_var), static_cast<T*>(y), static_cast<T>(num_per_sum),
                               static_cast<T>(decay), static_cast<T>(eps)};
        if (ordered_launch(n, c, s, {&tx}, ty, {x}, y, a, team_state, team_polls, st))
            return issued();
    }
    if (team_polls)
        return H2X_ERR_UNSUPPORTED;
    return forward_local<T>(n, c, s, tx, ty, x, scale, bias, num_per_sum, decay, eps, mean, var, running_mean,
                            running_var, y, ws, st);
}

template <typename T>
int backward_once(int n, size_t num_per_sum, const h2x_tensor_geometry* gx, const h2x_tensor_geometry* gd,
                  const h2x_tensor_geometry* go, const void* x, const void* dy, const void* mean, const void* var,
                  const void* scale, void* dscale, void* dbias, void* dmean, void* dvar, void* dx, double eps,
                  void* ws, void* team_state, hipStream_t st,
                   const uint32_t* team_polls = nullptr)
{
    HostTensor tx, td, to;
    int c;
    size_t s;
    const int err = three_tensors<T>(n, gx, gd, go, x, dy, dx, &tx, &td, &to, &c, &s);
    if (err)
        return err;
    if constexpr (sizeof(T) == 4) // see once_geometry
    {
        OnceGeometry g;
        if (x && dy && dx && n > 0 && c > 0 && s > 0 && once_geometry(n, c, s, {&tx, &td, &to}, &g))
        {
            const OnceBackward<T> a{static_cast<const T*>(x), static_cast<const T*>(dy), static_cast<const T*>(mean),
                                    static_cast<const T*>(var), static_cast<const T*>(scale), static_cast<T*>(dscale),
                                    static_cast<T*>(dbias), static_cast<T*>(dmean), static_cast<T*>(dvar),
                                    static_cast<T*>(dx), static_cast<T>(num_per_sum),
                                    static_cast<T>(num_per_sum - 1), static_cast<T>(eps)};
            if (team_polls)
                return launch_by_teams(g, a, n, {x, dy}, dx, true, *team_polls, team_state, st) ? issued()
                                                                                                : H2X_ERR_UNSUPPORTED;
            const auto by_teams = [&] { return launch_by_teams(g, a, n, {x, dy}, dx, false, kTeamPolls, team_state, st); };
            const bool teams = teams_first(g);
            if ((teams && by_teams()) || once_launch(g, a, n, st) || (!teams && by_teams()))
                return issued();
        }
    }
    else if (x && dy && dx && n > 0 && c > 0 && s > 0)
    {
        const OnceBackward<T> a{static_cast<const T*>(x), static_cast<const T*>(dy), static_cast<const T*>(mean),
                                static_cast<const T*>(var), static_cast<const T*>(scale), static_cast<T*>(dscale),
                                static_cast<T*>(dbias), static_cast<T*>(dmean), static_cast<T*>(dvar),
                                static_cast<T*>(dx), static_cast<T>(num_per_sum),
                                static_cast<T>(num_per_sum - 1), static_cast<T>(eps)};
        if (ordered_launch(n, c, s, {&tx, &td}, to, {x, dy}, dx, a, team_state, team_polls, st))
            return issued();
    }
    if (team_polls)
        return H2X_ERR_UNSUPPORTED;
    return backward_local<T>(n, c, s, tx, td, to, num_per_sum, x, dy, mean, var, scale, dscale, dbias, dmean, dvar,
                             dx, eps, ws, st);
}

// Tensors of one haloed geometry whose outputs' halos are cleared, as whole allocations: up to 2^28
// elements.  A last vector that is not whole starts early, where the cells it shares with the vector before
// it belong to the halo (forward + backward, halo of 1, in the staged calls and so: N 7, C 601, 37 x 32 57.2 and
// 30.3 us; N 64, C 256, 7 x 7 42.7 and 11.8; N 8, C 64, 31^3 102 and 76).
// bytes: of a tensor.
int clear_geometry(const h2x_haloed_geometry* h, ClearGeometry* g, size_t* bytes)
{
    size_t real;
    const int err = real_box(h, &g->box, &real);
    if (err)
        return err;
    constexpr size_t vec = full_vec<float>();
    const int nd = h->num_dims;
    const size_t n = h->local_shape[nd - 1], c = h->local_shape[nd - 2];
    size_t interior = 1;
    for (int d = 0; d < nd - 2; ++d)
        interior *= h->local_shape[d];
    if (n == 0 || c == 0 || interior == 0 || n * c * real >= (1ull << 28) || c > 0x7fffffffull)
        return H2X_ERR_UNSUPPORTED;
    const RealBox& b = g->box;
    const size_t inside = (static_cast<size_t>(b.hi[2] - 1) * b.hr.divisor + b.hi[1] - 1) * b.wr.divisor + b.hi[0];
    if (real % vec != 0 && real - inside < vec)
        return H2X_ERR_UNSUPPORTED;
    const size_t vectors = (real + vec - 1) / vec;
    g->per_segment = make_fastdiv(static_cast<uint32_t>(vectors));
    g->last = static_cast<uint32_t>(real - vec);
    g->vectors = static_cast<uint32_t>(n * vectors);
    g->stride_n = static_cast<uint32_t>(c * real);
    g->stride_c = static_cast<int64_t>(real);
    g->num_channels = static_cast<uint32_t>(c);
    *bytes = n * c * real * sizeof(float);
    return H2X_SUCCESS;
}

// Double tensors of one haloed geometry, as the calls that leave the halo alone see them, and the halo cells of a channel.
int haloed_tensor(const h2x_haloed_geometry* h, const void* buffer, HostTensor* t, const void** interior, int* channels,
                  size_t* spatial, HaloCells* halo)
{
    RealBox box;
    size_t real;
    int err = real_box(h, &box, &real);
    if (err)
        return err;
    const int nd = h->num_dims, ns = nd - 2;
    const size_t n = h->local_shape[nd - 1], c = h->local_shape[nd - 2];
    if (n == 0 || c == 0 || c > 0x7fffffffull || n > 0x7fffffffull || n * c * real >= (1ull << 30))
        return H2X_ERR_UNSUPPORTED;
    h2x_tensor_geometry g = {};
    g.num_dims = nd;
    int64_t stride = 1, origin = 0;
    for (int d = 0; d < nd; ++d)
    {
        if (h->local_shape[d] == 0)
            return H2X_ERR_UNSUPPORTED;
        g.local_shape[d] = h->local_shape[d];
        g.strides[d] = stride;
        origin += h->lower_halo[d] * stride;
        stride *= h->real_shape[d];
    }
    *interior = static_cast<const double*>(buffer) + origin;
    err = strided_tensor<double>(&g, *interior, static_cast<int>(n), t, channels, spatial);
    if (err)
        return err;
    uint32_t local[3] = {1, 1, 1}, extent[3] = {1, 1, 1}, lo[3] = {0, 0, 0};
    for (int d = 0; d < ns; ++d)
    {
        local[d] = static_cast<uint32_t>(h->local_shape[d]);
        extent[d] = static_cast<uint32_t>(h->real_shape[d]);
        lo[d] = static_cast<uint32_t>(h->lower_halo[d]);
    }
    const uint32_t samples = static_cast<uint32_t>(n);
    halo->before = lo[0];
    halo->after = extent[0] - lo[0] - local[0];
    halo->width = local[0];
    halo->h = make_fastdiv(local[1]);
    halo->d = make_fastdiv(local[2]);
    halo->pitch = extent[0];
    halo->units = make_fastdiv((extent[0] + 1) / 2);
    halo->real_h = make_fastdiv(extent[1]);
    const uint32_t beside = extent[1] - local[1];
    halo->beside = make_fastdiv(std::max(beside, 1u));
    halo->outer = (extent[2] - local[2]) * extent[1];
    const uint32_t rows = halo->outer + local[2] * beside;
    halo->rows = make_fastdiv(std::max(rows, 1u));
    halo->lo_y = lo[1];
    halo->lo_z = lo[2];
    halo->real_plane = extent[0] * extent[1];
    halo->ends = extent[0] > local[0] ? samples * local[1] * local[2] : 0;
    halo->whole = samples * rows * halo->units.divisor;
    halo->stride_n = static_cast<uint32_t>(g.strides[nd - 1]);
    halo->origin = origin;
    return H2X_SUCCESS;
}

// A whole pass over double tensors that clears the halo, with the bits of the staged calls; H2X_ERR_UNSUPPORTED: in these.
// `inputs`, `output`: pointers of `a`, of buffers first and then of their interiors.
template <typename A>
int clearing_ordered(const h2x_haloed_geometry* h, A* a, std::initializer_list<const double**> inputs, double** output,
                     void* team_state, hipStream_t st)
{
    HostTensor in[2], out;
    HaloCells halo;
    int c;
    size_t s, k = 0;
    const void* interior;
    for (const double** p : inputs)
    {
        const int err = *p ? haloed_tensor(h, *p, &in[k++], &interior, &c, &s, &halo) : H2X_ERR_UNSUPPORTED;
        if (err)
            return err;
        *p = static_cast<const double*>(interior);
    }
    const int err = *output ? haloed_tensor(h, *output, &out, &interior, &c, &s, &halo) : H2X_ERR_UNSUPPORTED;
    if (err)
        return err;
    *output = static_cast<double*>(const_cast<void*>(interior));
    const int n = static_cast<int>(h->local_shape[h->num_dims - 1]);
    bool launched;
    if constexpr (std::is_same<A, OnceForward<double>>::value)
        launched = ordered_launch(n, c, s, {&in[0]}, out, {a->x}, a->y, *a, team_state, nullptr, st, &halo);
    else
        launched = ordered_launch(n, c, s, {&in[0], &in[1]}, out, {a->x, a->dy}, a->dx, *a, team_state, nullptr, st, &halo);
    return launched ? issued() : H2X_ERR_UNSUPPORTED;
}

// The same for such tensors, by one workgroup or a team a channel; H2X_ERR_UNSUPPORTED: in the
// staged calls.
template <typename A>
int clearing_once(const h2x_haloed_geometry* h, const A& a, std::initializer_list<const void*> inputs, void* output,
                  void* team_state, hipStream_t st)
{
    ClearGeometry g;
    size_t bytes;
    const int err = clear_geometry(h, &g, &bytes);
    if (err)
        return err;
    bool fit = aligned16(output) && output;
    for (const void* p : inputs)
        fit = fit && p && aligned16(p);
    if (!fit)
        return H2X_ERR_UNSUPPORTED;
    const auto by_teams = [&] {
        return launch_by_teams(g, a, bytes, true, inputs, output, false, kTeamPolls, team_state, st);
    };
    const bool teams = teams_first(g);
    if ((teams && by_teams()) || once_launch<true>(g, a, st) || (!teams && by_teams()))
        return issued();
    return H2X_ERR_UNSUPPORTED;
}

} // namespace

namespace bn
{
LaunchLog* install_launch_log(LaunchLog* log)
{
    LaunchLog* before = t_launch_log;
    t_launch_log = log;
    return before;
}
} // namespace bn
} // namespace h2x

using namespace h2x;

#define H2X_BY_DTYPE(dtype, CALL_F32, CALL_F64)                                                    \
    switch (dtype)                                                                                 \
    {                                                                                              \
    case H2X_F32: return CALL_F32;                                                                 \
    case H2X_F64: return CALL_F64;                                                                 \
    }                                                                                              \
    return H2X_ERR_UNSUPPORTED

extern "C" size_t h2x_bn_workspace_bytes(int num_channels)
{
    if (num_channels <= 0)
        return 256;
    return (partials_bytes(num_channels) + 255) / 256 * 256;
}

extern "C" int h2x_bn_channel_sums_and_sqsums(h2x_dtype dtype, int num_samples, int num_channels,
                                              size_t spatial_size, size_t spatial_real_size,
                                              const void* x, void* sums, void* sqsums,
                                              void* workspace, h2x_stream_t stream)
{
    if (bad_geometry(num_samples, num_channels, spatial_size, spatial_real_size) || !sums || !sqsums
        || !workspace || (!x && num_samples > 0 && spatial_size > 0 && num_channels > 0))
        return H2X_ERR_INVALID_ARGUMENT;
    H2X_BY_DTYPE(dtype,
                 sums_dense<float>(num_samples, num_channels, spatial_size, spatial_real_size, x, sums,
                                   sqsums, workspace, as_stream(stream)),
                 sums_dense<double>(num_samples, num_channels, spatial_size, spatial_real_size, x,
                                    sums, sqsums, workspace, as_stream(stream)));
}

extern "C" size_t h2x_bn_static_max_channels(void)
{
    // largest channel count whose partial sums fit in the scratch array
    int lo = 0, hi = 65535;
    while (lo < hi)
    {
        const int mid = (lo + hi + 1) / 2;
        if (h2x_bn_workspace_bytes(mid) <= kStaticScratchBytes)
            lo = mid;
        else
            hi = mid - 1;
    }
    return static_cast<size_t>(lo);
}

extern "C" int h2x_bn_channel_sums_and_sqsums_static(h2x_dtype dtype, int num_samples,
                                                     int num_channels, size_t spatial_size,
                                                     size_t spatial_real_size, const void* x,
                                                     void* sums, void* sqsums, h2x_stream_t stream)
{
    if (num_channels > 0 && h2x_bn_workspace_bytes(num_channels) > kStaticScratchBytes)
        return H2X_ERR_SCRATCH_LIMIT;
    void* workspace = nullptr;
    const int err = static_scratch(&workspace);
    if (err != 0)
        return err;
    // The partial sums need no clearing: every slot the finishing kernel reads
    // is written by this call's reduction kernel first.
    return h2x_bn_channel_sums_and_sqsums(dtype, num_samples, num_channels, spatial_size,
                                          spatial_real_size, x, sums, sqsums, workspace, stream);
}

extern "C" int h2x_bn_channel_sums_and_sqsums_strided(h2x_dtype dtype, int num_samples,
                                                      const h2x_tensor_geometry* x_geometry,
                                                      const void* x, void* sums, void* sqsums,
                                                      void* workspace, h2x_stream_t stream)
{
    if (num_samples < 0 || !x_geometry || !sums || !sqsums || !workspace)
        return H2X_ERR_INVALID_ARGUMENT;
    H2X_BY_DTYPE(dtype,
                 sums_strided<float>(num_samples, x_geometry, x, sums, sqsums, workspace,
                                     as_stream(stream)),
                 sums_strided<double>(num_samples, x_geometry, x, sums, sqsums, workspace,
                                      as_stream(stream)));
}

extern "C" int h2x_bn_sums_to_statistics(h2x_dtype dtype, int num_channels, size_t num_per_sum,
                                         double decay, void* mean_inout, void* var_inout,
                                         void* running_mean, void* running_var,
                                         h2x_stream_t stream)
{
    if (num_channels < 0 || !mean_inout || !var_inout || !running_mean || !running_var)
        return H2X_ERR_INVALID_ARGUMENT;
    H2X_BY_DTYPE(dtype,
                 statistics_impl<float>(num_channels, num_per_sum, decay, mean_inout, var_inout,
                                        running_mean, running_var, as_stream(stream)),
                 statistics_impl<double>(num_channels, num_per_sum, decay, mean_inout, var_inout,
                                         running_mean, running_var, as_stream(stream)));
}

extern "C" int h2x_bn_batch_normalization(h2x_dtype dtype, int num_samples, int num_channels,
                                          size_t spatial_size, size_t x_spatial_real_size,
                                          size_t y_spatial_real_size, const void* x,
                                          const void* mean, const void* var, const void* scale,
                                          const void* bias, void* y, double epsilon,
                                          h2x_stream_t stream)
{
    if (bad_geometry(num_samples, num_channels, spatial_size, x_spatial_real_size)
        || y_spatial_real_size < spatial_size || !mean || !var || !scale || !bias)
        return H2X_ERR_INVALID_ARGUMENT;
    if ((!x || !y) && static_cast<size_t>(num_samples) * num_channels * spatial_size > 0)
        return H2X_ERR_INVALID_ARGUMENT;
    const int n = num_samples, c = num_channels;
    const size_t s = spatial_size;
    H2X_BY_DTYPE(dtype,
                 apply_impl<float>(n, c, s, dense_tensor<float>(x, c, s, x_spatial_real_size),
                                   dense_tensor<float>(y, c, s, y_spatial_real_size), x, mean, var,
                                   scale, bias, y, epsilon, as_stream(stream)),
                 apply_impl<double>(n, c, s, dense_tensor<double>(x, c, s, x_spatial_real_size),
                                    dense_tensor<double>(y, c, s, y_spatial_real_size), x, mean, var,
                                    scale, bias, y, epsilon, as_stream(stream)));
}

extern "C" int h2x_bn_batch_normalization_strided(h2x_dtype dtype, int num_samples,
                                                  const h2x_tensor_geometry* x_geometry,
                                                  const h2x_tensor_geometry* y_geometry,
                                                  const void* x, const void* mean, const void* var,
                                                  const void* scale, const void* bias, void* y,
                                                  double epsilon, h2x_stream_t stream)
{
    if (num_samples < 0 || !x_geometry || !y_geometry || !mean || !var || !scale || !bias)
        return H2X_ERR_INVALID_ARGUMENT;
    H2X_BY_DTYPE(dtype,
                 apply_strided<float>(num_samples, x_geometry, y_geometry, x, mean, var, scale, bias,
                                      y, epsilon, as_stream(stream)),
                 apply_strided<double>(num_samples, x_geometry, y_geometry, x, mean, var, scale,
                                       bias, y, epsilon, as_stream(stream)));
}

extern "C" int h2x_bn_backprop1(h2x_dtype dtype, int num_samples, int num_channels,
                                size_t spatial_size, size_t x_spatial_real_size,
                                size_t dy_spatial_real_size, const void* x, const void* dy,
                                const void* mean, const void* var, const void* scale, void* dscale,
                                void* dbias, void* dmean, void* dvar, double epsilon,
                                void* workspace, h2x_stream_t stream)
{
    if (bad_geometry(num_samples, num_channels, spatial_size, x_spatial_real_size)
        || dy_spatial_real_size < spatial_size || !mean || !var || !scale || !dscale || !dbias
        || !dmean || !dvar || !workspace)
        return H2X_ERR_INVALID_ARGUMENT;
    if ((!x || !dy) && static_cast<size_t>(num_samples) * num_channels * spatial_size > 0)
        return H2X_ERR_INVALID_ARGUMENT;
    const int n = num_samples, c = num_channels;
    const size_t s = spatial_size;
    H2X_BY_DTYPE(dtype,
                 backprop1_impl<float>(n, c, s, dense_tensor<float>(x, c, s, x_spatial_real_size),
                                       dense_tensor<float>(dy, c, s, dy_spatial_real_size), x, dy,
                                       mean, var, scale, dscale, dbias, dmean, dvar, epsilon,
                                       workspace, as_stream(stream)),
                 backprop1_impl<double>(n, c, s, dense_tensor<double>(x, c, s, x_spatial_real_size),
                                        dense_tensor<double>(dy, c, s, dy_spatial_real_size), x, dy,
                                        mean, var, scale, dscale, dbias, dmean, dvar, epsilon,
                                        workspace, as_stream(stream)));
}

extern "C" int h2x_bn_backprop1_strided(h2x_dtype dtype, int num_samples,
                                        const h2x_tensor_geometry* x_geometry,
                                        const h2x_tensor_geometry* dy_geometry, const void* x,
                                        const void* dy, const void* mean, const void* var,
                                        const void* scale, void* dscale, void* dbias, void* dmean,
                                        void* dvar, double epsilon, void* workspace,
                                        h2x_stream_t stream)
{
    if (num_samples < 0 || !x_geometry || !dy_geometry || !mean || !var || !scale || !dscale
        || !dbias || !dmean || !dvar || !workspace)
        return H2X_ERR_INVALID_ARGUMENT;
    H2X_BY_DTYPE(dtype,
                 backprop1_strided<float>(num_samples, x_geometry, dy_geometry, x, dy, mean, var,
                                          scale, dscale, dbias, dmean, dvar, epsilon, workspace,
                                          as_stream(stream)),
                 backprop1_strided<double>(num_samples, x_geometry, dy_geometry, x, dy, mean, var,
                                           scale, dscale, dbias, dmean, dvar, epsilon, workspace,
                                           as_stream(stream)));
}

extern "C" int h2x_bn_backprop2(h2x_dtype dtype, int num_samples, int num_channels,
                                size_t spatial_size, size_t x_spatial_real_size,
                                size_t dy_spatial_real_size, size_t dx_spatial_real_size,
                                size_t num_per_sum, const void* x, const void* dy,
                                const void* mean, const void* var, const void* scale,
                                const void* dmean, const void* dvar, void* dx, double epsilon,
                                h2x_stream_t stream)
{
    if (bad_geometry(num_samples, num_channels, spatial_size, x_spatial_real_size)
        || dy_spatial_real_size < spatial_size || dx_spatial_real_size < spatial_size || !mean
        || !var || !scale || !dmean || !dvar)
        return H2X_ERR_INVALID_ARGUMENT;
    if ((!x || !dy || !dx) && static_cast<size_t>(num_samples) * num_channels * spatial_size > 0)
        return H2X_ERR_INVALID_ARGUMENT;
    const int n = num_samples, c = num_channels;
    const size_t s = spatial_size;
    H2X_BY_DTYPE(dtype,
                 backprop2_impl<float>(n, c, s, num_per_sum,
                                       dense_tensor<float>(x, c, s, x_spatial_real_size),
                                       dense_tensor<float>(dy, c, s, dy_spatial_real_size),
                                       dense_tensor<float>(dx, c, s, dx_spatial_real_size), x, dy,
                                       mean, var, scale, dmean, dvar, dx, epsilon, as_stream(stream)),
                 backprop2_impl<double>(n, c, s, num_per_sum,
                                        dense_tensor<double>(x, c, s, x_spatial_real_size),
                                        dense_tensor<double>(dy, c, s, dy_spatial_real_size),
                                        dense_tensor<double>(dx, c, s, dx_spatial_real_size), x, dy,
                                        mean, var, scale, dmean, dvar, dx, epsilon,
                                        as_stream(stream)));
}

extern "C" int h2x_bn_backprop2_strided(h2x_dtype dtype, int num_samples, size_t num_per_sum,
                                        const h2x_tensor_geometry* x_geometry,
                                        const h2x_tensor_geometry* dy_geometry,
                                        const h2x_tensor_geometry* dx_geometry, const void* x,
                                        const void* dy, const void* mean, const void* var,
                                        const void* scale, const void* dmean, const void* dvar,
                                        void* dx, double epsilon, h2x_stream_t stream)
{
    if (num_samples < 0 || !x_geometry || !dy_geometry || !dx_geometry || !mean || !var || !scale
        || !dmean || !dvar)
        return H2X_ERR_INVALID_ARGUMENT;
    H2X_BY_DTYPE(dtype,
                 backprop2_strided<float>(num_samples, num_per_sum, x_geometry, dy_geometry,
                                          dx_geometry, x, dy, mean, var, scale, dmean, dvar, dx,
                                          epsilon, as_stream(stream)),
                 backprop2_strided<double>(num_samples, num_per_sum, x_geometry, dy_geometry,
                                           dx_geometry, x, dy, mean, var, scale, dmean, dvar, dx,
                                           epsilon, as_stream(stream)));
}

extern "C" int h2x_bn_batch_normalization_clearing(h2x_dtype dtype,
                                                   const h2x_haloed_geometry* geometry,
                                                   const void* x_buffer, const void* mean,
                                                   const void* var, const void* scale,
                                                   const void* bias, void* y_buffer, double epsilon,
                                                   h2x_stream_t stream)
{
    if (!geometry || !mean || !var || !scale || !bias)
        return H2X_ERR_INVALID_ARGUMENT;
    H2X_BY_DTYPE(dtype,
                 clearing_impl<float>(false, 0, geometry, x_buffer, nullptr, mean, var, scale, bias,
                                      nullptr, nullptr, y_buffer, epsilon, as_stream(stream)),
                 clearing_impl<double>(false, 0, geometry, x_buffer, nullptr, mean, var, scale, bias,
                                       nullptr, nullptr, y_buffer, epsilon, as_stream(stream)));
}

extern "C" int h2x_bn_backprop2_clearing(h2x_dtype dtype, size_t num_per_sum,
                                         const h2x_haloed_geometry* geometry, const void* x_buffer,
                                         const void* dy_buffer, const void* mean, const void* var,
                                         const void* scale, const void* dmean, const void* dvar,
                                         void* dx_buffer, double epsilon, h2x_stream_t stream)
{
    if (!geometry || !mean || !var || !scale || !dmean || !dvar)
        return H2X_ERR_INVALID_ARGUMENT;
    H2X_BY_DTYPE(dtype,
                 clearing_impl<float>(true, num_per_sum, geometry, x_buffer, dy_buffer, mean, var,
                                      scale, nullptr, dmean, dvar, dx_buffer, epsilon,
                                      as_stream(stream)),
                 clearing_impl<double>(true, num_per_sum, geometry, x_buffer, dy_buffer, mean, var,
                                       scale, nullptr, dmean, dvar, dx_buffer, epsilon,
                                       as_stream(stream)));
}

extern "C" int h2x_bn_forward_local(h2x_dtype dtype, int num_samples, int num_channels,
                                    size_t spatial_size, size_t x_spatial_real_size,
                                    size_t y_spatial_real_size, const void* x, const void* scale,
                                    const void* bias, size_t num_per_sum, double decay,
                                    double epsilon, void* mean, void* var, void* running_mean,
                                    void* running_var, void* y, void* workspace,
                                    h2x_stream_t stream)
{
    if (bad_geometry(num_samples, num_channels, spatial_size, x_spatial_real_size)
        || y_spatial_real_size < spatial_size || !scale || !bias || !mean || !var || !running_mean
        || !running_var || !workspace)
        return H2X_ERR_INVALID_ARGUMENT;
    if ((!x || !y) && static_cast<size_t>(num_samples) * num_channels * spatial_size > 0)
        return H2X_ERR_INVALID_ARGUMENT;
    H2X_BY_DTYPE(dtype,
                 forward_local<float>(
                     num_samples, num_channels, spatial_size,
                     dense_tensor<float>(x, num_channels, spatial_size, x_spatial_real_size),
                     dense_tensor<float>(y, num_channels, spatial_size, y_spatial_real_size), x, scale,
                     bias, num_per_sum, decay, epsilon, mean, var, running_mean, running_var, y,
                     workspace, as_stream(stream)),
                 forward_local<double>(
                     num_samples, num_channels, spatial_size,
                     dense_tensor<double>(x, num_channels, spatial_size, x_spatial_real_size),
                     dense_tensor<double>(y, num_channels, spatial_size, y_spatial_real_size), x, scale,
                     bias, num_per_sum, decay, epsilon, mean, var, running_mean, running_var, y,
                     workspace, as_stream(stream)));
}

extern "C" int h2x_bn_forward_local_strided(h2x_dtype dtype, int num_samples,
                                            const h2x_tensor_geometry* x_geometry,
                                            const h2x_tensor_geometry* y_geometry, const void* x,
                                            const void* scale, const void* bias, size_t num_per_sum,
                                            double decay, double epsilon, void* mean, void* var,
                                            void* running_mean, void* running_var, void* y,
                                            void* workspace, h2x_stream_t stream)
{
    if (num_samples < 0 || !x_geometry || !y_geometry || !scale || !bias || !mean || !var
        || !running_mean || !running_var || !workspace)
        return H2X_ERR_INVALID_ARGUMENT;
    H2X_BY_DTYPE(dtype,
                 forward_local_strided<float>(num_samples, x_geometry, y_geometry, x, scale, bias,
                                              num_per_sum, decay, epsilon, mean, var, running_mean,
                                              running_var, y, workspace, as_stream(stream)),
                 forward_local_strided<double>(num_samples, x_geometry, y_geometry, x, scale, bias,
                                               num_per_sum, decay, epsilon, mean, var, running_mean,
                                               running_var, y, workspace, as_stream(stream)));
}

extern "C" int h2x_bn_backward_local(h2x_dtype dtype, int num_samples, int num_channels,
                                     size_t spatial_size, size_t x_spatial_real_size,
                                     size_t dy_spatial_real_size, size_t dx_spatial_real_size,
                                     size_t num_per_sum, const void* x, const void* dy,
                                     const void* mean, const void* var, const void* scale,
                                     void* dscale, void* dbias, void* dmean, void* dvar, void* dx,
                                     double epsilon, void* workspace, h2x_stream_t stream)
{
    if (bad_geometry(num_samples, num_channels, spatial_size, x_spatial_real_size)
        || dy_spatial_real_size < spatial_size || dx_spatial_real_size < spatial_size || !mean
        || !var || !scale || !dscale || !dbias || !dmean || !dvar || !workspace)
        return H2X_ERR_INVALID_ARGUMENT;
    if ((!x || !dy || !dx) && static_cast<size_t>(num_samples) * num_channels * spatial_size > 0)
        return H2X_ERR_INVALID_ARGUMENT;
    H2X_BY_DTYPE(dtype,
                 backward_local<float>(
                     num_samples, num_channels, spatial_size,
                     dense_tensor<float>(x, num_channels, spatial_size, x_spatial_real_size),
                     dense_tensor<float>(dy, num_channels, spatial_size, dy_spatial_real_size),
                     dense_tensor<float>(dx, num_channels, spatial_size, dx_spatial_real_size),
                     num_per_sum, x, dy, mean, var, scale, dscale, dbias, dmean, dvar, dx, epsilon,
                     workspace, as_stream(stream)),
                 backward_local<double>(
                     num_samples, num_channels, spatial_size,
                     dense_tensor<double>(x, num_channels, spatial_size, x_spatial_real_size),
                     dense_tensor<double>(dy, num_channels, spatial_size, dy_spatial_real_size),
                     dense_tensor<double>(dx, num_channels, spatial_size, dx_spatial_real_size),
                     num_per_sum, x, dy, mean, var, scale, dscale, dbias, dmean, dvar, dx, epsilon,
                     workspace, as_stream(stream)));
}

extern "C" int h2x_bn_backward_local_strided(h2x_dtype dtype, int num_samples, size_t num_per_sum,
                                             const h2x_tensor_geometry* x_geometry,
                                             const h2x_tensor_geometry* dy_geometry,
                                             const h2x_tensor_geometry* dx_geometry, const void* x,
                                             const void* dy, const void* mean, const void* var,
                                             const void* scale, void* dscale, void* dbias,
                                             void* dmean, void* dvar, void* dx, double epsilon,
                                             void* workspace, h2x_stream_t stream)
{
    if (num_samples < 0 || !x_geometry || !dy_geometry || !dx_geometry || !mean || !var || !scale
        || !dscale || !dbias || !dmean || !dvar || !workspace)
        return H2X_ERR_INVALID_ARGUMENT;
    H2X_BY_DTYPE(dtype,
                 backward_local_strided<float>(num_samples, num_per_sum, x_geometry, dy_geometry,
                                               dx_geometry, x, dy, mean, var, scale, dscale, dbias,
                                               dmean, dvar, dx, epsilon, workspace, as_stream(stream)),
                 backward_local_strided<double>(num_samples, num_per_sum, x_geometry, dy_geometry,
                                                dx_geometry, x, dy, mean, var, scale, dscale, dbias,
                                                dmean, dvar, dx, epsilon, workspace,
                                                as_stream(stream)));
}

extern "C" size_t h2x_bn_team_state_bytes(int num_channels)
{
    return team_state_at(std::max(num_channels, 1)) * sizeof(unsigned long long);
}

extern "C" size_t h2x_bn_team_state_needed(h2x_dtype dtype, int num_samples, const h2x_tensor_geometry* geometry)
{
    HostTensor t;
    OnceGeometry g;
    int c;
    size_t s;
    // (an address: only its alignment is looked at, and that decides nothing here)
    if (dtype != H2X_F32 || num_samples <= 0 || !geometry
        || strided_tensor<float>(geometry, geometry, num_samples, &t, &c, &s) || c <= 0 || s == 0
        || !once_geometry(num_samples, c, s, {&t}, &g) || !for_teams(g, num_samples))
        return 0;
    return team_state_needed(g);
}

extern "C" size_t h2x_bn_ordered_state_needed(int num_samples, const h2x_tensor_geometry* geometry)
{
    HostTensor t;
    OrderedGeometry g;
    int c;
    size_t s;
    bool rows, forward = false, backward = false;
    // the address counts by its alignment: as of tensors made by an allocator
    const void* const aligned = reinterpret_cast<const void*>(uintptr_t(256));
    if (num_samples <= 0 || !geometry || strided_tensor<double>(geometry, aligned, num_samples, &t, &c, &s) || c <= 0 || s == 0)
        return 0;
    const size_t moved = moved_bytes(t, num_samples, c, s);
    const OnceForward<double>* const f = nullptr;
    const OnceBackward<double>* const b = nullptr;
    const uint32_t most = most_members();
    forward = ordered_geometry(num_samples, c, s, {&t}, t, &g, &rows)
              && ordered_variant(g, f, moved, rows, true, most, false, nullptr, nullptr, &forward) && forward;
    backward = ordered_geometry(num_samples, c, s, {&t, &t}, t, &g, &rows)
               && ordered_variant(g, b, moved, rows, true, most, false, nullptr, nullptr, &backward) && backward;
    return forward || backward ? h2x_bn_team_state_bytes(c) : 0;
}

extern "C" size_t h2x_bn_team_state_needed_clearing(h2x_dtype dtype, const h2x_haloed_geometry* geometry)
{
    ClearGeometry g;
    size_t bytes;
    if (dtype != H2X_F32 || !geometry || clear_geometry(geometry, &g, &bytes))
        return 0;
    return team_state_needed(g);
}

extern "C" int h2x_bn_forward_once(h2x_dtype dtype, int num_samples,
                                            const h2x_tensor_geometry* x_geometry,
                                            const h2x_tensor_geometry* y_geometry, const void* x,
                                            const void* scale, const void* bias, size_t num_per_sum,
                                            double decay, double epsilon, void* mean, void* var,
                                            void* running_mean, void* running_var, void* y,
                                            void* workspace, void* team_state, h2x_stream_t stream)
{
    if (num_samples < 0 || !x_geometry || !y_geometry || !scale || !bias || !mean || !var
        || !running_mean || !running_var || !workspace)
        return H2X_ERR_INVALID_ARGUMENT;
    H2X_BY_DTYPE(dtype,
                 forward_once<float>(num_samples, x_geometry, y_geometry, x, scale, bias,
                                              num_per_sum, decay, epsilon, mean, var, running_mean,
                                              running_var, y, workspace, team_state, as_stream(stream)),
                 forward_once<double>(num_samples, x_geometry, y_geometry, x, scale, bias,
                                               num_per_sum, decay, epsilon, mean, var, running_mean,
                                               running_var, y, workspace, team_state, as_stream(stream)));
}

extern "C" int h2x_bn_backward_once(h2x_dtype dtype, int num_samples, size_t num_per_sum,
                                             const h2x_tensor_geometry* x_geometry,
                                             const h2x_tensor_geometry* dy_geometry,
                                             const h2x_tensor_geometry* dx_geometry, const void* x,
                                             const void* dy, const void* mean, const void* var,
                                             const void* scale, void* dscale, void* dbias,
                                             void* dmean, void* dvar, void* dx, double epsilon,
                                             void* workspace, void* team_state, h2x_stream_t stream)
{
    if (num_samples < 0 || !x_geometry || !dy_geometry || !dx_geometry || !mean || !var || !scale
        || !dscale || !dbias || !dmean || !dvar || !workspace)
        return H2X_ERR_INVALID_ARGUMENT;
    H2X_BY_DTYPE(dtype,
                 backward_once<float>(num_samples, num_per_sum, x_geometry, dy_geometry,
                                               dx_geometry, x, dy, mean, var, scale, dscale, dbias,
                                               dmean, dvar, dx, epsilon, workspace, team_state, as_stream(stream)),
                 backward_once<double>(num_samples, num_per_sum, x_geometry, dy_geometry,
                                                dx_geometry, x, dy, mean, var, scale, dscale, dbias,
                                                dmean, dvar, dx, epsilon, workspace, team_state,
                                                as_stream(stream)));
}

extern "C" int h2x_bn_forward_team(h2x_dtype dtype, int num_samples, const h2x_tensor_geometry* x_geometry,
                                   const h2x_tensor_geometry* y_geometry, const void* x, const void* scale,
                                   const void* bias, size_t num_per_sum, double decay, double epsilon, void* mean,
                                   void* var, void* running_mean, void* running_var, void* y, void* team_state,
                                   unsigned int max_polls, h2x_stream_t stream)
{
    if (num_samples < 0 || !x_geometry || !y_geometry || !scale || !bias || !mean || !var || !running_mean
        || !running_var || !team_state)
        return H2X_ERR_INVALID_ARGUMENT;
    H2X_BY_DTYPE(dtype,
                 forward_once<float>(num_samples, x_geometry, y_geometry, x, scale, bias, num_per_sum, decay, epsilon,
                                     mean, var, running_mean, running_var, y, nullptr, team_state, as_stream(stream), &max_polls),
                 forward_once<double>(num_samples, x_geometry, y_geometry, x, scale, bias, num_per_sum, decay, epsilon,
                                      mean, var, running_mean, running_var, y, nullptr, team_state, as_stream(stream),
                                      &max_polls));
}

extern "C" int h2x_bn_backward_team(h2x_dtype dtype, int num_samples, size_t num_per_sum,
                                    const h2x_tensor_geometry* x_geometry, const h2x_tensor_geometry* dy_geometry,
                                    const h2x_tensor_geometry* dx_geometry, const void* x, const void* dy,
                                    const void* mean, const void* var, const void* scale, void* dscale, void* dbias,
                                    void* dmean, void* dvar, void* dx, double epsilon, void* team_state,
                                    unsigned int max_polls, h2x_stream_t stream)
{
    if (num_samples < 0 || !x_geometry || !dy_geometry || !dx_geometry || !mean || !var || !scale || !dscale || !dbias
        || !dmean || !dvar || !team_state)
        return H2X_ERR_INVALID_ARGUMENT;
    H2X_BY_DTYPE(dtype,
                 backward_once<float>(num_samples, num_per_sum, x_geometry, dy_geometry, dx_geometry, x, dy, mean, var,
                                      scale, dscale, dbias, dmean, dvar, dx, epsilon, nullptr, team_state, as_stream(stream),
                                      &max_polls),
                 backward_once<double>(num_samples, num_per_sum, x_geometry, dy_geometry, dx_geometry, x, dy, mean, var,
                                       scale, dscale, dbias, dmean, dvar, dx, epsilon, nullptr, team_state, as_stream(stream),
                                       &max_polls));
}

extern "C" int h2x_bn_forward_clearing(h2x_dtype dtype, const h2x_haloed_geometry* geometry, const void* x_buffer,
                                       const void* scale, const void* bias, size_t num_per_sum, double decay,
                                       double epsilon, void* mean, void* var, void* running_mean, void* running_var,
                                       void* y_buffer, void* team_state, h2x_stream_t stream)
{
    if (!geometry || !scale || !bias || !mean || !var || !running_mean || !running_var)
        return H2X_ERR_INVALID_ARGUMENT;
    if ((dtype != H2X_F32 && dtype != H2X_F64) || num_per_sum == 0)
        return H2X_ERR_UNSUPPORTED;
    if (dtype == H2X_F64)
    {
        typedef double T;
        OnceForward<T> a{static_cast<const T*>(x_buffer), static_cast<const T*>(scale), static_cast<const T*>(bias),
                         static_cast<T*>(mean), static_cast<T*>(var), static_cast<T*>(running_mean),
                         static_cast<T*>(running_var), static_cast<T*>(y_buffer), static_cast<T>(num_per_sum),
                         static_cast<T>(decay), static_cast<T>(epsilon)};
        return clearing_ordered(geometry, &a, {&a.x}, &a.y, team_state, as_stream(stream));
    }
    typedef float T;
    const OnceForward<T> a{static_cast<const T*>(x_buffer), static_cast<const T*>(scale), static_cast<const T*>(bias),
                           static_cast<T*>(mean), static_cast<T*>(var), static_cast<T*>(running_mean),
                           static_cast<T*>(running_var), static_cast<T*>(y_buffer), static_cast<T>(num_per_sum),
                           static_cast<T>(decay), static_cast<T>(epsilon)};
    return clearing_once(geometry, a, {x_buffer}, y_buffer, team_state, as_stream(stream));
}

extern "C" int h2x_bn_backward_clearing(h2x_dtype dtype, size_t num_per_sum, const h2x_haloed_geometry* geometry,
                                        const void* x_buffer, const void* dy_buffer, const void* mean,
                                        const void* var, const void* scale, void* dscale, void* dbias, void* dmean,
                                        void* dvar, void* dx_buffer, double epsilon, void* team_state,
                                        h2x_stream_t stream)
{
    if (!geometry || !mean || !var || !scale || !dscale || !dbias || !dmean || !dvar)
        return H2X_ERR_INVALID_ARGUMENT;
    if (dtype == H2X_F64)
    {
        typedef double T;
        OnceBackward<T> a{static_cast<const T*>(x_buffer), static_cast<const T*>(dy_buffer),
                          static_cast<const T*>(mean), static_cast<const T*>(var), static_cast<const T*>(scale),
                          static_cast<T*>(dscale), static_cast<T*>(dbias), static_cast<T*>(dmean),
                          static_cast<T*>(dvar), static_cast<T*>(dx_buffer), static_cast<T>(num_per_sum),
                          static_cast<T>(num_per_sum - 1), static_cast<T>(epsilon)};
        return clearing_ordered(geometry, &a, {&a.x, &a.dy}, &a.dx, team_state, as_stream(stream));
    }
    if (dtype != H2X_F32)
        return H2X_ERR_UNSUPPORTED;
    typedef float T;
    const OnceBackward<T> a{static_cast<const T*>(x_buffer), static_cast<const T*>(dy_buffer),
                            static_cast<const T*>(mean), static_cast<const T*>(var), static_cast<const T*>(scale),
                            static_cast<T*>(dscale), static_cast<T*>(dbias), static_cast<T*>(dmean),
                            static_cast<T*>(dvar), static_cast<T*>(dx_buffer), static_cast<T>(num_per_sum),
                            static_cast<T>(num_per_sum - 1), static_cast<T>(epsilon)};
    return clearing_once(geometry, a, {x_buffer, dy_buffer}, dx_buffer, team_state, as_stream(stream));
}

// Plays on the host which elements the workgroups that hold channels in registers touch.
extern "C" int h2x_bn_audit_once(int num_samples, const h2x_tensor_geometry* geometry, unsigned int member_vectors,
                                 unsigned char* counted, unsigned char* stored, size_t elements)
{
    if (!geometry || !counted || !stored)
        return H2X_ERR_INVALID_ARGUMENT;
    HostTensor t;
    int c;
    size_t s;
    const int err = strided_tensor<float>(geometry, counted, num_samples, &t, &c, &s);
    if (err)
        return err;
    OnceGeometry g;
    if (num_samples <= 0 || c <= 0 || s == 0 || !once_geometry(num_samples, c, s, {&t}, &g))
        return H2X_ERR_UNSUPPORTED;
    constexpr int VEC = full_vec<float>();
    const uint32_t span = member_vectors ? member_vectors : g.vectors;
    for (uint32_t ch = 0; ch < g.num_channels; ++ch)
        for (uint32_t first = 0; first < g.vectors; first += span)
            for (uint32_t i = first; i < std::min(first + span, g.vectors); ++i)
            {
                const uint32_t at = once_place<VEC>(g, i);
                const size_t e = static_cast<size_t>(ch * g.stride_c) + OnceGeometry::offset(at);
                if (e + VEC > elements)
                    return H2X_ERR_INVALID_ARGUMENT;
                for (int j = 0; j < VEC; ++j)
                {
                    stored[e + j] = 1;
                    counted[e + j] += OnceGeometry::counts(at, j);
                }
            }
    return H2X_SUCCESS;
}

// Plays on the host which elements the workgroups that keep the staged order touch.
extern "C" int h2x_bn_audit_ordered(int num_samples, const h2x_tensor_geometry* geometry, int backward,
                                    unsigned int passes, unsigned char* counted, unsigned char* stored,
                                    unsigned short* group, size_t elements)
{
    if (!geometry || !counted || !stored || !group || passes == 0)
        return H2X_ERR_INVALID_ARGUMENT;
    HostTensor t;
    OrderedGeometry g;
    int c;
    size_t s;
    bool rows;
    // (as of tensors made by an allocator)
    const int err = strided_tensor<double>(geometry, reinterpret_cast<const void*>(uintptr_t(256)), num_samples, &t, &c, &s);
    if (err)
        return err;
    if (num_samples <= 0 || c <= 0 || s == 0
        || !(backward ? ordered_geometry(num_samples, c, s, {&t, &t}, t, &g, &rows)
                      : ordered_geometry(num_samples, c, s, {&t}, t, &g, &rows)))
        return H2X_ERR_UNSUPPORTED;
    constexpr int kTeam = 2 * kBlockSize;
    g.passes = passes;
    const uint32_t members = (g.groups + 2 * passes - 1) / (2 * passes);
    for (uint32_t ch = 0; ch < g.num_channels; ++ch)
        for (uint32_t i = 0; i < members; ++i)
            for (uint32_t p = 0; p < passes; ++p)
                for (uint32_t thread = 0; thread < kTeam; ++thread)
                    for (uint32_t u = 0; u < g.group_batches.divisor * kOrderedBatch; ++u)
                    {
                        const uint32_t k = ordered_group<kTeam>(g, team_member(i, members), p, thread / kBlockSize);
                        const uint32_t b = u / kOrderedBatch, j = u % kOrderedBatch, th = thread % kBlockSize;
                        const uint32_t at = rows ? ordered_place<true>(g, k, b, j, th) : ordered_place<false>(g, k, b, j, th);
                        if (at == kNowhere)
                            continue;
                        const size_t e = static_cast<size_t>(ch * g.map.stride_c) + (at >> 1);
                        if (e + 2 > elements)
                            return H2X_ERR_INVALID_ARGUMENT;
                        for (uint32_t v = 0; v < 2; ++v)
                        {
                            stored[e + v] = 1;
                            if (v < (at & 1))
                                continue;
                            ++counted[e + v];
                            group[e + v] = static_cast<unsigned short>(k + 1);
                        }
                    }
    return H2X_SUCCESS;
}

// Plays on the host which elements the workgroups that hold short segments of doubles touch.
extern "C" int h2x_bn_audit_short(int num_samples, const h2x_tensor_geometry* geometry, int backward, unsigned int threads,
                                  unsigned int vectors, unsigned char* counted, unsigned char* stored, unsigned short* range,
                                  size_t elements)
{
    if (!geometry || !counted || !stored || !range)
        return H2X_ERR_INVALID_ARGUMENT;
    HostTensor t;
    ShortOnceGeometry g;
    int c;
    size_t s;
    const int err = strided_tensor<double>(geometry, reinterpret_cast<const void*>(uintptr_t(256)), num_samples, &t, &c, &s);
    if (err)
        return err;
    if (num_samples <= 0 || c <= 0 || s == 0
        || !(backward ? short_once_geometry(num_samples, c, s, {&t, &t}, t, &g) : short_once_geometry(num_samples, c, s, {&t}, t, &g)))
        return H2X_ERR_UNSUPPORTED;
    const auto same = [&](auto w) { return decltype(w)::threads == threads && decltype(w)::vectors == vectors; };
    if (!(backward ? any_short_workgroup<false>(same) : any_short_workgroup<true>(same)))
        return H2X_ERR_INVALID_ARGUMENT;
    const uint32_t windows = short_once_windows(&g, threads, vectors, short_once_passes(vectors, !backward)), vec = g.row == 1 ? 1 : 2;
    if (windows == 0)
        return H2X_ERR_UNSUPPORTED;
    for (uint32_t w = 0; w < windows; ++w)
        for (uint32_t thread = 0; thread < threads; ++thread)
        {
            const ShortOnceLane l = vec == 1 ? short_once_lane<1>(g, w, thread) : short_once_lane<2>(g, w, thread);
            for (uint32_t u = 0; l.live && u < g.passes * g.turns.divisor; ++u)
            {
                const uint32_t p = u / g.turns.divisor, n = short_once_sample(g, l, p, u - p * g.turns.divisor);
                if (n >= g.num_samples)
                    continue;
                const size_t e = static_cast<size_t>(w * g.channels.divisor * g.stride_c) + (l.at + n * g.stride_n);
                if (e + vec > elements)
                    return H2X_ERR_INVALID_ARGUMENT;
                for (uint32_t v = 0; v < vec; ++v)
                {
                    stored[e + v] = 1;
                    if (v < l.skip)
                        continue;
                    ++counted[e + v];
                    range[e + v] = static_cast<unsigned short>(p * g.together + l.q + 1);
                }
            }
        }
    return H2X_SUCCESS;
}

// Plays on the host which cells the passes over double tensors clear, by so many threads a channel.
extern "C" int h2x_bn_audit_cleared(const h2x_haloed_geometry* geometry, unsigned int threads, unsigned char* cleared, size_t cells)
{
    if (!geometry || !cleared || threads == 0)
        return H2X_ERR_INVALID_ARGUMENT;
    HostTensor t;
    HaloCells halo;
    int c;
    size_t s;
    const void* interior;
    const int err = haloed_tensor(geometry, reinterpret_cast<const void*>(uintptr_t(256)), &t, &interior, &c, &s, &halo);
    if (err)
        return err;
    size_t outside = 0;
    for (int channel = 0; channel < c; ++channel)
    {
        // (the kernels start from the interior's first element of the channel)
        const int64_t first = static_cast<const double*>(interior) - reinterpret_cast<const double*>(uintptr_t(256))
                              + channel * t.map.stride_c - halo.origin;
        const auto one = [&](uint32_t i) {
            if (static_cast<size_t>(first + i) < cells)
                cleared[first + i] = 1;
            else
                ++outside;
        };
        for (uint32_t at = 0; at < threads; ++at)
            each_halo_cell(halo, at, threads, one, [&](uint32_t i) {
                one(i);
                one(i + 1);
            });
    }
    return outside ? H2X_ERR_INVALID_ARGUMENT : H2X_SUCCESS;
}

// What a whole pass over tensors of one geometry launches, by the entry points' own choice.
extern "C" int h2x_bn_planned(int backward, h2x_dtype dtype, int num_samples, const h2x_tensor_geometry* geometry,
                              const h2x_haloed_geometry* cleared, int with_state, h2x_bn_planned_launch* launches,
                              int* num_launches)
{
    if (!geometry == !cleared || !launches || !num_launches)
        return H2X_ERR_INVALID_ARGUMENT;
    // addresses that nobody follows, apart from one another
    const auto at = [](int i) { return reinterpret_cast<void*>(static_cast<uintptr_t>(i) << 40); };
    void *const x = at(1), *const dy = at(2), *const out = at(3), *const ws = at(4), *const state = with_state ? at(5) : nullptr;
    void *const mean = at(6), *const var = at(7), *const scale = at(8), *const s0 = at(9), *const s1 = at(10), *const s2 = at(11),
               *const s3 = at(12);
    constexpr size_t kPerSum = 2;
    constexpr double kDecay = 0.9, kEpsilon = 1e-5;
    LaunchLog log;
    ScopedLaunchLog scope(&log);
    int err;
    if (cleared)
        err = backward ? h2x_bn_backward_clearing(dtype, kPerSum, cleared, x, dy, mean, var, scale, s0, s1, s2, s3, out, kEpsilon,
                                                  state, nullptr)
                       : h2x_bn_forward_clearing(dtype, cleared, x, scale, s0, kPerSum, kDecay, kEpsilon, mean, var, s1, s2, out,
                                                 state, nullptr);
    else
        err = backward ? h2x_bn_backward_once(dtype, num_samples, kPerSum, geometry, geometry, geometry, x, dy, mean, var, scale,
                                              s0, s1, s2, s3, out, kEpsilon, ws, state, nullptr)
                       : h2x_bn_forward_once(dtype, num_samples, geometry, geometry, x, scale, s0, kPerSum, kDecay, kEpsilon,
                                             mean, var, s1, s2, out, ws, state, nullptr);
    if (err)
        return err;
    if (log.records.size() > H2X_BN_AUDIT_MAX_LAUNCHES)
        return H2X_ERR_TOO_LARGE;
    *num_launches = static_cast<int>(log.records.size());
    for (size_t i = 0; i < log.records.size(); ++i)
    {
        const LaunchRecord& r = log.records[i];
        launches[i] = {r.kernel, r.grid_x * r.grid_y, static_cast<uint32_t>(r.threads), static_cast<uint32_t>(r.vectors)};
    }
    return H2X_SUCCESS;
}
