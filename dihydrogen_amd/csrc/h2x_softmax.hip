// Channel softmax (forward, backward) for gfx950 and the C entry points.
//
// Tensors are dense [N][C][S]; the softmax runs over C, so the C values of one
// pixel are S elements apart while neighbouring pixels are contiguous.  A
// thread owns VEC neighbouring pixels and keeps all C values of them in
// registers (the channel loop is unrolled to a compile-time bound CMAX >= C),
// so x (or y and dy) is read from HBM exactly once with fully coalesced
// 4*VEC-byte accesses and no LDS staging; the reference stages a
// C x 256 tile in LDS and walks it three times
// (legacy/src/dnn_backend/softmax.cu:538-593,621-669).  Above 32 channels the
// waves of a workgroup share the channels of 64 * VEC pixels, still in
// registers; channel counts beyond the largest such tile fall back to a kernel
// that re-reads its inputs; tensors with one pixel per sample have kernels
// that put the channels, which are contiguous then, on the lanes of a wave or,
// beyond 2048 channels, on the threads of a workgroup.
#include "h2x_device.hpp"

#include <cfloat>
#include <cmath>
#include <limits>
#include <type_traits>

namespace h2x
{
namespace
{

template <typename T>
struct Limits;
template <>
struct Limits<float>
{
    static constexpr float min_normal = FLT_MIN;
};
template <>
struct Limits<double>
{
    static constexpr double min_normal = DBL_MIN;
};

__device__ __forceinline__ float exp_t(float v)
{
    return expf(v);
}
__device__ __forceinline__ double exp_t(double v)
{
    return exp(v);
}
__device__ __forceinline__ float fma_t(float a, float b, float c)
{
    return __builtin_fmaf(a, b, c);
}
__device__ __forceinline__ double fma_t(double a, double b, double c)
{
    return __builtin_fma(a, b, c);
}

// VEC neighbouring pixels of one channel.
template <typename T, int VEC>
struct Pack
{
    T e[VEC];
    __device__ __forceinline__ T& operator[](int j) { return e[j]; }
    __device__ __forceinline__ const T& operator[](int j) const { return e[j]; }

    // STREAM: past the caches
    template <bool STREAM = false>
    static __device__ __forceinline__ Pack load(const T* p)
    {
        Pack r;
        if constexpr (VEC == 1)
        {
            r.e[0] = STREAM ? __builtin_nontemporal_load(p) : *p;
        }
        else
        {
            typedef T V __attribute__((ext_vector_type(VEC)));
            const V* const q = reinterpret_cast<const V*>(p);
            const V t = STREAM ? __builtin_nontemporal_load(q) : *q;
#pragma unroll
            for (int j = 0; j < VEC; ++j)
                r.e[j] = t[j];
        }
        return r;
    }
    template <bool STREAM = false>
    static __device__ __forceinline__ void store(T* p, const Pack& r)
    {
        if constexpr (VEC == 1)
        {
            if constexpr (STREAM)
                __builtin_nontemporal_store(r.e[0], p);
            else
                *p = r.e[0];
        }
        else
        {
            typedef T V __attribute__((ext_vector_type(VEC)));
            V t;
#pragma unroll
            for (int j = 0; j < VEC; ++j)
                t[j] = r.e[j];
            if constexpr (STREAM)
                __builtin_nontemporal_store(t, reinterpret_cast<V*>(p));
            else
                *reinterpret_cast<V*>(p) = t;
        }
    }
};

// The wave of a thread, as the scalar that it is: which channels a wave takes, and where they
// lie, is then worked out once a wave and not in every lane.
__device__ __forceinline__ int wave_index()
{
    return __builtin_amdgcn_readfirstlane(threadIdx.x / kWaveSize);
}

// Where the VEC pixels of a lane start (offset of their first channel) and
// whether they exist; `index` counts the lanes of the grid's x dimension in tile
// order.  Tensors with few pixels per sample (flat_samples > 0; one pixel a lane)
// count their pixels through all samples, so that a tile of 64 or 256 pixels is
// full whatever the size of a sample.
template <int VEC>
__device__ __forceinline__ bool lane_pixels(size_t index, int num_channels, size_t spatial,
                                            int flat_samples, size_t* base, unsigned int sample)
{
    const size_t p = index * VEC;
    if (flat_samples > 0)
    {
        const unsigned int n = static_cast<unsigned int>(p) / static_cast<unsigned int>(spatial);
        const bool exists = n < static_cast<unsigned int>(flat_samples);
        *base = exists ? static_cast<size_t>(n) * num_channels * spatial + (p - n * spatial) : 0;
        return exists;
    }
    const bool exists = p < spatial;
    *base = static_cast<size_t>(sample) * num_channels * spatial + (exists ? p : 0);
    return exists;
}

// The tiles of 64 lanes that a launch consists of: blockIdx.y counts the samples, or (one
// row of workgroups) per_sample tiles of one sample are followed by those of the next.
struct WideTiles
{
    FastDiv per_sample;
    unsigned int samples;
};

// One pixel a lane.
__device__ __forceinline__ bool tile_pixels(const WideTiles& t, int num_channels, size_t spatial, int flat_samples,
                                            size_t* base)
{
    const unsigned int tile = xcd_contiguous(blockIdx.x, gridDim.x);
    const unsigned int n = fastdiv(tile, t.per_sample);
    const unsigned int sample = blockIdx.y + n;
    const size_t first = static_cast<size_t>(tile - n * t.per_sample.divisor) * kWaveSize;
    return lane_pixels<1>(first + threadIdx.x % kWaveSize, num_channels, spatial, flat_samples, base, sample)
           && sample < t.samples;
}

// What a workgroup of the split kernels serves: the first element of its tile, the same for all its threads,
// and from there the bytes to the lane's first pixel (of a lane without pixels: 0, which can be read).
struct TilePlace
{
    size_t first;
    uint32_t offset;
    bool active; // the lane has pixels
    bool any;    // the tile has
};

template <typename T, int VEC, int LANES>
__device__ __forceinline__ TilePlace tile_place(const WideTiles& t, int num_channels, size_t spatial, int flat_samples)
{
    TilePlace p;
    const unsigned int tile = xcd_contiguous(blockIdx.x, gridDim.x);
    const unsigned int lane = threadIdx.x % LANES;
    const size_t sample_size = num_channels * spatial;
    if (flat_samples > 0)
    {
        const unsigned int size = static_cast<unsigned int>(spatial), pixel = tile * LANES + lane;
        const unsigned int n0 = tile * LANES / size, n = pixel / size;
        p.first = n0 * sample_size + (tile * LANES - n0 * size);
        p.any = n0 < static_cast<unsigned int>(flat_samples);
        p.active = n < static_cast<unsigned int>(flat_samples);
        const size_t at = n * sample_size + (pixel - n * size);
        p.offset = p.active ? static_cast<uint32_t>(at - p.first) * sizeof(T) : 0;
        return p;
    }
    const unsigned int n = fastdiv(tile, t.per_sample), sample = blockIdx.y + n;
    const size_t pixel = static_cast<size_t>(tile - n * t.per_sample.divisor) * (LANES * VEC);
    p.first = sample * sample_size + pixel;
    p.any = sample < t.samples && pixel < spatial;
    p.active = pixel + lane * VEC < spatial;
    p.offset = p.active ? lane * (VEC * sizeof(T)) : 0;
    return p;
}

// The element `offset` bytes behind p, which all lanes share: scalar registers and one vector register address it.
template <typename T>
__device__ __forceinline__ T* element(T* p, uint32_t offset)
{
    using C = std::conditional_t<std::is_const_v<T>, const char, char>;
    return reinterpret_cast<T*>(reinterpret_cast<C*>(p) + offset);
}

// The larger of the two, b where a is no number (b is one).
__device__ __forceinline__ float larger(float a, float b)
{
    return __builtin_amdgcn_fmed3f(a, b, __builtin_inff());
}
__device__ __forceinline__ double larger(double a, double b)
{
    return a > b ? a : b;
}

// Cache policy.  The backward pass reads the y that the forward pass has written; x and dy are read
// and dx is written once.  Tensors of 24 MiB and more are streamed (STREAM): x and dy are loaded and dx is stored past
// the caches, y alone stays.  (x, y, dy and dx of such a layer, 96 MiB, fit the 256 MB memory-side cache by themselves; with
// those of its neighbours, or of two more layers like it, they do not, and that is what was measured.)
// Forward + backward, us going round three sets of tensors, before -> streamed: N 16, C 21, 256 x 256, 88 MB,
// 74.6 -> 69.8; N 8, C 32, 256 x 256, 67 MB, 60.3 -> 53.5; N 16, C 500, 48 x 48, 74 MB, 90.5 -> 82.5; N 6, C 19,
// 256 x 256, 30 MB, 29.8 -> 28.2; N 4, C 100, 128 x 128, 26 MB, 27.3 -> 25.6; below, the caches hold what is read: N 4, C 19,
// 256 x 256, 20 MB, 20.8 and 21.3, N 2, C 16, 384 x 384, 19 MB, 24.1 and 26.8.  Rows that are no whole
// vectors share their lines with the tile next door and are not streamed (N 30, C 179, 43 x 43, 40 MB,
// 49.3 and 52.2; N 16, C 21, 255 x 257 78.5 both ways).  With y past the caches too the first takes 76.9.
// That is the call alone.  Between neighbours that write x, make dy of y and read dx (one set of tensors,
// elementwise kernels, all five launches, normally -> streamed): N 16, C 21, 256 x 256 188.8 -> 167.7, N 8, C 32 134.4 ->
// 126.2, N 16, C 500, 48 x 48 164.2 -> 156.8, N 6, C 19 63.7 and 63.9, N 4, C 100, 128 x 128 57.5 -> 57.0, but N 2,
// C 64, 32 MB, 67.8 -> 69.1.  The kernel behind it reads a streamed dx from memory: backward + consumer of 64 MB
// 49.3 -> 53.4, of 28 MB 24.0 -> 27.0; y and what else is live stay cached instead and give back as much or
// more.  Called over and over on one set of 63 MB, with nothing in between, 48.7 -> 55.7.
constexpr size_t kStreamBytes = size_t(24) << 20;

template <typename T>
bool streamed(int vector, int n, int c, size_t s)
{
    return vector == static_cast<int>(16 / sizeof(T)) && static_cast<size_t>(n) * c * s * sizeof(T) >= kStreamBytes;
}

// forward, register-resident.  Replaces fp_channel_kernel, softmax.cu:538-593:
// running maximum starts at min_normal (positive), the sum is taken in channel
// order, y = max(e * (1 / sum), min_normal).
template <typename T, int VEC, int CMAX, bool STREAM>
__global__ __launch_bounds__(kBlockSize) void softmax_fwd_reg_kernel(
    const T* __restrict__ x, T* __restrict__ y, int num_channels, size_t spatial, int flat_samples)
{
    using P = Pack<T, VEC>;
    size_t base;
    if (!lane_pixels<VEC>(static_cast<size_t>(xcd_contiguous(blockIdx.x, gridDim.x)) * kBlockSize
                              + threadIdx.x,
                          num_channels, spatial, flat_samples, &base, blockIdx.y))
        return;
    const T* xp = x + base;
    T* yp = y + base;
    constexpr T kMin = Limits<T>::min_normal;

    P v[CMAX];
#pragma unroll
    for (int c = 0; c < CMAX; ++c)
        if (c < num_channels)
            v[c] = P::template load<STREAM>(xp + static_cast<size_t>(c) * spatial);

    T mx[VEC], sum[VEC];
#pragma unroll
    for (int j = 0; j < VEC; ++j)
    {
        mx[j] = kMin;
        sum[j] = T(0);
    }
#pragma unroll
    for (int c = 0; c < CMAX; ++c)
        if (c < num_channels)
#pragma unroll
            for (int j = 0; j < VEC; ++j)
                mx[j] = v[c][j] > mx[j] ? v[c][j] : mx[j];
#pragma unroll
    for (int c = 0; c < CMAX; ++c)
        if (c < num_channels)
#pragma unroll
            for (int j = 0; j < VEC; ++j)
            {
                const T e = exp_t(v[c][j] - mx[j]);
                v[c][j] = e;
                sum[j] += e;
            }
#pragma unroll
    for (int j = 0; j < VEC; ++j)
        sum[j] = T(1) / sum[j];
#pragma unroll
    for (int c = 0; c < CMAX; ++c)
        if (c < num_channels)
        {
#pragma unroll
            for (int j = 0; j < VEC; ++j)
            {
                const T r = v[c][j] * sum[j];
                v[c][j] = r > kMin ? r : kMin;
            }
            P::store(yp + static_cast<size_t>(c) * spatial, v[c]);
        }
}

constexpr int kWideBatch = 8;

// forward, any channel count.  A workgroup serves 64 neighbouring pixels; its
// four waves share the channels (wave g takes c = g, g + 4, ...), combine their
// maxima and sums through LDS in wave order, and walk their channels again for
// the second and third pass; the tile is 64 * C elements, so those re-reads are
// served by the L2.  The sum is formed from four partial sums instead of one
// running sum over all channels (softmax.cu:565-580).
template <typename T>
__global__ __launch_bounds__(kBlockSize) void softmax_fwd_wide_kernel(
    const T* __restrict__ x, T* __restrict__ y, int num_channels, size_t spatial, int flat_samples,
    const WideTiles tiles)
{
    __shared__ T lds[kWavesPerBlock][kWaveSize];
    const int lane = threadIdx.x % kWaveSize;
    const int g = wave_index();
    size_t base;
    const bool active = tile_pixels(tiles, num_channels, spatial, flat_samples, &base);
    const T* xp = x + base;
    T* yp = y + base;
    constexpr T kMin = Limits<T>::min_normal;

    // kWideBatch loads are issued together in every pass: the channel loop of a
    // wave is a chain of dependent operations on values that are a memory
    // latency away each (N 8, C 1000, 64 x 64 backward: 334 us one by one)
    constexpr int kStep = kWavesPerBlock * kWideBatch;
    T mx = kMin;
    if (active)
        for (int c0 = g; c0 < num_channels; c0 += kStep)
        {
            T v[kWideBatch];
#pragma unroll
            for (int u = 0; u < kWideBatch; ++u)
                if (c0 + u * kWavesPerBlock < num_channels)
                    v[u] = xp[static_cast<size_t>(c0 + u * kWavesPerBlock) * spatial];
#pragma unroll
            for (int u = 0; u < kWideBatch; ++u)
                if (c0 + u * kWavesPerBlock < num_channels)
                    mx = v[u] > mx ? v[u] : mx;
        }
    lds[g][lane] = mx;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kWavesPerBlock; ++w)
        mx = lds[w][lane] > mx ? lds[w][lane] : mx;
    __syncthreads();

    T sum = T(0);
    if (active)
        for (int c0 = g; c0 < num_channels; c0 += kStep)
        {
            T v[kWideBatch];
#pragma unroll
            for (int u = 0; u < kWideBatch; ++u)
                if (c0 + u * kWavesPerBlock < num_channels)
                    v[u] = xp[static_cast<size_t>(c0 + u * kWavesPerBlock) * spatial];
#pragma unroll
            for (int u = 0; u < kWideBatch; ++u)
                if (c0 + u * kWavesPerBlock < num_channels)
                    sum += exp_t(v[u] - mx);
        }
    lds[g][lane] = sum;
    __syncthreads();
    sum = lds[0][lane];
#pragma unroll
    for (int w = 1; w < kWavesPerBlock; ++w)
        sum += lds[w][lane];
    const T inv = T(1) / sum;

    if (active)
        for (int c0 = g; c0 < num_channels; c0 += kStep)
        {
            T v[kWideBatch];
#pragma unroll
            for (int u = 0; u < kWideBatch; ++u)
                if (c0 + u * kWavesPerBlock < num_channels)
                    v[u] = xp[static_cast<size_t>(c0 + u * kWavesPerBlock) * spatial];
#pragma unroll
            for (int u = 0; u < kWideBatch; ++u)
                if (c0 + u * kWavesPerBlock < num_channels)
                {
                    const T r = exp_t(v[u] - mx) * inv;
                    yp[static_cast<size_t>(c0 + u * kWavesPerBlock) * spatial] = r > kMin ? r : kMin;
                }
        }
}

// backward, register-resident.  Replaces bp_channel_kernel, softmax.cu:621-669:
// dp accumulates y*dy in channel order with fused multiply-adds.
template <typename T, int VEC, int CMAX, bool STREAM>
__global__ __launch_bounds__(kBlockSize) void softmax_bwd_reg_kernel(
    const T* __restrict__ y, const T* __restrict__ dy, T* __restrict__ dx, int num_channels,
    size_t spatial, int flat_samples)
{
    using P = Pack<T, VEC>;
    size_t base;
    if (!lane_pixels<VEC>(static_cast<size_t>(xcd_contiguous(blockIdx.x, gridDim.x)) * kBlockSize
                              + threadIdx.x,
                          num_channels, spatial, flat_samples, &base, blockIdx.y))
        return;
    const T* yp = y + base;
    const T* gp = dy + base;
    T* op = dx + base;
    constexpr T kMin = Limits<T>::min_normal;

    P yv[CMAX], gv[CMAX];
#pragma unroll
    for (int c = 0; c < CMAX; ++c)
        if (c < num_channels)
        {
            yv[c] = P::load(yp + static_cast<size_t>(c) * spatial);
            gv[c] = P::template load<STREAM>(gp + static_cast<size_t>(c) * spatial);
        }
    T dp[VEC];
#pragma unroll
    for (int j = 0; j < VEC; ++j)
        dp[j] = T(0);
#pragma unroll
    for (int c = 0; c < CMAX; ++c)
        if (c < num_channels)
#pragma unroll
            for (int j = 0; j < VEC; ++j)
                dp[j] = fma_t(yv[c][j], gv[c][j], dp[j]);
#pragma unroll
    for (int c = 0; c < CMAX; ++c)
        if (c < num_channels)
        {
#pragma unroll
            for (int j = 0; j < VEC; ++j)
                yv[c][j] = yv[c][j] > kMin ? yv[c][j] * (gv[c][j] - dp[j]) : T(0);
            P::template store<STREAM>(op + static_cast<size_t>(c) * spatial, yv[c]);
        }
}

// backward, any channel count: the same tiling; dp is formed from the four
// waves' partial dot products.
template <typename T>
__global__ __launch_bounds__(kBlockSize) void softmax_bwd_wide_kernel(
    const T* __restrict__ y, const T* __restrict__ dy, T* __restrict__ dx, int num_channels,
    size_t spatial, int flat_samples,
    const WideTiles tiles)
{
    __shared__ T lds[kWavesPerBlock][kWaveSize];
    const int lane = threadIdx.x % kWaveSize;
    const int g = wave_index();
    size_t base;
    const bool active = tile_pixels(tiles, num_channels, spatial, flat_samples, &base);
    const T* yp = y + base;
    const T* gp = dy + base;
    T* op = dx + base;
    constexpr T kMin = Limits<T>::min_normal;

    constexpr int kStep = kWavesPerBlock * kWideBatch;
    T dp = T(0);
    if (active)
        for (int c0 = g; c0 < num_channels; c0 += kStep)
        {
            T yv[kWideBatch], gv[kWideBatch];
#pragma unroll
            for (int u = 0; u < kWideBatch; ++u)
                if (c0 + u * kWavesPerBlock < num_channels)
                {
                    yv[u] = yp[static_cast<size_t>(c0 + u * kWavesPerBlock) * spatial];
                    gv[u] = gp[static_cast<size_t>(c0 + u * kWavesPerBlock) * spatial];
                }
#pragma unroll
            for (int u = 0; u < kWideBatch; ++u)
                if (c0 + u * kWavesPerBlock < num_channels)
                    dp = fma_t(yv[u], gv[u], dp);
        }
    lds[g][lane] = dp;
    __syncthreads();
    dp = lds[0][lane];
#pragma unroll
    for (int w = 1; w < kWavesPerBlock; ++w)
        dp += lds[w][lane];

    if (active)
        for (int c0 = g; c0 < num_channels; c0 += kStep)
        {
            T yv[kWideBatch], gv[kWideBatch];
#pragma unroll
            for (int u = 0; u < kWideBatch; ++u)
                if (c0 + u * kWavesPerBlock < num_channels)
                {
                    yv[u] = yp[static_cast<size_t>(c0 + u * kWavesPerBlock) * spatial];
                    gv[u] = gp[static_cast<size_t>(c0 + u * kWavesPerBlock) * spatial];
                }
#pragma unroll
            for (int u = 0; u < kWideBatch; ++u)
                if (c0 + u * kWavesPerBlock < num_channels)
                    op[static_cast<size_t>(c0 + u * kWavesPerBlock) * spatial] =
                        yv[u] > kMin ? yv[u] * (gv[u] - dp) : T(0);
        }
}

// The waves' partial sums in place i, added pairwise: a chain of WAVES additions would give
// back the accuracy that the waves' shorter chains gain.
template <typename T, int WAVES, int N>
__device__ __forceinline__ T sum_of_waves(const T (&lds)[WAVES][N], int i)
{
    T t[WAVES];
#pragma unroll
    for (int w = 0; w < WAVES; ++w)
        t[w] = lds[w][i];
#pragma unroll
    for (int step = WAVES / 2; step >= 1; step /= 2)
#pragma unroll
        for (int w = 0; w < step; ++w)
            t[w] += t[w + step];
    return t[0];
}

// The values of the lanes that serve a pixel, LANES apart, combined.
template <int LANES, typename T, typename F>
__device__ __forceinline__ T pixel_combine(T v, const F& f)
{
    if constexpr (LANES <= 32)
        v = combine_apart<32>(v, f);
    if constexpr (LANES <= 16)
        v = combine_apart<16>(v, f);
    return v;
}

// forward, up to WAVES * CPW channels, register-resident.  A workgroup serves
// 64 * VEC neighbouring pixels; its WAVES waves share the channels (wave g takes
// c = g, g + WAVES, ...: CPW of them at most) and keep their values in registers,
// so x is read once; maxima and sums are combined through LDS in a fixed order.
// softmax_fwd_wide_kernel, with the same terms, re-reads its tile twice, and its
// tiles of 64 * C elements the L2 does not hold once every CU runs eight of them
// (N 16, C 150, 128 x 128: 100 us there, 63 us with the tile in registers).  Bound by
// memory where there are several tiles a CU, else by a wave's chain of loads,
// exponentials and sums.
// Where there are few tiles, a pixel is for 64 / LANES lanes of a wave instead of one: a workgroup serves LANES
// pixels, lane l of wave g the channels (g + k * WAVES) * 64 / LANES + l / LANES, the chain is that many times shorter
// and there are as many more workgroups, for rows of 64 or 128 bytes (see launch_split_for).
// The chain of a wave counts: 19 vector and 6 scalar instructions a channel forward, of which the exponential takes 13.
// So the first CERTAIN channels of a wave, which the smallest channel count of the variant has, are not asked for; a
// channel that is not there is -infinity (backward 0), with no further question but, where a wave lacks it as a whole,
// one ahead of its exponential; lanes without pixels work on the tile's first one and store nothing; and addresses are
// a running scalar pointer and a lane's offset in bytes. Asking before each load, term and store, with addresses of 64
// bits a lane (23 and 22 instructions, backward 13 and 30 with registers spilled), forward + backward in us -> so: N 4,
// C 150, 65 x 97 17.5 -> 16.8; N 2, C 209, 15 x 15 6.85 -> 5.75; N 5, C 308, 56 x 52 21.8 -> 20.6; N 2, C 322, 75 x 110
// 26.7 -> 24.0; N 4, C 431, 99 x 126 111 -> 102; doubles N 4, C 472, 49 x 44 47.3 -> 43.6; of 47 calls the mean is
// 0.950. The question ahead of the exponential is for tiles that are half empty, without it and with it: N 1, C 39, 316
// x 354 (asking each time 17.9) 18.0 and 17.1; N 13, C 42, 220 x 134 (56.2) 57.4 and 56.2; doubles N 4, C 33, 128 x 128
// (18.0) 18.4 and 17.4. One round of workgroups of full tiles whose tensors are streamed does lose, a wave's loads now
// being together: N 1, C 60, 316 x 354 28.7 -> 29.5, N 8, C 60, 112 x 125 28.2 -> 29.0 (two rounds, N 2, C 60, 316 x
// 354 52.5 -> 49.8).
template <typename T, int VEC, int CPW, int CERTAIN, int WAVES, int LANES, bool STREAM>
__global__ __launch_bounds__(WAVES * kWaveSize) void softmax_fwd_split_kernel(
    const T* __restrict__ x, T* __restrict__ y, int num_channels, size_t spatial, int flat_samples,
    const WideTiles tiles)
{
    using P = Pack<T, VEC>;
    __shared__ T lds[WAVES][LANES * VEC];
    constexpr int kApart = kWaveSize / LANES; // channels that a wave takes at once
    const int lane = threadIdx.x % LANES, q = threadIdx.x % kWaveSize / LANES;
    const int g = wave_index();
    const TilePlace place = tile_place<T, VEC, LANES>(tiles, num_channels, spatial, flat_samples);
    if (!place.any) // the whole workgroup
        return;
    const uint32_t offset = place.offset + static_cast<uint32_t>(q * spatial * sizeof(T));
    const size_t first = place.first + g * kApart * spatial, step = WAVES * kApart * spatial;
    const auto exists = [&](int k) { return k < CERTAIN || (g + k * WAVES) * kApart + q < num_channels; };
    constexpr T kMin = Limits<T>::min_normal;

    P v[CPW];
    T mx[VEC], sum[VEC];
    const T* xp = x + first;
#pragma unroll
    for (int k = 0; k < CPW; ++k, xp += step)
    {
        if (exists(k))
            v[k] = P::template load<STREAM>(element(xp, offset));
        else
#pragma unroll
            for (int j = 0; j < VEC; ++j)
                v[k][j] = -std::numeric_limits<T>::infinity(); // no maximum, and exactly 0 in the sum
    }
#pragma unroll
    for (int j = 0; j < VEC; ++j)
    {
        mx[j] = kMin;
#pragma unroll
        for (int k = 0; k < CPW; ++k)
            mx[j] = larger(v[k][j], mx[j]);
        mx[j] = pixel_combine<LANES>(mx[j], [](T p, T r) { return larger(p, r); });
        if (q == 0)
            lds[g][lane * VEC + j] = mx[j];
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < VEC; ++j)
#pragma unroll
        for (int w = 0; w < WAVES; ++w)
            mx[j] = larger(lds[w][lane * VEC + j], mx[j]);
    __syncthreads();

#pragma unroll
    for (int j = 0; j < VEC; ++j)
        sum[j] = T(0);
#pragma unroll
    for (int k = 0; k < CPW; ++k)
    {
        if (LANES == kWaveSize && !exists(k)) // uniform, and so are all that follow
            break;
#pragma unroll
        for (int j = 0; j < VEC; ++j)
        {
            const T e = exp_t(v[k][j] - mx[j]);
            v[k][j] = e;
            sum[j] += e;
        }
    }
#pragma unroll
    for (int j = 0; j < VEC; ++j)
    {
        sum[j] = pixel_combine<LANES>(sum[j], [](T p, T r) { return p + r; });
        if (q == 0)
            lds[g][lane * VEC + j] = sum[j];
    }
    __syncthreads();
    T inv[VEC];
#pragma unroll
    for (int j = 0; j < VEC; ++j)
    {
        inv[j] = T(1) / sum_of_waves<T, WAVES>(lds, lane * VEC + j);
    }
    if (!place.active)
        return;
    T* yp = y + first;
#pragma unroll
    for (int k = 0; k < CPW; ++k, yp += step)
        if (exists(k))
        {
#pragma unroll
            for (int j = 0; j < VEC; ++j)
                v[k][j] = larger(v[k][j] * inv[j], kMin);
            P::store(element(yp, offset), v[k]);
        }
}

// backward likewise: y and dy of up to WAVES * CPW channels in registers.  All of y is
// asked for before any of dy: alternating, the wave waited more often (N 4, C 150,
// 65 x 97 in four waves 15.9 us against 10.2).
template <typename T, int VEC, int CPW, int CERTAIN, int WAVES, int LANES, bool STREAM>
__global__ __launch_bounds__(WAVES * kWaveSize) void softmax_bwd_split_kernel(
    const T* __restrict__ y, const T* __restrict__ dy, T* __restrict__ dx, int num_channels,
    size_t spatial, int flat_samples,
    const WideTiles tiles)
{
    using P = Pack<T, VEC>;
    __shared__ T lds[WAVES][LANES * VEC];
    constexpr int kApart = kWaveSize / LANES; // channels that a wave takes at once
    const int lane = threadIdx.x % LANES, q = threadIdx.x % kWaveSize / LANES;
    const int g = wave_index();
    const TilePlace place = tile_place<T, VEC, LANES>(tiles, num_channels, spatial, flat_samples);
    if (!place.any) // the whole workgroup
        return;
    const uint32_t offset = place.offset + static_cast<uint32_t>(q * spatial * sizeof(T));
    const size_t first = place.first + g * kApart * spatial, step = WAVES * kApart * spatial;
    const auto exists = [&](int k) { return k < CERTAIN || (g + k * WAVES) * kApart + q < num_channels; };
    constexpr T kMin = Limits<T>::min_normal;

    P yv[CPW], gv[CPW];
    const auto load = [&](const T* p, P(&v)[CPW], auto stream) {
#pragma unroll
        for (int k = 0; k < CPW; ++k, p += step)
        {
            if (exists(k))
                v[k] = P::template load<decltype(stream)::value>(element(p, offset));
            else
#pragma unroll
                for (int j = 0; j < VEC; ++j)
                    v[k][j] = T(0);
        }
    };
    load(y + first, yv, std::false_type());
    load(dy + first, gv, std::bool_constant<STREAM>());
    T dp[VEC];
#pragma unroll
    for (int j = 0; j < VEC; ++j)
    {
        dp[j] = T(0);
#pragma unroll
        for (int k = 0; k < CPW; ++k)
            dp[j] = fma_t(yv[k][j], gv[k][j], dp[j]);
        dp[j] = pixel_combine<LANES>(dp[j], [](T p, T r) { return p + r; });
        if (q == 0)
            lds[g][lane * VEC + j] = dp[j];
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < VEC; ++j)
    {
        dp[j] = sum_of_waves<T, WAVES>(lds, lane * VEC + j);
    }
    if (!place.active)
        return;
    T* op = dx + first;
#pragma unroll
    for (int k = 0; k < CPW; ++k, op += step)
        if (exists(k))
        {
#pragma unroll
            for (int j = 0; j < VEC; ++j)
                yv[k][j] = yv[k][j] > kMin ? yv[k][j] * (gv[k][j] - dp[j]) : T(0);
            P::template store<STREAM>(element(op, offset), yv[k]);
        }
}

// Up to 32 channels of few pixels: a workgroup of 256 threads serves LANES pixels, thread group g their channels g, g +
// 256 / LANES, ... A lane's chain of loads, exponentials and stores is that many times shorter, and there are as many
// more workgroups. The exponentials (backward the values) go through LDS, where each thread adds those of its pixel in
// channel order: the same bits as by one thread a pixel.
template <typename T, int CMAX, int LANES>
__global__ __launch_bounds__(kBlockSize) void softmax_fwd_shared_kernel(
    const T* __restrict__ x, T* __restrict__ y, int num_channels, size_t spatial, int flat_samples, const WideTiles tiles)
{
    constexpr int kGroups = kBlockSize / LANES, kEach = (CMAX + kGroups - 1) / kGroups;
    __shared__ T largest[kGroups][LANES];
    __shared__ T terms[CMAX][LANES];
    const int lane = threadIdx.x % LANES, g = threadIdx.x / LANES;
    const TilePlace place = tile_place<T, 1, LANES>(tiles, num_channels, spatial, flat_samples);
    if (!place.any) // the whole workgroup
        return;
    constexpr T kMin = Limits<T>::min_normal;
    const auto exists = [&](int k) { return g + k * kGroups < num_channels; };
    const T* const xp = element(x + place.first, place.offset) + g * spatial;
    T v[kEach], mx = kMin;
#pragma unroll
    for (int k = 0; k < kEach; ++k)
        if (exists(k))
            v[k] = xp[k * kGroups * spatial];
#pragma unroll
    for (int k = 0; k < kEach; ++k)
        if (exists(k))
            mx = v[k] > mx ? v[k] : mx;
    largest[g][lane] = mx;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kGroups; ++i)
        mx = largest[i][lane] > mx ? largest[i][lane] : mx;
#pragma unroll
    for (int k = 0; k < kEach; ++k)
        if (exists(k))
            terms[g + k * kGroups][lane] = v[k] = exp_t(v[k] - mx);
    __syncthreads();
    T sum = T(0);
#pragma unroll
    for (int c = 0; c < CMAX; ++c)
        if (c < num_channels)
            sum += terms[c][lane];
    sum = T(1) / sum;
    if (!place.active)
        return;
    T* const yp = element(y + place.first, place.offset) + g * spatial;
#pragma unroll
    for (int k = 0; k < kEach; ++k)
        if (exists(k))
        {
            const T r = v[k] * sum;
            yp[k * kGroups * spatial] = r > kMin ? r : kMin;
        }
}

template <typename T, int CMAX, int LANES>
__global__ __launch_bounds__(kBlockSize) void softmax_bwd_shared_kernel(
    const T* __restrict__ y, const T* __restrict__ dy, T* __restrict__ dx, int num_channels, size_t spatial, int flat_samples,
    const WideTiles tiles)
{
    constexpr int kGroups = kBlockSize / LANES, kEach = (CMAX + kGroups - 1) / kGroups;
    __shared__ T terms[2][CMAX][LANES];
    const int lane = threadIdx.x % LANES, g = threadIdx.x / LANES;
    const TilePlace place = tile_place<T, 1, LANES>(tiles, num_channels, spatial, flat_samples);
    if (!place.any) // the whole workgroup
        return;
    constexpr T kMin = Limits<T>::min_normal;
    const auto exists = [&](int k) { return g + k * kGroups < num_channels; };
    const T* const yp = element(y + place.first, place.offset) + g * spatial;
    const T* const gp = element(dy + place.first, place.offset) + g * spatial;
    T yv[kEach], gv[kEach];
#pragma unroll
    for (int k = 0; k < kEach; ++k)
        if (exists(k))
        {
            yv[k] = yp[k * kGroups * spatial];
            gv[k] = gp[k * kGroups * spatial];
        }
#pragma unroll
    for (int k = 0; k < kEach; ++k)
        if (exists(k))
        {
            terms[0][g + k * kGroups][lane] = yv[k];
            terms[1][g + k * kGroups][lane] = gv[k];
        }
    __syncthreads();
    T dp = T(0);
#pragma unroll
    for (int c = 0; c < CMAX; ++c)
        if (c < num_channels)
            dp = fma_t(terms[0][c][lane], terms[1][c][lane], dp);
    if (!place.active)
        return;
    T* const op = element(dx + place.first, place.offset) + g * spatial;
#pragma unroll
    for (int k = 0; k < kEach; ++k)
        if (exists(k))
            op[k * kGroups * spatial] = yv[k] > kMin ? yv[k] * (gv[k] - dp) : T(0);
}

// One pixel per sample (the output of a fully connected layer): the channels of
// a sample are contiguous, so a wave takes a sample, lane l the channels l,
// l + 64, ... (CPL of them at most), and maxima, sums and dot products are
// combined across the lanes with a butterfly of permutes.  The kernels above
// would put one sample on each lane and read with a stride of C elements
// (N 256, C 1000: 176 us).
template <typename T>
__device__ __forceinline__ T wave_butterfly_sum(T v)
{
    return wave_combine(v, [](T p, T q) { return p + q; });
}

// Maximum or sum over a workgroup: the lanes of a wave as a butterfly, the waves pairwise.
template <int WAVES, typename T>
__device__ __forceinline__ T block_combine(T v, bool is_max, T* lds)
{
    const auto both = [is_max](T p, T q) { return is_max ? (q > p ? q : p) : p + q; };
    v = wave_combine(v, both);
    __syncthreads(); // lds may still be read from the previous call
    if ((threadIdx.x & (kWaveSize - 1)) == 0)
        lds[threadIdx.x / kWaveSize] = v;
    __syncthreads();
    T r[WAVES];
#pragma unroll
    for (int w = 0; w < WAVES; ++w)
        r[w] = lds[w];
#pragma unroll
    for (int step = WAVES / 2; step >= 1; step /= 2)
#pragma unroll
        for (int w = 0; w < step; ++w)
            r[w] = both(r[w], r[w + step]);
    return r[0];
}

template <typename T>
__device__ __forceinline__ T wave_max(T v)
{
    return wave_combine(v, [](T p, T q) { return q > p ? q : p; });
}

// The same over the LANES threads that serve a sample: a wave, or a workgroup of that many threads.
template <int LANES, typename T>
__device__ __forceinline__ T lanes_max(T v, T* lds)
{
    if constexpr (LANES == kWaveSize)
        return wave_max(v);
    else
        return block_combine<LANES / kWaveSize>(v, true, lds);
}

template <int LANES, typename T>
__device__ __forceinline__ T lanes_sum(T v, T* lds)
{
    if constexpr (LANES == kWaveSize)
        return wave_butterfly_sum(v);
    else
        return block_combine<LANES / kWaveSize>(v, false, lds);
}

template <int LANES>
constexpr int lanes_block()
{
    return LANES < kBlockSize ? kBlockSize : LANES;
}

// LANES: a wave, or a workgroup where a wave would not hold the channels or samples are few
// (N 16, C 4096: forward 9.0 us, backward 7.3 in a kernel that walked them three times).
template <typename T, int CPL, int LANES>
__global__ __launch_bounds__(lanes_block<LANES>()) void softmax_fwd_row_kernel(
    const T* __restrict__ x, T* __restrict__ y, int num_channels, int num_samples)
{
    __shared__ T lds[lanes_block<LANES>() / kWaveSize];
    const int lane = threadIdx.x % LANES;
    const int n = blockIdx.x * (lanes_block<LANES>() / LANES) + threadIdx.x / LANES;
    if (n >= num_samples) // all lanes of a sample
        return;
    const T* xp = x + static_cast<size_t>(n) * num_channels;
    T* yp = y + static_cast<size_t>(n) * num_channels;
    constexpr T kMin = Limits<T>::min_normal;
    T v[CPL];
    T mx = kMin;
#pragma unroll
    for (int k = 0; k < CPL; ++k)
        if (lane + k * LANES < num_channels)
            v[k] = xp[lane + k * LANES];
#pragma unroll
    for (int k = 0; k < CPL; ++k)
        if (lane + k * LANES < num_channels)
            mx = v[k] > mx ? v[k] : mx;
    mx = lanes_max<LANES>(mx, lds);
    T sum = T(0);
#pragma unroll
    for (int k = 0; k < CPL; ++k)
        if (lane + k * LANES < num_channels)
        {
            v[k] = exp_t(v[k] - mx);
            sum += v[k];
        }
    const T inv = T(1) / lanes_sum<LANES>(sum, lds);
#pragma unroll
    for (int k = 0; k < CPL; ++k)
        if (lane + k * LANES < num_channels)
        {
            const T r = v[k] * inv;
            yp[lane + k * LANES] = r > kMin ? r : kMin;
        }
}

template <typename T, int CPL, int LANES>
__global__ __launch_bounds__(lanes_block<LANES>()) void softmax_bwd_row_kernel(
    const T* __restrict__ y, const T* __restrict__ dy, T* __restrict__ dx, int num_channels,
    int num_samples)
{
    __shared__ T lds[lanes_block<LANES>() / kWaveSize];
    const int lane = threadIdx.x % LANES;
    const int n = blockIdx.x * (lanes_block<LANES>() / LANES) + threadIdx.x / LANES;
    if (n >= num_samples)
        return;
    const size_t base = static_cast<size_t>(n) * num_channels;
    constexpr T kMin = Limits<T>::min_normal;
    T yv[CPL], gv[CPL];
    T dp = T(0);
#pragma unroll
    for (int k = 0; k < CPL; ++k)
        if (lane + k * LANES < num_channels)
        {
            yv[k] = y[base + lane + k * LANES];
            gv[k] = dy[base + lane + k * LANES];
        }
#pragma unroll
    for (int k = 0; k < CPL; ++k)
        if (lane + k * LANES < num_channels)
            dp = fma_t(yv[k], gv[k], dp);
    dp = lanes_sum<LANES>(dp, lds);
#pragma unroll
    for (int k = 0; k < CPL; ++k)
        if (lane + k * LANES < num_channels)
            dx[base + lane + k * LANES] = yv[k] > kMin ? yv[k] * (gv[k] - dp) : T(0);
}

// One pixel per sample and more channels than a workgroup holds in registers: a
// workgroup takes a sample and walks its channels (contiguous) three times
// forward, twice backward; the re-reads come from the L2.  Thread t adds up the
// channels t, t + 256, ....
template <typename T>
__global__ __launch_bounds__(kBlockSize) void softmax_fwd_long_row_kernel(
    const T* __restrict__ x, T* __restrict__ y, int num_channels)
{
    __shared__ T lds[kWavesPerBlock];
    const T* xp = x + static_cast<size_t>(blockIdx.x) * num_channels;
    T* yp = y + static_cast<size_t>(blockIdx.x) * num_channels;
    constexpr T kMin = Limits<T>::min_normal;
    T mx = kMin;
    for (int c = threadIdx.x; c < num_channels; c += kBlockSize)
        mx = xp[c] > mx ? xp[c] : mx;
    mx = block_combine<kWavesPerBlock>(mx, true, lds);
    T sum = T(0);
    for (int c = threadIdx.x; c < num_channels; c += kBlockSize)
        sum += exp_t(xp[c] - mx);
    const T inv = T(1) / block_combine<kWavesPerBlock>(sum, false, lds);
    for (int c = threadIdx.x; c < num_channels; c += kBlockSize)
    {
        const T r = exp_t(xp[c] - mx) * inv;
        yp[c] = r > kMin ? r : kMin;
    }
}

template <typename T>
__global__ __launch_bounds__(kBlockSize) void softmax_bwd_long_row_kernel(
    const T* __restrict__ y, const T* __restrict__ dy, T* __restrict__ dx, int num_channels)
{
    __shared__ T lds[kWavesPerBlock];
    const size_t base = static_cast<size_t>(blockIdx.x) * num_channels;
    constexpr T kMin = Limits<T>::min_normal;
    T dp = T(0);
    for (int c = threadIdx.x; c < num_channels; c += kBlockSize)
        dp = fma_t(y[base + c], dy[base + c], dp);
    dp = block_combine<kWavesPerBlock>(dp, false, lds);
    for (int c = threadIdx.x; c < num_channels; c += kBlockSize)
    {
        const T yi = y[base + c];
        dx[base + c] = yi > kMin ? yi * (dy[base + c] - dp) : T(0);
    }
}

// Largest vector (elements) usable for all of the given pointers.
template <typename T>
int vector_width(size_t spatial, int want, std::initializer_list<const void*> ptrs)
{
    int v = want;
    while (v > 1)
    {
        bool ok = spatial % v == 0;
        for (const void* p : ptrs)
            ok = ok && (reinterpret_cast<uintptr_t>(p) % (v * sizeof(T)) == 0);
        if (ok)
            break;
        v /= 2;
    }
    return v;
}

dim3 pixel_grid(size_t spatial, int vec, int num_samples)
{
    const size_t per_block = static_cast<size_t>(kBlockSize) * vec;
    return dim3(static_cast<unsigned int>((spatial + per_block - 1) / per_block), num_samples);
}

// Samples of fewer pixels than this have their pixels counted through all
// samples (one pixel a lane): a tile is full whatever the size of a sample
// (N 256, C 100, 7 x 7: one workgroup a sample with 49 of its 64 pixels, 17 us).
constexpr size_t kFlatBelow = 128;

int flat_samples(int num_samples, size_t spatial)
{
    return spatial < kFlatBelow && spatial * static_cast<size_t>(num_samples) < (1ull << 31)
               ? num_samples
               : 0;
}

// Tiles of lanes * vec pixels, padded to a multiple of the XCD count for kernels
// that reorder their tiles with xcd_contiguous (tiles past the end do nothing).
dim3 tile_grid(size_t spatial, int lanes, int vec, int num_samples, int flat)
{
    const size_t per_block = static_cast<size_t>(lanes) * vec;
    const size_t pixels = flat > 0 ? spatial * static_cast<size_t>(flat) : spatial;
    const size_t blocks = (pixels + per_block - 1) / per_block;
    return dim3(static_cast<unsigned int>((blocks + kNumXcd - 1) / kNumXcd * kNumXcd),
                flat > 0 ? 1 : num_samples);
}

dim3 pixel_grid_xcd(size_t spatial, int vec, int num_samples, int flat)
{
    return tile_grid(spatial, kBlockSize, vec, num_samples, flat);
}

// 64 * vec pixels per workgroup.  Tiles are counted through all samples where filling up each
// sample's to a multiple of the XCDs would leave more than one of nine idle, on the same
// XCDs for every sample (forward + backward, us, filled up and counted through: N 32, C 300, 14 x 14, 4 tiles
// a sample, 23.3 and 18.0; N 25, C 120, 24 x 24, 9 tiles, 14.9 and 10.9; N 29, C 338, 24 x 37, 14 tiles,
// 43.6 and 41.4; but N 30, C 179, 43 x 43, 29 tiles, 47.3 and 48.0, N 8, C 40, 128 x 128, 128 tiles,
// 20.1 and 21.4: samples one after another reach the memory more evenly).  Also where only the filling makes them more
// than two a CU: a third would start when the first two are done, on the XCDs that have it (N 11, C 135, 45 x 61, 473
// tiles filled up to 528, 19.3 and 17.4; N 5, C 151, 92 x 67, 485 to 520, 20.7 and 18.8).
dim3 wide_grid(size_t spatial, int lanes, int vec, int num_samples, int flat, WideTiles* t)
{
    const dim3 by_sample = tile_grid(spatial, lanes, vec, num_samples, flat);
    const size_t per_block = static_cast<size_t>(lanes) * vec;
    const size_t tiles = (spatial + per_block - 1) / per_block;
    t->samples = flat > 0 ? 1 : num_samples;
    const size_t launched = by_sample.x * static_cast<size_t>(num_samples), all = tiles * num_samples;
    const size_t two = 2 * chip_units();
    const bool through = flat == 0 && (launched * 8 > all * 9 || (lanes == kWaveSize && all <= two && launched > two));
    t->per_sample = make_fastdiv(through ? static_cast<uint32_t>(tiles) : by_sample.x);
    if (!through)
        return by_sample;
    return dim3((static_cast<unsigned int>(tiles) * num_samples + kNumXcd - 1) / kNumXcd * kNumXcd);
}

template <typename T, int VEC, int CMAX>
void launch_fwd(const T* x, T* y, int n, int c, size_t s, bool stream, hipStream_t st)
{
    const int flat = VEC == 1 ? flat_samples(n, s) : 0;
    const dim3 grid = pixel_grid_xcd(s, VEC, n, flat);
    if (stream)
        launch(softmax_fwd_reg_kernel<T, VEC, CMAX, true>, grid, kBlockSize, st, x, y, c, s, flat);
    else
        launch(softmax_fwd_reg_kernel<T, VEC, CMAX, false>, grid, kBlockSize, st, x, y, c, s, flat);
}

template <typename T, int VEC, int CMAX>
void launch_bwd(const T* y, const T* dy, T* dx, int n, int c, size_t s, bool stream, hipStream_t st)
{
    const int flat = VEC == 1 ? flat_samples(n, s) : 0;
    const dim3 grid = pixel_grid_xcd(s, VEC, n, flat);
    if (stream)
        launch(softmax_bwd_reg_kernel<T, VEC, CMAX, true>, grid, kBlockSize, st, y, dy, dx, c, s, flat);
    else
        launch(softmax_bwd_reg_kernel<T, VEC, CMAX, false>, grid, kBlockSize, st, y, dy, dx, c, s, flat);
}

// More samples than this fill the chip with a wave each; and more than kSomeSamples (channel softmax of floats,
// forward: kSomeRows) leave its waves little to wait for where samples are short.
constexpr int kManySamples = 2048, kSomeSamples = 768, kSomeRows = 512;

// Which kernel serves which channel count (measured on MI355X).  Up to 32 channels a
// thread keeps all channels of its pixels (softmax_*_reg_kernel: 21 channels of
// N 16, 256 x 256 in 28 / 40 us).  Beyond, the waves of a workgroup share the channels
// (softmax_*_split_kernel) with the smallest register tile that holds them: tiles wider
// than needed cost time, since every lane walks the whole tile under a predicate (N 1, C 79, 135 x 192 in
// tiles of 128 channels 12.0, of 96 11.0 us; N 2, C 89, 115 x 115 13.2 and 11.9; N 2, C 393, 78 x 126 in 512 43.7, in
// 448 42.0; but of 257 to 320 channels some are 4 % faster in 320 than in 384, and others 2 % slower).  Eight
// waves against four, N 4, C 150, 65 x 97: forward 10.2 and 11.7 us; N 1: 5.7 and 8.0; N 16:
// 29.8 and 34.3.  More channels than the largest tile holds (1024 forward, 768 backward, 1024 where
// tiles are few; double: 512, or 1024; N 18, C 270, 27 x 40 backward, re-reading 40.3 us, in
// registers 27.9) take the re-reading kernel.
constexpr int kNoSplit = -1000; // not the status of a launch

template <int VEC, int CPW, int CERTAIN, int WAVES, int LANES = kWaveSize, bool MAY_STREAM = true, typename T>
int launch_split(const T* x, T* y, int n, int c, size_t s, bool stream, hipStream_t st)
{
    if (c < CERTAIN * WAVES * (kWaveSize / LANES))
        return kNoSplit;
    const int flat = VEC == 1 ? flat_samples(n, s) : 0;
    WideTiles tiles;
    const dim3 grid = wide_grid(s, LANES, VEC, n, flat, &tiles);
    if (MAY_STREAM && stream)
        launch(softmax_fwd_split_kernel<T, VEC, CPW, CERTAIN, WAVES, LANES, MAY_STREAM>, grid, WAVES * kWaveSize, st, x, y, c,
               s, flat, tiles);
    else
        launch(softmax_fwd_split_kernel<T, VEC, CPW, CERTAIN, WAVES, LANES, false>, grid, WAVES * kWaveSize, st, x, y, c, s,
               flat, tiles);
    return launch_status();
}

template <int VEC, int CPW, int CERTAIN, int WAVES, int LANES = kWaveSize, bool MAY_STREAM = true, typename T>
int launch_split(const T* y, const T* dy, T* dx, int n, int c, size_t s, bool stream, hipStream_t st)
{
    if (c < CERTAIN * WAVES * (kWaveSize / LANES))
        return kNoSplit;
    const int flat = VEC == 1 ? flat_samples(n, s) : 0;
    WideTiles tiles;
    const dim3 grid = wide_grid(s, LANES, VEC, n, flat, &tiles);
    if (MAY_STREAM && stream)
        launch(softmax_bwd_split_kernel<T, VEC, CPW, CERTAIN, WAVES, LANES, MAY_STREAM>, grid, WAVES * kWaveSize, st, y, dy, dx, c, s,
               flat, tiles);
    else
        launch(softmax_bwd_split_kernel<T, VEC, CPW, CERTAIN, WAVES, LANES, false>, grid, WAVES * kWaveSize, st, y, dy, dx, c, s,
               flat, tiles);
    return launch_status();
}

// The split kernel for 33 channels and more, or kNoSplit.  (Tiles are of 64 pixels; their numbers below are those for 256 CUs.)
// Forward + backward, us, by such tiles (16 waves up to 256 of them, else 8) -> as now:
// * Up to 256 tiles, no more than the CUs: 16 pixels a tile and 8 waves, four times the workgroups, each with half the
//   channels a lane.  N 1, C 447, 17 x 13 16.9 -> 8.7; N 7, C 507, 13 x 16 19.9 -> 9.7; N 4, C 341, 50 x 40 17.8 ->
//   14.3; doubles, whose exponentials are longer: N 2, C 421, 20 x 19 40.6 -> 12.2, N 5, C 217, 14 x 13 17.3 -> 8.7.
//   Up to 96 channels (64 of doubles) the launches are all there is (8.1 both ways), and beyond 16 MiB (20) the parts
//   of lines cost as much: N 28, C 420, 25 x 15 23.3 and 25.6, N 19, C 237, 26 x 26 of doubles 29.5 and 31.2.
// * From 257 tiles to about two a CU: forward, floats of 65 to 256 channels, 16 pixels and 4 waves, a lane's chain as
//   short as with 16 waves of 64 (32 pixels and 8 waves: N 4, C 150, 65 x 97 0.6 us more, N 3, C 129, 84 x 65 13.5 for
//   12.7; but N 20, C 197, 32 x 25 15.4 for 16.1); else 32 pixels and 8 waves, backward to one and a half tiles a CU
//   (beyond, N 4, C 150, 65 x 97 0.2 us more).  N 27, C 133, 23 x 28 16.3 -> 13.1; N 4, C 150, 65 x 97 18.4 -> 17.0; N
//   22, C 143, 38 x 33 18.3 -> 17.1.  Not where the tensors are streamed (N 1, C 306, 195 x 164 43.2 and 50.2: whole
//   lines count there), nor beyond 384 channels (N 2, C 398, 119 x 107 52 and 57).
// * Doubles of 257 to 512 channels, of any size: 32 pixels and 8 waves, whose values fit the registers (16 waves of 64
//   pixels kept five words in scratch, and beyond 384 channels backward read everything twice).  N 17, C 490, 46 x 51 244 -> 185;
//   N 1, C 267, 197 x 189 112 -> 89.
// * Sixteen waves of 64 pixels remain for at most 256 tiles of few or of very many channels, and beyond 512 of floats
//   (N 8, C 400, 64 x 64, 512 tiles: 32.3 forward and 36.8 backward, eight waves 30.1 and 35.3).
// * Two pixels a lane where that leaves two tiles a CU
//   forward, one backward (N 1, C 60, 384 x 384, 1152 tiles of two pixels a lane: 13.3 and 22.2 us,
//   one pixel 14.3 and 25.4; N 8, C 256, 64 x 64, 256 of them: 17.8 and 21.6, one pixel 16.5 and 23.7).
template <typename T, typename... P>
int launch_split_for(int v, int n, int c, size_t s, hipStream_t st, P... p)
{
    constexpr bool kForward = sizeof...(P) == 2;
    constexpr bool kFloat = sizeof(T) == 4;
    const bool stream = streamed<T>(v, n, c, s);
    const int flat = flat_samples(n, s);
    const size_t pixels = flat > 0 ? s * n : s, samples = flat > 0 ? 1 : n;
    const size_t tiles = (pixels + kWaveSize - 1) / kWaveSize * samples;
    const size_t elements = s * c * n, cus = chip_units();
    if (tiles <= cus && c > (kFloat ? 96 : 64) && c <= 1024 && elements * sizeof(T) <= size_t(kFloat ? 16 : 20) << 20)
    {
        if (c <= 128) return launch_split<1, 4, 2, 8, 16, false>(p..., n, c, s, stream, st);
        if (c <= 192) return launch_split<1, 6, 4, 8, 16, false>(p..., n, c, s, stream, st);
        if (c <= 256) return launch_split<1, 8, 6, 8, 16, false>(p..., n, c, s, stream, st);
        if (c <= 384) return launch_split<1, 12, 8, 8, 16, false>(p..., n, c, s, stream, st);
        if (c <= 512) return launch_split<1, 16, 12, 8, 16, false>(p..., n, c, s, stream, st);
        if (c <= 768) return launch_split<1, 24, 16, 8, 16, false>(p..., n, c, s, stream, st);
        return launch_split<1, 32, 24, 8, 16, false>(p..., n, c, s, stream, st);
    }
    if constexpr (kForward && kFloat)
    {
        if (tiles > cus && tiles <= cus * 9 / 4 && c > 64 && c <= 256 && !stream)
        {
            if (c <= 96) return launch_split<1, 6, 4, 4, 16, false>(p..., n, c, s, stream, st);
            if (c <= 128) return launch_split<1, 8, 6, 4, 16, false>(p..., n, c, s, stream, st);
            if (c <= 160) return launch_split<1, 10, 8, 4, 16, false>(p..., n, c, s, stream, st);
            if (c <= 192) return launch_split<1, 12, 10, 4, 16, false>(p..., n, c, s, stream, st);
            return launch_split<1, 16, 12, 4, 16, false>(p..., n, c, s, stream, st);
        }
    }
    if (tiles > cus && tiles <= (kFloat && !kForward ? cus * 3 / 2 : cus * 2) && c > 64 && c <= (kFloat ? 384 : 256) && !stream)
    {
        if constexpr (!(kFloat && kForward))
        {
            if (c <= 128) return launch_split<1, 8, 4, 8, 32, false>(p..., n, c, s, stream, st);
            if (c <= 192) return launch_split<1, 12, 8, 8, 32, false>(p..., n, c, s, stream, st);
            if (c <= 256) return launch_split<1, 16, 12, 8, 32, false>(p..., n, c, s, stream, st);
        }
        if constexpr (kFloat)
            return launch_split<1, 24, 16, 8, 32, false>(p..., n, c, s, stream, st);
    }
    if constexpr (!kFloat)
    {
        if (c > 512) return kNoSplit;
        if (c > 384) return launch_split<1, 32, 24, 8, 32>(p..., n, c, s, stream, st);
        if (c > 256) return launch_split<1, 24, 16, 8, 32>(p..., n, c, s, stream, st);
    }
    if ((tiles <= cus && c > 64) || c > 512)
    {
        if constexpr (kFloat)
        {
            if (c <= 96) return launch_split<1, 8, 4, 16, kWaveSize, false>(p..., n, c, s, stream, st);
            if (c <= 384) return launch_split<1, 24, 6, 16>(p..., n, c, s, stream, st);
            if (c <= 512) return launch_split<1, 32, 24, 16>(p..., n, c, s, stream, st);
            if (c <= 768) return launch_split<1, 48, 32, 16>(p..., n, c, s, stream, st);
        }
        else
            return launch_split<1, 16, 4, 16>(p..., n, c, s, stream, st);
        if constexpr (kFloat && kForward)
        {
            if (c <= 1024) return launch_split<1, 64, 48, 16>(p..., n, c, s, stream, st);
        }
        return kNoSplit;
    }
    if constexpr (kFloat)
    {
        if (v >= 2 && c <= 256 && (s + 2 * kWaveSize - 1) / (2 * kWaveSize) * n >= (kForward ? 2 : 1) * cus)
        {
            if (c <= 64) return launch_split<2, 8, 4, 8>(p..., n, c, s, stream, st);
            if (c <= 96) return launch_split<2, 12, 8, 8>(p..., n, c, s, stream, st);
            if (c <= 128) return launch_split<2, 16, 12, 8>(p..., n, c, s, stream, st);
            if (c <= 160) return launch_split<2, 20, 16, 8>(p..., n, c, s, stream, st);
            if (c <= 192) return launch_split<2, 24, 20, 8>(p..., n, c, s, stream, st);
            if (c <= 224) return launch_split<2, 28, 24, 8>(p..., n, c, s, stream, st);
            return launch_split<2, 32, 28, 8>(p..., n, c, s, stream, st);
        }
    }
    // (floats that are streamed have, with few channels, the pixels for two a lane)
    constexpr bool kStreams96 = !kFloat, kStreams192 = !kFloat || kForward;
    if (c <= 64) return launch_split<1, 8, 4, 8, kWaveSize, kStreams96>(p..., n, c, s, stream, st);
    if (c <= 96) return launch_split<1, 12, 8, 8, kWaveSize, kStreams96>(p..., n, c, s, stream, st);
    if (c <= 128) return launch_split<1, 16, 12, 8, kWaveSize, kStreams192>(p..., n, c, s, stream, st);
    if (c <= 160) return launch_split<1, 20, 16, 8, kWaveSize, kStreams192>(p..., n, c, s, stream, st);
    if (c <= 192) return launch_split<1, 24, 20, 8, kWaveSize, kStreams192>(p..., n, c, s, stream, st);
    if (c <= 224) return launch_split<1, 28, 24, 8>(p..., n, c, s, stream, st);
    if (c <= 256) return launch_split<1, 32, 28, 8>(p..., n, c, s, stream, st);
    if constexpr (kFloat)
    {
        if (c <= 384) return launch_split<1, 48, 32, 8>(p..., n, c, s, stream, st);
        if (c <= 448) return launch_split<1, 56, 48, 8>(p..., n, c, s, stream, st);
        if (c <= 512) return launch_split<1, 64, 56, 8>(p..., n, c, s, stream, st);
    }
    return kNoSplit;
}

template <int CMAX, int LANES, typename T>
int launch_shared(const T* x, T* y, int n, int c, size_t s, hipStream_t st)
{
    WideTiles tiles;
    const int flat = flat_samples(n, s);
    const dim3 grid = wide_grid(s, LANES, 1, n, flat, &tiles);
    launch(softmax_fwd_shared_kernel<T, CMAX, LANES>, grid, kBlockSize, st, x, y, c, s, flat, tiles);
    return launch_status();
}

template <int CMAX, int LANES, typename T>
int launch_shared(const T* y, const T* dy, T* dx, int n, int c, size_t s, hipStream_t st)
{
    WideTiles tiles;
    const int flat = flat_samples(n, s);
    const dim3 grid = wide_grid(s, LANES, 1, n, flat, &tiles);
    launch(softmax_bwd_shared_kernel<T, CMAX, LANES>, grid, kBlockSize, st, y, dy, dx, c, s, flat, tiles);
    return launch_status();
}

// Up to 32 channels: the threads of a workgroup share them, or kNoSplit. Where one thread a pixel leaves CUs waiting
// for its chain; with more pixels the sums that every thread forms cost more than the chain. Us in a graph, a thread a
// pixel and so (32 pixels forward, 16 backward; 64 pixels are slower throughout, and at 2^17 pixels all of them are):
//   floats, C 32, 4608 pixels 4.9 / 4.1 and 3.6 / 3.3, 2^14 5.1 / 4.3 and 4.0 / 3.9, 2^15 5.3 / 4.5 and 4.4 / 4.8, 2^16
//   6.0 / 6.4 and 6.0 / 8.6; C 12, 2^14 3.1 / 2.7 and 2.9 / 2.7; C 8, 2^15 2.8 / 2.4 and 2.8 / 2.8;
//   doubles, whose exponentials are longer, C 32, 4608 pixels 8.6 / 5.2 and 4.1 / 3.8, 2^16 12.3 / 10.0 and 9.8 / 12.3,
//   3 x 2^16 23.3 and 24.1 forward; C 12, 2^14 4.6 / 3.2 and 3.4 / 2.9, 2^16 5.2 and 5.1 forward; C 6, 2^15 3.3 / 2.6
//   and 3.0 / 3.0.
template <typename T, typename... P>
int launch_shared_for(int n, int c, size_t s, hipStream_t st, P... p)
{
    constexpr bool kForward = sizeof...(P) == 2, kFloat = sizeof(T) == 4;
    const size_t pixels = s * n, cus = chip_units();
    if (c > 32 || pixels > cus * (!kForward ? 64 : kFloat ? 128 : 256) || c <= (kForward && !kFloat ? 4 : 8))
        return kNoSplit;
    constexpr int kLanes = kForward ? 32 : 16;
    if constexpr (kForward && !kFloat)
    {
        if (c <= 8) return launch_shared<8, kLanes>(p..., n, c, s, st);
    }
    if (c <= 16) return launch_shared<16, kLanes>(p..., n, c, s, st);
    return launch_shared<32, kLanes>(p..., n, c, s, st);
}

// Calls f(elements a lane, lanes) with constants for samples of `size` contiguous elements that
// lanes hold in registers: a wave while samples are short, or many (it needs no barrier), else
// a workgroup, of 1024 threads with up to MAX_LARGE elements each where 256 would have more than 16.
// A workgroup from 257 elements on, and from 513 also of more than `some` samples: a wave's chain of up to 32 loads,
// exponentials and stores is what else is waited for (sums of the data's type have fewer terms in a row so; the last
// bits of a sample of channels differ between the two, and so go with the number of samples). GPU time, a wave a sample
// -> a workgroup, forward / backward in us: channels, floats N 16, 1000 3.1 / 2.4 -> 2.2 / 1.8, N 466, 1983 5.1 / 4.2
// -> 3.3 / 2.9, N 1418, 1480 6.7 / 6.0 -> 5.6 / 5.4; doubles N 59, 1480 6.6 / 3.8 -> 3.3 / 2.3, N 700, 1000 5.7 / 4.5
// -> 4.3 / 3.8, N 1418, 704 6.4 / 5.6 -> 5.7 / 5.2; instances of doubles N 128, 1983 8.6 / 4.6 -> 4.0 / 2.7 (at the
// line, channels, floats N 2048, 600 4.0 / 3.3 -> 4.2 / 3.3, 1000 5.2 / 5.2 both ways). Up to 512 elements, a wave and
// a workgroup: channels, floats, 300 and 400 elements, N 466 2.3 / 1.9 and 2.3 / 1.8, N 512 2.3 / 2.0 and 2.3 / 1.9, N
// 600 2.4 / 2.0 and 2.4 / 1.9, N 700 2.3 / 1.9 and 2.4 / 1.8, N 768 2.4 / 2.0 and 2.6 / 1.9, N 1000 2.4 / 1.9 and 2.8 /
// 1.9; doubles, 400, N 512 3.4 / 2.4 and 2.7 / 2.1, N 768 3.5 / 2.4 and 3.0 / 2.3; instances, floats, 400, N 700 3.0 /
// 2.2 and 2.7 / 2.1, N 850 3.1 / 2.2 and 3.0 / 2.2, N 1418 3.1 / 2.3 and 3.4 / 2.6; N 2600 the same either way.
template <int MAX_LARGE = 0, typename F>
int with_lanes(int n, size_t size, int some, const F& f)
{
#define H2X_LANES(CPL, LANES)                                                                      \
    return f(std::integral_constant<int, CPL>(), std::integral_constant<int, LANES>())
    if (size <= 1 * kWaveSize) H2X_LANES(1, kWaveSize);
    if (size <= 2 * kWaveSize) H2X_LANES(2, kWaveSize);
    if (size <= 4 * kWaveSize) H2X_LANES(4, kWaveSize);
    if (n > (size <= 2 * kBlockSize ? some : kManySamples))
    {
        if (size <= 8 * kWaveSize) H2X_LANES(8, kWaveSize);
        if (size <= 16 * kWaveSize) H2X_LANES(16, kWaveSize);
        if (size <= 32 * kWaveSize) H2X_LANES(32, kWaveSize);
    }
    if (size <= 4 * kBlockSize) H2X_LANES(4, kBlockSize);
    if (size <= 8 * kBlockSize) H2X_LANES(8, kBlockSize);
    if (size <= 16 * kBlockSize) H2X_LANES(16, kBlockSize);
    if constexpr (MAX_LARGE == 0)
    {
        H2X_LANES(32, kBlockSize);
    }
    else
    {
        if (size <= 8 * 1024) H2X_LANES(8, 1024);
        if (MAX_LARGE > 16 && size <= 16 * 1024) H2X_LANES(16, 1024);
        H2X_LANES(MAX_LARGE, 1024);
    }
#undef H2X_LANES
}

template <int LANES>
unsigned int lanes_grid(int n)
{
    constexpr unsigned int samples = lanes_block<LANES>() / LANES;
    return (static_cast<unsigned int>(n) + samples - 1) / samples;
}

// Pixels a lane up to 32 channels, of those that alignment and registers allow.  A lane runs a chain of loads,
// exponentials and stores as long as the channels times its pixels: with fewer than 2^18 pixels one, which
// leaves more wavefronts, to 2^20 two; two also where tensors are large enough to come from memory.  Forward + backward,
// us, 4, 2 and 1 a lane, going round three sets of tensors: N 1, C 16, 128 x 128 11.5, 7.9, 6.9; N 2, C 12,
// 256 x 256 12.9, 10.3, 9.3; N 4, C 16, 256 x 256 21.2, 17.7, 17.7; N 8, C 16, 256 x 256 32.8, 29.7, 33.1; N 16, C 16,
// 256 x 256 52.8 and 55.0; N 32, C 16, 256 x 256 108 and 104; N 1, C 32, 256 x 256, by 2 and 1, 15.7 and 12.4.
// (Still fewer pixels go to launch_shared_for.)
int pixels_a_lane(int widest, size_t pixels, size_t bytes)
{
    constexpr size_t kOnePixel = size_t(1) << 18, kTwoPixels = size_t(1) << 20, kFromMemory = size_t(68) << 20;
    return pixels < kOnePixel ? 1 : pixels < kTwoPixels || bytes >= kFromMemory ? std::min(widest, 2) : widest;
}

template <typename T>
int forward_impl(int n, int c, size_t s, const void* xv, void* yv, hipStream_t st)
{
    const T* x = static_cast<const T*>(xv);
    T* y = static_cast<T*>(yv);
    constexpr int kWords = sizeof(T) / 4;
    if (s == 1 && c <= 32 * kBlockSize)
        return with_lanes(n, c, kWords == 1 ? kSomeRows : kSomeSamples, [&](auto cpl, auto lanes) {
            constexpr int CPL = decltype(cpl)::value, LANES = decltype(lanes)::value;
            launch(softmax_fwd_row_kernel<T, CPL, LANES>, lanes_grid<LANES>(n), lanes_block<LANES>(), st, x, y, c, n);
            return launch_status();
        });
    if (s == 1)
    {
        launch(softmax_fwd_long_row_kernel<T>, n, kBlockSize, st, x, y, c);
        return launch_status();
    }
    const int widest = s < kFlatBelow ? 1 : vector_width<T>(s, 4 / kWords, {xv, yv});
    const bool stream = streamed<T>(widest, n, c, s);
    const int v4 = pixels_a_lane(widest, n * s, n * s * c * sizeof(T));
    if (const int shared = launch_shared_for<T>(n, c, s, st, x, y); shared != kNoSplit)
        return shared;
#define H2X_FWD(V, CM)                                                                             \
    do                                                                                             \
    {                                                                                              \
        launch_fwd<T, V, CM>(x, y, n, c, s, stream, st);                                                \
        return launch_status();                                                                    \
    } while (0)
    if constexpr (sizeof(T) == 4)
    {
        // 4 pixels per thread only while the channel values fit in 64 registers;
        // above that 2 pixels per thread run faster (config 4, 21 channels:
        // 29.5 us against 32.5 us), with twice the workgroups in flight
        if (v4 == 4)
        {
            if (c <= 8) H2X_FWD(4, 8);
            if (c <= 16) H2X_FWD(4, 16);
        }
        if (v4 >= 2)
        {
            if (c <= 8) H2X_FWD(2, 8);
            if (c <= 16) H2X_FWD(2, 16);
            if (c <= 32) H2X_FWD(2, 32);
        }
        if (c <= 8) H2X_FWD(1, 8);
        if (c <= 16) H2X_FWD(1, 16);
        if (c <= 32) H2X_FWD(1, 32);
    }
    else
    {
        if (v4 == 2)
        {
            if (c <= 8) H2X_FWD(2, 8);
            if (c <= 16) H2X_FWD(2, 16);
            if (c <= 32) H2X_FWD(2, 32);
        }
        if (c <= 8) H2X_FWD(1, 8);
        if (c <= 16) H2X_FWD(1, 16);
        if (c <= 32) H2X_FWD(1, 32);
    }
#undef H2X_FWD
    const int status = launch_split_for<T>(widest, n, c, s, st, x, y);
    if (status != kNoSplit)
        return status;
    const int flat = flat_samples(n, s);
    WideTiles tiles;
    const dim3 grid = wide_grid(s, kWaveSize, 1, n, flat, &tiles);
    launch(softmax_fwd_wide_kernel<T>, grid, kBlockSize, st, x, y, c, s, flat, tiles);
    return launch_status();
}

template <typename T>
int backward_impl(int n, int c, size_t s, const void* yv, const void* dyv, void* dxv,
                  hipStream_t st)
{
    const T* y = static_cast<const T*>(yv);
    const T* dy = static_cast<const T*>(dyv);
    T* dx = static_cast<T*>(dxv);
    constexpr int kWords = sizeof(T) / 4;
    if (s == 1 && c <= 32 * kBlockSize)
        return with_lanes(n, c, kSomeSamples, [&](auto cpl, auto lanes) {
            constexpr int CPL = decltype(cpl)::value, LANES = decltype(lanes)::value;
            launch(softmax_bwd_row_kernel<T, CPL, LANES>, lanes_grid<LANES>(n), lanes_block<LANES>(), st, y, dy,
                   dx, c, n);
            return launch_status();
        });
    if (s == 1)
    {
        launch(softmax_bwd_long_row_kernel<T>, n, kBlockSize, st, y, dy, dx, c);
        return launch_status();
    }
    const int widest = s < kFlatBelow ? 1 : vector_width<T>(s, 4 / kWords, {yv, dyv, dxv});
    const bool stream = streamed<T>(widest, n, c, s);
    const int v4 = pixels_a_lane(widest, n * s, n * s * c * sizeof(T));
    if (const int shared = launch_shared_for<T>(n, c, s, st, y, dy, dx); shared != kNoSplit)
        return shared;
#define H2X_BWD(V, CM)                                                                             \
    do                                                                                             \
    {                                                                                              \
        launch_bwd<T, V, CM>(y, dy, dx, n, c, s, stream, st);                                           \
        return launch_status();                                                                    \
    } while (0)
    if constexpr (sizeof(T) == 4)
    {
        if (v4 == 4)
        {
            if (c <= 8) H2X_BWD(4, 8);
            if (c <= 16) H2X_BWD(4, 16);
        }
        if (v4 >= 2)
        {
            if (c <= 8) H2X_BWD(2, 8);
            if (c <= 16) H2X_BWD(2, 16);
            if (c <= 32) H2X_BWD(2, 32);
        }
        if (c <= 8) H2X_BWD(1, 8);
        if (c <= 16) H2X_BWD(1, 16);
        if (c <= 32) H2X_BWD(1, 32);
    }
    else
    {
        if (v4 == 2)
        {
            if (c <= 8) H2X_BWD(2, 8);
            if (c <= 16) H2X_BWD(2, 16);
        }
        if (c <= 8) H2X_BWD(1, 8);
        if (c <= 16) H2X_BWD(1, 16);
        if (c <= 32) H2X_BWD(1, 32);
    }
#undef H2X_BWD
    const int status = launch_split_for<T>(widest, n, c, s, st, y, dy, dx);
    if (status != kNoSplit)
        return status;
    const int flat = flat_samples(n, s);
    WideTiles tiles;
    const dim3 grid = wide_grid(s, kWaveSize, 1, n, flat, &tiles);
    launch(softmax_bwd_wide_kernel<T>, grid, kBlockSize, st, y, dy, dx, c, s, flat, tiles);
    return launch_status();
}

// ---- instance mode -----------------------------------------------------------
// Softmax over all elements of a sample (legacy/src/dnn_backend/softmax.cu:179-536,
// 705-784): per-sample maximum, exp(x - max) with per-sample sum, y / sum clamped
// to sqrt(min_normal); backward: per-sample dot product, then the gradient.  The
// reference finishes its per-sample reductions with atomics; here every
// workgroup stores a partial (fp64 for sums) and a second small kernel combines
// them in index order.  A sample is a contiguous block of `sample_size`
// elements (dense tensor), so every pass is a plain 16-byte stream.

constexpr int kInstUnroll = 4;
constexpr int kInstTargetGroups = 4096;
constexpr int kInstMaxGroupsPerSample = 2048;

int inst_groups_per_sample_max(int num_samples)
{
    const int g = (kInstTargetGroups + num_samples - 1) / (num_samples > 0 ? num_samples : 1);
    return g < 8 ? 8 : (g > kInstMaxGroupsPerSample ? kInstMaxGroupsPerSample : g);
}

enum InstReduce : int
{
    kInstMax = 0,   // max x                       -> T partial
    kInstExpSum = 1, // y = exp(x - max); sum y     -> double partial
    kInstDot = 2,    // sum y * dy                  -> double partial
    kInstSumExp = 3  // sum exp(x - max), y untouched -> double partial
};

// Partials of a reduction that the kernel which needs its result combines itself: a launch of one
// workgroup a sample between the two costs 4 to 5 us, each workgroup reading up to a few
// hundred partials less than one.  (First workgroup of a sample: stores the result.)
template <typename T>
struct InstPartials
{
    const double* first; // of sample 0
    int groups;
    T* result;
};

// The maximum over a workgroup, in every thread.
__device__ __forceinline__ double inst_block_max(double m, double* lds)
{
    m = wave_max(m);
    if ((threadIdx.x & (kWaveSize - 1)) == 0)
        lds[threadIdx.x / kWaveSize] = m;
    __syncthreads();
    double r = lds[0];
#pragma unroll
    for (int w = 1; w < kWavesPerBlock; ++w)
        r = lds[w] > r ? lds[w] : r;
    return r;
}

// The maximum of a sample from its partials, in every thread.
template <typename T>
__device__ __forceinline__ T inst_combine_max(const double* mine, int groups, double* lds)
{
    double m = static_cast<double>(Limits<T>::min_normal);
    for (int g = threadIdx.x; g < groups; g += kBlockSize)
        m = mine[g] > m ? mine[g] : m;
    return static_cast<T>(inst_block_max(m, lds));
}

// The sum likewise, in index order.
template <typename T>
__device__ __forceinline__ T inst_combine_sum(const double* mine, int groups, double* lds)
{
    double t[1] = {0.0};
    for (int g = threadIdx.x; g < groups; g += kBlockSize)
        t[0] += mine[g];
    block_sum<1>(t, lds);
    return static_cast<T>(t[0]);
}

// One pass over the chunk [begin, end) of sample n.  a: x (max, exp) or y (dot);
// b: dy (dot); out: y (exp).  Partials are stored as doubles in all modes.
// COMBINE: kInstSumExp makes the maximum of its partials.
template <typename T, int VEC, int MODE, bool COMBINE>
__global__ __launch_bounds__(kBlockSize) void softmax_inst_reduce_kernel(
    const T* __restrict__ a, const T* __restrict__ b, T* __restrict__ out,
    const T* __restrict__ sample_param, double* partials, size_t sample_size, size_t chunk,
    int groups_max, const InstPartials<T> max_partials)
{
    using P = Pack<T, VEC>;
    __shared__ double lds[kWavesPerBlock];
    const int n = blockIdx.y;
    const size_t begin = static_cast<size_t>(blockIdx.x) * chunk;
    const size_t end = begin + chunk < sample_size ? begin + chunk : sample_size;
    const T* ap = a + static_cast<size_t>(n) * sample_size;
    const T* bp = MODE == kInstDot ? b + static_cast<size_t>(n) * sample_size : nullptr;
    T* op = MODE == kInstExpSum ? out + static_cast<size_t>(n) * sample_size : nullptr;
    T shift = T(0);
    if constexpr (COMBINE)
    {
        shift = inst_combine_max<T>(max_partials.first + static_cast<size_t>(n) * groups_max, max_partials.groups, lds);
        if (blockIdx.x == 0 && threadIdx.x == 0)
            max_partials.result[n] = shift;
    }
    else if (MODE == kInstExpSum || MODE == kInstSumExp)
    {
        shift = sample_param[n];
    }
    constexpr size_t kStride = static_cast<size_t>(kBlockSize) * VEC;

    T mx = Limits<T>::min_normal; // softmax.cu:88-99: the maximum starts at min_normal
    double acc = 0.0;
    for (size_t i = begin + threadIdx.x * VEC; i < end; i += kStride * kInstUnroll)
    {
        P va[kInstUnroll], vb[kInstUnroll];
#pragma unroll
        for (int u = 0; u < kInstUnroll; ++u)
            if (i + u * kStride < end)
            {
                va[u] = P::load(ap + i + u * kStride);
                if constexpr (MODE == kInstDot)
                    vb[u] = P::load(bp + i + u * kStride);
            }
#pragma unroll
        for (int u = 0; u < kInstUnroll; ++u)
            if (i + u * kStride < end)
            {
#pragma unroll
                for (int j = 0; j < VEC; ++j)
                {
                    if constexpr (MODE == kInstMax)
                    {
                        mx = va[u][j] >= mx ? va[u][j] : mx;
                    }
                    else if constexpr (MODE == kInstExpSum || MODE == kInstSumExp)
                    {
                        const T e = exp_t(va[u][j] - shift);
                        va[u][j] = e;
                        acc += static_cast<double>(e);
                    }
                    else
                    {
                        acc = __builtin_fma(static_cast<double>(va[u][j]),
                                            static_cast<double>(vb[u][j]), acc);
                    }
                }
                if constexpr (MODE == kInstExpSum)
                    P::store(op + i + u * kStride, va[u]);
            }
    }
    double part;
    if constexpr (MODE == kInstMax)
    {
        mx = wave_max(mx);
        if ((threadIdx.x & (kWaveSize - 1)) == 0)
            lds[threadIdx.x / kWaveSize] = static_cast<double>(mx);
        __syncthreads();
        part = lds[0];
#pragma unroll
        for (int w = 1; w < kWavesPerBlock; ++w)
            part = lds[w] > part ? lds[w] : part;
    }
    else
    {
        double v[1] = {acc};
        block_sum<1>(v, lds);
        part = v[0];
    }
    if (threadIdx.x == 0)
        partials[static_cast<size_t>(n) * groups_max + blockIdx.x] = part;
}

// Combines the partials of every sample in index order.
template <typename T, bool IS_MAX>
__global__ __launch_bounds__(kBlockSize) void softmax_inst_finish_kernel(
    const double* __restrict__ partials, int groups, int groups_max, T* __restrict__ out)
{
    __shared__ double lds[kWavesPerBlock];
    const int n = blockIdx.x;
    const double* mine = partials + static_cast<size_t>(n) * groups_max;
    const T r = IS_MAX ? inst_combine_max<T>(mine, groups, lds) : inst_combine_sum<T>(mine, groups, lds);
    if (threadIdx.x == 0)
        out[n] = r;
}

// kMapNormalize: y = max(y / sum, sqrt(min_normal))  (SoftmaxOp, softmax.cu:424-435);
// kMapGradient:  dx = y > sqrt(min_normal) ? y * (dy - dp) : 0  (bp_compute_func, :483-500);
// kMapFromInput: y = max(exp(x - max) / sum, sqrt(min_normal)): the exponentials are
// made again from x instead of being read back (the same bits: the same function of
// the same arguments), for samples that are whole on this rank.
enum InstMap : int
{
    kMapNormalize = 0,
    kMapGradient = 1,
    kMapFromInput = 2
};

// COMBINE: the sum (or dot product) is made of its partials, not read from sample_param.
template <typename T, int VEC, int KIND, bool COMBINE>
__global__ __launch_bounds__(kBlockSize) void softmax_inst_map_kernel(
    const T* y_in, const T* __restrict__ dy, const T* __restrict__ sample_param,
    const T* __restrict__ sample_shift, T* out, size_t sample_size, T min_output,
    const InstPartials<T> sum_partials, int groups_max)
{
    using P = Pack<T, VEC>;
    const int n = blockIdx.y;
    const size_t i = (static_cast<size_t>(blockIdx.x) * kBlockSize + threadIdx.x) * VEC;
    T p;
    if constexpr (COMBINE)
    {
        __shared__ double lds[kWavesPerBlock];
        p = inst_combine_sum<T>(sum_partials.first + static_cast<size_t>(n) * groups_max, sum_partials.groups, lds);
        if (blockIdx.x == 0 && threadIdx.x == 0)
            sum_partials.result[n] = p;
    }
    if (i >= sample_size)
        return;
    const size_t off = static_cast<size_t>(n) * sample_size + i;
    if constexpr (!COMBINE)
        p = sample_param[n];
    P v = P::load(y_in + off);
    if constexpr (KIND == kMapGradient)
    {
        const P g = P::load(dy + off);
#pragma unroll
        for (int j = 0; j < VEC; ++j)
            v[j] = v[j] > min_output ? v[j] * (g[j] - p) : T(0);
    }
    else
    {
        T shift = T(0);
        if constexpr (KIND == kMapFromInput)
            shift = sample_shift[n];
#pragma unroll
        for (int j = 0; j < VEC; ++j)
        {
            const T e = KIND == kMapFromInput ? exp_t(v[j] - shift) : v[j];
            const T r = e / p;
            v[j] = r > min_output ? r : min_output;
        }
    }
    P::store(out + off, v);
}

// Samples that the lanes of a wave or a workgroup hold in registers (the softmax behind a
// classifier: 10 to a few thousand classes; up to 32 K elements): a reduction is one launch
// without partials, and a whole pass of samples that are whole on this rank is one
// launch too.  Sums are accumulated in fp64, lane by lane and then across the lanes;
// the staged and the fused path add in the same order.
enum InstSmall : int
{
    kSmallMax = 0,     // result[n] = max x
    kSmallExpSum = 1,  // out = exp(x - param[n]); result[n] = sum
    kSmallSumExp = 2,  // result[n] = sum exp(x - param[n])
    kSmallDot = 3,     // result[n] = sum a * b
    kSmallForward = 4, // result[n] = max, result2[n] = sum, out = max(exp(x - max) / sum, min_output)
    kSmallBackward = 5 // result[n] = sum a * b, out = a > min_output ? a * (b - result[n]) : 0
};

template <typename T, int CPL, int MODE, int LANES>
__global__ __launch_bounds__(lanes_block<LANES>()) void softmax_inst_small_kernel(
    const T* __restrict__ a, const T* __restrict__ b, T* __restrict__ out,
    const T* __restrict__ sample_param, T* __restrict__ result, T* __restrict__ result2,
    int sample_size, int num_samples, T min_output)
{
    constexpr bool kDot = MODE == kSmallDot || MODE == kSmallBackward;
    __shared__ double lds[lanes_block<LANES>() / kWaveSize];
    const int lane = threadIdx.x % LANES;
    const int n = blockIdx.x * (lanes_block<LANES>() / LANES) + threadIdx.x / LANES;
    if (n >= num_samples) // all lanes of a sample
        return;
    const size_t base = static_cast<size_t>(n) * sample_size;
    T va[CPL], vb[kDot ? CPL : 1];
#pragma unroll
    for (int k = 0; k < CPL; ++k)
        if (lane + k * LANES < sample_size)
        {
            va[k] = a[base + lane + k * LANES];
            if constexpr (kDot)
                vb[k] = b[base + lane + k * LANES];
        }
    T shift = T(0);
    if constexpr (MODE == kSmallMax || MODE == kSmallForward)
    {
        T mx = Limits<T>::min_normal; // softmax.cu:88-99: the maximum starts at min_normal
#pragma unroll
        for (int k = 0; k < CPL; ++k)
            if (lane + k * LANES < sample_size)
                mx = va[k] >= mx ? va[k] : mx;
        if constexpr (LANES == kWaveSize)
            mx = wave_max(mx);
        else
            mx = static_cast<T>(block_combine<LANES / kWaveSize>(static_cast<double>(mx), true, lds));
        if (lane == 0)
            result[n] = mx;
        if constexpr (MODE == kSmallMax)
            return;
        shift = mx;
    }
    else if constexpr (!kDot)
    {
        shift = sample_param[n];
    }
    double acc = 0.0;
#pragma unroll
    for (int k = 0; k < CPL; ++k)
        if (lane + k * LANES < sample_size)
        {
            if constexpr (kDot)
            {
                acc = __builtin_fma(static_cast<double>(va[k]), static_cast<double>(vb[k]), acc);
            }
            else
            {
                va[k] = exp_t(va[k] - shift);
                acc += static_cast<double>(va[k]);
            }
        }
    const T total = static_cast<T>(lanes_sum<LANES>(acc, lds));
    if (lane == 0)
        (MODE == kSmallForward ? result2 : result)[n] = total;
    if constexpr (MODE == kSmallExpSum || MODE == kSmallForward || MODE == kSmallBackward)
    {
#pragma unroll
        for (int k = 0; k < CPL; ++k)
            if (lane + k * LANES < sample_size)
            {
                if constexpr (MODE == kSmallForward)
                {
                    const T r = va[k] / total;
                    va[k] = r > min_output ? r : min_output;
                }
                else if constexpr (MODE == kSmallBackward)
                {
                    va[k] = va[k] > min_output ? va[k] * (vb[k] - total) : T(0);
                }
                out[base + lane + k * LANES] = va[k];
            }
    }
}

// Elements a lane of 1024 holds.  Twice as many leave one CU too much to do
// (30 samples of 57600: forward 22.0 us, in five launches 16.7).
template <typename T>
constexpr int kInstLargeLanes = 128 / sizeof(T);
template <typename T>
constexpr size_t kInstSmallSample = kInstLargeLanes<T> * size_t(1024);

// Elements of a chunk of samples that a workgroup holds (inst_chunking cuts them so).
template <typename T>
constexpr size_t kInstSmallChunk = size_t(kBlockSize) * (16 / sizeof(T)) * kInstUnroll;

// Whether a workgroup holds a sample whose sums are added in the order of chunks, as those of larger samples are, so
// that a team can run a whole pass (softmax_inst_team_*_kernel), and a workgroup, in whole vectors, any
// (softmax_inst_rounds_kernel). vec: elements of a vector. Single elements: only what teams may take, of the upper
// half; forward + backward, one workgroup's lanes -> in rounds in us, N 2, 12001 floats 10.4 and 10.2, but N 256, 17101
// 22.5 and 23.2, dot products and gradients alone 32 and 34. Lane by lane -> by teams: N 4, 17101 floats 13.7 -> 10.8,
// N 64 15.4 -> 13.7, N 2, 28225 16.7 -> 10.9; N 4, 9001 doubles 13.4 -> 10.0; in place, in rounds, 14.0 -> 12.2, 15.4
// -> 13.6, 16.9 -> 14.9, 13.6 -> 12.4.
template <typename T>
bool inst_by_chunks(int n, size_t sample_size, int vec)
{
    if (n <= 0 || sample_size > kInstSmallSample<T> || sample_size <= kInstSmallChunk<T>)
        return false;
    const size_t chunks = (sample_size + kInstSmallChunk<T> - 1) / kInstSmallChunk<T>;
    return vec == 16 / sizeof(T) || (chunks > 4 && chunks * n <= 2 * chip_units());
}

// Elements of a vector that the tensors of a call allow.
template <typename T>
int inst_vector(size_t sample_size, const void* a, const void* b, const void* out)
{
    return vector_width<T>(sample_size, 16 / sizeof(T), {a, b ? b : a, out ? out : a});
}

// Whether the lanes of a wave or a workgroup hold a sample, each adding up its own elements. (Asked before anything is
// cut: the host's part of a small call is what it is bound by, and samples of one chunk go by lanes whatever the
// vectors are.)
template <typename T>
bool inst_by_lanes(int n, size_t sample_size, const void* a, const void* b, const void* out)
{
    return n > 0 && sample_size <= kInstSmallSample<T>
           && (sample_size <= kInstSmallChunk<T> || !inst_by_chunks<T>(n, sample_size, inst_vector<T>(sample_size, a, b, out)));
}

template <typename T, int MODE>
int inst_small(int n, size_t sample_size, const void* a, const void* b, void* out,
               const void* param, void* result, void* result2, T min_output, hipStream_t st)
{
    return with_lanes<kInstLargeLanes<T>>(n, sample_size, kSomeSamples, [&](auto cpl, auto lanes) {
        constexpr int CPL = decltype(cpl)::value, LANES = decltype(lanes)::value;
        launch(softmax_inst_small_kernel<T, CPL, MODE, LANES>, lanes_grid<LANES>(n), lanes_block<LANES>(), st,
               static_cast<const T*>(a), static_cast<const T*>(b), static_cast<T*>(out),
               static_cast<const T*>(param), static_cast<T*>(result), static_cast<T*>(result2),
               static_cast<int>(sample_size), n, min_output);
        return launch_status();
    });
}

#include "h2x_softmax_team.hpp"

template <typename T>
T inst_min_output()
{
    return static_cast<T>(std::sqrt(static_cast<double>(Limits<T>::min_normal))); // softmax.cu:156-160
}

struct InstChunking
{
    size_t chunk;
    int groups;
};

// Partials of a sample that a workgroup combines for itself: one a thread.  Samples of more are large enough
// for the finishing launch not to count.
constexpr int kInstCombine = kBlockSize;

// Bytes of a chunk up to which a sample is cut into no more chunks than a workgroup combines, or a team
// holds: 16, 32 or 64 KB for one, two or more samples, which leaves a reduction its workgroups (N 1, 3,000,001
// floats: max and sum of exponentials 5.8 and 8.0 us, in chunks of 48 KB 6.4 and 10.1; N 2, 2,097,152 4.6 and 8.1 us, in
// chunks of 32 KB 4.7 and 7.8).
size_t inst_chunk_bytes(int num_samples)
{
    return size_t(kBlockSize) * 16 * (num_samples <= 1 ? 4 : num_samples == 2 ? 8 : 16);
}

// Samples that are no whole vectors are cut as those of whole vectors are: with chunks a quarter of that, members of four chunks
// hold 16 KB, and there are four times as many (forward + backward, by teams, N 23, 142,071 floats 59.7 -> 27.5 us, N 12, 241,997
// 50.7 -> 26.9; separate launches 37 and 35). Few samples leave CUs idle with members of four such chunks, and are cut
// finer up to three quarters of a round of the chip (N 2, 138,475 doubles, 34 and 68 members, 17.3 and 16.0; N 2,
// 439,890 floats 19.6 and 18.7). Chunks of more than 32 KB pay there only if members of four fill most of one round of
// the chip (N 5, 3,054,213 floats, 315 members, 143 us, in chunks of 16 KB, and no teams, 122; N 3, 2,097,657, 129
// members, 59 and 54; with 144 to 256 members the same either way).
InstChunking inst_chunking(size_t sample_size, int num_samples, int vec, size_t elem_bytes)
{
    const size_t gmax = inst_groups_per_sample_max(num_samples);
    const auto cut = [&](size_t bytes, size_t tile) {
        const size_t chunk = std::max((sample_size + gmax - 1) / gmax,
                                      std::min((sample_size + kInstCombine - 1) / kInstCombine, bytes / elem_bytes));
        InstChunking c;
        c.chunk = (chunk + tile - 1) / tile * tile;
        c.groups = static_cast<int>((sample_size + c.chunk - 1) / c.chunk);
        return c;
    };
    const size_t most = inst_chunk_bytes(num_samples), tile = kBlockSize * (16 / elem_bytes) * kInstUnroll;
    const InstChunking c = cut(most, tile);
    if (vec * elem_bytes == 16)
        return c;
    const auto members = [&](const InstChunking& of) { return static_cast<size_t>((of.groups + 3) / 4) * num_samples; };
    if (c.chunk * elem_bytes <= (size_t(32) << 10))
    {
        const InstChunking fine = cut(most, tile / (16 / elem_bytes));
        return c.groups > kInstCombine / 4 && fine.groups <= kInstCombine && members(fine) <= 192 ? fine : c;
    }
    return c.groups <= kInstCombine && members(c) > 140 && members(c) <= 256 ? c : cut(size_t(16) << 10, tile);
}

// How a reduction over samples is cut.  out: takes part in the choice of the vector width.
template <typename T>
InstChunking inst_plan(int n, size_t sample_size, const void* a, const void* b, const void* out, int* v)
{
    *v = inst_vector<T>(sample_size, a, b, out);
    return inst_chunking(sample_size, n, *v, sizeof(T));
}

// One reduction, or a whole pass, of few samples that a workgroup holds, added in the order of chunks.
template <typename T, int MODE>
int inst_rounds(int n, size_t sample_size, const void* a, const void* b, void* out, const void* param, void* result, void* result2,
                T min_output, hipStream_t st)
{
    constexpr int kFull = 16 / sizeof(T);
    int v;
    // (dx of a whole pass is as aligned as its inputs)
    const InstChunking ch = inst_plan<T>(n, sample_size, a, b, MODE == kSmallBackward ? nullptr : out, &v);
    if (ch.chunk != kInstSmallChunk<T> || ch.groups > 8)
        return H2X_ERR_INVALID_ARGUMENT; // (never: see inst_chunking)
    const auto run = [&](auto vec, auto rounds) {
        constexpr int VEC = decltype(vec)::value, ROUNDS = decltype(rounds)::value;
        launch(softmax_inst_rounds_kernel<T, VEC, kInstSmallChunk<T> / kBlockSize / VEC, ROUNDS, MODE>, n, 4 * kBlockSize, st,
               static_cast<const T*>(a), static_cast<const T*>(b), static_cast<T*>(out), static_cast<const T*>(param),
               static_cast<T*>(result), static_cast<T*>(result2), static_cast<uint32_t>(sample_size), min_output);
    };
    const auto wide = [&](auto vec) {
        if (ch.groups <= 4)
            run(vec, std::integral_constant<int, 1>());
        else
            run(vec, std::integral_constant<int, 2>());
    };
    if (v == kFull)
        wide(std::integral_constant<int, kFull>());
    else // (teams have more than four chunks)
        run(std::integral_constant<int, 1>(), std::integral_constant<int, 2>());
    return launch_status();
}

// The partial sums of a reduction at `partials` (groups_max of them a sample); no finishing launch.
template <typename T, int MODE, bool COMBINE = false>
void inst_partials(int n, size_t sample_size, const void* a, const void* b, void* out, const void* param,
                   double* partials, hipStream_t st,
                   const InstPartials<T>& max_partials = InstPartials<T>())
{
    constexpr int kFull = 16 / sizeof(T);
    int v;
    const InstChunking ch = inst_plan<T>(n, sample_size, a, b, out, &v);
    const int gmax = inst_groups_per_sample_max(n);
    const dim3 grid(ch.groups, n);
    if (v == kFull)
        launch(softmax_inst_reduce_kernel<T, kFull, MODE, COMBINE>, grid, kBlockSize, st, static_cast<const T*>(a),
               static_cast<const T*>(b), static_cast<T*>(out), static_cast<const T*>(param), partials, sample_size,
               ch.chunk, gmax, max_partials);
    else
        launch(softmax_inst_reduce_kernel<T, 1, MODE, COMBINE>, grid, kBlockSize, st, static_cast<const T*>(a),
               static_cast<const T*>(b), static_cast<T*>(out), static_cast<const T*>(param), partials, sample_size,
               ch.chunk, gmax, max_partials);
}

template <typename T, int MODE>
int inst_reduce(int n, size_t sample_size, const void* a, const void* b, void* out,
                const void* param, void* result, void* workspace, hipStream_t st)
{
    if ((MODE == kInstMax && n > 0 && sample_size <= kInstSmallSample<T>) // (a maximum in any order)
        || inst_by_lanes<T>(n, sample_size, a, b, out))
    {
        constexpr int kSmallMode = MODE == kInstMax      ? kSmallMax
                                   : MODE == kInstExpSum ? kSmallExpSum
                                   : MODE == kInstSumExp ? kSmallSumExp
                                                         : kSmallDot;
        return inst_small<T, kSmallMode>(n, sample_size, a, b, out, param, result, nullptr, T(0), st);
    }
    int v;
    const int groups = inst_plan<T>(n, sample_size, a, b, out, &v).groups;
    if constexpr (MODE == kInstExpSum || MODE == kInstDot) // (kInstSumExp is of whole passes of larger samples)
        if (inst_by_chunks<T>(n, sample_size, v))
            return inst_rounds<T, MODE == kInstDot ? kSmallDot : kSmallExpSum>(n, sample_size, a, b, out, param, result, nullptr, T(0), st);
    double* partials = static_cast<double*>(workspace);
    inst_partials<T, MODE>(n, sample_size, a, b, out, param, partials, st);
    launch(softmax_inst_finish_kernel<T, MODE == kInstMax>, n, kBlockSize, st, partials,
           groups, inst_groups_per_sample_max(n), static_cast<T*>(result));
    return launch_status();
}

template <typename T, int KIND, bool COMBINE = false>
int inst_map(int n, size_t sample_size, const void* y, const void* dy, const void* param,
             const void* shift, void* out, hipStream_t st,
             const InstPartials<T>& sum_partials = InstPartials<T>())
{
    constexpr int kFull = 16 / sizeof(T);
    const int v = vector_width<T>(sample_size, kFull, {y, dy ? dy : y, out});
    const int gmax = inst_groups_per_sample_max(n);
    const T min_output = inst_min_output<T>();
    if (v == kFull)
        launch(softmax_inst_map_kernel<T, kFull, KIND, COMBINE>, pixel_grid(sample_size, kFull, n), kBlockSize, st,
               static_cast<const T*>(y), static_cast<const T*>(dy), static_cast<const T*>(param),
               static_cast<const T*>(shift), static_cast<T*>(out), sample_size, min_output, sum_partials, gmax);
    else
        launch(softmax_inst_map_kernel<T, 1, KIND, COMBINE>, pixel_grid(sample_size, 1, n), kBlockSize, st,
               static_cast<const T*>(y), static_cast<const T*>(dy), static_cast<const T*>(param),
               static_cast<const T*>(shift), static_cast<T*>(out), sample_size, min_output, sum_partials, gmax);
    return launch_status();
}

// Vectors of 16 bytes a thread that members of four chunks hold at most: beyond, 1024 threads lack the registers.
constexpr int kInstMostForward = 16, kInstMostBackward = 8;

// What a forward pass by members of four chunks takes more than one in separate launches, in us: by the bytes, and for every
// round of the chip, which holds two members of up to four vectors a thread a CU, or one larger one (of eight, whose
// team may fill a quarter of the chip, the second ones start late), what it needs for its loads, two exchanges and
// stores. Fitted to 353 calls, forward with backward; the way it names makes both 0.1 to 0.2 % longer than the faster
// one on average (also of 170 calls not fitted to), 3.9 at most, always teams 0.6, 0.5 and (single elements) 0.1, never
// 6.8, 6.4 and 15.7 %. Members of one chunk, and backward passes, which exchange once, are never slower than separate
// launches. Forward + backward, separate launches, by teams: N 1, 760,320 floats 16.7 and 17.8; N 2, 1,853,544 27.3 and
// 28.1; N 7, 1,280,796, more than a round, 62 and 61; N 24, 318,008 45.2 and 38.8; N 7, 264,306 23.2 and 19.2; N 4,
// 915,840 doubles 43.3 and 38.7.
struct InstForwardCost
{
    float base, per_mb, per_mb_beyond, per_round[3], wait; // beyond: 40 MB; per_round: of 64, 128, 256 KB; wait: of a round, for 64 members
};
// whole vectors of floats and of doubles, single elements
constexpr InstForwardCost kInstForwardCost[3] = {{-2.19f, -0.179f, -0.292f, {0.71f, 2.1f, 4.91f}, 4.17f},
                                                 {-0.52f, -0.182f, -0.155f, {-0.75f, 0.51f, 7.41f}, 3.17f},
                                                 {-7.29f, -0.419f, 0.04f, {5.79f, 5.13f, 15.2f}, 3.93f}};

bool inst_forward_pays(const InstForwardCost& cost, size_t bytes, size_t members, size_t n, int each)
{
    const float mb = bytes * 1e-6f, on_chip = static_cast<float>(chip_units() * (each <= 4 ? 2 : 1));
    const float round = cost.per_round[each <= 4 ? 0 : each <= 8 ? 1 : 2] + cost.wait * members / 64;
    return cost.base + cost.per_mb * mb + cost.per_mb_beyond * std::max(mb - 40, 0.0f) + std::ceil(members * n / on_chip) * round < 0;
}

// A team for samples cut as the staged sums are, or false: of up to 64 members of one chunk, or of four (see
// h2x_softmax_team.hpp).  Members fit a CU once at least, so a team is within a quarter of the chip.
template <typename T, bool FORWARD>
bool inst_team(int n, size_t sample_size, const void* a, const void* b, const void* out, int* v, InstTeam* g)
{
    constexpr int most = FORWARD ? kInstMostForward : kInstMostBackward;
    if (n <= 0 || sample_size <= kInstSmallChunk<T>)
        return false;
    if (inst_by_lanes<T>(n, sample_size, a, b, out))
        return false;
    const InstChunking ch = inst_plan<T>(n, sample_size, a, b, out, v);
    const int each = static_cast<int>(ch.chunk / kBlockSize / (16 / sizeof(T))); // vectors of 16 bytes
    const int chunks = ch.groups <= static_cast<int>(kInstMembers) ? 1 : 4;
    const int members = (ch.groups + chunks - 1) / chunks;
    // Of what a workgroup holds, samples of more than four chunks, of which there are few. One workgroup each and by
    // teams, us: N 64, 5 chunks of floats 11.6 and 12.2, of doubles 11.3 and 11.9, N 32 11.0 and 9.9; N 128, 5 chunks
    // 15.2 and 15.9, doubles 14.1 and 15.6; N 96, 7 chunks 19.7 and 17.4, N 128 22.0 and 20.8; N 128, 8 chunks 23.8 and
    // 22.6, N 256 39.4 and 38.1 before a workgroup's first round went without comparisons (37.5 so).
    if (inst_by_chunks<T>(n, sample_size, *v))
    {
        const int cus = static_cast<int>(compute_units());
        if (ch.groups <= 4 || !(2 * members * n <= 3 * cus || (ch.groups >= 6 && 2 * n <= cus)))
            return false;
    }
    static_assert(4 * kInstMembers >= kInstCombine, "members of four hold all chunks");
    if (ch.groups > kInstCombine || each > (chunks == 1 ? 16 : most) || 4 * members > static_cast<int>(compute_units()))
        return false;
    if (FORWARD && chunks == 4 && each >= 4 // (members of finer chunks are few, and pay)
        && !inst_forward_pays(kInstForwardCost[*v != 16 / sizeof(T) ? 2 : sizeof(T) == 8], n * sample_size * sizeof(T), members, n, each))
        return false;
    g->members = make_fastdiv(static_cast<uint32_t>(members));
    g->chunks = static_cast<uint32_t>(chunks);
    g->sample_size = static_cast<uint32_t>(sample_size); // up to 256 chunks of 64 KB
    g->chunk = static_cast<uint32_t>(ch.chunk);
    return true;
}

// Calls f(threads, elements a vector, vectors a thread) with constants.
template <typename T, int MOST, typename F>
void inst_team_variant(const InstTeam& g, int v, const F& f)
{
    using std::integral_constant;
    constexpr int kFull = 16 / sizeof(T);
    const size_t each = g.chunk / kBlockSize; // elements of a thread
    const auto with = [&](auto team, auto vec) {
        constexpr int kMost = kFull * 16 / decltype(vec)::value;
        constexpr bool kAll = decltype(team)::value == kBlockSize;
        if (each <= kFull * 4)
            f(team, vec, integral_constant<int, kMost / 4>());
        else if (kAll || MOST >= 8)
        {
            if (each <= kFull * 8)
                f(team, vec, integral_constant<int, kAll || MOST >= 8 ? kMost / 2 : kMost / 4>());
            else if (kAll || MOST >= 16)
                f(team, vec, integral_constant<int, kAll || MOST >= 16 ? kMost : kMost / 4>());
        }
    };
    const auto wide = [&](auto vec) {
        if (g.chunks == 1)
            with(integral_constant<int, kBlockSize>(), vec);
        else
            with(integral_constant<int, 4 * kBlockSize>(), vec);
    };
    if (v == kFull)
        wide(integral_constant<int, kFull>());
    else
        wide(integral_constant<int, 1>());
}

// Forward pass of samples that are whole on this rank: maximum, sum of the
// exponentials (y is not written), y from x: 4 tensor passes instead of 5, and three
// launches instead of five where a sample has few partials (N 1, 158 652 elements 15.1 -> 9.8 us, backward, which saves
// one of three, 9.9 -> 7.2; N 16, 86 016 15.0 -> 11.6 and 9.8 -> 8.4).
template <typename T>
int inst_forward_local(int n, size_t sample_size, const void* x, void* y, void* sample_max,
                       void* sample_exp, void* workspace, hipStream_t st)
{
    if (inst_by_lanes<T>(n, sample_size, x, nullptr, y))
        return inst_small<T, kSmallForward>(n, sample_size, x, nullptr, y, nullptr, sample_max,
                                            sample_exp, inst_min_output<T>(), st);
    int v;
    const int sums = inst_plan<T>(n, sample_size, x, nullptr, y, &v).groups;
    if (inst_by_chunks<T>(n, sample_size, v))
        return inst_rounds<T, kSmallForward>(n, sample_size, x, nullptr, y, nullptr, sample_max, sample_exp, inst_min_output<T>(), st);
    // `y` takes part in the choice of the vector width only, as in the staged call,
    // so that the sum is cut up and added in the same order
    int v_x;
    const int maxima = inst_plan<T>(n, sample_size, x, nullptr, nullptr, &v_x).groups;
    // the partials of both reductions lie side by side in the workspace
    if (n > 0 && maxima <= kInstCombine && sums <= kInstCombine && maxima + sums <= inst_groups_per_sample_max(n))
    {
        double* const partials = static_cast<double*>(workspace);
        inst_partials<T, kInstMax>(n, sample_size, x, nullptr, nullptr, nullptr, partials, st);
        inst_partials<T, kInstSumExp, true>(n, sample_size, x, nullptr, y, nullptr, partials + maxima, st,
                                            InstPartials<T>{partials, maxima, static_cast<T*>(sample_max)});
        return inst_map<T, kMapFromInput, true>(n, sample_size, x, nullptr, nullptr, sample_max, y, st,
                                                InstPartials<T>{partials + maxima, sums, static_cast<T*>(sample_exp)});
    }
    int err = inst_reduce<T, kInstMax>(n, sample_size, x, nullptr, nullptr, nullptr, sample_max,
                                       workspace, st);
    if (!err)
        err = inst_reduce<T, kInstSumExp>(n, sample_size, x, nullptr, y, sample_max, sample_exp,
                                          workspace, st);
    return err ? err : inst_map<T, kMapFromInput>(n, sample_size, x, nullptr, sample_exp, sample_max, y, st);
}

template <typename T>
int inst_backward_local(int n, size_t sample_size, const void* y, const void* dy, void* dx, void* sample_dp,
                        void* workspace, hipStream_t st)
{
    if (inst_by_lanes<T>(n, sample_size, y, dy, nullptr))
        return inst_small<T, kSmallBackward>(n, sample_size, y, dy, dx, nullptr, sample_dp, nullptr,
                                             inst_min_output<T>(), st);
    int v;
    const int sums = inst_plan<T>(n, sample_size, y, dy, nullptr, &v).groups;
    const bool by_chunks = inst_by_chunks<T>(n, sample_size, v);
    if (by_chunks && vector_width<T>(sample_size, v, {dx}) == v) // dx takes no part in the cut
        return inst_rounds<T, kSmallBackward>(n, sample_size, y, dy, dx, nullptr, sample_dp, nullptr, inst_min_output<T>(), st);
    if (n > 0 && sums <= kInstCombine && !by_chunks)
    {
        double* const partials = static_cast<double*>(workspace);
        inst_partials<T, kInstDot>(n, sample_size, y, dy, nullptr, nullptr, partials, st);
        return inst_map<T, kMapGradient, true>(n, sample_size, y, dy, nullptr, nullptr, dx, st,
                                         InstPartials<T>{partials, sums, static_cast<T*>(sample_dp)});
    }
    const int err = inst_reduce<T, kInstDot>(n, sample_size, y, dy, nullptr, nullptr, sample_dp, workspace, st);
    return err ? err : inst_map<T, kMapGradient>(n, sample_size, y, dy, sample_dp, nullptr, dx, st);
}

// By teams, or false.  polls: looks at what the others have stored, of about a microsecond.
template <typename T>
bool inst_forward_team(int n, size_t sample_size, const void* x, void* y, void* sample_max, void* sample_exp,
                       void* state, uint32_t polls, hipStream_t st)
{
    InstTeam g;
    int v;
    if (!state || !inst_team<T, true>(n, sample_size, x, nullptr, y, &v, &g)
        || !apart(x, y, n * sample_size * sizeof(T)))
        return false;
    g.max_polls = polls;
    g.states = static_cast<unsigned long long*>(state);
    inst_team_variant<T, kInstMostForward>(g, v, [&](auto team, auto vec, auto vectors) {
        constexpr int TEAM = decltype(team)::value, VEC = decltype(vec)::value, V = decltype(vectors)::value;
        launch(softmax_inst_team_forward_kernel<T, TEAM, VEC, V>, g.members.divisor * n, TEAM, st,
               static_cast<const T*>(x), static_cast<T*>(y), static_cast<T*>(sample_max), static_cast<T*>(sample_exp),
               g, inst_min_output<T>());
    });
    return true;
}

template <typename T>
bool inst_backward_team(int n, size_t sample_size, const void* y, const void* dy, void* dx, void* sample_dp,
                        void* state, uint32_t polls, hipStream_t st)
{
    InstTeam g;
    int v;
    const size_t bytes = n * sample_size * sizeof(T);
    if (!state || !inst_team<T, false>(n, sample_size, y, dy, nullptr, &v, &g) || !apart(y, dx, bytes)
        || !apart(dy, dx, bytes) || vector_width<T>(sample_size, v, {dx}) != v) // the outputs take no part in the cut
        return false;
    g.max_polls = polls;
    g.states = static_cast<unsigned long long*>(state);
    inst_team_variant<T, kInstMostBackward>(g, v, [&](auto team, auto vec, auto vectors) {
        constexpr int TEAM = decltype(team)::value, VEC = decltype(vec)::value, V = decltype(vectors)::value;
        launch(softmax_inst_team_backward_kernel<T, TEAM, VEC, V>, g.members.divisor * n, TEAM, st,
               static_cast<const T*>(y), static_cast<const T*>(dy), static_cast<T*>(dx), static_cast<T*>(sample_dp), g,
               inst_min_output<T>());
    });
    return true;
}

bool inst_bad(int num_samples, size_t sample_size)
{
    return num_samples < 0 || num_samples > 65535
           || (sample_size + kBlockSize - 1) / kBlockSize > 0x7fffffffull;
}

} // namespace
} // namespace h2x

using namespace h2x;

extern "C" int h2x_softmax_channel_forward(h2x_dtype dtype, int num_samples, int num_channels,
                                           size_t spatial_size, const void* x, void* y,
                                           h2x_stream_t stream)
{
    if (num_samples < 0 || num_channels < 0)
        return H2X_ERR_INVALID_ARGUMENT;
    if (num_samples == 0 || num_channels == 0 || spatial_size == 0)
        return H2X_SUCCESS; // empty local tensor: softmax.cu:600-603
    if (!x || !y)
        return H2X_ERR_INVALID_ARGUMENT;
    if (num_samples > 65535 || (spatial_size + kWaveSize - 1) / kWaveSize > 0x7ffffff0ull)
        return H2X_ERR_TOO_LARGE;
    switch (dtype)
    {
    case H2X_F32:
        return forward_impl<float>(num_samples, num_channels, spatial_size, x, y, as_stream(stream));
    case H2X_F64:
        return forward_impl<double>(num_samples, num_channels, spatial_size, x, y, as_stream(stream));
    }
    return H2X_ERR_UNSUPPORTED;
}

extern "C" int h2x_softmax_channel_backward(h2x_dtype dtype, int num_samples, int num_channels,
                                            size_t spatial_size, const void* y, const void* dy,
                                            void* dx, h2x_stream_t stream)
{
    if (num_samples < 0 || num_channels < 0)
        return H2X_ERR_INVALID_ARGUMENT;
    if (num_samples == 0 || num_channels == 0 || spatial_size == 0)
        return H2X_SUCCESS;
    if (!y || !dy || !dx)
        return H2X_ERR_INVALID_ARGUMENT;
    if (num_samples > 65535 || (spatial_size + kWaveSize - 1) / kWaveSize > 0x7ffffff0ull)
        return H2X_ERR_TOO_LARGE;
    switch (dtype)
    {
    case H2X_F32:
        return backward_impl<float>(num_samples, num_channels, spatial_size, y, dy, dx, as_stream(stream));
    case H2X_F64:
        return backward_impl<double>(num_samples, num_channels, spatial_size, y, dy, dx, as_stream(stream));
    }
    return H2X_ERR_UNSUPPORTED;
}

// ---- instance mode -------------------------------------------------------------

extern "C" size_t h2x_softmax_instance_workspace_bytes(int num_samples)
{
    const size_t n = num_samples > 0 ? num_samples : 1;
    return (n * inst_groups_per_sample_max(num_samples) * sizeof(double) + 255) / 256 * 256;
}

#define H2X_INST_ENTRY(CALL_F32, CALL_F64)                                                         \
    if (inst_bad(num_samples, sample_size))                                                        \
        return num_samples < 0 ? H2X_ERR_INVALID_ARGUMENT : H2X_ERR_TOO_LARGE;                     \
    if (num_samples == 0 || sample_size == 0)                                                      \
        return H2X_SUCCESS;                                                                        \
    switch (dtype)                                                                                 \
    {                                                                                              \
    case H2X_F32: return CALL_F32;                                                                 \
    case H2X_F64: return CALL_F64;                                                                 \
    }                                                                                              \
    return H2X_ERR_UNSUPPORTED

extern "C" int h2x_softmax_instance_max(h2x_dtype dtype, int num_samples, size_t sample_size,
                                        const void* x, void* sample_max, void* workspace,
                                        h2x_stream_t stream)
{
    if (!x || !sample_max || !workspace)
        return num_samples == 0 || sample_size == 0 ? H2X_SUCCESS : H2X_ERR_INVALID_ARGUMENT;
    H2X_INST_ENTRY((inst_reduce<float, kInstMax>(num_samples, sample_size, x, nullptr, nullptr, nullptr,
                                                 sample_max, workspace, as_stream(stream))),
                   (inst_reduce<double, kInstMax>(num_samples, sample_size, x, nullptr, nullptr,
                                                  nullptr, sample_max, workspace, as_stream(stream))));
}

extern "C" int h2x_softmax_instance_exp(h2x_dtype dtype, int num_samples, size_t sample_size,
                                        const void* x, const void* sample_max, void* y,
                                        void* sample_exp, void* workspace, h2x_stream_t stream)
{
    if (!x || !sample_max || !y || !sample_exp || !workspace)
        return num_samples == 0 || sample_size == 0 ? H2X_SUCCESS : H2X_ERR_INVALID_ARGUMENT;
    H2X_INST_ENTRY((inst_reduce<float, kInstExpSum>(num_samples, sample_size, x, nullptr, y, sample_max,
                                                    sample_exp, workspace, as_stream(stream))),
                   (inst_reduce<double, kInstExpSum>(num_samples, sample_size, x, nullptr, y,
                                                     sample_max, sample_exp, workspace,
                                                     as_stream(stream))));
}

extern "C" int h2x_softmax_instance_normalize(h2x_dtype dtype, int num_samples, size_t sample_size,
                                              const void* sample_exp, void* y, h2x_stream_t stream)
{
    if (!sample_exp || !y)
        return num_samples == 0 || sample_size == 0 ? H2X_SUCCESS : H2X_ERR_INVALID_ARGUMENT;
    H2X_INST_ENTRY((inst_map<float, kMapNormalize>(num_samples, sample_size, y, nullptr, sample_exp,
                                                   nullptr, y, as_stream(stream))),
                   (inst_map<double, kMapNormalize>(num_samples, sample_size, y, nullptr, sample_exp,
                                                    nullptr, y, as_stream(stream))));
}

extern "C" int h2x_softmax_instance_dot(h2x_dtype dtype, int num_samples, size_t sample_size,
                                        const void* y, const void* dy, void* sample_dp,
                                        void* workspace, h2x_stream_t stream)
{
    if (!y || !dy || !sample_dp || !workspace)
        return num_samples == 0 || sample_size == 0 ? H2X_SUCCESS : H2X_ERR_INVALID_ARGUMENT;
    H2X_INST_ENTRY((inst_reduce<float, kInstDot>(num_samples, sample_size, y, dy, nullptr, nullptr,
                                                 sample_dp, workspace, as_stream(stream))),
                   (inst_reduce<double, kInstDot>(num_samples, sample_size, y, dy, nullptr, nullptr,
                                                  sample_dp, workspace, as_stream(stream))));
}

extern "C" int h2x_softmax_instance_gradient(h2x_dtype dtype, int num_samples, size_t sample_size,
                                             const void* y, const void* dy, const void* sample_dp,
                                             void* dx, h2x_stream_t stream)
{
    if (!y || !dy || !sample_dp || !dx)
        return num_samples == 0 || sample_size == 0 ? H2X_SUCCESS : H2X_ERR_INVALID_ARGUMENT;
    H2X_INST_ENTRY((inst_map<float, kMapGradient>(num_samples, sample_size, y, dy, sample_dp, nullptr,
                                                  dx, as_stream(stream))),
                   (inst_map<double, kMapGradient>(num_samples, sample_size, y, dy, sample_dp, nullptr,
                                                   dx, as_stream(stream))));
}

extern "C" int h2x_softmax_instance_forward_local(h2x_dtype dtype, int num_samples,
                                                  size_t sample_size, const void* x, void* y,
                                                  void* sample_max, void* sample_exp,
                                                  void* workspace, h2x_stream_t stream)
{
    if (!x || !y || !sample_max || !sample_exp || !workspace)
        return num_samples == 0 || sample_size == 0 ? H2X_SUCCESS : H2X_ERR_INVALID_ARGUMENT;
    H2X_INST_ENTRY((inst_forward_local<float>(num_samples, sample_size, x, y, sample_max, sample_exp,
                                              workspace, as_stream(stream))),
                   (inst_forward_local<double>(num_samples, sample_size, x, y, sample_max, sample_exp,
                                               workspace, as_stream(stream))));
}

extern "C" int h2x_softmax_instance_backward_local(h2x_dtype dtype, int num_samples, size_t sample_size,
                                                   const void* y, const void* dy, void* dx, void* sample_dp,
                                                   void* workspace, h2x_stream_t stream)
{
    if (!y || !dy || !dx || !sample_dp || !workspace)
        return num_samples == 0 || sample_size == 0 ? H2X_SUCCESS : H2X_ERR_INVALID_ARGUMENT;
    H2X_INST_ENTRY((inst_backward_local<float>(num_samples, sample_size, y, dy, dx, sample_dp, workspace,
                                               as_stream(stream))),
                   (inst_backward_local<double>(num_samples, sample_size, y, dy, dx, sample_dp, workspace,
                                                as_stream(stream))));
}

// Looks from which a member works out what it misses (2 ms against the microseconds of a launch).
constexpr int kInstPolls = 2048;

extern "C" size_t h2x_softmax_instance_state_needed(h2x_dtype dtype, int num_samples, size_t sample_size)
{
    if ((dtype != H2X_F32 && dtype != H2X_F64) || num_samples <= 0 || inst_bad(num_samples, sample_size))
        return 0;
    const auto team = [&](auto zero) {
        InstTeam g;
        int v;
        return inst_team<decltype(zero), true>(num_samples, sample_size, nullptr, nullptr, nullptr, &v, &g)
               || inst_team<decltype(zero), false>(num_samples, sample_size, nullptr, nullptr, nullptr, &v, &g);
    };
    return (dtype == H2X_F32 ? team(0.0f) : team(0.0)) ? num_samples * kInstStateWords * sizeof(unsigned long long) : 0;
}

extern "C" int h2x_softmax_instance_forward_once(h2x_dtype dtype, int num_samples, size_t sample_size, const void* x,
                                                 void* y, void* sample_max, void* sample_exp, void* workspace,
                                                 void* state, int max_polls, h2x_stream_t stream)
{
    if (!x || !y || !sample_max || !sample_exp || !workspace)
        return num_samples == 0 || sample_size == 0 ? H2X_SUCCESS : H2X_ERR_INVALID_ARGUMENT;
    const uint32_t polls = max_polls < 0 ? kInstPolls : max_polls;
    if (!inst_bad(num_samples, sample_size)
        && (dtype == H2X_F32   ? inst_forward_team<float>(num_samples, sample_size, x, y, sample_max, sample_exp, state,
                                                          polls, as_stream(stream))
            : dtype == H2X_F64 ? inst_forward_team<double>(num_samples, sample_size, x, y, sample_max, sample_exp,
                                                           state, polls, as_stream(stream))
                               : false))
        return launch_status();
    return h2x_softmax_instance_forward_local(dtype, num_samples, sample_size, x, y, sample_max, sample_exp, workspace,
                                              stream);
}

extern "C" int h2x_softmax_instance_backward_once(h2x_dtype dtype, int num_samples, size_t sample_size, const void* y,
                                                  const void* dy, void* dx, void* sample_dp, void* workspace,
                                                  void* state, int max_polls, h2x_stream_t stream)
{
    if (!y || !dy || !dx || !sample_dp || !workspace)
        return num_samples == 0 || sample_size == 0 ? H2X_SUCCESS : H2X_ERR_INVALID_ARGUMENT;
    const uint32_t polls = max_polls < 0 ? kInstPolls : max_polls;
    if (!inst_bad(num_samples, sample_size)
        && (dtype == H2X_F32   ? inst_backward_team<float>(num_samples, sample_size, y, dy, dx, sample_dp, state, polls,
                                                           as_stream(stream))
            : dtype == H2X_F64 ? inst_backward_team<double>(num_samples, sample_size, y, dy, dx, sample_dp, state,
                                                            polls, as_stream(stream))
                               : false))
        return launch_status();
    return h2x_softmax_instance_backward_local(dtype, num_samples, sample_size, y, dy, dx, sample_dp, workspace,
                                               stream);
}
