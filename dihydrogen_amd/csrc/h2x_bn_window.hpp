// Batch-norm of a rank that shares its statistics with no one, for dense segments of a few hundred
// bytes: a workgroup loads a window of neighbouring whole channels, all samples, into registers,
// sums them, and writes y (dx) from the registers.  Included by h2x_bn.hip after h2x_bn_once.hpp,
// whose arguments, terms and rounding these kernels share; only the order of the fp64 sums is another.
//
// A segment of 7 x 7 floats lies in two or three lines, most of which the neighbours' segments share.  A
// workgroup a channel, as in h2x_bn_once.hpp, asks for them once each; where two channels are
// served together, an instruction of a wave covers runs of 392 bytes instead of 196, with two thirds of
// the requests.  Bound by memory, and by the wait of a round of workgroups for its last loads:
// N 128, C 1024, 7 x 7, going round three sets of tensors, forward + backward 32.1 -> 26.5 us (4.0 -> 4.85 TB/s of the
// bytes that cannot be done without; copies in the same order and phases 24.9).  Windows of four
// channels 28.7, of two by 512 threads 28.1.
//
// A thread serves one vector of the window, the same in all of its samples: its channel, the elements it skips and the step
// from sample to sample are worked out once.
#pragma once

constexpr uint32_t kWindowChannels = 4; // at most

struct WindowGeometry
{
    uint32_t width;        // elements of a segment
    uint32_t num_channels, samples, channels; // of a window: two or four
    FastDiv spr;           // vectors a segment is padded to
    FastDiv slots;         // vectors of a window
    uint32_t rows;         // samples that a workgroup serves at once
    uint32_t stride_n;     // the last element of a channel is less than 2^30 elements from its first
    int64_t stride_c;
};

// What thread t of a window serves, the same in each of its samples row, row + rows, ...
struct WindowPlace
{
    uint32_t row, first, skip; // element offset within a sample of the window; elements that belong to the vector before
    uint32_t channel, vector;  // of the window, of the segment
    bool live;
};

template <int VEC>
__device__ __forceinline__ WindowPlace window_place(const WindowGeometry& g, uint32_t window, uint32_t t)
{
    WindowPlace p;
    p.row = fastdiv(t, g.slots);
    const uint32_t slot = t - p.row * g.slots.divisor;
    p.channel = fastdiv(slot, g.spr);
    p.vector = slot - p.channel * g.spr.divisor;
    const uint32_t x = p.vector * VEC, last = g.width - VEC;
    const uint32_t at = x < last ? x : last;
    p.skip = x - at;
    p.first = p.channel * static_cast<uint32_t>(g.stride_c) + at;
    p.live = p.row < g.rows && window * g.channels + p.channel < g.num_channels;
    return p;
}

// The N sums of the thread's channel over the threads that share it, in a fixed order: a wave adds up a sum of a channel, whose
// terms lie side by side in LDS.
template <int BLOCK, int N>
__device__ __forceinline__ void window_sum(const WindowGeometry& g, const WindowPlace& p, double (&s)[N],
                                           double (&parts)[N][BLOCK], double (&totals)[kWindowChannels][N])
{
    static_assert(BLOCK / kWaveSize >= kWindowChannels * N, "a wave a sum");
    const uint32_t count = g.rows * g.spr.divisor; // threads of a channel
    if (p.row < g.rows)
#pragma unroll
        for (int k = 0; k < N; ++k)
            parts[k][p.channel * count + p.row * g.spr.divisor + p.vector] = s[k];
    __syncthreads();
    const uint32_t lane = threadIdx.x % kWaveSize, i = threadIdx.x / kWaveSize;
    if (i < g.channels * N) // uniform
    {
        const double* const from = &parts[i % N][i / N * count];
        double v = 0.0;
        for (uint32_t j = lane; j < count; j += 2 * kWaveSize)
            v += from[j] + (j + kWaveSize < count ? from[j + kWaveSize] : 0.0);
        v = wave_sum(v);
        if (lane == 0)
            totals[i / N][i % N] = v;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < N; ++k)
        s[k] = totals[p.channel][k];
}

template <typename T, int BLOCK, int K>
__global__ __launch_bounds__(BLOCK) void bn_window_forward_kernel(const WindowGeometry g, const OnceForward<T> a)
{
    constexpr int VEC = 16 / sizeof(T);
    __shared__ double parts[2][BLOCK], totals[kWindowChannels][2];
    const uint32_t window = xcd_contiguous(blockIdx.x, gridDim.x);
    if (window * g.channels >= g.num_channels)
        return;
    const WindowPlace p = window_place<VEC>(g, window, threadIdx.x);
    const uint32_t c = window * g.channels + p.channel;
    const int64_t base = window * g.channels * g.stride_c;
    const ChannelParams<T> params(a, p.live ? c : 0);
    const T* const x = a.x + base;
    const auto at = [&](int u) { return (p.row + u * g.rows) * g.stride_n + p.first; };
    const auto live = [&](int u) { return p.live && p.row + u * g.rows < g.samples; };
    T v[K][VEC];
#pragma unroll
    for (int u = 0; u < K; ++u)
        if (live(u))
            load_vec<T, VEC, false>(x + at(u), v[u]);
    double s[2] = {0.0, 0.0};
#pragma unroll
    for (int u = 0; u < K; ++u)
        if (live(u))
        {
#pragma unroll
            for (int j = 0; j < VEC; ++j)
                if (j >= static_cast<int>(p.skip))
                {
                    const double d = static_cast<double>(v[u][j]);
                    s[0] += d;
                    s[1] = __builtin_fma(d, d, s[1]);
                }
        }
    window_sum<BLOCK, 2>(g, p, s, parts, totals);
    if (!p.live)
        return;
    T m, variance;
    sums_to_mean_var(static_cast<T>(s[0]), static_cast<T>(s[1]), a.n, &m, &variance);
    if (p.row == 0 && p.vector == 0)
        params.store_statistics(a, c, m, variance);
    const T inv_stdev = inv_sqrt_t(variance + a.epsilon);
    T* const y = a.y + base;
#pragma unroll
    for (int u = 0; u < K; ++u)
        if (live(u))
        {
#pragma unroll
            for (int j = 0; j < VEC; ++j)
                v[u][j] = fma_t((v[u][j] - m) * inv_stdev, params.scale, params.bias);
            store_once<T, VEC, false>(y + at(u), v[u]);
        }
}

template <typename T, int BLOCK, int K>
__global__ __launch_bounds__(BLOCK) void bn_window_backward_kernel(const WindowGeometry g, const OnceBackward<T> a)
{
    constexpr int VEC = 16 / sizeof(T);
    __shared__ double parts[4][BLOCK], totals[kWindowChannels][4];
    const uint32_t window = xcd_contiguous(blockIdx.x, gridDim.x);
    if (window * g.channels >= g.num_channels)
        return;
    const WindowPlace p = window_place<VEC>(g, window, threadIdx.x);
    const uint32_t c = p.live ? window * g.channels + p.channel : 0;
    const int64_t base = window * g.channels * g.stride_c;
    const T m = a.mean[c], sc = a.scale[c], variance = a.var[c];
    const auto at = [&](int u) { return (p.row + u * g.rows) * g.stride_n + p.first; };
    const auto live = [&](int u) { return p.live && p.row + u * g.rows < g.samples; };
    T xv[K][VEC], dv[K][VEC];
#pragma unroll
    for (int u = 0; u < K; ++u)
        if (live(u))
        {
            load_vec<T, VEC, false>(a.x + base + at(u), xv[u]);
            load_vec<T, VEC, false>(a.dy + base + at(u), dv[u]);
        }
    const T inv_stdev = inv_sqrt_t(variance + a.epsilon);
    const T dvar_factor = inv_stdev * inv_stdev * inv_stdev / T(2);
    double s[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int u = 0; u < K; ++u)
        if (live(u))
        {
#pragma unroll
            for (int j = 0; j < VEC; ++j)
                if (j >= static_cast<int>(p.skip))
                {
                    const T xm = xv[u][j] - m;
                    const T dxhat = dv[u][j] * sc;
                    const double dd = static_cast<double>(dv[u][j]);
                    s[0] = __builtin_fma(dd, static_cast<double>(xm * inv_stdev), s[0]);
                    s[1] += dd;
                    s[2] += static_cast<double>(dxhat);
                    s[3] += static_cast<double>(dxhat * xm);
                }
        }
    window_sum<BLOCK, 4>(g, p, s, parts, totals);
    if (!p.live)
        return;
    const T dmean = static_cast<T>(s[2] * -static_cast<double>(inv_stdev));
    const T dvar = static_cast<T>(s[3] * -static_cast<double>(dvar_factor));
    if (p.row == 0 && p.vector == 0)
    {
        a.dscale[c] = static_cast<T>(s[0]);
        a.dbias[c] = static_cast<T>(s[1]);
        a.dmean[c] = dmean;
        a.dvar[c] = dvar;
    }
    const T dmean_term = dmean / a.n;
    const T dvar_term = dvar * T(2) / a.n_minus_1;
#pragma unroll
    for (int u = 0; u < K; ++u)
        if (live(u))
        {
#pragma unroll
            for (int j = 0; j < VEC; ++j)
                xv[u][j] = fma_t(xv[u][j] - m, dvar_term, fma_t(dv[u][j] * sc, inv_stdev, dmean_term));
            store_once<T, VEC, false>(a.dx + base + at(u), xv[u]);
        }
}
