// Batch-norm of double tensors of a rank that shares its statistics with no one, for short segments:
// every element read once, with the bits of the staged calls.  Included by h2x_bn.hip after h2x_bn_ordered.hpp.
//
// The staged short-segment reduction gives each slot (vector) of a channel's segment a lane a row, which adds the
// samples row, row + rows, ... of a range; the slots of a row are added as a tree, then the rows and the ranges one
// after the other.  Which channels share a workgroup does not matter to that order.  Here a workgroup holds all samples of a
// few neighbouring channels in its registers: a lane plays a slot and a row of some ranges, the sums of its ranges go
// to LDS, waves add the trees there, and y (dx) is written from the registers.
//
// Bound by launches and waits where tensors are small, else by memory and by registers that a range which is no whole number
// of a lane's vectors leaves idle.  Two launches each way -> this, forward + backward, us going round three sets of tensors:
//   N 8, C 1685, 3 x 3       17.8 -> 11.6      N 30, C 1225, 10 x 11    56.9 -> 42.6
//   N 128, C 512, 7 x 7      52.5 -> 33.8      N 32, C 2048, 7 x 7      47.1 -> 32.8
//   N 64, C 256, 14 x 14     43.9 -> 31.7      N 60, C 1406, 4 x 6, halo of 1   55.2 -> 39.8
// and 150 drawn calls on average 0.76 of their time.
#pragma once

struct ShortOnceGeometry
{
    uint32_t row;          // elements that are contiguous
    FastDiv slots_per_row; // vectors a row is padded to
    FastDiv slots;         // of a segment
    FastDiv h;             // rows of a plane
    int64_t sy, sz;        // strides of rows and planes
    uint32_t stride_n;     // the last element of a channel is less than 2^30 elements from its first
    int64_t stride_c;
    FastDiv channels;      // of a workgroup
    FastDiv rows;          // of lanes, a range of samples
    FastDiv turns;         // samples of a lane in a range
    uint32_t per, ranges;  // samples of a range, ranges
    uint32_t together;     // ranges that are played at once
    uint32_t passes;       // and how often: range p * together + q is that of lane group q in pass p
    uint32_t num_samples, num_channels;
};

// Haloed tensors of one geometry whose output's halo is cleared.
struct ShortOnceClearing : ShortOnceGeometry
{
    HaloCells halo;
};

// What a lane plays.
struct ShortOnceLane
{
    uint32_t at;      // of its slot, from the start of the window's first channel and of the sample
    uint32_t skip;    // leading elements of its vector that belong to the slot before it
    uint32_t channel; // of the window
    uint32_t q, row;
    bool live;
};

template <int VEC>
__host__ __device__ __forceinline__ ShortOnceLane short_once_lane(const ShortOnceGeometry& g, uint32_t window, uint32_t t)
{
    ShortOnceLane l;
    const uint32_t run = fastdiv(t, g.slots), slot = t - run * g.slots.divisor;
    const uint32_t lane_row = fastdiv(run, g.channels);
    l.channel = run - lane_row * g.channels.divisor;
    l.q = fastdiv(lane_row, g.rows);
    l.row = lane_row - l.q * g.rows.divisor;
    const uint32_t line = fastdiv(slot, g.slots_per_row);
    const uint32_t x = (slot - line * g.slots_per_row.divisor) * VEC, last = g.row - VEC;
    const uint32_t first = x < last ? x : last;
    const uint32_t z = fastdiv(line, g.h), y = line - z * g.h.divisor;
    l.skip = x - first;
    l.at = static_cast<uint32_t>(l.channel * g.stride_c + first + y * g.sy + z * g.sz);
    l.live = l.q < g.together && window * g.channels.divisor + l.channel < g.num_channels;
    return l;
}

// Sample of the lane's vector i of pass p; at least num_samples: there is none.
__host__ __device__ __forceinline__ uint32_t short_once_sample(const ShortOnceGeometry& g, const ShortOnceLane& l, uint32_t p,
                                                               uint32_t i)
{
    const uint32_t range = p * g.together + l.q, of_range = l.row + i * g.rows.divisor;
    return of_range < g.per && range < g.ranges ? range * g.per + of_range : ~0u;
}

// Terms 0 to n - 1, one after the other; n is uniform and at least 1. An addition that waits for the read before it
// takes 100 clocks: they are read ahead of the additions, eight at a time. (The sums of a range and those of the ranges
// by a thread each, reads ahead, against one thread a channel, read by read, forward + backward in us: N 254, C 149, 3
// x 3 16.5 -> 13.1, N 243, C 1065, 1 x 1 13.2 -> 10.7; N 18, C 776, 15 x 15 43.5 -> 35.8; N 148, C 334, 5 x 5 23.7 ->
// 22.5; 55 drawn calls 0.97. In finish_short, whose workgroups have two to eight rows, the reads beyond the last row
// cost more than they save: N 67, C 55, 9 x 11 21.1 and 22.4.)
template <typename F>
__device__ __forceinline__ double sum_in_order(uint32_t n, const F& term)
{
    constexpr uint32_t kBatch = 8;
    double t = term(0);
    for (uint32_t i = 1; i < n; i += kBatch)
    {
        double w[kBatch];
#pragma unroll
        for (uint32_t j = 0; j < kBatch; ++j)
            w[j] = term(i + j < n ? i + j : n - 1);
#pragma unroll
        for (uint32_t j = 0; j < kBatch; ++j)
            if (i + j < n)
                t += w[j];
    }
    return t;
}

// The N sums of a lane's channel from what the lanes have left in sums[k][pass][thread], in the order of finish_short and
// sequential_totals.
template <int TEAM, int PASSES, int N, typename G>
__device__ __forceinline__ void short_once_totals(const G& g, const ShortOnceLane& l, double (&v)[N],
                                                  double (&sums)[N][PASSES][TEAM])
{
    const uint32_t slots = g.slots.divisor, channels = g.channels.divisor, rows = g.rows.divisor;
    const uint32_t lane = threadIdx.x % kWaveSize, wave = threadIdx.x / kWaveSize;
    __syncthreads();
    if (slots > 1) // uniform
    {
        // a tree is one lane's, or of as many lanes as its slots are padded to, up to a wave
        const uint32_t width = 2u << (31 - __builtin_clz(slots - 1)), lanes = width < kWaveSize ? width : kWaveSize;
        const uint32_t at_once = kWaveSize / lanes, slot = lane & (lanes - 1);
        const uint32_t runs = g.together * rows * channels, trees = runs * g.passes * N;
        uint32_t first = wave * at_once; // uniform
        // Backward, which has twice the trees: two of them at once wait for their exchanges together (forward +
        // backward in us, one by one and so: N 18, C 386, 8 x 9 15.5 and 14.9; N 15, C 136, 7 x 10 with a halo 11.8 and
        // 11.2; N 42, C 271, 4 x 6 12.4 and 11.9; forward, four at once, or trees wider than a wave 2 to 10 % longer;
        // where a large output's halo is cleared, and what waits longer spreads the stores, N 158, C 610, 7 x 4 68.5
        // and 70.4).
        if constexpr (N == 4 && !std::is_same<G, ShortOnceClearing>::value)
            if (width <= kWaveSize)
                for (constexpr uint32_t kStep = TEAM / kWaveSize; first + kStep * at_once < trees; first += 2 * kStep * at_once)
                {
                    double* leaves[2];
                    double t[2];
                    bool mine[2];
#pragma unroll
                    for (int i = 0; i < 2; ++i)
                    {
                        const uint32_t tree = first + i * kStep * at_once + lane / lanes;
                        const uint32_t kind = tree / runs, run = tree - kind * runs;
                        leaves[i] = &sums[0][0][0] + (kind % N * PASSES + kind / N) * TEAM + run * slots;
                        mine[i] = tree < trees;
                        t[i] = mine[i] && slot < slots ? leaves[i][slot] : 0.0;
                    }
                    for (uint32_t step = lanes / 2; step >= 1; step /= 2)
                    {
                        const double o[2] = {__shfl_down(t[0], step), __shfl_down(t[1], step)};
                        if (slot < step && slot + step < slots)
                        {
                            t[0] += o[0];
                            t[1] += o[1];
                        }
                    }
#pragma unroll
                    for (int i = 0; i < 2; ++i)
                        if (mine[i] && slot == 0)
                            leaves[i][0] = t[i]; // read by this wave alone, above
                }
        for (; first < trees; first += TEAM / kWaveSize * at_once)
        {
            const uint32_t tree = first + lane / lanes;
            const uint32_t kind = tree / runs, run = tree - kind * runs;
            const uint32_t k = kind % N, p = kind / N;
            double* const leaves = &sums[0][0][0] + (k * PASSES + p) * TEAM + run * slots;
            const bool mine = tree < trees;
            double t = mine && slot < slots ? leaves[slot] : 0.0;
            if (width > kWaveSize)
            {
                if (width > 2 * kWaveSize && slot + 2 * kWaveSize < slots)
                    t += leaves[slot + 2 * kWaveSize];
                if (slot + kWaveSize < slots)
                {
                    double o = leaves[slot + kWaveSize];
                    if (width > 2 * kWaveSize && slot + 3 * kWaveSize < slots)
                        o += leaves[slot + 3 * kWaveSize];
                    t += o;
                }
            }
            for (uint32_t step = lanes / 2; step >= 1; step /= 2)
            {
                const double o = __shfl_down(t, step);
                if (slot < step && slot + step < slots)
                    t += o;
            }
            if (mine && slot == 0)
                leaves[0] = t; // read by this wave alone, above
        }
        __syncthreads();
    }
    // the rows of each range, then the ranges, each of them by a thread
    const auto top = [&](uint32_t k, uint32_t range, uint32_t c) {
        uint32_t p = 0;
#pragma unroll
        for (int i = 1; i < PASSES; ++i)
            p += range >= i * g.together;
        return &sums[k][p][((range - p * g.together) * rows * channels + c) * slots];
    };
    if (rows > 1) // uniform
        for (uint32_t i = threadIdx.x; i < channels * N * g.ranges; i += TEAM)
        {
            const uint32_t of_sum = fastdiv(i, g.channels);
            uint32_t k = 0;
#pragma unroll
            for (int n = 1; n < N; ++n)
                k += of_sum >= n * g.ranges;
            double* const first = top(k, of_sum - k * g.ranges, i - of_sum * channels);
            *first = sum_in_order(rows, [&](uint32_t r) { return first[r * channels * slots]; }); // read by this thread alone
        }
    if (g.ranges > 1)
    {
        __syncthreads();
        for (uint32_t i = threadIdx.x; i < channels * N; i += TEAM)
        {
            const uint32_t k = fastdiv(i, g.channels), c = i - k * channels;
            sums[k][0][c * slots] = sum_in_order(g.ranges, [&](uint32_t range) { return *top(k, range, c); });
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < N; ++k)
        v[k] = sums[k][0][l.channel * slots];
}

// Ranges that one thread plays, at most: a workgroup keeps the sums of each of its threads for each.  Backward no more than leave
// the CU as many workgroups as its registers do (four ranges, or two by 1024 threads, 1.012 times as long on average, N
// 10, C 52, 13 x 15 11.7 and 15.0 us).
constexpr int short_once_passes(int vectors, bool forward)
{
    return forward ? 4 : vectors / 4;
}

// The vectors of a lane: f(u, n) for vector u of sample n, between them done(p) where those of a pass end.
template <int K, typename F, typename D>
__device__ __forceinline__ void short_once_each(const ShortOnceGeometry& g, const ShortOnceLane& l, const F& f, const D& done)
{
#pragma unroll
    for (int u = 0; u < K; ++u)
    {
        const uint32_t p = fastdiv(u, g.turns), i = u - p * g.turns.divisor;
        if (p >= g.passes) // uniform
            continue;
        const uint32_t n = short_once_sample(g, l, p, i);
        if (n < g.num_samples)
            f(u, n);
        if (i + 1 == g.turns.divisor)
            done(p);
    }
}

template <int VEC, int TEAM, int K, typename G>
__global__ __launch_bounds__(TEAM) void bn_short_once_forward_kernel(const G g, const OnceForward<double> a)
{
    typedef double T;
    constexpr int kPasses = short_once_passes(K, true);
    __shared__ double sums[2][kPasses][TEAM];
    const uint32_t window = xcd_contiguous(blockIdx.x, gridDim.x);
    if (window * g.channels.divisor >= g.num_channels)
        return;
    const ShortOnceLane l = short_once_lane<VEC>(g, window, threadIdx.x);
    const uint32_t first = window * g.channels.divisor, c = l.live ? first + l.channel : first;
    const ChannelParams<T> params(a, c);
    const T* const x = a.x + first * g.stride_c;
    T v[K][VEC];
    const auto none = [](uint32_t) {};
    if (l.live)
        short_once_each<K>(
            g, l, [&](int u, uint32_t n) { load_vec<T, VEC, false>(x + (l.at + n * g.stride_n), v[u]); }, none);
    double s[2] = {0.0, 0.0};
    if (l.live)
        short_once_each<K>(
            g, l,
            [&](int u, uint32_t) {
#pragma unroll
                for (int j = 0; j < VEC; ++j)
                    if (j >= static_cast<int>(l.skip))
                    {
                        s[0] += v[u][j];
                        s[1] += v[u][j] * v[u][j];
                    }
            },
            [&](uint32_t p) {
#pragma unroll
                for (int k = 0; k < 2; ++k)
                {
                    sums[k][p][threadIdx.x] = s[k];
                    s[k] = 0.0;
                }
            });
    short_once_totals<TEAM, kPasses, 2>(g, l, s, sums);
    if constexpr (std::is_same<G, ShortOnceClearing>::value)
        for (uint32_t i = 0; i < g.channels.divisor && first + i < g.num_channels; ++i)
            clear_halo_cells(g.halo, a.y + (first + i) * g.stride_c, threadIdx.x, TEAM);
    if (!l.live)
        return;
    T m, variance;
    sums_to_mean_var(s[0], s[1], a.n, &m, &variance);
    if (threadIdx.x == l.channel * g.slots.divisor)
        params.store_statistics(a, c, m, variance);
    const T inv_stdev = inv_sqrt_t(variance + a.epsilon);
    const T sc = params.scale, bi = params.bias;
    T* const y = a.y + first * g.stride_c;
    short_once_each<K>(
        g, l,
        [&](int u, uint32_t n) {
#pragma unroll
            for (int j = 0; j < VEC; ++j)
                v[u][j] = fma_t((v[u][j] - m) * inv_stdev, sc, bi);
            store_once<T, VEC, false>(y + (l.at + n * g.stride_n), v[u]);
        },
        none);
}

template <int VEC, int TEAM, int K, typename G>
__global__ __launch_bounds__(TEAM) void bn_short_once_backward_kernel(const G g, const OnceBackward<double> a)
{
    typedef double T;
    constexpr int kPasses = short_once_passes(K, false);
    __shared__ double sums[4][kPasses][TEAM];
    const uint32_t window = xcd_contiguous(blockIdx.x, gridDim.x);
    if (window * g.channels.divisor >= g.num_channels)
        return;
    const ShortOnceLane l = short_once_lane<VEC>(g, window, threadIdx.x);
    const uint32_t first = window * g.channels.divisor, c = l.live ? first + l.channel : first;
    const T m = a.mean[c];
    const T sc = a.scale[c];
    const T var = a.var[c];
    const int64_t base = first * g.stride_c;
    T xv[K][VEC], dv[K][VEC];
    const auto none = [](uint32_t) {};
    if (l.live)
        short_once_each<K>(
            g, l,
            [&](int u, uint32_t n) {
                load_vec<T, VEC, false>(a.x + base + (l.at + n * g.stride_n), xv[u]);
                load_vec<T, VEC, false>(a.dy + base + (l.at + n * g.stride_n), dv[u]);
            },
            none);
    const T inv_stdev = inv_sqrt_t(var + a.epsilon);
    const T dvar_factor = inv_stdev * inv_stdev * inv_stdev / T(2);
    const double neg_inv = -inv_stdev, neg_fac = -dvar_factor;
    double s[4] = {0.0, 0.0, 0.0, 0.0};
    if (l.live)
        short_once_each<K>(
            g, l,
            [&](int u, uint32_t) {
                // as in bn_backprop1_short_kernel
#pragma unroll
                for (int j = 0; j < VEC; ++j)
                    if (j >= static_cast<int>(l.skip))
                    {
                        const T xm = xv[u][j] - m;
                        const T dxhat = dv[u][j] * sc;
                        s[0] = __builtin_fma(dv[u][j], xm * inv_stdev, s[0]);
                        s[1] += dv[u][j];
                        s[2] = __builtin_fma(dxhat, neg_inv, s[2]);
                        s[3] = __builtin_fma(dxhat * xm, neg_fac, s[3]);
                    }
            },
            [&](uint32_t p) {
#pragma unroll
                for (int k = 0; k < 4; ++k)
                {
                    sums[k][p][threadIdx.x] = s[k];
                    s[k] = 0.0;
                }
            });
    short_once_totals<TEAM, kPasses, 4>(g, l, s, sums);
    if constexpr (std::is_same<G, ShortOnceClearing>::value)
        for (uint32_t i = 0; i < g.channels.divisor && first + i < g.num_channels; ++i)
            clear_halo_cells(g.halo, a.dx + (first + i) * g.stride_c, threadIdx.x, TEAM);
    if (!l.live)
        return;
    if (threadIdx.x == l.channel * g.slots.divisor)
    {
        a.dscale[c] = s[0];
        a.dbias[c] = s[1];
        a.dmean[c] = s[2];
        a.dvar[c] = s[3];
    }
    const T dmean_term = s[2] / a.n;
    const T dvar_term = s[3] * T(2) / a.n_minus_1;
    short_once_each<K>(
        g, l,
        [&](int u, uint32_t n) {
#pragma unroll
            for (int j = 0; j < VEC; ++j)
                xv[u][j] = fma_t(xv[u][j] - m, dvar_term, fma_t(dv[u][j] * sc, inv_stdev, dmean_term));
            store_once<T, VEC, false>(a.dx + base + (l.at + n * g.stride_n), xv[u]);
        },
        none);
}
