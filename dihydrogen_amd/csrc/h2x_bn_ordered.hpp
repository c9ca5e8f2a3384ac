// Batch-norm of double tensors of a rank that shares its statistics with no one, every
// element read once, with the bits of the staged calls.  Included by h2x_bn.hip after
// h2x_bn_team.hpp.
//
// The staged calls of double tensors are promised bit for bit, so the sums have to be
// added in their order: bn_sums_kernel and bn_backprop1_kernel give each group of 256
// threads some units (chunks of a segment) and leave one partial sum a group, and
// channel_totals adds those, thread t starting with partial t.  Here a workgroup, or a
// team of workgroups where a channel is larger or channels are few, holds the vectors
// of several such groups in its registers: 256 neighbouring threads play one group, one
// after another its passes; the sums of a group are those of the staged workgroup, and the
// partial sums are added along the staged tree.  What the members of a team exchange
// are sums of two or four neighbouring partials, the first steps of that tree.
//
// Bound by memory, and by the wait for the last member of a team.  Two launches each way ->
// this, forward + backward, us going round three sets of tensors:
//   N 8, C 32, 33^3              98 -> 75       N 4, C 64, 56 x 56            19 -> 12.5
//   N 64, C 512, 20 x 20        137 -> 101      N 8, C 100, 64 x 64           40 -> 26
//   N 16, C 32, 112 x 112        70 -> 49       N 12, C 9, 113 x 123, halo    27 -> 21
//   N 4, C 213, 17 x 20 x 23, halo of 1  85 -> 72
// (33^3 is 18 units a segment, the last of them half empty: 144 groups, 36 members.)
#pragma once

struct OrderedGeometry
{
    TensorMap map;         // of every tensor of the call
    uint32_t spatial;      // elements of a (padded) segment
    uint32_t chunk;        // elements of a unit, a multiple of four vectors a thread
    FastDiv per_segment;   // units of a segment
    FastDiv unit_batches;  // batches of four vectors a thread of a unit
    FastDiv group_batches; // of all units of a group
    uint32_t units;        // of a channel; group k takes units k, k + groups, ...
    uint32_t groups;       // of a channel, at most kBlockSize
    uint32_t passes;       // groups that 256 threads of a workgroup play one after another
    uint32_t num_channels;
    FastDiv members;       // of a team
    uint32_t max_polls;
    bool streams_gradient; // backward: dy past the caches
};

// Haloed tensors of one geometry whose output's halo is cleared.
struct OrderedClearing : OrderedGeometry
{
    HaloCells halo;
};

// Zeros in the halo cells of a channel, by threads `at`, at + threads, ... (Whole passes of doubles, forward + backward
// in us, in the staged calls, up to seven launches, and so: N 1, C 115, 49 x 58, halo of 2 30.9 -> 10.7; N 24, C 542, 6
// x 6 36.7 -> 17.8; N 12, C 61, 85 x 84 69 -> 56; 80 drawn calls 0.76 of their time.) Stored normally, as the interior
// is, whose lines they complete in the cache: behind it, or, by the kernels of short segments, before it.
template <typename T>
__device__ __forceinline__ void clear_halo_cells(const HaloCells& g, T* interior, uint32_t at, uint32_t threads)
{
    T* const y = interior - g.origin;
    each_halo_cell(
        g, at, threads, [&](uint32_t i) { y[i] = T(0); },
        [&](uint32_t i) {
            const T zeros[2] = {T(0), T(0)};
            store_once<T, 2, false>(y + i, zeros);
        });
}

constexpr int kOrderedBatch = 4; // vectors a thread: kUnroll of the staged kernels
constexpr uint32_t kNowhere = ~0u;

// Vector j of batch `batch` of a group, of its thread t: element offset from the start of the
// channel, times two, plus the element it skips; kNowhere: there is none.  (Offsets below 2^30.)
template <bool ROWS>
__host__ __device__ __forceinline__ uint32_t ordered_place(const OrderedGeometry& g, uint32_t group, uint32_t batch,
                                                           uint32_t j, uint32_t t)
{
    const uint32_t round = fastdiv(batch, g.unit_batches);
    const uint32_t unit = group + round * g.groups;
    if (group >= g.groups || unit >= g.units)
        return kNowhere;
    const uint32_t n = fastdiv(unit, g.per_segment);
    const uint32_t begin = (unit - n * g.per_segment.divisor) * g.chunk;
    const uint32_t end = begin + g.chunk < g.spatial ? begin + g.chunk : g.spatial;
    const uint32_t slot = (batch - round * g.unit_batches.divisor) * kOrderedBatch + j;
    const uint32_t i = begin + (slot * kBlockSize + t) * 2;
    if (i + 2 > end)
        return kNowhere;
    const uint32_t start = n * static_cast<uint32_t>(g.map.stride_n);
    if constexpr (!ROWS)
        return (start + i) * 2;
    Place pl{0, 0, 0, 0};
    place_vector<2>(g.map, row_split<2>(g.map, i, &pl), &pl);
    return (start + static_cast<uint32_t>(row_offset(g.map, pl)) + static_cast<uint32_t>(pl.first)) * 2 + pl.skip;
}

// The group that a thread plays in its pass p, as member `member` of its team.
template <int TEAM>
__host__ __device__ __forceinline__ uint32_t ordered_group(const OrderedGeometry& g, uint32_t member, uint32_t p,
                                                           uint32_t quarter)
{
    return (member * g.passes + p) * (TEAM / kBlockSize) + quarter;
}

// The partial sums of the groups that a member plays, in lds as the sums of their four waves:
// sums[group of the member][wave][k].  add(u, s): the terms of a thread's vector u.
template <int TEAM, int K, int N, typename F>
__device__ __forceinline__ void ordered_partials(const OrderedGeometry& g, double* sums, const F& add)
{
    constexpr int kQuarters = TEAM / kBlockSize;
    const uint32_t wave = threadIdx.x / kWaveSize;
    double s[N];
#pragma unroll
    for (int k = 0; k < N; ++k)
        s[k] = 0.0;
#pragma unroll
    for (int b = 0; b < K / kOrderedBatch; ++b)
    {
        const uint32_t p = fastdiv(b, g.group_batches);
        if (p >= g.passes) // uniform
            continue;
#pragma unroll
        for (int j = 0; j < kOrderedBatch; ++j)
            add(b * kOrderedBatch + j, s);
        if (b - p * g.group_batches.divisor + 1 < g.group_batches.divisor)
            continue;
        const double t = wave_sums_in_order<N>(s);
        if (threadIdx.x % kWaveSize < N)
            sums[((p * kQuarters + wave / kWavesPerBlock) * kWavesPerBlock + wave % kWavesPerBlock) * N
                 + threadIdx.x % kWaveSize] = t;
#pragma unroll
        for (int k = 0; k < N; ++k)
            s[k] = 0.0;
    }
}

// Partial sum k of a group of the member, as block_sum adds its waves; nothing beyond the last group.
template <int N>
__device__ __forceinline__ double ordered_partial(const double* sums, uint32_t local, bool there, int k)
{
    if (!there)
        return 0.0;
    const double* const w = sums + local * kWavesPerBlock * N + k;
    double t = w[0];
#pragma unroll
    for (int i = 1; i < kWavesPerBlock; ++i)
        t += w[i * N];
    return 0.0 + t; // as channel_totals starts
}

// What the waves of a workgroup leave one another.
template <int TEAM, int K, int N, bool TEAMS>
struct OrderedShared
{
    double sums[TEAM / kBlockSize * (K / kOrderedBatch) * kWavesPerBlock * N];
    double waves[N][kWavesPerBlock];              // of the waves of a staged finishing workgroup
    unsigned long long late[TEAMS ? kWavesPerBlock : 1]; // lanes whose sum was not there in time
};

// The totals of those waves.
template <int N>
__device__ __forceinline__ void ordered_totals(double (&v)[N], const double (&waves)[N][kWavesPerBlock])
{
#pragma unroll
    for (int k = 0; k < N; ++k)
    {
        double t = waves[k][0];
#pragma unroll
        for (int w = 1; w < kWavesPerBlock; ++w)
            t += waves[k][w];
        v[k] = t;
    }
}

// The sums of the channel in v[] of every thread, from the partial sums in `shared`.  Teams: a counter, tags and looks as in
// team_exchange; recompute(m) leaves the partial sums of member m in `shared`.  What a thread of channel_totals starts
// with, or the thread in steps of two or four where the members exchange sums of as many partials, the same lane of the
// first four waves looks for; the lanes in between take the other sums, so that the steps of the tree that are left add
// all of them at once. (With a lane an item, all its sums one after another, N 8, C 32, 33^3 forward + backward, took
// 86.2 us, so 75.4; N 24, C 461, 24 x 30 with a halo of 1 98.8 and 86.0; N 16, C 32, 112 x 112 54.7 and 49.0.)
template <int TEAM, int K, int N, bool TEAMS, typename F>
__device__ __forceinline__ void ordered_exchange(double (&v)[N], const OrderedGeometry& g, uint32_t member,
                                                 unsigned long long* state, uint32_t tag,
                                                 OrderedShared<TEAM, K, N, TEAMS>& shared, const F& recompute)
{
    constexpr uint32_t kQuarters = TEAM / kBlockSize;
    const uint32_t t = threadIdx.x, own = g.passes * kQuarters; // groups of a member
    const uint32_t lane = t % kWaveSize, wave = t / kWaveSize;
    __syncthreads();
    if constexpr (!TEAMS)
    {
        if (t < kBlockSize)
        {
#pragma unroll
            for (int k = 0; k < N; ++k)
                v[k] = t < own ? ordered_partial<N>(shared.sums, t, t < g.groups, k) : 0.0;
            const double total = wave_sums_in_order<N>(v);
            if (lane < N)
                shared.waves[lane][wave] = total;
        }
        __syncthreads();
        ordered_totals<N>(v, shared.waves);
    }
    else
    {
        // an item: what the tree makes of two or four neighbouring partial sums
        const uint32_t width = own % 4 == 0 ? 4 : 2, per_member = own / width;
        const uint32_t items = (g.groups + width - 1) / width;
        const auto item_of = [&](uint32_t m, uint32_t i, int k) {
            const auto at = [&](uint32_t j) {
                return ordered_partial<N>(shared.sums, i * width + j, m * own + i * width + j < g.groups, k);
            };
            const double low = at(0) + at(1);
            return width == 2 ? low : low + (at(2) + at(3));
        };
        unsigned long long* const words = state + kCounterWords;
        if (t < per_member * N && member * per_member + t / N < items)
            team_put(words + 2 * (t % N) * items, items, member * per_member + t / N, tag, item_of(member, t / N, t % N));
        // the sums of its item that a lane looks for: one, or, of four with items on every other lane, two
        const uint32_t item = t / width, first = t % width;
        const bool two = N == 4 && width == 2; // uniform
        const bool reads = t < kBlockSize && item < items && first < N;
        double s[2] = {0.0, 0.0};
        const auto leave_waves = [&] {
            if (t >= kBlockSize)
                return;
#pragma unroll
            for (int i = 0; i < 2; ++i)
                if (i == 0 || two)
                {
                    const double total = wave_sum_from(s[i], width);
                    const uint32_t k = first + i * 2;
                    if (lane < width && k < N)
                        shared.waves[k][wave] = total;
                }
        };
        if (t < kBlockSize) // whole waves
        {
            const unsigned long long* const at = words + 2 * first * items + item;
            bool there = !reads;
            uint32_t looks = g.max_polls; // uniform
            if (items > kSmallTeam)
                for (; looks > 1 && __any(!there && first == 0 && team_load(at) >> 32 != tag); --looks)
                {
                    __builtin_amdgcn_s_sleep(4);
                    if (gridDim.x > kCrowd) // uniform
                        __builtin_amdgcn_s_sleep(40);
                }
            for (; looks > 0; --looks)
            {
                if (!there)
                {
                    there = team_look(at, items, tag, &s[0]);
                    if (two)
                        there = team_look(at + 4 * items, items, tag, &s[1]) && there;
                }
                if (__all(there))
                    break;
                __builtin_amdgcn_s_sleep(4);
            }
            if (!there || !reads)
                s[0] = s[1] = 0.0;
            const unsigned long long late = __ballot(!there);
            if (lane == 0)
                shared.late[wave] = late;
            leave_waves();
        }
        __syncthreads();
        if (t == 0)
            team_leave(state);
        unsigned long long late = 0;
#pragma unroll
        for (int w = 0; w < kWavesPerBlock; ++w)
            late |= shared.late[w];
        if (late) // uniform
        {
            for (uint32_t m = 0; m < g.members.divisor; ++m)
            {
                bool missing = false;
                for (uint32_t i = m * per_member; i < (m + 1) * per_member && i < items; ++i)
                    missing = missing
                              || (shared.late[i * width / kWaveSize] >> i * width % kWaveSize & ((1u << width) - 1)) != 0;
                if (!missing) // uniform
                    continue;
                __syncthreads(); // the sums may still be read
                recompute(m);
                __syncthreads();
                if (reads && item / per_member == m)
                {
                    s[0] = item_of(m, item - m * per_member, first);
                    if (two)
                        s[1] = item_of(m, item - m * per_member, first + 2);
                }
            }
            leave_waves();
            __syncthreads();
        }
        ordered_totals<N>(v, shared.waves);
    }
}

// Channel and member of a workgroup.
template <bool TEAMS>
__device__ __forceinline__ uint32_t ordered_channel(const OrderedGeometry& g, uint32_t* member)
{
    if constexpr (!TEAMS)
    {
        *member = 0;
        return xcd_contiguous(blockIdx.x, gridDim.x);
    }
    const uint32_t c = fastdiv(blockIdx.x, g.members);
    *member = team_member(blockIdx.x - c * g.members.divisor, g.members.divisor);
    return c;
}

template <int TEAM, int K, bool TEAMS, bool ROWS, bool STREAM, typename G>
__global__ __launch_bounds__(TEAM, TEAMS ? 4 : 1) void bn_ordered_forward_kernel(const G g, const OnceForward<double> a,
                                                                  unsigned long long* states)
{
    typedef double T;
    constexpr int VEC = 2;
    __shared__ OrderedShared<TEAM, K, 2, TEAMS> shared;
    uint32_t member;
    const uint32_t c = ordered_channel<TEAMS>(g, &member);
    if (c >= g.num_channels)
        return;
    unsigned long long* const state = TEAMS ? states + team_state_at(c) : nullptr;
    uint32_t tag = TEAMS ? team_tag(state) : 0;
    const uint32_t quarter = __builtin_amdgcn_readfirstlane(threadIdx.x / kBlockSize), t = threadIdx.x % kBlockSize;
    const ChannelParams<T> params(a, c);
    const T* const x = a.x + c * g.map.stride_c;
    const auto place = [&](uint32_t m, int u) {
        const uint32_t p = fastdiv(u / kOrderedBatch, g.group_batches);
        return p >= g.passes ? kNowhere
                             : ordered_place<ROWS>(g, ordered_group<TEAM>(g, m, p, quarter),
                                                   u / kOrderedBatch - p * g.group_batches.divisor, u % kOrderedBatch, t);
    };
    const auto terms = [](double (&s)[2], const T (&v)[VEC], uint32_t at) {
#pragma unroll
        for (int j = 0; j < VEC; ++j)
            if (!ROWS || j >= static_cast<int>(at & 1))
            {
                s[0] += v[j];
                s[1] += v[j] * v[j];
            }
    };
    T v[K][VEC];
    uint32_t at[K];
#pragma unroll
    for (int u = 0; u < K; ++u)
    {
        at[u] = place(member, u);
        if (at[u] != kNowhere)
            load_vec<T, VEC, !ROWS>(x + (at[u] >> 1), v[u]);
    }
    ordered_partials<TEAM, K, 2>(g, shared.sums, [&](int u, double (&s)[2]) {
        if (at[u] != kNowhere)
            terms(s, v[u], at[u]);
    });
    if constexpr (TEAMS)
        asm volatile("" : "+v"(tag)); // every wave has it before any stores
    double s[2];
    ordered_exchange<TEAM, K, 2, TEAMS>(s, g, member, state, tag, shared, [&](uint32_t other) {
        ordered_partials<TEAM, K, 2>(g, shared.sums, [&](int u, double (&r)[2]) {
            const uint32_t p = place(other, u);
            if (p == kNowhere)
                return;
            T w[VEC];
            load_vec<T, VEC, !ROWS>(x + (p >> 1), w);
            terms(r, w, p);
        });
    });
    T m, variance;
    sums_to_mean_var(s[0], s[1], a.n, &m, &variance);
    if (member == 0 && threadIdx.x == 0)
        params.store_statistics(a, c, m, variance);
    const T inv_stdev = inv_sqrt_t(variance + a.epsilon);
    const T sc = params.scale, bi = params.bias;
    T* const y = a.y + c * g.map.stride_c;
#pragma unroll
    for (int u = 0; u < K; ++u)
        if (at[u] != kNowhere)
        {
#pragma unroll
            for (int j = 0; j < VEC; ++j)
                v[u][j] = fma_t((v[u][j] - m) * inv_stdev, sc, bi);
            store_once<T, VEC, STREAM>(y + (at[u] >> 1), v[u]);
        }
    if constexpr (std::is_same<G, OrderedClearing>::value)
        clear_halo_cells(g.halo, a.y + c * g.map.stride_c, member * TEAM + threadIdx.x, g.members.divisor * TEAM);
}

template <int TEAM, int K, bool TEAMS, bool ROWS, bool STREAM, bool GRADIENT, typename G>
__global__ __launch_bounds__(TEAM, TEAMS ? 4 : 1) void bn_ordered_backward_kernel(const G g,
                                                                   const OnceBackward<double> a,
                                                                   unsigned long long* states)
{
    typedef double T;
    constexpr int VEC = 2;
    __shared__ OrderedShared<TEAM, K, 4, TEAMS> shared;
    uint32_t member;
    const uint32_t c = ordered_channel<TEAMS>(g, &member);
    if (c >= g.num_channels)
        return;
    unsigned long long* const state = TEAMS ? states + team_state_at(c) : nullptr;
    uint32_t tag = TEAMS ? team_tag(state) : 0;
    const uint32_t quarter = __builtin_amdgcn_readfirstlane(threadIdx.x / kBlockSize), t = threadIdx.x % kBlockSize;
    const int64_t base = c * g.map.stride_c;
    const auto place = [&](uint32_t m, int u) {
        const uint32_t p = fastdiv(u / kOrderedBatch, g.group_batches);
        return p >= g.passes ? kNowhere
                             : ordered_place<ROWS>(g, ordered_group<TEAM>(g, m, p, quarter),
                                                   u / kOrderedBatch - p * g.group_batches.divisor, u % kOrderedBatch, t);
    };
    T xv[K][VEC], dv[K][VEC];
    uint32_t at[K];
#pragma unroll
    for (int u = 0; u < K; ++u)
    {
        at[u] = place(member, u);
        if (at[u] != kNowhere)
        {
            load_vec<T, VEC, !ROWS>(a.x + base + (at[u] >> 1), xv[u]);
            load_vec<T, VEC, !ROWS, GRADIENT>(a.dy + base + (at[u] >> 1), dv[u]);
        }
    }
    const T m = a.mean[c];
    const T sc = a.scale[c];
    const T inv_stdev = inv_sqrt_t(a.var[c] + a.epsilon);
    const T dvar_factor = inv_stdev * inv_stdev * inv_stdev / T(2);
    const double neg_inv = -inv_stdev, neg_fac = -dvar_factor;
    // as in bn_backprop1_kernel
    const auto terms = [&](double (&s)[4], const T (&x)[VEC], const T (&d)[VEC], uint32_t p) {
#pragma unroll
        for (int j = 0; j < VEC; ++j)
            if (!ROWS || j >= static_cast<int>(p & 1))
            {
                const T xm = x[j] - m;
                const T dxhat = d[j] * sc;
                s[0] = __builtin_fma(d[j], xm * inv_stdev, s[0]);
                s[1] += d[j];
                s[2] = __builtin_fma(dxhat, neg_inv, s[2]);
                s[3] = __builtin_fma(dxhat * xm, neg_fac, s[3]);
            }
    };
    ordered_partials<TEAM, K, 4>(g, shared.sums, [&](int u, double (&s)[4]) {
        if (at[u] != kNowhere)
            terms(s, xv[u], dv[u], at[u]);
    });
    if constexpr (TEAMS)
        asm volatile("" : "+v"(tag)); // every wave has it before any stores
    double s[4];
    ordered_exchange<TEAM, K, 4, TEAMS>(s, g, member, state, tag, shared, [&](uint32_t other) {
        ordered_partials<TEAM, K, 4>(g, shared.sums, [&](int u, double (&r)[4]) {
            const uint32_t p = place(other, u);
            if (p == kNowhere)
                return;
            T w[VEC], d[VEC];
            load_vec<T, VEC, !ROWS>(a.x + base + (p >> 1), w);
            load_vec<T, VEC, !ROWS>(a.dy + base + (p >> 1), d);
            terms(r, w, d, p);
        });
    });
    if (member == 0 && threadIdx.x == 0)
    {
        a.dscale[c] = s[0];
        a.dbias[c] = s[1];
        a.dmean[c] = s[2];
        a.dvar[c] = s[3];
    }
    const T dmean_term = s[2] / a.n;
    const T dvar_term = s[3] * T(2) / a.n_minus_1;
#pragma unroll
    for (int u = 0; u < K; ++u)
        if (at[u] != kNowhere)
        {
#pragma unroll
            for (int j = 0; j < VEC; ++j)
                xv[u][j] = fma_t(xv[u][j] - m, dvar_term, fma_t(dv[u][j] * sc, inv_stdev, dmean_term));
            store_once<T, VEC, STREAM>(a.dx + base + (at[u] >> 1), xv[u]);
        }
    if constexpr (std::is_same<G, OrderedClearing>::value)
        clear_halo_cells(g.halo, a.dx + base, member * TEAM + threadIdx.x, g.members.divisor * TEAM);
}
