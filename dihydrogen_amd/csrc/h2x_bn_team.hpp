// Batch-norm of a rank that shares its statistics with no one, for channels that are
// too large for one workgroup: the workgroups of a team hold a channel in their
// registers together, exchange their partial sums through memory and write y (dx)
// from the registers.  Included by h2x_bn.hip after h2x_bn_once.hpp, whose geometry,
// terms and stores these kernels share.
//
// The two-launch kernels are bound by memory and read x (backward: x and dy) twice, at
// 5 to 7 TB/s; here every element is read once.  Bound by memory and by the wait for the
// last member of a team.  Forward, backward in us, two launches each way -> by teams, going round
// three sets of tensors:
//   N 8, C 64, 30^3, halo of 1      38, 54 -> 34, 40     N 32, C 256, 56 x 56     48, 85 -> 39, 58
//   N 4, C 64, 64^3                116, 189 -> 101, 152  N 64, C 128, 40 x 40     27, 45 -> 18, 28
//   N 8, C 64, 64^3                257, 411 -> 200, 344  N 2, C 32, 48^3          16, 28 -> 12, 15
//   N 1, C 64, 96^3                 98, 160 -> 87, 131   N 64, C 64, 57^2, halo   31, 51 -> 31, 38
//   N 2, C 16, 48^3, halo of 1      12, 17 -> 10, 12     N 8, C 64, 56 x 56      8.6, 10.6 -> 5.7, 7.0
// Looking at a counter of arrivals instead of the sums themselves was slower the
// larger the team (64 members, N 4, C 64, 64^3: 119 us against 98): one address.
//
// The exchange is that of h2x_device.hpp, with a counter a channel (a fill launch before the kernel instead of
// tags cost 4.7 us behind streaming stores).  A member works out the sums it misses with the additions of the
// member they belong to, and gets the same bits.  Members are neighbouring
// workgroups, and workgroups start in order, so a team is on the chip together unless
// other streams fill it; the launch rule keeps a team within half of it.
#pragma once

// (A wave looks after 64 / N members with N lanes each, N sums: 8 waves after 128 of four sums, the most that
// team_exchange takes.)
constexpr uint32_t kMaxMembers = 128;

// State of a channel, zero before its first call: the counter on a line of its own, then
// two words a sum.  A channel has room for 256 sums, members times sums of a member: 128 forward, 64 backward.  Larger teams are
// for channels of more than 8 MB, of which a tensor has few: the first 32 channels have room for twice that.
// (Where a channel's state lies is the same for all calls on one state, whatever their sizes.)
constexpr uint32_t kTeamSums = 256, kWideChannels = 32;

__host__ __device__ __forceinline__ uint32_t most_team_sums(uint32_t channels)
{
    return channels <= kWideChannels ? 2 * kTeamSums : kTeamSums;
}
// Words before channel c.
__host__ __device__ __forceinline__ size_t team_state_at(uint32_t c)
{
    return static_cast<size_t>(c) * (kCounterWords + 2 * kTeamSums) + (c < kWideChannels ? c : kWideChannels) * 2 * kTeamSums;
}

template <typename G>
struct TeamGeometry
{
    G once;
    FastDiv members;   // of a team
    uint32_t span;     // vectors of a member, a multiple of its threads
    uint32_t max_polls;
};

// Which member of a team of `members` the team's workgroup i is.  Workgroups go to the XCDs in
// turn, and each XCD's members take neighbouring pieces of the channel: with piece i for workgroup
// i the pieces of one XCD lie 8 pieces apart, and the samples of a channel a power of two, and the
// memory behind them is reached unevenly.  Forward, backward in us, piece i -> this (going round three sets of
// tensors): N 4, C 64, 64^3 108, 175 -> 103, 166; N 8, C 32, 64^3 113, 193 -> 107, 185; copies in these orders 114 -> 98.
// (Whole teams on one XCD would wait for the slots of that XCD.)
__host__ __device__ __forceinline__ uint32_t team_member(uint32_t i, uint32_t members)
{
    const uint32_t xcd = i % kNumXcd, left = members % kNumXcd;
    return xcd * (members / kNumXcd) + (xcd < left ? xcd : left) + i / kNumXcd;
}

// Teams of up to kSmallTeam members look at all words at once.  Larger ones look at one word of each member until all have
// come, and then at the others: what waiting workgroups read takes the memory from those that load.  Between looks they sleep
// 4 x 64 clocks, 0.1 us, and 44 x 64, 1.2 us, where a launch has more than kCrowd workgroups, about those that the chip holds at
// once, hundreds of which wait all the time.  N 4, C 64, 64^3, teams of 32 and 64, forward + backward going round three sets
// of tensors: all words every 0.1 us 266 us, one word every 0.15 us 245, every 0.4 us 242, every 1.2 us 240, every 1.9
// us 242, every 2.9 us 246. Small teams lose by one word every 1.2 us (of 4, N 8, C 64, 56 x 56, 11.7 us and 13.5; of 8
// and 15, N 8, C 64, 30^3 with a halo, 73.8 and 74.7), small launches by the long sleep (N 3, C 6, 43 x 50 x 38 15.1
// us, with the short one 13.6; N 15, C 4, 22 x 17 x 22, doubles, 15.1 and 13.9; up to 1024 workgroups, N 23, C 21, 144
// x 155, 45.0 and 42.0), doubles by all words there (N 81, C 9, 33 x 41 16.9 and 19.0).
constexpr uint32_t kSmallTeam = 16, kCrowd = 1024;

// What the waves of a member leave one another, and what a member knows of the others.
template <int TEAM, int N>
struct TeamShared
{
    static constexpr uint32_t kGroup = kWaveSize / N; // lanes, and members that a wave looks after
    double waves[2][N * TEAM / kWaveSize];
    double theirs[N][kMaxMembers];
    double parts[kMaxMembers / kGroup][N];        // what the members of a wave make together
    unsigned long long late[kMaxMembers / kGroup]; // lanes whose sum was not there in time
};

// The N sums of all members in v[] of every thread, given this member's own as lane_sums leaves them, and the tag it
// made of the counter.  The lanes of the first wave that hold the sums store them; a wave looks after as many members as a group
// has lanes, group k after their k-th sums, and leaves what it adds up to all.  recompute(member, sums): the terms of a thread,
// called by the whole workgroup.  (With the first thread storing all sums, a thread a member looking at all of its
// words and two more reductions through LDS, N 8, C 64, 56 x 56, forward + backward, took 13.8 us; so 11.75.)
template <int TEAM, int N, typename G, typename F>
__device__ __forceinline__ void team_exchange(double own, double (&v)[N], const TeamGeometry<G>& g, uint32_t member,
                                              unsigned long long* state, uint32_t tag, TeamShared<TEAM, N>& shared,
                                              const F& recompute)
{
    constexpr uint32_t kGroup = kWaveSize / N;
    static_assert(TEAM / kWaveSize * kGroup >= kMaxMembers, "a wave for a group of members");
    const uint32_t members = g.members.divisor, lane = threadIdx.x % kWaveSize, wave = threadIdx.x / kWaveSize;
    const uint32_t k = lane / kGroup, m = wave * kGroup + lane % kGroup;
    const uint32_t lookers = (members + kGroup - 1) / kGroup; // waves
    unsigned long long* const words = state + kCounterWords + 2 * k * members;
    if (threadIdx.x < kWaveSize && lane % kGroup == 0)
        team_put(words, members, member, tag, own);
    if (wave < lookers) // uniform
    {
        const unsigned long long* const at = words + m;
        double s = 0.0;
        bool there = m >= members;
        uint32_t looks = g.max_polls; // uniform
        if (members > kSmallTeam)     // (the last look is one at all words: it takes what has come, whoever is missing)
            for (; looks > 1 && __any(!there && k == N - 1 && team_load(at) >> 32 != tag); --looks)
            {
                __builtin_amdgcn_s_sleep(4);
                if (gridDim.x > kCrowd) // uniform
                    __builtin_amdgcn_s_sleep(40);
            }
        for (; looks > 0; --looks)
        {
            if (!there)
                there = team_look(at, members, tag, &s);
            if (__all(there))
                break;
            __builtin_amdgcn_s_sleep(4);
        }
        shared.theirs[k][m] = s;
        const unsigned long long late = __ballot(!there);
        if (lane == 0)
            shared.late[wave] = late;
        const double part = lane_group_sum<N>(s);
        if (lane % kGroup == 0)
            shared.parts[wave][k] = part;
    }
    __syncthreads();
    if (threadIdx.x == 0)
        team_leave(state);
    unsigned long long late = shared.late[0];
    for (uint32_t w = 1; w < lookers; ++w)
        late |= shared.late[w];
    if (late) // uniform
    {
        for (uint32_t i = 0; i < members; ++i)
        {
            unsigned long long lanes = 0;
#pragma unroll
            for (int n = 0; n < N; ++n)
                lanes |= shared.late[i / kGroup] >> (n * kGroup + i % kGroup);
            if (!(lanes & 1)) // uniform
                continue;
            double r[N];
#pragma unroll
            for (int n = 0; n < N; ++n)
                r[n] = 0.0;
            recompute(i, r);
            const double t = lane_sums<TEAM, N>(r, shared.waves[1]);
            if (threadIdx.x < kWaveSize && lane % kGroup == 0)
                shared.theirs[k][i] = t;
            __syncthreads(); // waves[1] is written again
        }
        if (wave < lookers)
        {
            const double part = lane_group_sum<N>(shared.theirs[k][m]);
            if (lane % kGroup == 0)
                shared.parts[wave][k] = part;
        }
        __syncthreads();
    }
#pragma unroll
    for (int n = 0; n < N; ++n)
    {
        double t = shared.parts[0][n];
        for (uint32_t w = 1; w < lookers; ++w)
            t += shared.parts[w][n];
        v[n] = t;
    }
}

// The terms of the vector at place `at`.
template <typename G, typename T, int VEC>
__device__ __forceinline__ void add_forward_terms(double (&s)[2], const T (&v)[VEC], uint32_t at)
{
#pragma unroll
    for (int j = 0; j < VEC; ++j)
        if (G::counts(at, j))
        {
            const double d = static_cast<double>(v[j]);
            s[0] += d;
            s[1] = __builtin_fma(d, d, s[1]);
        }
}

template <typename G, typename T, int VEC>
__device__ __forceinline__ void add_backward_terms(double (&s)[4], const T (&x)[VEC], const T (&d)[VEC], uint32_t at,
                                                   T m, T sc, T inv_stdev)
{
#pragma unroll
    for (int j = 0; j < VEC; ++j)
        if (G::counts(at, j))
        {
            const T xm = x[j] - m;
            const T dxhat = d[j] * sc;
            const double dd = static_cast<double>(d[j]);
            s[0] = __builtin_fma(dd, static_cast<double>(xm * inv_stdev), s[0]);
            s[1] += dd;
            s[2] += static_cast<double>(dxhat);
            s[3] += static_cast<double>(dxhat * xm);
        }
}

// Scale and bias are loaded behind the elements: they are scalars, and a wave that asks for them first waits for them
// before its first element. The exchange hides them (forward in us, loaded behind the exchange, before the elements and
// so: N 3, C 17, 31 x 22 x 18 5.4, 5.1 and 5.1; N 32, C 256, 56 x 56 41.0, 40.2 and 39.6, over one set of tensors 33.0,
// 34.7 and 33.5; N 4, C 64, 64^3 102.8, 102.7 and 101.8, over one set 83.7, 86.3 and 84.8, where what is loaded late
// spreads the stores). kOneByOne: a wave of a large member whose output's halo is cleared waits for each of its stores
// (forward in us, at once and so: N 29, C 24, 19 x 32 x 29 31.3 and 29.5; N 9, C 128, 124 x 107 30.8 and 28.4; N 3, C
// 373, 27 x 29 x 38, halo of 2 83.6 and 78.2; N 188, C 301, 8 x 7 x 8 89.6 and 84.9). Members of 8 vectors a thread
// lose by it (N 3, C 655, 121 x 88 31.1 and 33.2; N 166, C 201, 14 x 20, halo of 2 22.4 and 23.4), dense tensors too
// where they go round several sets (N 1, C 64, 128 x 128 x 64 95.8 and 100).
template <typename T, int TEAM, int K, bool STREAM, typename G>
__global__ __launch_bounds__(TEAM) void bn_team_forward_kernel(const TeamGeometry<G> g, const OnceForward<T> a,
                                                                      unsigned long long* states)
{
    constexpr int VEC = 16 / sizeof(T);
    constexpr bool kOneByOne = G::kClears && K == 16;
    __shared__ TeamShared<TEAM, 2> shared;
    const uint32_t c = fastdiv(blockIdx.x, g.members);
    const uint32_t member = team_member(blockIdx.x - c * g.members.divisor, g.members.divisor);
    const T* const x = a.x + c * g.once.stride_c;
    unsigned long long* const state = states + team_state_at(c);
    uint32_t tag = team_tag(state);
    const uint32_t first = member * g.span;
    const uint32_t end = first + g.span < g.once.vectors ? first + g.span : g.once.vectors;
    T v[K][VEC];
    uint32_t at[K];
    const auto live = [&](int u) { return first + u * TEAM < end && first + u * TEAM + threadIdx.x < end; };
#pragma unroll
    for (int u = 0; u < K; ++u)
        if (live(u))
        {
            at[u] = once_place<VEC>(g.once, first + u * TEAM + threadIdx.x);
            load_vec<T, VEC, false>(x + G::offset(at[u]), v[u]);
        }
    const T sc = a.scale[c], bi = a.bias[c];
    double s[2] = {0.0, 0.0};
#pragma unroll
    for (int u = 0; u < K; ++u)
        if (live(u))
            add_forward_terms<G, T, VEC>(s, v[u], at[u]);
    asm volatile("" : "+v"(tag)); // every wave has it before any stores: beyond the barrier others may leave
    const double own = lane_sums<TEAM, 2>(s, shared.waves[0]);
    team_exchange<TEAM, 2>(own, s, g, member, state, tag, shared, [&](uint32_t other, double (&r)[2]) {
        const uint32_t stop = (other + 1) * g.span < g.once.vectors ? (other + 1) * g.span : g.once.vectors;
        for (uint32_t i = other * g.span + threadIdx.x; i < stop; i += TEAM)
        {
            const uint32_t p = once_place<VEC>(g.once, i);
            T w[VEC];
            load_vec<T, VEC, false>(x + G::offset(p), w);
            add_forward_terms<G, T, VEC>(r, w, p);
        }
    });
    T m, variance;
    sums_to_mean_var(static_cast<T>(s[0]), static_cast<T>(s[1]), a.n, &m, &variance);
    if (member == 0 && threadIdx.x == 0)
        update_statistics(a, c, m, variance);
    const T inv_stdev = inv_sqrt_t(variance + a.epsilon);
    T* const y = a.y + c * g.once.stride_c;
#pragma unroll
    for (int u = 0; u < K; ++u)
        if (live(u))
        {
#pragma unroll
            for (int j = 0; j < VEC; ++j)
                v[u][j] = G::kClears && !G::counts(at[u], j) ? T(0) : fma_t((v[u][j] - m) * inv_stdev, sc, bi);
            if constexpr (kOneByOne)
                __builtin_amdgcn_s_waitcnt(0x0f70); // vector memory only
            store_once<T, VEC, STREAM>(y + G::offset(at[u]), v[u]);
        }
}

// GRADIENT: dy, read for the last time, past the caches (see streams_gradient, where it is launched).
template <typename T, int TEAM, int K, bool STREAM, bool GRADIENT, typename G>
__global__ __launch_bounds__(TEAM) void bn_team_backward_kernel(const TeamGeometry<G> g, const OnceBackward<T> a,
                                                                       unsigned long long* states)
{
    constexpr int VEC = 16 / sizeof(T);
    __shared__ TeamShared<TEAM, 4> shared;
    const uint32_t c = fastdiv(blockIdx.x, g.members);
    const uint32_t member = team_member(blockIdx.x - c * g.members.divisor, g.members.divisor);
    const int64_t base = c * g.once.stride_c;
    unsigned long long* const state = states + team_state_at(c);
    uint32_t tag = team_tag(state);
    const uint32_t first = member * g.span;
    const uint32_t end = first + g.span < g.once.vectors ? first + g.span : g.once.vectors;
    T xv[K][VEC], dv[K][VEC];
    uint32_t at[K];
    const auto live = [&](int u) { return first + u * TEAM < end && first + u * TEAM + threadIdx.x < end; };
#pragma unroll
    for (int u = 0; u < K; ++u)
        if (live(u))
        {
            at[u] = once_place<VEC>(g.once, first + u * TEAM + threadIdx.x);
            load_vec<T, VEC, false>(a.x + base + G::offset(at[u]), xv[u]);
            load_vec<T, VEC, false, GRADIENT>(a.dy + base + G::offset(at[u]), dv[u]);
        }
    const T m = a.mean[c];
    const T sc = a.scale[c];
    const T inv_stdev = inv_sqrt_t(a.var[c] + a.epsilon);
    const T dvar_factor = inv_stdev * inv_stdev * inv_stdev / T(2);
    double s[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int u = 0; u < K; ++u)
        if (live(u))
            add_backward_terms<G, T, VEC>(s, xv[u], dv[u], at[u], m, sc, inv_stdev);
    asm volatile("" : "+v"(tag)); // every wave has it before any stores: beyond the barrier others may leave
    const double own = lane_sums<TEAM, 4>(s, shared.waves[0]);
    team_exchange<TEAM, 4>(own, s, g, member, state, tag, shared, [&](uint32_t other, double (&r)[4]) {
        const uint32_t stop = (other + 1) * g.span < g.once.vectors ? (other + 1) * g.span : g.once.vectors;
        for (uint32_t i = other * g.span + threadIdx.x; i < stop; i += TEAM)
        {
            const uint32_t p = once_place<VEC>(g.once, i);
            T w[VEC], d[VEC];
            load_vec<T, VEC, false>(a.x + base + G::offset(p), w);
            load_vec<T, VEC, false>(a.dy + base + G::offset(p), d);
            add_backward_terms<G, T, VEC>(r, w, d, p, m, sc, inv_stdev);
        }
    });
    const T dmean = static_cast<T>(s[2] * -static_cast<double>(inv_stdev));
    const T dvar = static_cast<T>(s[3] * -static_cast<double>(dvar_factor));
    if (member == 0 && threadIdx.x == 0)
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
                xv[u][j] = G::kClears && !G::counts(at[u], j)
                               ? T(0)
                               : fma_t(xv[u][j] - m, dvar_term, fma_t(dv[u][j] * sc, inv_stdev, dmean_term));
            store_once<T, VEC, STREAM>(a.dx + base + G::offset(at[u]), xv[u]);
        }
}
