// Instance softmax of samples of several chunks, in one launch each way.  Teams (samples beyond one
// workgroup, and few of more than four chunks): the workgroups of a team hold a sample in their registers,
// one or four chunks of the staged reductions each, and exchange their partial results through memory.
// One workgroup that plays the chunks of a sample, four a round (softmax_inst_rounds_kernel, below): the
// other samples of several chunks that it holds.  Included by h2x_softmax.hip.
//
// The launches for the maximum, the sum and the map read the sample three times and are
// bound by their starts; here every element is read once, and what is bound is the wait
// for the last member, twice forward and once backward.  The bits are those of the
// staged calls: 256 neighbouring threads play the workgroup of a chunk, and the partial sums
// are added along the tree in which a kernel combines stored ones, thread t starting with
// partial t.  Members of four chunks exchange sums of four neighbouring partials, the first
// steps of that tree.  Separate launches -> by teams, forward + backward, us, going round three
// sets of tensors:
//   N 1, 33,759 elements     15.8 -> 10.9      N 8, 800,000             48.0 -> 39.6
//   N 16, 86,016             19.2 -> 15.8      N 32, 344,064            74.7 -> 56.9
//   N 2, 58,100              16.0 -> 9.8       N 32, 688,128           134.9 -> 102
//   N 1, 773,145             23.3 -> 18.9      N 4, 3,932,160           98.2 -> 86.3
// A member looks at what all others store: with members of one chunk throughout, 256 of them, N 2,
// 1,048,576 elements took 29.6 us, of four 22.6.  Up to 64 chunks more CUs are worth more (16 x 86,016
// in members of four 17.3, N 1, 158,652 15.3 and 13.8).
//
// The exchange is that of h2x_device.hpp, with a counter a sample; the two of a forward pass share a tag.
#pragma once

// State of a sample, zero before its first call: the counter on a line of its own, then two
// words a member for each of the two exchanges.
// (256 chunks in members of four, or 64 in members of one.)
constexpr uint32_t kInstMembers = 64;
constexpr uint32_t kInstStateWords = kCounterWords + 2 * 2 * kInstMembers;

struct InstTeam
{
    FastDiv members; // of a team
    uint32_t chunks; // of a sample
    uint32_t sample_size, chunk;
    uint32_t max_polls;
    unsigned long long* states;
};

// What the waves of a member leave one another.  Each array is written once, so nothing waits for it to be read.
template <int TEAM>
struct InstShared
{
    double waves[2][TEAM / kWaveSize]; // of each exchange
    double again[TEAM / kWaveSize];    // of a member whose result is worked out here
    double totals[2][kWavesPerBlock];
    unsigned long long late[2][kWavesPerBlock]; // lanes whose result was not there in time
};

// f(k, bytes) for the vectors of a thread in its chunk of a member, in the order of the staged reductions; they
// lie where inst_at says (one offset in a vector register for all of them).
template <typename T, int TEAM, int VEC, int V, typename F>
__device__ __forceinline__ void inst_chunk(const InstTeam& g, uint32_t member, const F& f)
{
    const uint32_t begin = (member * (TEAM / kBlockSize) + threadIdx.x / kBlockSize) * g.chunk;
    const uint32_t end = begin + g.chunk < g.sample_size ? begin + g.chunk : g.sample_size;
    const uint32_t first = begin + threadIdx.x % kBlockSize * VEC;
#pragma unroll
    for (int k = 0; k < V; ++k)
        if (first + k * kBlockSize * VEC < end)
            f(k, first * static_cast<uint32_t>(sizeof(T)));
}

template <int VEC, typename T>
__device__ __forceinline__ T* inst_at(T* sample, int k, uint32_t bytes)
{
    using Byte = typename std::conditional<std::is_const<T>::value, const char, char>::type;
    return reinterpret_cast<T*>(reinterpret_cast<Byte*>(sample + k * kBlockSize * VEC) + bytes);
}

// What a member exchanges, in every lane: the maximum over the workgroup, or the sum of its chunk, as block_sum adds, or of
// four.  waves: a double for each wave.
template <int TEAM, bool SUM>
__device__ __forceinline__ double inst_partial(double mine, double* waves)
{
    constexpr int kWaves = TEAM / kWaveSize, kChunks = TEAM / kBlockSize;
    mine = SUM ? wave_sum(mine) : wave_max(mine);
    if (threadIdx.x % kWaveSize == 0)
        waves[threadIdx.x / kWaveSize] = mine;
    __syncthreads();
    if constexpr (SUM)
    {
        const double* const w = waves + threadIdx.x % kChunks * kWavesPerBlock;
        double p = w[0];
#pragma unroll
        for (int i = 1; i < kWavesPerBlock; ++i)
            p += w[i];
        p = 0.0 + p; // as inst_combine_sum starts
        if constexpr (kChunks == 4)
        {
            p += dpp_move<kDppQuadSwap1>(p);
            p += dpp_move<kDppQuadSwap2>(p);
        }
        return p;
    }
    else
    {
        const auto larger = [](double a, double b) { return a > b ? a : b; };
        double r = waves[threadIdx.x % kWaves];
        r = larger(r, dpp_move<kDppQuadSwap1>(r));
        r = larger(r, dpp_move<kDppQuadSwap2>(r));
        if constexpr (kWaves == 16)
        {
            r = larger(r, dpp_move<kDppRowRor4>(r));
            r = larger(r, dpp_move<kDppRowRor8>(r));
        }
        return r;
    }
}

// The result of all members, given this member's own and the tag that it made of the counter.  Lanes 0, 1, ... of the first wave
// look after a member each, or, members of four chunks, lanes 0, 4, ... of the first four: where a thread of the
// staged combination holds the first of the partials that member has added up, so that the steps left of its tree
// are wave_sum_from's.  recompute(member): what a thread adds to it, called by the whole workgroup.
// (With the first thread storing, a reduction through LDS before and behind the look and two barriers each, N 13, 44,880
// elements, forward + backward, took 11.6 us, so 10.2; N 12, 66,912 12.5 and 10.9.)
template <int TEAM, int WHICH, bool SUM, typename F>
__device__ __forceinline__ double inst_exchange(double part, const InstTeam& g, uint32_t member,
                                                unsigned long long* state, uint32_t tag, InstShared<TEAM>& shared,
                                                const F& recompute)
{
    constexpr uint32_t kChunks = TEAM / kBlockSize;
    const uint32_t members = g.members.divisor, t = threadIdx.x, mine = t / kChunks;
    const uint32_t lane = t % kWaveSize, wave = t / kWaveSize;
    const bool reads = t % kChunks == 0 && mine < members;
    unsigned long long* const words = state + kCounterWords + WHICH * 2 * kInstMembers;
    const auto leave_wave = [&](double s) {
        s = SUM ? wave_sum_from(s, kChunks) : wave_max(s);
        if (lane == 0)
            shared.totals[WHICH][wave] = s;
    };
    const auto total = [&] {
        double r = shared.totals[WHICH][0];
#pragma unroll
        for (uint32_t w = 1; w < kChunks; ++w)
        {
            const double x = shared.totals[WHICH][w];
            r = SUM ? r + x : x > r ? x : r;
        }
        return r;
    };
    if (t == 0)
        team_put(words, kInstMembers, member, tag, part);
    double s = 0.0; // less than any maximum
    if (wave < kChunks) // uniform
    {
        const bool there = !reads || team_get(words + mine, kInstMembers, tag, g.max_polls, &s);
        if (!there)
            s = 0.0;
        const unsigned long long late = __ballot(!there);
        if (lane == 0)
            shared.late[WHICH][wave] = late;
        leave_wave(s);
    }
    __syncthreads();
    unsigned long long late = shared.late[WHICH][0];
#pragma unroll
    for (uint32_t w = 1; w < kChunks; ++w)
        late |= shared.late[WHICH][w];
    if (late) // uniform
    {
        for (uint32_t m = 0; m < members; ++m)
        {
            if (!(shared.late[WHICH][m * kChunks / kWaveSize] >> m * kChunks % kWaveSize & 1)) // uniform
                continue;
            const double r = inst_partial<TEAM, SUM>(recompute(m), shared.again);
            if (t == m * kChunks)
                s = r;
            __syncthreads(); // shared.again is written again
        }
        if (wave < kChunks)
            leave_wave(s);
        __syncthreads();
    }
    return total();
}

template <typename T, int VEC>
__device__ __forceinline__ void add_max(T& mx, const Pack<T, VEC>& v)
{
#pragma unroll
    for (int j = 0; j < VEC; ++j)
        mx = v[j] >= mx ? v[j] : mx;
}

template <typename T, int VEC>
__device__ __forceinline__ void add_exponentials(double& acc, Pack<T, VEC>& v, T shift)
{
#pragma unroll
    for (int j = 0; j < VEC; ++j)
    {
        v[j] = exp_t(v[j] - shift);
        acc += static_cast<double>(v[j]);
    }
}

template <typename T, int VEC>
__device__ __forceinline__ void add_products(double& acc, const Pack<T, VEC>& y, const Pack<T, VEC>& dy)
{
#pragma unroll
    for (int j = 0; j < VEC; ++j)
        acc = __builtin_fma(static_cast<double>(y[j]), static_cast<double>(dy[j]), acc);
}

// Waves of a SIMD: two members of 1024 threads a CU, for which a thread may have 64 registers, where it holds up to 32 (HELD
// elements; doubles in single elements spill then). Without the bound the compiler gives forward floats of 8 vectors 67
// registers, doubles 69, backward floats of 4 vectors 66, and single elements (61 and 59) too many scalars: one member
// a CU. us, without -> with, going round three sets of tensors: forward N 16, 1,225,728 floats 59.3 -> 51.5, N 23,
// 632,400 doubles 82.2 -> 68.0; backward N 11, 527,040 floats 17.3 -> 15.5; single elements N 24, 318,009 24.6 -> 20.8
// forward, 21.7 -> 18.9 backward, but, where all members have a CU of their own, N 4, 500,001 12.8 -> 13.0 and 9.1 ->
// 9.45, N 11, 263,537 12.6 -> 12.8 and 10.1 -> 10.4.
template <typename T, int TEAM, int HELD, bool SINGLE>
constexpr int inst_waves()
{
    return TEAM == kBlockSize ? 2 : HELD * sizeof(T) <= 4 * 32 && !(sizeof(T) == 8 && SINGLE) ? 8 : 4;
}

// VEC elements a vector, up to V vectors a thread.
template <typename T, int TEAM, int VEC, int V>
__global__ __launch_bounds__(TEAM, (inst_waves<T, TEAM, VEC * V, VEC == 1>())) void softmax_inst_team_forward_kernel(
    const T* __restrict__ x, T* __restrict__ y, T* __restrict__ sample_max, T* __restrict__ sample_exp,
    const InstTeam g, T min_output)
{
    using P = Pack<T, VEC>;
    __shared__ InstShared<TEAM> shared;
    const uint32_t n = fastdiv(blockIdx.x, g.members);
    const uint32_t member = blockIdx.x - n * g.members.divisor;
    unsigned long long* const state = g.states + static_cast<size_t>(n) * kInstStateWords;
    uint32_t tag = team_tag(state);
    const T* const xp = x + static_cast<size_t>(n) * g.sample_size;
    P v[V];
    inst_chunk<T, TEAM, VEC, V>(g, member, [&](int k, uint32_t i) { v[k] = P::load(inst_at<VEC>(xp, k, i)); });

    T mx = Limits<T>::min_normal;
    inst_chunk<T, TEAM, VEC, V>(g, member, [&](int k, uint32_t) { add_max<T, VEC>(mx, v[k]); });
    asm volatile("" : "+v"(tag)); // every wave has it before any stores: beyond the barrier others may leave
    const T shift = static_cast<T>(inst_exchange<TEAM, 0, false>(
        inst_partial<TEAM, false>(static_cast<double>(mx), shared.waves[0]), g, member, state, tag, shared, [&](uint32_t m) {
            T r = Limits<T>::min_normal;
            inst_chunk<T, TEAM, VEC, V>(g, m, [&](int k, uint32_t i) {
                add_max<T, VEC>(r, P::load(inst_at<VEC>(xp, k, i)));
            });
            return static_cast<double>(r);
        }));

    double acc = 0.0;
    inst_chunk<T, TEAM, VEC, V>(g, member, [&](int k, uint32_t) { add_exponentials<T, VEC>(acc, v[k], shift); });
    const T sum = static_cast<T>(inst_exchange<TEAM, 1, true>(
        inst_partial<TEAM, true>(acc, shared.waves[1]), g, member, state, tag, shared, [&](uint32_t m) {
            double r = 0.0;
            inst_chunk<T, TEAM, VEC, V>(g, m, [&](int k, uint32_t i) {
                P w = P::load(inst_at<VEC>(xp, k, i));
                add_exponentials<T, VEC>(r, w, shift);
            });
            return r;
        }));
    if (threadIdx.x == 0)
        team_leave(state);
    if (member == 0 && threadIdx.x == 0)
    {
        sample_max[n] = shift;
        sample_exp[n] = sum;
    }
    T* const yp = y + static_cast<size_t>(n) * g.sample_size;
    inst_chunk<T, TEAM, VEC, V>(g, member, [&](int k, uint32_t i) {
#pragma unroll
        for (int j = 0; j < VEC; ++j)
        {
            const T r = v[k][j] / sum;
            v[k][j] = r > min_output ? r : min_output;
        }
        P::store(inst_at<VEC>(yp, k, i), v[k]);
    });
}

template <typename T, int TEAM, int VEC, int V>
__global__ __launch_bounds__(TEAM, (inst_waves<T, TEAM, 2 * VEC * V, VEC == 1>())) void softmax_inst_team_backward_kernel(
    const T* __restrict__ y, const T* __restrict__ dy, T* __restrict__ dx, T* __restrict__ sample_dp,
    const InstTeam g, T min_output)
{
    using P = Pack<T, VEC>;
    __shared__ InstShared<TEAM> shared;
    const uint32_t n = fastdiv(blockIdx.x, g.members);
    const uint32_t member = blockIdx.x - n * g.members.divisor;
    unsigned long long* const state = g.states + static_cast<size_t>(n) * kInstStateWords;
    uint32_t tag = team_tag(state);
    const T* const yp = y + static_cast<size_t>(n) * g.sample_size;
    const T* const dp = dy + static_cast<size_t>(n) * g.sample_size;
    P v[V], d[V];
    inst_chunk<T, TEAM, VEC, V>(g, member, [&](int k, uint32_t i) {
        v[k] = P::load(inst_at<VEC>(yp, k, i));
        d[k] = P::load(inst_at<VEC>(dp, k, i));
    });
    double acc = 0.0;
    inst_chunk<T, TEAM, VEC, V>(g, member, [&](int k, uint32_t) { add_products<T, VEC>(acc, v[k], d[k]); });
    asm volatile("" : "+v"(tag)); // every wave has it before any stores: beyond the barrier others may leave
    const T dot = static_cast<T>(inst_exchange<TEAM, 0, true>(
        inst_partial<TEAM, true>(acc, shared.waves[0]), g, member, state, tag, shared, [&](uint32_t m) {
            double r = 0.0;
            inst_chunk<T, TEAM, VEC, V>(g, m, [&](int k, uint32_t i) {
                add_products<T, VEC>(r, P::load(inst_at<VEC>(yp, k, i)), P::load(inst_at<VEC>(dp, k, i)));
            });
            return r;
        }));
    if (threadIdx.x == 0)
        team_leave(state);
    if (member == 0 && threadIdx.x == 0)
        sample_dp[n] = dot;
    T* const op = dx + static_cast<size_t>(n) * g.sample_size;
    inst_chunk<T, TEAM, VEC, V>(g, member, [&](int k, uint32_t i) {
#pragma unroll
        for (int j = 0; j < VEC; ++j)
            v[k][j] = v[k][j] > min_output ? v[k][j] * (d[k][j] - dot) : T(0);
        P::store(inst_at<VEC>(op, k, i), v[k]);
    });
}

// Samples of several chunks that one workgroup holds, where a team is not for the call (many samples, smaller ones, in
// place, a single reduction, no state): the workgroup plays the chunks, four a round, and adds their sums as the
// combination of stored ones does: a round's are what a member of four chunks exchanges, and one addition, the last
// that is not of zeros, is left. All rounds but the last are of whole chunks. Bound by the work of a CU and by waits in
// a row. The kernel that adds lane by lane, which loads single elements and compares for each, -> this, forward +
// backward in us, going round three sets of tensors:
//   floats  N 16, 4100    8.4 -> 7.3      N 16, 12000   10.5 -> 8.7     N 128, 16400  17.0 -> 14.3    N 256, 32768  41.1 -> 37.5
//   doubles N 16, 4200    9.1 -> 7.7      N 128, 8200   15.4 -> 13.7    N 500, 12000  58.7 -> 52.1    N 500, 16384  78.0 -> 66.7
//   in place, floats  N 2, 32768  18.2 -> 14.5    N 64, 20000  16.1 -> 12.8    N 256, 28224  29.5 -> 27.5
// (With comparisons in all rounds N 2, 32768 in place 16.4.)
template <typename T, int VEC, int V, int ROUNDS, int MODE>
__global__ __launch_bounds__(4 * kBlockSize) void softmax_inst_rounds_kernel(const T* a, const T* b, T* out, const T* sample_param,
                                                                             T* __restrict__ result, T* __restrict__ result2,
                                                                             uint32_t sample_size, T min_output)
{
    using P = Pack<T, VEC>;
    constexpr int TEAM = 4 * kBlockSize;
    constexpr bool kDot = MODE == kSmallDot || MODE == kSmallBackward;
    __shared__ double waves[ROUNDS + 1][TEAM / kWaveSize];
    const uint32_t n = blockIdx.x;
    InstTeam g = {};
    g.sample_size = sample_size;
    g.chunk = kBlockSize * VEC * V;
    const size_t base = static_cast<size_t>(n) * sample_size;
    // f(k, bytes) for the vectors of a thread in a round
    const auto of_round = [&](int r, const auto& f) {
        if (r + 1 == ROUNDS)
        {
            inst_chunk<T, TEAM, VEC, V>(g, r, f);
            return;
        }
        const uint32_t first = (r * 4 + threadIdx.x / kBlockSize) * g.chunk + threadIdx.x % kBlockSize * VEC;
#pragma unroll
        for (int k = 0; k < V; ++k)
            f(k, first * static_cast<uint32_t>(sizeof(T)));
    };
    P va[ROUNDS][V], vb[kDot ? ROUNDS : 1][V];
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r)
        of_round(r, [&](int k, uint32_t i) {
            va[r][k] = P::load(inst_at<VEC>(a + base, k, i));
            if constexpr (kDot)
                vb[r][k] = P::load(inst_at<VEC>(b + base, k, i));
        });
    T shift = T(0);
    if constexpr (MODE == kSmallForward)
    {
        T mx = Limits<T>::min_normal;
#pragma unroll
        for (int r = 0; r < ROUNDS; ++r)
            of_round(r, [&](int k, uint32_t) { add_max<T, VEC>(mx, va[r][k]); });
        shift = static_cast<T>(inst_partial<TEAM, false>(static_cast<double>(mx), waves[ROUNDS]));
        if (threadIdx.x == 0)
            result[n] = shift;
    }
    else if constexpr (!kDot)
    {
        shift = sample_param[n];
    }
    double total = 0.0;
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r)
    {
        double acc = 0.0;
        of_round(r, [&](int k, uint32_t) {
            if constexpr (kDot)
                add_products<T, VEC>(acc, va[r][k], vb[r][k]);
            else
                add_exponentials<T, VEC>(acc, va[r][k], shift);
        });
        total += inst_partial<TEAM, true>(acc, waves[r]);
    }
    const T sum = static_cast<T>(total);
    if (threadIdx.x == 0)
        (MODE == kSmallForward ? result2 : result)[n] = sum;
    if constexpr (MODE != kSmallDot)
#pragma unroll
        for (int r = 0; r < ROUNDS; ++r)
            of_round(r, [&](int k, uint32_t i) {
                if constexpr (MODE != kSmallExpSum)
                {
#pragma unroll
                    for (int j = 0; j < VEC; ++j)
                        if constexpr (MODE == kSmallForward)
                        {
                            const T q = va[r][k][j] / sum;
                            va[r][k][j] = q > min_output ? q : min_output;
                        }
                        else
                        {
                            va[r][k][j] = va[r][k][j] > min_output ? va[r][k][j] * (vb[r][k][j] - sum) : T(0);
                        }
                }
                P::store(inst_at<VEC>(out + base, k, i), va[r][k]);
            });
}
