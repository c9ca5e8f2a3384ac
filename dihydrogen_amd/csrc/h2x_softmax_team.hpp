// Instance softmax of samples beyond one workgroup, in one launch each way: the
// workgroups of a team hold a sample in their registers, one or four chunks of the staged
// reductions each, and exchange their partial results through memory.  Included by
// h2x_softmax.hip.
//
// The launches for the maximum, the sum and the map read the sample three times and are
// bound by their starts; here every element is read once, and what is bound is the wait
// for the last member, twice forward and once backward.  The bits are those of the
// staged calls: 256 neighbouring threads play the workgroup of a chunk, and the partial sums
// are added along the tree in which a kernel combines stored ones, thread t starting with
// partial t.  Members of four chunks exchange sums of four neighbouring partials, the first
// steps of that tree.  Separate launches -> by teams, forward + backward, us, going round three
// sets of tensors:
//   N 1, 33,759 elements     15.8 -> 11.8      N 8, 800,000             48.0 -> 39.5
//   N 16, 86,016             19.2 -> 16.6      N 32, 344,064            74.7 -> 61.9
//   N 2, 58,100              16.0 -> 12.8      N 32, 688,128           134.9 -> 114
//   N 1, 773,145             23.3 -> 19.6      N 4, 3,932,160           98.2 -> 87.2
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

// What member m exchanges in thread TEAM / kBlockSize * m, given this member's own in thread 0.
// recompute(member) is called by the whole workgroup.  shared: kInstMembers + 2 words.
template <int TEAM, int WHICH, typename F>
__device__ __forceinline__ double inst_exchange(double part, const InstTeam& g, uint32_t member,
                                                unsigned long long* state, uint32_t* tag, uint32_t* shared,
                                                const F& recompute)
{
    constexpr uint32_t kChunks = TEAM / kBlockSize;
    const uint32_t members = g.members.divisor, t = threadIdx.x;
    unsigned long long* const words = state + kCounterWords + WHICH * 2 * kInstMembers;
    if (t == 0)
    {
        const double own[1] = {part};
        team_put<1>(words, kInstMembers, member, *tag, own);
        shared[kInstMembers] = 0;
        shared[kInstMembers + 1] = *tag;
    }
    __syncthreads();
    *tag = shared[kInstMembers + 1];
    double s = 0.0;
    const uint32_t mine = t / kChunks;
    if (t % kChunks == 0 && mine < members)
    {
        double theirs[1] = {0.0};
        const bool there = team_get<1>(words, kInstMembers, mine, *tag, g.max_polls, theirs);
        s = theirs[0];
        shared[mine] = !there;
        if (!there)
            shared[kInstMembers] = 1; // every writer stores the same
    }
    __syncthreads();
    if (shared[kInstMembers])
        for (uint32_t m = 0; m < members; ++m)
            if (shared[m]) // uniform
            {
                const double r = recompute(m);
                if (t == m * kChunks)
                    s = r;
            }
    return s;
}

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

// The maximum over the workgroup.
template <int TEAM>
__device__ __forceinline__ double inst_maximum(double mine, double* lds)
{
    mine = wave_max(mine);
    __syncthreads(); // lds may still be read
    if (threadIdx.x % kWaveSize == 0)
        lds[threadIdx.x / kWaveSize] = mine;
    __syncthreads();
    double r = lds[0];
#pragma unroll
    for (int w = 1; w < TEAM / kWaveSize; ++w)
        r = lds[w] > r ? lds[w] : r;
    return r;
}

// The sum that a member exchanges: of its chunk, as block_sum adds, or of four.
template <int TEAM>
__device__ __forceinline__ double inst_partial(double mine, double* lds)
{
    constexpr int kChunks = TEAM / kBlockSize;
    mine = wave_sum(mine);
    __syncthreads();
    if (threadIdx.x % kWaveSize == 0)
        lds[threadIdx.x / kWaveSize] = mine;
    __syncthreads();
    double p[kChunks];
#pragma unroll
    for (int q = 0; q < kChunks; ++q)
    {
        p[q] = lds[q * kWavesPerBlock];
#pragma unroll
        for (int w = 1; w < kWavesPerBlock; ++w)
            p[q] += lds[q * kWavesPerBlock + w];
        p[q] = 0.0 + p[q]; // as inst_combine_sum starts
    }
    if constexpr (kChunks == 1)
        return p[0];
    else
        return (p[0] + p[1]) + (p[2] + p[3]);
}

// The sum of what the members have exchanged.
template <int TEAM>
__device__ __forceinline__ double inst_total(double mine, double* lds)
{
    mine = wave_sum_from(mine, TEAM / kBlockSize);
    __syncthreads();
    if (threadIdx.x % kWaveSize == 0)
        lds[threadIdx.x / kWaveSize] = mine;
    __syncthreads();
    double r = lds[0];
#pragma unroll
    for (int w = 1; w < kWavesPerBlock; ++w)
        r += lds[w];
    return r;
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

// VEC elements a vector, up to V vectors a thread.
template <typename T, int TEAM, int VEC, int V>
__global__ __launch_bounds__(TEAM, TEAM == kBlockSize ? 2 : 4) void softmax_inst_team_forward_kernel(
    const T* __restrict__ x, T* __restrict__ y, T* __restrict__ sample_max, T* __restrict__ sample_exp,
    const InstTeam g, T min_output)
{
    using P = Pack<T, VEC>;
    __shared__ double lds[TEAM / kWaveSize];
    __shared__ uint32_t shared[kInstMembers + 2];
    const uint32_t n = fastdiv(blockIdx.x, g.members);
    const uint32_t member = blockIdx.x - n * g.members.divisor;
    unsigned long long* const state = g.states + static_cast<size_t>(n) * kInstStateWords;
    uint32_t tag = threadIdx.x == 0 ? team_tag(state) : 0;
    const T* const xp = x + static_cast<size_t>(n) * g.sample_size;
    P v[V];
    inst_chunk<T, TEAM, VEC, V>(g, member, [&](int k, uint32_t i) { v[k] = P::load(inst_at<VEC>(xp, k, i)); });

    T mx = Limits<T>::min_normal;
    inst_chunk<T, TEAM, VEC, V>(g, member, [&](int k, uint32_t) { add_max<T, VEC>(mx, v[k]); });
    double s = inst_exchange<TEAM, 0>(
        inst_maximum<TEAM>(static_cast<double>(mx), lds), g, member, state, &tag, shared, [&](uint32_t m) {
            T r = Limits<T>::min_normal;
            inst_chunk<T, TEAM, VEC, V>(g, m, [&](int k, uint32_t i) {
                add_max<T, VEC>(r, P::load(inst_at<VEC>(xp, k, i)));
            });
            return inst_maximum<TEAM>(static_cast<double>(r), lds);
        });
    const double least = static_cast<double>(Limits<T>::min_normal); // what threads without a partial hold is less
    const T shift = static_cast<T>(inst_maximum<TEAM>(s > least ? s : least, lds));

    double acc = 0.0;
    inst_chunk<T, TEAM, VEC, V>(g, member, [&](int k, uint32_t) { add_exponentials<T, VEC>(acc, v[k], shift); });
    s = inst_exchange<TEAM, 1>(inst_partial<TEAM>(acc, lds), g, member, state, &tag, shared, [&](uint32_t m) {
        double r = 0.0;
        inst_chunk<T, TEAM, VEC, V>(g, m, [&](int k, uint32_t i) {
            P w = P::load(inst_at<VEC>(xp, k, i));
            add_exponentials<T, VEC>(r, w, shift);
        });
        return inst_partial<TEAM>(r, lds);
    });
    if (threadIdx.x == 0)
        team_leave(state);
    const T sum = static_cast<T>(inst_total<TEAM>(s, lds));
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
__global__ __launch_bounds__(TEAM, TEAM == kBlockSize ? 2 : 4) void softmax_inst_team_backward_kernel(
    const T* __restrict__ y, const T* __restrict__ dy, T* __restrict__ dx, T* __restrict__ sample_dp,
    const InstTeam g, T min_output)
{
    using P = Pack<T, VEC>;
    __shared__ double lds[TEAM / kWaveSize];
    __shared__ uint32_t shared[kInstMembers + 2];
    const uint32_t n = fastdiv(blockIdx.x, g.members);
    const uint32_t member = blockIdx.x - n * g.members.divisor;
    unsigned long long* const state = g.states + static_cast<size_t>(n) * kInstStateWords;
    uint32_t tag = threadIdx.x == 0 ? team_tag(state) : 0;
    const T* const yp = y + static_cast<size_t>(n) * g.sample_size;
    const T* const dp = dy + static_cast<size_t>(n) * g.sample_size;
    P v[V], d[V];
    inst_chunk<T, TEAM, VEC, V>(g, member, [&](int k, uint32_t i) {
        v[k] = P::load(inst_at<VEC>(yp, k, i));
        d[k] = P::load(inst_at<VEC>(dp, k, i));
    });
    double acc = 0.0;
    inst_chunk<T, TEAM, VEC, V>(g, member, [&](int k, uint32_t) { add_products<T, VEC>(acc, v[k], d[k]); });
    const double s = inst_exchange<TEAM, 0>(inst_partial<TEAM>(acc, lds), g, member, state, &tag, shared, [&](uint32_t m) {
        double r = 0.0;
        inst_chunk<T, TEAM, VEC, V>(g, m, [&](int k, uint32_t i) {
            add_products<T, VEC>(r, P::load(inst_at<VEC>(yp, k, i)), P::load(inst_at<VEC>(dp, k, i)));
        });
        return inst_partial<TEAM>(r, lds);
    });
    if (threadIdx.x == 0)
        team_leave(state);
    const T dot = static_cast<T>(inst_total<TEAM>(s, lds));
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
