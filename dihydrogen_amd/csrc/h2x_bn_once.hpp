// Batch-norm of a rank that shares its statistics with no one, in one launch each
// way: a team of threads loads every element of a channel into registers, sums
// them, and writes y (dx) from the registers.  Included by h2x_bn.hip.
//
// The two-launch kernels read x (backward: x and dy) twice, and the second launch
// waits for the first; up to tens of megabytes both cost more than what has to be
// moved.  Forward + backward, fp32, two launches each way -> one:
//   N 128, C 1024, 7 x 7           51.8 -> 25.3 us      N 16, C 512, 14 x 14   21.0 -> 9.8
//   N 16, C 256, 28 x 28           25.4 -> 12.5         N 4, C 64, 56 x 56     16.5 -> 11.0
//   N 64, C 1024, 14 x 14          78.2 -> 43.7         N 4, C 512, 56 x 56    43.4 -> 19.8
//   N 16, C 512, 7^3, halo of 1    54.7 -> 19.3         N 8, C 1024, 7 x 7     17.0 -> 7.7
// (one set of tensors over and over: up to 256 MB of it stay in the memory-side cache)
//
// A channel is as large as the registers of one CU allow: 512 KB, of which the
// largest variants hold 320 KB forward, 256 KB and 128 KB of LDS backward.  Larger ones, few, and those that would leave
// CUs idle or alone with one workgroup are for teams of workgroups (h2x_bn_team.hpp), where the caller has a state for them and
// outputs lie apart from inputs.
//
// The elements are those of the other kernels: rows in vectors of 16 bytes that may
// start on any element, the last vector of a row that is no whole number of vectors
// starting early; its `skip` leading elements belong to the vector before it and are
// not counted, and both vectors store the same values.  That also holds in place:
// the whole channel has been loaded before anything is stored.  Every term of the
// sums is rounded as in the two-launch kernels and added in fp64; only the order of
// the fp64 additions differs.
//
// Neighbouring channels go to one XCD (xcd_contiguous): short segments share their
// first and last cache line with the neighbours', and the L2 that has read the line
// serves the other half and merges the halves written.
#pragma once

// Tensors that lie alike: rows of interior elements.
struct OnceGeometry
{
    static constexpr bool kClears = false;
    // of a place: the element offset of a vector, and whether its element j counts
    static __host__ __device__ __forceinline__ uint32_t offset(uint32_t at) { return at >> 2; }
    static __host__ __device__ __forceinline__ bool counts(uint32_t at, int j) { return j >= static_cast<int>(at & 3); }

    uint32_t vectors;           // of one channel, all samples
    uint32_t width;             // elements of a row
    FastDiv spr;                // vectors a row is padded to
    FastDiv h, d;               // rows of a plane, planes of a segment
    uint32_t sy, sz;            // strides of rows and planes
    uint32_t stride_n;          // the last element of a channel is less than 2^30 elements from its first
    int64_t stride_c;
    uint32_t num_channels;
};

// Element offset of vector i of a channel, times four, plus the elements it skips.
template <int VEC>
__host__ __device__ __forceinline__ uint32_t once_place(const OnceGeometry& g, uint32_t i)
{
    static_assert(VEC <= 4, "two bits hold the elements skipped");
    const uint32_t r = fastdiv(i, g.spr);
    const uint32_t x = (i - r * g.spr.divisor) * VEC;
    const uint32_t last = g.width - VEC;
    const uint32_t first = x < last ? x : last;
    uint32_t n = r, at = first;
    if (g.h.divisor * g.d.divisor != 1) // uniform: a dense segment is one row
    {
        const uint32_t q = fastdiv(r, g.h);
        n = fastdiv(q, g.d);
        at += (r - q * g.h.divisor) * g.sy + (q - n * g.d.divisor) * g.sz;
    }
    return (at + n * g.stride_n) * 4 + (x - first);
}

// Tensors of one haloed geometry whose outputs' halos are cleared: the vectors of the
// whole allocation; halo elements are read and not counted, and stored as zeros.  Their
// stores leave no partial lines (forward + backward, N 8, C 64, 30^3 with a halo of 1, us
// going round three sets of tensors: 87 in six launches, 68 here, 78 without clearing).
struct ClearGeometry
{
    static constexpr bool kClears = true;
    static __host__ __device__ __forceinline__ uint32_t offset(uint32_t at) { return at >> 4; }
    static __host__ __device__ __forceinline__ bool counts(uint32_t at, int j) { return (at >> j) & 1; }

    uint32_t vectors;     // of one channel, all samples
    FastDiv per_segment;  // vectors of a segment
    uint32_t last;        // of these: the elements before it
    RealBox box;
    uint32_t stride_n;    // the last element of a channel is less than 2^28 elements from its first
    int64_t stride_c;
    uint32_t num_channels;
};

// Element offset of vector i of a channel, times sixteen, plus a bit for each interior element.
template <int VEC>
__host__ __device__ __forceinline__ uint32_t once_place(const ClearGeometry& g, uint32_t i)
{
    static_assert(VEC <= 4, "four bits hold the interior elements");
    const uint32_t n = fastdiv(i, g.per_segment);
    // (a last vector that starts early shares only halo cells with the one before it, which stores the same zeros)
    const uint32_t first = (i - n * g.per_segment.divisor) * VEC;
    const uint32_t e = first < g.last ? first : g.last;
    return (e + n * g.stride_n) * 16 + interior_bits<VEC>(g.box, e);
}

// STREAM: past the caches.  Rows of a few hundred bytes are stored normally: their
// ends are partial lines, which the L2 merges with the neighbours' (N 128, C 1024,
// 7 x 7 forward 10.3 us, streaming 17.1; N 4, C 512, 56 x 56 10.3 and 8.8), unless
// the tensors are haloed and large.
template <typename T, int VEC, bool STREAM>
__device__ __forceinline__ void store_once(T* p, const T (&r)[VEC])
{
    if constexpr (STREAM)
    {
        store_vec<T, VEC, false>(p, r);
    }
    else
    {
        typedef T V __attribute__((ext_vector_type(VEC), aligned(sizeof(T))));
        V t;
#pragma unroll
        for (int j = 0; j < VEC; ++j)
            t[j] = r[j];
        *reinterpret_cast<V*>(p) = t;
    }
}

// N sums over the TEAM threads that share a channel, a wave or a whole workgroup: group k of the lanes of each wave
// returns the k-th (wave_sums).  lds: N doubles a wave.
template <int TEAM, int N>
__device__ __forceinline__ double lane_sums(const double (&s)[N], double* lds)
{
    double v = wave_sums<N>(s);
    if constexpr (TEAM > kWaveSize)
    {
        constexpr int kWaves = TEAM / kWaveSize;
        constexpr uint32_t kGroup = kWaveSize / N;
        static_assert(kWaves <= 16, "a group of lanes adds what the waves have left");
        const uint32_t lane = threadIdx.x % kWaveSize, k = lane / kGroup, w = lane % kGroup;
        if (w == 0)
            lds[k * kWaves + threadIdx.x / kWaveSize] = v;
        __syncthreads();
        v = lane_group_sum<N>(w < kWaves ? lds[k * kWaves + w] : 0.0);
    }
    return v;
}
template <int TEAM, int N>
__device__ __forceinline__ void team_sum(double (&v)[N], double* lds)
{
    const double t = lane_sums<TEAM, N>(v, lds);
#pragma unroll
    for (int k = 0; k < N; ++k)
        v[k] = read_lane(t, k * (kWaveSize / N));
}

// TEAM threads with K vectors each serve a channel; teams of one wave share a
// workgroup of 256 threads (and then meet at no barrier).
template <int TEAM>
constexpr int once_block()
{
    return TEAM < kBlockSize ? kBlockSize : TEAM;
}

template <typename T>
struct OnceForward
{
    const T *x, *scale, *bias;
    T *mean, *var, *running_mean, *running_var, *y;
    T n, decay, epsilon;
    // a program that keeps no running statistics may give the buffers of mean and variance for them, or one for both
    bool shared = running_mean == mean || running_mean == var || running_var == mean || running_var == var || running_var == running_mean;
};

// By one thread a channel; the running statistics are read where they are due.
template <typename T>
__device__ __forceinline__ void update_statistics(const OnceForward<T>& a, uint32_t c, T m, T variance)
{
    a.mean[c] = m;
    a.var[c] = variance;
    a.running_mean[c] = fma_t(a.decay, a.running_mean[c], (T(1) - a.decay) * m);
    a.running_var[c] = fma_t(a.decay, a.running_var[c], (T(1) - a.decay) * variance);
}

// What the threads of channel c need once its sums are there, loaded before the elements: behind the sums nothing else hides the
// wait (forward in us, loaded behind the sums and so: N 24, C 224, 5 x 4 3.40 and 3.08; N 16, C 256, 28 x 28 6.59 and
// 6.42; N 64, C 512, 14 x 14 12.2 and 12.0; from 20 us on equal).
template <typename T>
struct ChannelParams
{
    T scale, bias, running_mean, running_var;
    __device__ __forceinline__ ChannelParams(const OnceForward<T>& a, uint32_t c)
        : scale(a.scale[c]), bias(a.bias[c]), running_mean(a.running_mean[c]), running_var(a.running_var[c])
    {
    }
    // by one thread a channel
    __device__ __forceinline__ void store_statistics(const OnceForward<T>& a, uint32_t c, T m, T variance) const
    {
        if (a.shared) // uniform
            return update_statistics(a, c, m, variance);
        a.mean[c] = m;
        a.var[c] = variance;
        a.running_mean[c] = fma_t(a.decay, running_mean, (T(1) - a.decay) * m);
        a.running_var[c] = fma_t(a.decay, running_var, (T(1) - a.decay) * variance);
    }
};

template <typename T, int TEAM, int K, bool STREAM, typename G>
__global__ __launch_bounds__(once_block<TEAM>()) void bn_once_forward_kernel(const G g,
                                                                            const OnceForward<T> a)
{
    static_assert(TEAM == kWaveSize || TEAM >= kBlockSize, "a wave or a workgroup");
    constexpr int VEC = 16 / sizeof(T);
    __shared__ double lds[TEAM > kWaveSize ? 2 * TEAM / kWaveSize : 1];
    const uint32_t c = xcd_contiguous(blockIdx.x, gridDim.x) * (once_block<TEAM>() / TEAM) + threadIdx.x / TEAM;
    const uint32_t t = threadIdx.x % TEAM;
    if (c >= g.num_channels) // a whole team
        return;
    const ChannelParams<T> params(a, c);
    const T* const x = a.x + c * g.stride_c;
    T v[K][VEC];
    uint32_t at[K];
#pragma unroll
    for (int u = 0; u < K; ++u)
        if (u * TEAM < g.vectors && u * TEAM + t < g.vectors)
        {
            at[u] = once_place<VEC>(g, u * TEAM + t);
            load_vec<T, VEC, false>(x + G::offset(at[u]), v[u]);
        }
    double s[2] = {0.0, 0.0};
#pragma unroll
    for (int u = 0; u < K; ++u)
        if (u * TEAM < g.vectors && u * TEAM + t < g.vectors)
        {
#pragma unroll
            for (int j = 0; j < VEC; ++j)
                if (G::counts(at[u], j))
                {
                    const double d = static_cast<double>(v[u][j]);
                    s[0] += d;
                    s[1] = __builtin_fma(d, d, s[1]);
                }
        }
    team_sum<TEAM>(s, lds);
    T m, variance;
    sums_to_mean_var(static_cast<T>(s[0]), static_cast<T>(s[1]), a.n, &m, &variance);
    if (t == 0)
        params.store_statistics(a, c, m, variance);
    const T inv_stdev = inv_sqrt_t(variance + a.epsilon);
    const T sc = params.scale, bi = params.bias;
    T* const y = a.y + c * g.stride_c;
#pragma unroll
    for (int u = 0; u < K; ++u)
        if (u * TEAM < g.vectors && u * TEAM + t < g.vectors)
        {
#pragma unroll
            for (int j = 0; j < VEC; ++j)
                v[u][j] = G::kClears && !G::counts(at[u], j) ? T(0) : fma_t((v[u][j] - m) * inv_stdev, sc, bi);
            store_once<T, VEC, STREAM>(y + G::offset(at[u]), v[u]);
        }
}

template <typename T>
struct OnceBackward
{
    const T *x, *dy, *mean, *var, *scale;
    T *dscale, *dbias, *dmean, *dvar, *dx;
    T n, n_minus_1, epsilon;
};

// IN_LDS: that many of a thread's K vectors of dy stay in LDS, where the registers
// of a CU do not hold both tensors (each thread reads what it has written).
template <typename T, int TEAM, int K, bool STREAM, int IN_LDS, typename G>
__global__ __launch_bounds__(once_block<TEAM>()) void bn_once_backward_kernel(const G g,
                                                                             const OnceBackward<T> a)
{
    static_assert(TEAM == kWaveSize || TEAM >= kBlockSize, "a wave or a workgroup");
    constexpr int VEC = 16 / sizeof(T);
    // the places of the vectors: where registers are short they are worked out again in each step, unless that is long
    constexpr bool kKept = IN_LDS == 0 || G::kClears;
    typedef T V __attribute__((ext_vector_type(VEC)));
    __shared__ double lds[TEAM > kWaveSize ? 4 * TEAM / kWaveSize : 1];
    __shared__ V parked[IN_LDS > 0 ? IN_LDS * TEAM : 1];
    const uint32_t c = xcd_contiguous(blockIdx.x, gridDim.x) * (once_block<TEAM>() / TEAM) + threadIdx.x / TEAM;
    const uint32_t t = threadIdx.x % TEAM;
    if (c >= g.num_channels)
        return;
    const int64_t base = c * g.stride_c;
    T xv[K][VEC], dv[K > IN_LDS ? K - IN_LDS : 1][VEC];
    uint32_t at[K];
    auto live = [&](int u) { return u * TEAM < g.vectors && u * TEAM + t < g.vectors; };
    auto gradient = [&](int u, T (&d)[VEC]) {
#pragma unroll
        for (int j = 0; j < VEC; ++j)
            d[j] = u < IN_LDS ? parked[(u < IN_LDS ? u : 0) * TEAM + t][j] : dv[u < IN_LDS ? 0 : u - IN_LDS][j];
    };
#pragma unroll
    for (int u = 0; u < K; ++u)
        if (live(u))
        {
            at[u] = once_place<VEC>(g, u * TEAM + t);
            load_vec<T, VEC, false>(a.x + base + G::offset(at[u]), xv[u]);
            if (u < IN_LDS)
            {
                T d[VEC];
                load_vec<T, VEC, false>(a.dy + base + G::offset(at[u]), d);
                V p;
#pragma unroll
                for (int j = 0; j < VEC; ++j)
                    p[j] = d[j];
                parked[(u < IN_LDS ? u : 0) * TEAM + t] = p;
            }
            else
            {
                load_vec<T, VEC, false>(a.dy + base + G::offset(at[u]), dv[u < IN_LDS ? 0 : u - IN_LDS]);
            }
        }
    const T m = a.mean[c];
    const T sc = a.scale[c];
    const T inv_stdev = inv_sqrt_t(a.var[c] + a.epsilon);
    const T dvar_factor = inv_stdev * inv_stdev * inv_stdev / T(2);
    double s[4] = {0.0, 0.0, 0.0, 0.0};
    [[maybe_unused]] uint32_t again = t; // of the present step: where nothing is kept the compiler shall not keep it either
    if constexpr (!kKept)
        asm volatile("" : "+v"(again));
#pragma unroll
    for (int u = 0; u < K; ++u)
        if (live(u))
        {
            if constexpr (!kKept)
                at[u] = once_place<VEC>(g, u * TEAM + again);
            T d[VEC];
            gradient(u, d);
#pragma unroll
            for (int j = 0; j < VEC; ++j)
                if (G::counts(at[u], j))
                {
                    const T xm = xv[u][j] - m;
                    const T dxhat = d[j] * sc;
                    const double dd = static_cast<double>(d[j]);
                    s[0] = __builtin_fma(dd, static_cast<double>(xm * inv_stdev), s[0]);
                    s[1] += dd;
                    s[2] += static_cast<double>(dxhat);
                    s[3] += static_cast<double>(dxhat * xm);
                }
        }
    team_sum<TEAM>(s, lds);
    const T dmean = static_cast<T>(s[2] * -static_cast<double>(inv_stdev));
    const T dvar = static_cast<T>(s[3] * -static_cast<double>(dvar_factor));
    if (t == 0)
    {
        a.dscale[c] = static_cast<T>(s[0]);
        a.dbias[c] = static_cast<T>(s[1]);
        a.dmean[c] = dmean;
        a.dvar[c] = dvar;
    }
    const T dmean_term = dmean / a.n;
    const T dvar_term = dvar * T(2) / a.n_minus_1;
    if constexpr (!kKept)
        asm volatile("" : "+v"(again));
#pragma unroll
    for (int u = 0; u < K; ++u)
        if (live(u))
        {
            if constexpr (!kKept)
                at[u] = once_place<VEC>(g, u * TEAM + again);
            T d[VEC];
            gradient(u, d);
#pragma unroll
            for (int j = 0; j < VEC; ++j)
                xv[u][j] = G::kClears && !G::counts(at[u], j)
                               ? T(0)
                               : fma_t(xv[u][j] - m, dvar_term, fma_t(d[j] * sc, inv_stdev, dmean_term));
            store_once<T, VEC, STREAM>(a.dx + base + G::offset(at[u]), xv[u]);
        }
}
