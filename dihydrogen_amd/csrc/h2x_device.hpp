// Device-side helpers shared by the gfx950 kernels: wave64 reductions built on
// DPP lane permutes, a fixed-order block reduction through LDS, unaligned
// 16-byte vector types, and the host-side status plumbing.
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>

#include <cstdint>
#include <tuple>

#include "h2x.h"

namespace h2x
{

constexpr int kWaveSize = 64;
constexpr int kBlockSize = 256;
constexpr int kWavesPerBlock = kBlockSize / kWaveSize;

inline hipStream_t as_stream(h2x_stream_t s)
{
    return reinterpret_cast<hipStream_t>(s);
}

// Status of the launch that was just issued.
inline int launch_status()
{
    return static_cast<int>(hipGetLastError());
}

#ifdef __HIPCC__
// Launches a kernel as <<<grid, block, 0, stream>>> does, without handing the configuration to the
// runtime in a call of its own and fetching it back in another (2.30 us a launch so, 2.15 here).
template <typename... P, typename... A>
inline void launch(void (*kernel)(P...), dim3 grid, dim3 block, hipStream_t stream, A&&... args)
{
    static_assert(sizeof...(P) == sizeof...(A), "an argument for each parameter");
    std::tuple<P...> values(static_cast<P>(args)...);
    std::apply(
        [&](P&... v) {
            void* pointers[] = {const_cast<void*>(static_cast<const void*>(&v))...};
            (void) hipLaunchKernel(reinterpret_cast<const void*>(kernel), grid, block, pointers, 0, stream);
        },
        values);
}
#endif

inline bool aligned16(const void* p)
{
    return (reinterpret_cast<uintptr_t>(p) & 15u) == 0;
}

// ---- division by a launch-time constant ------------------------------------
// n / d for n < 2^31 by multiply-high and shift.
struct FastDiv
{
    uint32_t divisor;
    uint32_t multiplier;
    uint32_t shift;
};

inline FastDiv make_fastdiv(uint32_t d)
{
    FastDiv f{d, 0u, 0u};
    if (d > 1)
    {
        const uint32_t log2 = 32u - static_cast<uint32_t>(__builtin_clz(d - 1)); // ceil(log2 d), d >= 2
        const uint32_t p = 31 + log2;
        f.multiplier = static_cast<uint32_t>(((1ull << p) + d - 1) / d);
        f.shift = p - 32;
    }
    return f;
}

__host__ __device__ inline uint32_t fastdiv(uint32_t n, const FastDiv& f)
{
#ifdef __HIP_DEVICE_COMPILE__
    return f.divisor == 1 ? n : __umulhi(n, f.multiplier) >> f.shift;
#else
    return f.divisor == 1
               ? n
               : static_cast<uint32_t>((static_cast<uint64_t>(n) * f.multiplier) >> 32) >> f.shift;
#endif
}

#ifdef __HIPCC__

// ---- lane permutes --------------------------------------------------------
// DPP controls: quad_perm [1,0,3,2] and [2,3,0,1] swap lanes at distance 1 and
// 2 inside a quad; row_ror:n rotates a 16-lane row.
constexpr int kDppQuadSwap1 = 0xB1;
constexpr int kDppQuadSwap2 = 0x4E;
constexpr int kDppRowRor4 = 0x124;
constexpr int kDppRowRor8 = 0x128;

template <int Ctrl>
__device__ __forceinline__ float dpp_move(float v)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), Ctrl, 0xf, 0xf, false));
}
template <int Ctrl>
__device__ __forceinline__ double dpp_move(double v)
{
    const long long bits = __double_as_longlong(v);
    int lo = static_cast<int>(bits & 0xffffffffll);
    int hi = static_cast<int>(bits >> 32);
    lo = __builtin_amdgcn_update_dpp(0, lo, Ctrl, 0xf, 0xf, false);
    hi = __builtin_amdgcn_update_dpp(0, hi, Ctrl, 0xf, 0xf, false);
    return __longlong_as_double((static_cast<long long>(hi) << 32)
                                | static_cast<unsigned int>(lo));
}

// What the two lanes that are D (16 or 32) apart hold, in both of them: the one in the even row
// (lower half) first.  Swapped in the vector unit; a shuffle goes through LDS, and a reduction is a
// chain of them that a workgroup waits for (batch-norm forward + backward with shuffles -> with swaps: doubles, N 8,
// C 32, 33^3, 88.3 -> 86.8 us; N 8, C 64, 56 x 56 14.5 -> 14.3; N 8, C 64, 30^3 with a halo 77.1 -> 76.6).
template <int D>
__device__ __forceinline__ void lanes_apart(uint32_t v, uint32_t* even, uint32_t* odd)
{
    static_assert(D == 16 || D == 32, "rows of 16 lanes, or halves of the wave");
    const auto p = D == 16 ? __builtin_amdgcn_permlane16_swap(v, v, false, false)
                           : __builtin_amdgcn_permlane32_swap(v, v, false, false);
    *even = p[0];
    *odd = p[1];
}
template <int D>
__device__ __forceinline__ void lanes_apart(float v, float* even, float* odd)
{
    uint32_t e, o;
    lanes_apart<D>(__float_as_uint(v), &e, &o);
    *even = __uint_as_float(e);
    *odd = __uint_as_float(o);
}
template <int D>
__device__ __forceinline__ void lanes_apart(double v, double* even, double* odd)
{
    const unsigned long long bits = __double_as_longlong(v);
    uint32_t el, ol, eh, oh;
    lanes_apart<D>(static_cast<uint32_t>(bits), &el, &ol);
    lanes_apart<D>(static_cast<uint32_t>(bits >> 32), &eh, &oh);
    *even = __longlong_as_double(static_cast<long long>(static_cast<unsigned long long>(eh) << 32 | el));
    *odd = __longlong_as_double(static_cast<long long>(static_cast<unsigned long long>(oh) << 32 | ol));
}

// v combined with what the lane D apart holds; f is commutative.
template <int D, typename T, typename F>
__device__ __forceinline__ T combine_apart(T v, const F& f)
{
    T even, odd;
    lanes_apart<D>(v, &even, &odd);
    return f(even, odd);
}

// Sum over the 64 lanes of a wave; every lane returns the total.  The
// combination order is fixed (distance 1, 2, 4, 8 inside a row, then rows 16
// and 32 apart), so the result does not depend on scheduling.
__device__ __forceinline__ double wave_sum(double v)
{
    const auto add = [](double a, double b) { return a + b; };
    v += dpp_move<kDppQuadSwap1>(v);
    v += dpp_move<kDppQuadSwap2>(v);
    v += dpp_move<kDppRowRor4>(v);
    v += dpp_move<kDppRowRor8>(v);
    v = combine_apart<16>(v, add);
    return combine_apart<32>(v, add);
}

// Butterfly over the 64 lanes of a wave, 32 apart first: f is commutative, and every lane returns the same.
template <typename T, typename F>
__device__ __forceinline__ T wave_combine(T v, const F& f)
{
    v = combine_apart<32>(v, f);
    v = combine_apart<16>(v, f);
    v = f(v, dpp_move<kDppRowRor8>(v));
    v = f(v, dpp_move<kDppRowRor4>(v)); // lanes 8 apart hold the same: 4 to the right is as good as 4 apart
    v = f(v, dpp_move<kDppQuadSwap2>(v));
    return f(v, dpp_move<kDppQuadSwap1>(v));
}

// Several sums over the 64 lanes of a wave at once: the lanes are cut into N groups (two or four), and group k returns the
// total of v[k], all its lanes the same bits. In a fixed order. Four sums take seven additions in a row so, one after
// another 24.
template <int N>
__device__ __forceinline__ double lane_group_sum(double v)
{
    static_assert(N == 2 || N == 4, "groups of 32 or of 16 lanes");
    if constexpr (N == 2)
        v = combine_apart<16>(v, [](double a, double b) { return a + b; });
    v += dpp_move<kDppRowRor8>(v);
    v += dpp_move<kDppRowRor4>(v); // lanes 8 apart hold the same
    v += dpp_move<kDppQuadSwap2>(v);
    return v + dpp_move<kDppQuadSwap1>(v);
}
// Of each pair of lanes D (16 or 32) apart: the sum of a in the even row (lower half), that of b in the odd one.
template <int D>
__device__ __forceinline__ double add_apart(double a, double b)
{
    const unsigned long long x = __double_as_longlong(a), y = __double_as_longlong(b);
    const uint32_t xl = static_cast<uint32_t>(x), xh = static_cast<uint32_t>(x >> 32), yl = static_cast<uint32_t>(y),
                   yh = static_cast<uint32_t>(y >> 32);
    // what a has in the odd rows and b in the even ones change places
    const auto lo = D == 16 ? __builtin_amdgcn_permlane16_swap(xl, yl, false, false)
                            : __builtin_amdgcn_permlane32_swap(xl, yl, false, false);
    const auto hi = D == 16 ? __builtin_amdgcn_permlane16_swap(xh, yh, false, false)
                            : __builtin_amdgcn_permlane32_swap(xh, yh, false, false);
    const uint32_t l0 = lo[0], l1 = lo[1], h0 = hi[0], h1 = hi[1];
    return __longlong_as_double(static_cast<long long>(static_cast<unsigned long long>(h0) << 32 | l0))
           + __longlong_as_double(static_cast<long long>(static_cast<unsigned long long>(h1) << 32 | l1));
}
template <int N>
__device__ __forceinline__ double wave_sums(const double (&v)[N])
{
    if constexpr (N == 2)
        return lane_group_sum<2>(add_apart<32>(v[0], v[1]));
    else
        return lane_group_sum<4>(add_apart<16>(add_apart<32>(v[0], v[2]), add_apart<32>(v[1], v[3])));
}
// wave_sum of two or four sums at once, bit for bit: lane k (k < N) returns the total of v[k].  The first steps of the
// tree, lanes 1 apart and, of four sums, 2 apart, leave one sum a lane; the others take an addition each.
template <int N>
__device__ __forceinline__ double wave_sums_in_order(const double (&v)[N])
{
    static_assert(N == 2 || N == 4, "a sum a lane of a pair or a quad");
    // even lanes (of quads: the lower pair) keep the first of two and send the second
    const auto halve = [](bool upper, double a, double b, auto swap) {
        return (upper ? b : a) + swap(upper ? a : b);
    };
    const uint32_t lane = threadIdx.x;
    const auto next = [](double x) { return dpp_move<kDppQuadSwap1>(x); };
    const auto pair = [](double x) { return dpp_move<kDppQuadSwap2>(x); };
    double t = halve(lane & 1, v[0], v[1], next);
    if constexpr (N == 4)
        t = halve(lane & 2, t, halve(lane & 1, v[2], v[3], next), pair);
    else
        t += pair(t);
    t += dpp_move<kDppRowRor4>(t);
    t += dpp_move<kDppRowRor8>(t);
    const auto add = [](double a, double b) { return a + b; };
    t = combine_apart<16>(t, add);
    return combine_apart<32>(t, add);
}
// What lane `lane` holds, in a scalar register.
__device__ __forceinline__ double read_lane(double v, int lane)
{
    const unsigned long long bits = __double_as_longlong(v);
    const uint32_t lo = __builtin_amdgcn_readlane(static_cast<uint32_t>(bits), lane);
    const uint32_t hi = __builtin_amdgcn_readlane(static_cast<uint32_t>(bits >> 32), lane);
    return __longlong_as_double(static_cast<long long>(static_cast<unsigned long long>(hi) << 32 | lo));
}

// Steps of wave_sum from those that add lanes `first` apart (1, 2 or 4): lanes that leave the same remainder when divided by
// `first` are added, each such set by itself, and all of them return its sum.
__device__ __forceinline__ double wave_sum_from(double v, uint32_t first)
{
    if (first < 2)
        v += dpp_move<kDppQuadSwap1>(v);
    if (first < 4)
        v += dpp_move<kDppQuadSwap2>(v);
    v += dpp_move<kDppRowRor4>(v);
    v += dpp_move<kDppRowRor8>(v);
    const auto add = [](double a, double b) { return a + b; };
    v = combine_apart<16>(v, add);
    return combine_apart<32>(v, add);
}

// Sum of K values per thread over a 256-thread workgroup.  `lds` must hold
// K * kWavesPerBlock doubles.  Every thread returns the totals in v[].
template <int K>
__device__ __forceinline__ void block_sum(double (&v)[K], double* lds)
{
    const int lane = threadIdx.x & (kWaveSize - 1);
    const int wave = threadIdx.x / kWaveSize;
#pragma unroll
    for (int k = 0; k < K; ++k)
        v[k] = wave_sum(v[k]);
    __syncthreads(); // lds may still be read by a previous use
    if (lane == 0)
    {
#pragma unroll
        for (int k = 0; k < K; ++k)
            lds[k * kWavesPerBlock + wave] = v[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; ++k)
    {
        double t = lds[k * kWavesPerBlock];
#pragma unroll
        for (int w = 1; w < kWavesPerBlock; ++w)
            t += lds[k * kWavesPerBlock + w];
        v[k] = t;
    }
}

// ---- teams of workgroups ---------------------------------------------------------
// How the workgroups of a team exchange doubles through memory.  What is exchanged validates itself: half a double travels with
// the tag of the call in one 64-bit access of the whole device's scope, so nothing has to be ordered and nothing
// cleared.  The tag is the team's counter plus one: a member reads the counter before it stores anything, and
// adds one to it when it has all that it needs, so all members of a call find the same value, and no later call
// finds it again.  (A member that gave up waiting may add early; who then reads a larger counter is not
// believed, believes no one, and works all out.  The next call's counter is larger still.  Tags come round after 2^32
// arrivals; a word would have to lie untouched for just that long.)  Nobody waits for ever: after max_polls looks a
// member works out what it misses from memory, which is why outputs may not overlap inputs.
//
// A team's state: the counter, on a line of its own, then the words, zero before the first call.
constexpr uint32_t kCounterWords = 16;

__device__ __forceinline__ unsigned long long team_load(const unsigned long long* p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void team_store(unsigned long long* p, uint32_t tag, uint32_t half)
{
    __hip_atomic_store(p, static_cast<unsigned long long>(tag) << 32 | half, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The tag of a call.
__device__ __forceinline__ uint32_t team_tag(const unsigned long long* state)
{
    return static_cast<uint32_t>(team_load(state)) + 1;
}
// One to the counter, by one thread of a member that has all it needs.
__device__ __forceinline__ void team_leave(unsigned long long* state)
{
    __hip_atomic_fetch_add(state, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Stores v at place `at` of `places`; the same half of all places lies side by side, so that a look reads few lines.
__device__ __forceinline__ void team_put(unsigned long long* words, uint32_t places, uint32_t at, uint32_t tag, double v)
{
    const unsigned long long bits = __double_as_longlong(v);
    team_store(words + at, tag, static_cast<uint32_t>(bits));
    team_store(words + places + at, tag, static_cast<uint32_t>(bits >> 32));
}
// Whether a place, whose first half lies at `at`, holds what this call has stored; then that in *v.
__device__ __forceinline__ bool team_look(const unsigned long long* at, uint32_t places, uint32_t tag, double* v)
{
    const unsigned long long lo = team_load(at), hi = team_load(at + places);
    const bool there = lo >> 32 == tag && hi >> 32 == tag;
    if (there)
        *v = __longlong_as_double(hi << 32 | (lo & 0xffffffffull));
    return there;
}
// What it holds, once it holds it; false after max_polls looks.
__device__ __forceinline__ bool team_get(const unsigned long long* at, uint32_t places, uint32_t tag, uint32_t max_polls,
                                         double* v)
{
    bool there = false;
    for (uint32_t poll = 0; poll < max_polls && !there; ++poll)
    {
        if (poll > 0)
            __builtin_amdgcn_s_sleep(4);
        there = team_look(at, places, tag, v);
    }
    return there;
}

// Whether two tensors of so many bytes do not overlap.
inline bool apart(const void* a, const void* b, size_t bytes)
{
    const uintptr_t x = reinterpret_cast<uintptr_t>(a), y = reinterpret_cast<uintptr_t>(b);
    return x + bytes <= y || y + bytes <= x;
}

constexpr int kMaxDevices = 64;

// CUs of the current device (0: there is none), asked for once: a device does not change, and
// the question costs a small call most of a microsecond.
inline uint32_t compute_units()
{
    static std::atomic<int> known[kMaxDevices];
    int device = 0, cus = 0;
    if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= kMaxDevices)
        return 0;
    cus = known[device].load(std::memory_order_relaxed);
    if (cus == 0
        && hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) == hipSuccess)
        known[device].store(cus, std::memory_order_relaxed);
    return static_cast<uint32_t>(cus);
}

// CUs that a launch rule counts with: an MI355X's where no device can be asked.
inline uint32_t chip_units()
{
    const uint32_t cus = compute_units();
    return cus ? cus : 256;
}

// ---- workgroup order ---------------------------------------------------------
// Workgroups go to the eight XCDs round-robin (workgroup i runs on XCD i mod
// 8) and every XCD has its own L2 with its own address-interleaved channels.
// When consecutive workgroups walk through memory in equal steps, the
// workgroups of one XCD visit addresses 8 steps apart and can end up on a
// fraction of its L2 channels; with power-of-two strides between the streams
// of one workgroup this costs a quarter of the bandwidth (channel softmax,
// N 32, C 19, 1024 x 2048: 3.9 TB/s -> 5.4 TB/s).  xcd_contiguous gives each
// XCD one contiguous eighth of the tiles instead.  `padded_grid` is the grid
// size, a multiple of 8; the result may exceed the number of tiles needed.
constexpr unsigned int kNumXcd = 8;

__device__ __forceinline__ unsigned int xcd_contiguous(unsigned int block, unsigned int padded_grid)
{
    return (block % kNumXcd) * (padded_grid / kNumXcd) + block / kNumXcd;
}

// ---- vectors --------------------------------------------------------------
// 16-byte vectors that may sit on any element boundary.
template <typename T, int N>
struct alignas(sizeof(T)) UVec
{
    T v[N];
};

template <typename T, int N>
struct alignas(sizeof(T) * N) AVec
{
    T v[N];
};

#endif // __HIPCC__

} // namespace h2x
