// The forward halo exchange of a whole grid of ranks whose tensors share the
// device, in one launch, and the clearing of their halos in one launch.
//
// The exchange proceeds dimension by dimension in the reference (legacy/include/
// distconv/tensor/halo_exchange_cuda.hpp:56-106): the strip of a later dimension
// carries the halo cells that an earlier one has filled.  Where every tensor is
// addressable that order need not be played out: what ends up in a halo cell is
// the cell of the rank that is reached by stepping to the neighbour along every
// dimension in which the cell lies in the halo and a neighbour exists.  Along a
// dimension without a neighbour the cell keeps its halo coordinate; no phase
// writes such a cell of the source, so nothing that is read is written here and
// the whole exchange has no order.  Strips go straight from tensor to tensor.
//
// The halo of a rank is cut into regions, one per combination of {interior,
// lower, upper} of the outer two spatial dimensions, crossed with the two kinds
// of work along the rows.  "Runs" are the interior of the row in 16-byte vectors
// that may start on any element; the last vector of a row that is no whole number
// of vectors starts early and moves a few elements twice.  "Ends" are the halo
// cells at both ends of the row, for all ranks of a line along dimension 0 in the
// same thread.  They are bound by whole lines of memory: a cell of 4 bytes costs
// the read of a 128-byte line and its write-back.  The line of a row seam holds the
// two halo cells that one rank receives and the two cells that its neighbours take;
// serving the line of ranks together reads it once and writes it in the L2 that
// has just read it.  Measured on four ranks of 64 x 256 x 128 x 32 cells with
// halos of 3: 254 us, one rank per workgroup 300 us; eight ranks of 128^3 x 32
// (periodic, all dimensions) 273 and 288 us, packing and unpacking 338 us.
// Nontemporal loads lose the line before the store arrives (387 us).
//
// All regions of all ranks are one launch: an exchange of small shards is bound
// by launches (4 ranks of 29 x 29 x 64 channels x 4 samples, clear and exchange: 14
// launches 57 us, two 9.4 us).  Descriptors travel in the kernel arguments;
// nothing is allocated or kept.
#include "h2x_copy_kernel.hpp"

#include <algorithm>

namespace h2x
{
namespace grid
{
namespace
{

using copy::Audit;
using copy::current_audit;
using copy::DeviceMem;
using copy::TraceMem;
using copy::Words;

// A cell that a launch touches once for several strips: an audit, which expects a touch for each, counts so many (that
// it is one touch, and of one thread, the audit sees by the threads, see issue_fold_grid).
__device__ __forceinline__ const DeviceMem& of_strips(const DeviceMem& mem, int)
{
    return mem;
}
TraceMem of_strips(const TraceMem& mem, int strips)
{
    return TraceMem{mem.audit, strips};
}

constexpr int kMaxRanks = 16;
constexpr int kMaxSpatial = 3;
constexpr int kMaxRegions = 9 + 8;
constexpr int kBlock = 256;
constexpr uint64_t kMaxRankBlocks = 0x7fffff;         // indexes of one rank stay below 2^31
constexpr uint64_t kMaxBlocks = 0xffffffffu / kBlock; // a launch counts its threads in 32 bits
// Ranks of a line whose ends a thread loads before it stores any (measured: 1, 2, 4; two hold
// the fewest registers at the rate of four).
constexpr int kRanksPerTurn = 2;
// Rows of a rank from which on the reverse exchange goes line by line: fewer take as long as one thread does
// (5 x 2 x 14 x 6 x 47 of doubles on 2 x 1 x 4, 660 rows: line by line 8.4 us, rank by rank 7.9; 9 x 8 x 287 x 109
// on 4 x 2, 5,500 rows: 9.4 and 11.1).
constexpr int64_t kLineRows = 4096;
// Halo strips in bytes, of all ranks, up to which a reverse exchange of two or three dimensions is one launch.  It saves
// one launch or two, of 1.5 to 2.5 us each; its regions, a few times as many as strips, keep more workgroups waiting for
// few cells, which costs more with size.  Three launches or two and one, us:
//   three dimensions: 2 x 3 x 15 x 21 x 17 on 2^3 9.4 and 5.5; 1 x 11 x 46 x 67 x 50 on 2^3, 0.76 MB 10.2 and 6.8;
//   9 x 11 x 28 x 34 x 28 on 2^3, periodic, 4.3 MB 17.0 and 14.2; 6 x 50 x 27^2 x 25 on 2^3, halos of 2, 18 MB 35.9, 43;
//   two: 1 x 32 x 57 x 57 on 2 x 2 6.4 and 5.3; 2 x 44 x 264 x 116 on 4 x 2, 0.70 MB 6.9 and 6.5; 2 x 15 x 15 x 30 x 79
//   on 2 x 4, 0.98 MB 8.6 and 10.8.
// The line for two dimensions lies below the last two, on the safe side: just above it one launch gains a twentieth where
// it gains, and at 0.98 MB loses a quarter.
constexpr uint64_t kFoldBytes2 = 640 << 10, kFoldBytes3 = 4608 << 10;

// One end of a row of a rank, halo cell 0: where its values come from.
struct RowEnd
{
    char* from;     // halo cell 0 of row 0 lies here: at the neighbour's other end, without one at this end of this rank
    uint32_t pitch; // elements of a row there
    uint32_t filled; // there is a neighbour
};

// Whole words throughout: a byte cannot be read through the scalar cache, and a
// workgroup spends most of its time before its first access on what it reads here.  What can be
// followed on the host is: the rank that a region's cells come from, and the neighbours along a row.  (A chain of a
// dozen loads, some of them through the vector memory, to one of five scalar ones, us, exchange or clear and exchange: 4 x 64 x
// 57 x 57 on 2 x 2 6.95 -> 6.55, 3 x 40 x 127 x 327 on 2 x 4, halos of 2 6.23 -> 5.66, 2 x 97 x 187 x 181 on 2 x 2 5.25 -> 4.80,
// 3 x 50 x 16 x 36 x 72 on 2 x 4, halos of 3 26.3 -> 24.9. Asking for all of the arguments' lines at once before the
// chain gave no more.)
struct Rank
{
    char* tensor;                 // start of the real allocation
    RowEnd end[2];
    uint32_t source[kMaxSpatial]; // by the digit of dimension 2, eight bits by that of dimension 1: see kSourceRank
    int32_t local[kMaxSpatial];   // interior extents
    int32_t peer[kMaxSpatial][2]; // rank of the neighbour, or -1
    FastDiv units;                // by vectors (or elements) of an interior row
    FastDiv extent[2];            // by local[1], local[2]
    uint32_t clear;               // bit 2 * d + side: this strip is cleared (reverse: there is no neighbour); see kRestEmpty
    uint32_t vectors;             // the interior row holds at least one vector
};

struct Args
{
    uint32_t first[kMaxRegions]; // first workgroup of a region (beyond the last one: none)
    uint32_t code[kMaxRegions];  // ends + 4 * digit of dimension 1 + 16 * digit of dimension 2;
                                 // digits: 0 interior, 1 lower, 2 upper halo
    FastDiv halo[kMaxSpatial];     // by the halo width (1 where there is none)
    FastDiv both_ends;             // by twice the halo width of a row
    FastDiv ranks;                 // by num_ranks
    FastDiv lines;                 // by the number of lines
    int32_t line;                  // ranks in a line
    int32_t width[kMaxSpatial];
    uint32_t outer; // channels x samples
    Rank rank[kMaxRanks];
};

// The rank that the cells of a region come from, four bits, and in which dimensions it is another one.
constexpr uint32_t kSourceRank = 15, kStepped = 8; // bit 4 for dimension 1, bit 5 for dimension 2
constexpr uint32_t kSteppedAny = 3 * 2 * kStepped;
// Of Rank::clear, from here on: the strips of dimension d leave nothing of the rank's real extent.
constexpr uint32_t kRestEmpty = 2 * kMaxSpatial;

// Start of a region's cells in dimension d (1 or 2) of a rank of so many interior cells, and where
// they start in the neighbour `src` they come from: the lower halo is its last interior
// cells, the upper one its first.
__host__ __device__ __forceinline__ uint32_t region_start(int w, int local, uint32_t digit)
{
    return digit == 0 ? w : digit == 1 ? 0 : w + local;
}
__host__ __device__ __forceinline__ uint32_t source_start(int w, int local, uint32_t digit, bool stepped)
{
    return !stepped ? region_start(w, local, digit) : digit == 1 ? local : w;
}

// The same value, in a scalar register (all lanes hold it): two values that are read by scalar loads
// stay two, instead of one vector load from either place.
__host__ __device__ __forceinline__ uint32_t in_scalar(uint32_t v)
{
#ifdef __HIP_DEVICE_COMPILE__
    return __builtin_amdgcn_readfirstlane(v);
#else
    return v;
#endif
}
__host__ __device__ __forceinline__ uint64_t in_scalar(const char* p)
{
    const uint64_t v = reinterpret_cast<uintptr_t>(p);
    return static_cast<uint64_t>(in_scalar(static_cast<uint32_t>(v >> 32))) << 32 | in_scalar(static_cast<uint32_t>(v));
}
template <typename T>
__host__ __device__ __forceinline__ const T* global_place(uint64_t v)
{
#ifdef __HIP_DEVICE_COMPILE__
    return (const T*) reinterpret_cast<const T __attribute__((address_space(1)))*>(v);
#else
    return reinterpret_cast<const T*>(v);
#endif
}

// The loads of a turn go out one after another: what a thread loads together, twice the lines of memory
// between their load and their store, is slower where the line is all that bounds (N x C x extents on a grid,
// us, together and so: 4 x 3 x 314 x 77 x 155 on 4 x 1 x 2, periodic 35.9 and 33.1; 5 x 4 x 99 x 61 x 92 on 2 x 1 x 2, halos
// of 3 16.9 and 15.8; 15 x 11 x 15 x 25 x 18 on 2^3, halos of 2 12.7 and 12.0) and no faster elsewhere.
__host__ __device__ __forceinline__ void one_by_one()
{
#ifdef __HIP_DEVICE_COMPILE__
    __builtin_amdgcn_s_waitcnt(0x0f70); // vector memory only
#endif
}

template <typename T, bool CLEAR, typename Mem>
__host__ __device__ __forceinline__ void body(const Args& a, uint32_t block, uint32_t thread, const Mem& mem)
{
    constexpr int VEC = 16 / sizeof(T);
    using W = typename Words<T, VEC>::unaligned_t;
    uint32_t first = 0, code = a.code[0];
#pragma unroll
    for (int i = 1; i < kMaxRegions; ++i)
        if (block >= a.first[i])
        {
            first = a.first[i];
            code = a.code[i];
        }
    const bool ends = code & 1;
    // Lines or ranks take turns workgroup by workgroup.
    const FastDiv& turns = ends ? a.lines : a.ranks;
    const uint32_t local_block = fastdiv(block - first, turns);
    const int r = static_cast<int>((block - first - local_block * turns.divisor) * (ends ? a.line : 1));
    const Rank& me = a.rank[r]; // ends: the first one of its line

    const uint32_t digit_y = code >> 2 & 3, digit_z = code >> 4;
    const FastDiv div_y = digit_y == 0 ? me.extent[0] : a.halo[1], div_z = digit_z == 0 ? me.extent[1] : a.halo[2];
    // what of it lies in a strip that has a neighbour to copy from (CLEAR: that is cleared) along dimension 1 or 2
    const uint32_t source = CLEAR ? static_cast<uint32_t>(r) : me.source[digit_z] >> (8 * digit_y);
    const uint32_t src = CLEAR ? r : source & kSourceRank; // ends: the first one of a line
    const bool moved = CLEAR ? (digit_y && (me.clear >> (1 + digit_y) & 1)) || (digit_z && (me.clear >> (3 + digit_z) & 1))
                             : (source & kSteppedAny) != 0;
    const Rank& from_rank = a.rank[src];
    const uint32_t y_to = region_start(a.width[1], me.local[1], digit_y), z_to = region_start(a.width[2], me.local[2], digit_z);
    const FastDiv div_x = ends ? a.both_ends : me.units;
    const uint32_t at = local_block * kBlock + thread;
    if (at >= div_y.divisor * div_z.divisor * a.outer * div_x.divisor || (!ends && !moved))
        return;
    const uint32_t row = fastdiv(at, div_x);
    uint32_t x = at - row * div_x.divisor;
    const uint32_t yz = fastdiv(row, div_y);
    const uint32_t y = row - yz * div_y.divisor;
    const uint32_t o = fastdiv(yz, div_z);
    const uint32_t z = yz - o * div_z.divisor;
    // rows of the real tensors (whose elements are fewer than 2^31)
    const uint32_t w = a.width[0];
    const auto real = [&](const Rank& q, int d) { return static_cast<uint32_t>(q.local[d] + 2 * a.width[d]); };
    const uint32_t row_to = (o * real(me, 2) + z_to + z) * real(me, 1) + y_to + y;
    uint32_t row_from = row_to;
    if constexpr (!CLEAR)
        row_from = (o * real(from_rank, 2)
                    + source_start(a.width[2], from_rank.local[2], digit_z, source & 4 * kStepped) + z)
                       * real(from_rank, 1)
                   + source_start(a.width[1], from_rank.local[1], digit_y, source & 2 * kStepped) + y;
    if (!ends)
    {
        T* const to = reinterpret_cast<T*>(me.tensor) + row_to * real(me, 0) + w;
        const T* const from = reinterpret_cast<const T*>(from_rank.tensor) + row_from * real(from_rank, 0) + w;
        if (me.vectors)
        {
            x *= VEC;
            const uint32_t last = static_cast<uint32_t>(me.local[0]) - VEC;
            x = x < last ? x : last;
            W v;
            if constexpr (CLEAR)
                v = W(T(0));
            else
                v = mem.template load<VEC, false>(from + x);
            mem.template store<VEC, false>(to + x, v);
        }
        else
        {
            mem.store1(to + x, CLEAR ? T(0) : mem.load1(from + x));
        }
        return;
    }
    // The ends of a row in every rank of the line: the lower end's cells, then the upper end's, then
    // the next row's, so that what neighbouring lanes write at a row seam lies side by side.
    const bool upper = x >= w;
    const uint32_t j = upper ? x - w : x;
#pragma unroll 1
    for (int base = 0; base < a.line; base += kRanksPerTurn)
    {
        T v[kRanksPerTurn];
        bool live[kRanksPerTurn];
#pragma unroll
        for (int i = 0; i < kRanksPerTurn; ++i)
        {
            live[i] = false;
            if (base + i >= a.line)
                continue;
            if constexpr (CLEAR)
            {
                live[i] = moved || (a.rank[r + base + i].clear >> (upper ? 1 : 0) & 1);
                v[i] = T(0);
            }
            else
            {
                const RowEnd& lo = a.rank[src + base + i].end[0];
                const RowEnd& hi = a.rank[src + base + i].end[1];
                const uint64_t lo_from = in_scalar(lo.from), hi_from = in_scalar(hi.from);
                const uint32_t lo_pitch = in_scalar(lo.pitch), hi_pitch = in_scalar(hi.pitch);
                const uint32_t lo_filled = in_scalar(lo.filled), hi_filled = in_scalar(hi.filled);
                live[i] = moved || (upper ? hi_filled : lo_filled) != 0;
                if (live[i])
                    v[i] = mem.load1(global_place<T>(upper ? hi_from : lo_from)
                                     + (row_from * (upper ? hi_pitch : lo_pitch) + j));
                if (i + 1 < kRanksPerTurn)
                    one_by_one();
            }
        }
#pragma unroll
        for (int i = 0; i < kRanksPerTurn; ++i)
            if (live[i])
            {
                const Rank& q = a.rank[r + base + i];
                mem.store1(reinterpret_cast<T*>(q.tensor)
                               + (row_to * (q.local[0] + 2 * w) + (upper ? w + q.local[0] : 0) + j),
                           v[i]);
            }
    }
}

// A seam of two ranks in the dimension of a reverse exchange. What a workgroup reads of its arguments stands between
// its start and its first access, so all that can be followed is followed on the host: two scalar loads, one after the
// other, instead of five (reverse exchanges, us: 4 x 64 x 57 x 57 on 2 x 2 9.2 -> 7.9; 8 x 6 x 13 x 13 x 12 on 2^3,
// periodic, halos of 3 14.4 -> 12.5; 2 x 34 x 68 x 105 x 34 of doubles on 2 x 2 x 1 9.9 -> 8.3; 9 x 2 x 63 x 156 x 131
// on 1 x 2 x 2, periodic 25.5 -> 21.2; 1 x 32 x 256^3 on 2^3, periodic 304 -> 297).
struct FoldSeam
{
    char *lower, *upper;              // the lower rank's upper boundary cells, whose upper halo follows them; the upper rank's lower halo,
                                      // whose lower boundary cells follow it: in row 0
    uint32_t lower_pitch, upper_pitch; // elements from row to row
    uint32_t run, rows;               // elements of a strip that lie together; how often
    FastDiv units;                    // by vectors (or elements) of a run
    uint32_t vectors;                 // a run holds at least one vector
};

struct FoldArgs
{
    FastDiv turns; // by the number of seams, or lines of ranks, that take turns workgroup by workgroup
    int32_t line;  // seams of a line; of a ring, seam i is the upper one of rank i
    FastDiv cells; // by the threads that serve a row's ends
    FoldSeam seam[kMaxRanks];
};

// How a dimension is folded: strip by strip, or dimension 0 line by line, with both sides of every seam or one end of
// every rank's row in a thread.
enum Fold : int
{
    kStrips = 0,
    kOpenLines = 1,
    kRings = 2
};

// Where the cells of one side of a seam are and where what is added to them comes from, both from the start of a row.
template <typename T>
struct FoldSide
{
    T* to;
    const T* from;
};
template <typename T>
__host__ __device__ __forceinline__ FoldSide<T> fold_side(const FoldSeam& s, uint32_t row, bool of_upper)
{
    T* const lower = reinterpret_cast<T*>(s.lower) + row * s.lower_pitch;
    T* const upper = reinterpret_cast<T*>(s.upper) + row * s.upper_pitch;
    return of_upper ? FoldSide<T>{upper + s.run, lower + s.run} : FoldSide<T>{lower, upper};
}

// One dimension of the reverse exchange: the halo strips of the dimension are folded into
// the boundary cells of the ranks they belong to.  A strip spans the real extents
// of the other dimensions, so along memory it is runs of `width` times the real
// extents below it, one per index above it.  A thread serves the same vector of
// both strips of a seam, what each rank gives and takes there: four loads in
// flight, and what a rank gives lies beside what it takes, in a line of memory that
// they often share (both strips of a rank and, so, both of a seam, us, N x C x extents on
// a grid: 13 x 47 x 27 x 42 x 15 on 1 x 2 x 1, periodic, halo of 1 10.9 and 9.3; 2 x 12 x 116 x
// 316 x 84 on 2 x 4 x 1, periodic 15.0 and 13.8; 4 x 85 x 27 x 38 x 14 on 2 x 2 x 1, halos of 3
// 12.6 and 11.8; counting ranks without a seam too, whose XCDs then idle, 14.8).  Phases of
// different dimensions are launches of their own: a later one reads halo cells that
// an earlier one has added to (small ones go in one launch, fold_grid_body).
template <typename T, typename Op, typename Mem>
__host__ __device__ __forceinline__ void fold_body(const FoldArgs& a, uint32_t block, uint32_t thread, Op op,
                                                   const Mem& mem)
{
    constexpr int VEC = 16 / sizeof(T);
    using W = typename Words<T, VEC>::unaligned_t;
    const uint32_t local_block = fastdiv(block, a.turns);
    const FoldSeam& seam = a.seam[block - local_block * a.turns.divisor];
    const uint32_t at = local_block * kBlock + thread;
    const uint32_t row = fastdiv(at, seam.units);
    if (row >= seam.rows)
        return;
    const FoldSide<T> side[2] = {fold_side<T>(seam, row, false), fold_side<T>(seam, row, true)};
    uint32_t x = at - row * seam.units.divisor;
    uint32_t n = 1;
    if (seam.vectors)
    {
        x *= VEC;
        n = seam.run - x < VEC ? seam.run - x : VEC;
    }
    if (n == VEC)
    {
        W s[2], t[2];
#pragma unroll
        for (int i = 0; i < 2; ++i)
        {
            s[i] = mem.template load<VEC, false>(side[i].from + x);
            t[i] = mem.template load<VEC, false>(side[i].to + x);
        }
#pragma unroll
        for (int i = 0; i < 2; ++i)
        {
#pragma unroll
            for (int j = 0; j < VEC; ++j)
                t[i][j] = op(t[i][j], s[i][j]);
            mem.template store<VEC, false>(side[i].to + x, t[i]);
        }
        return;
    }
    for (const uint32_t end = x + n; x < end; ++x)
    {
        const T s0 = mem.load1(side[0].from + x), t0 = mem.load1(side[0].to + x);
        const T s1 = mem.load1(side[1].from + x), t1 = mem.load1(side[1].to + x);
        mem.store1(side[0].to + x, op(t0, s0));
        mem.store1(side[1].to + x, op(t1, s1));
    }
}

template <typename T, typename Op>
__global__ __launch_bounds__(kBlock, 8) void halo_fold_kernel(const FoldArgs a, Op op)
{
    fold_body<T, Op, DeviceMem>(a, blockIdx.x, threadIdx.x, op, DeviceMem());
}

// Dimension 0 for all ranks of a line in the same thread: the two lines of memory at a
// seam of two ranks hold what both give and take, and a workgroup per rank reads them
// twice and writes them back from two XCDs.  RINGS (every rank has both neighbours): a
// thread serves one end of a row in every rank, so that the upper ends and the next
// row's lower ends, which share a line of memory, are neighbouring lanes' work; open lines: both sides of every seam,
// so that no lane is idle.  Reverse exchanges, rank by rank and so (us; N x C x extents
// on a grid, halo 1 unless noted): 1 x 32 x 128^3 on 2^3, periodic 96.7 -> 87.8 (seam by
// seam 98.4), 4 x 32 x 64^3 on 1 x 2 x 4 110 -> 97, 8 x 16 x 64^3 of doubles on 2^3,
// halo 3 173 -> 135, 15 x 8 x 33 x 57 x 45 of doubles on 2^3 43.0 -> 39.5 (end by end
// 43.3), 8 x 64 x 112^2 on 2 x 2, periodic 15.8 -> 11.7.
template <typename T, typename Op, int BY, typename Mem>
__host__ __device__ __forceinline__ void fold_ends_body(const FoldArgs& a, uint32_t block, uint32_t thread, Op op,
                                                        const Mem& mem)
{
    constexpr int kCells = BY == kOpenLines ? 2 : 1;
    const uint32_t local_block = fastdiv(block, a.turns);
    const FoldSeam* const line = a.seam + (block - local_block * a.turns.divisor) * a.line;
    const uint32_t w = line[0].run;
    const uint32_t at = local_block * kBlock + thread;
    const uint32_t row = fastdiv(at, a.cells);
    if (row >= line[0].rows)
        return;
    const uint32_t x = at - row * a.cells.divisor;
    const bool lower_end = x < w; // of a rank's row
    const uint32_t j = lower_end ? x : x - w;
#pragma unroll 1
    for (int base = 0; base < a.line; base += kRanksPerTurn)
    {
        T s[kRanksPerTurn][kCells], t[kRanksPerTurn][kCells];
        T* to[kRanksPerTurn][kCells];
#pragma unroll
        for (int i = 0; i < kRanksPerTurn; ++i)
        {
            to[i][0] = nullptr;
            if (base + i >= a.line)
                continue;
            const FoldSeam& above = line[base + i];
            if constexpr (BY == kRings)
            {
                const FoldSeam& below = line[base + i > 0 ? base + i - 1 : a.line - 1];
                // (Taking the lower end of the next rank, at the same seam, is faster by up to a tenth where the ends
                // of the rows stay in the caches and slower by as much beyond: the upper end of a row and the lower end
                // of the next share a line.)
                const uint32_t lower_start = row * below.upper_pitch + below.run, upper_start = row * above.lower_pitch;
                to[i][0] = reinterpret_cast<T*>(lower_end ? below.upper : above.lower) + ((lower_end ? lower_start : upper_start) + j);
                s[i][0] = mem.load1(reinterpret_cast<const T*>(lower_end ? below.lower : above.upper)
                                    + (row * (lower_end ? below.lower_pitch : above.upper_pitch) + (lower_end ? w : 0) + j));
                t[i][0] = mem.load1(to[i][0]);
                continue;
            }
#pragma unroll
            for (int c = 0; c < kCells; ++c)
            {
                const FoldSide<T> side = fold_side<T>(above, row, c == 1);
                to[i][c] = side.to + j;
                s[i][c] = mem.load1(side.from + j);
                t[i][c] = mem.load1(to[i][c]);
            }
        }
#pragma unroll
        for (int i = 0; i < kRanksPerTurn; ++i)
            if (to[i][0])
            {
#pragma unroll
                for (int c = 0; c < kCells; ++c)
                    mem.store1(to[i][c], op(t[i][c], s[i][c]));
            }
    }
}

template <typename T, typename Op, int BY>
__global__ __launch_bounds__(kBlock, 8) void halo_fold_ends_kernel(const FoldArgs a, Op op)
{
    fold_ends_body<T, Op, BY, DeviceMem>(a, blockIdx.x, threadIdx.x, op, DeviceMem());
}

// A launch of a reverse exchange, played for an audit. Its threads have no order: each cell is loaded once at most and
// stored once at most, and who stores it is the only one to touch it, or the call fails.
template <typename F>
int play_fold(Audit* audit, uint32_t blocks, const F& body)
{
    const TraceMem mem{audit};
    for (uint32_t block = 0; block < blocks; ++block)
        for (uint32_t thread = 0; thread < kBlock; ++thread)
        {
            audit->thread = block * kBlock + thread + 1;
            body(block, thread, mem);
        }
    ++audit->launches;
    audit->workgroups += blocks;
    return audit->followed() ? H2X_SUCCESS : H2X_ERR_INVALID_ARGUMENT;
}

template <typename T, typename Op, int BY>
int issue_fold(const FoldArgs& a, uint32_t blocks, hipStream_t stream)
{
    if (Audit* const audit = current_audit())
    {
        return play_fold(audit, blocks, [&](uint32_t block, uint32_t thread, const TraceMem& mem) {
            if constexpr (BY == kStrips)
                fold_body<T, Op, TraceMem>(a, block, thread, Op(), mem);
            else
                fold_ends_body<T, Op, BY, TraceMem>(a, block, thread, Op(), mem);
        });
    }
    if constexpr (BY == kStrips)
        launch(halo_fold_kernel<T, Op>, dim3(blocks), kBlock, stream, a, Op());
    else
        launch(halo_fold_ends_kernel<T, Op, BY>, dim3(blocks), kBlock, stream, a, Op());
    return launch_status();
}

template <typename T, typename Op>
int issue_fold(const FoldArgs& a, uint32_t blocks, Fold by, hipStream_t stream)
{
    switch (by)
    {
    case kStrips: return issue_fold<T, Op, kStrips>(a, blocks, stream);
    case kOpenLines: return issue_fold<T, Op, kOpenLines>(a, blocks, stream);
    default: return issue_fold<T, Op, kRings>(a, blocks, stream);
    }
}

template <typename T>
int issue_fold(int op, const FoldArgs& a, uint32_t blocks, Fold by, hipStream_t stream)
{
    switch (op)
    {
    case H2X_HALO_ID: return issue_fold<T, copy::OpId>(a, blocks, by, stream);
    case H2X_HALO_SUM: return issue_fold<T, copy::OpSum>(a, blocks, by, stream);
    case H2X_HALO_MAX: return issue_fold<T, copy::OpMax>(a, blocks, by, stream);
    default: return issue_fold<T, copy::OpMin>(a, blocks, by, stream);
    }
}

// The reverse exchange of several dimensions in one launch. Phase after phase, every cell of a boundary strip takes in
// the halo cell of its neighbour along the phase's dimension, which has taken in others before. Cells whose values meet
// are a group: per dimension in which they lie at a seam, the boundary cell of one rank and the halo cell of its
// neighbour that stands for it. A halo cell is of one group alone (a rank has at least two halo widths of interior
// along such a dimension), so groups have no order: a thread loads the two, four or eight cells of one, plays the
// phases on them, with their roundings, and stores those that lie in a boundary strip.
//
// The groups of a rank are those whose cells in all boundary strips are its own: regions per {elsewhere, lower, upper
// boundary} of the outer two dimensions, as vectors along what of the rows is no end ("elsewhere" of dimension 0), and the ends.
template <typename F>
__host__ __device__ __forceinline__ void fold_outer(uint32_t dims, F combine)
{
#pragma unroll
    for (int i = 0; i < 4; i += 2)
        if ((dims & 1) && (i & ~dims) == 0)
            combine(i, i + 1);
#pragma unroll
    for (int i = 0; i < 2; ++i)
        if ((dims & 2) && (i & ~dims) == 0)
            combine(i, i + 2);
}

// Start of what a rank's seams along dimension d leave of its real extent.
__host__ __device__ __forceinline__ uint32_t rest_start(const Rank& k, int d, int w)
{
    return k.clear >> (2 * d) & 1 ? 0 : 2 * w;
}

template <typename T, typename Op, typename Mem>
__host__ __device__ __forceinline__ void fold_grid_body(const Args& a, uint32_t block, uint32_t thread, Op op, const Mem& mem)
{
    constexpr int VEC = 16 / sizeof(T);
    using W = typename Words<T, VEC>::unaligned_t;
    uint32_t first = 0, code = a.code[0];
#pragma unroll
    for (int i = 1; i < kMaxRegions; ++i)
        if (block >= a.first[i])
        {
            first = a.first[i];
            code = a.code[i];
        }
    const bool ends = code & 1;
    const FastDiv& turns = ends ? a.lines : a.ranks;
    const uint32_t local_block = fastdiv(block - first, turns);
    const uint32_t r = (block - first - local_block * turns.divisor) * (ends ? a.line : 1);
    const Rank& me = a.rank[r]; // ends: the first one of its line
    const uint32_t digit_y = code >> 2 & 3, digit_z = code >> 4;
    // bit 0: a seam along dimension 1, bit 1: along dimension 2; cell i of a group lies in the halo along those of its bits
    const uint32_t dims = (digit_y != 0) | (digit_z != 0) << 1;
    const uint32_t both = me.source[digit_z] >> (8 * digit_y);
    const uint32_t empty = (ends ? 0 : 1) | (digit_y ? 0 : 2) | (digit_z ? 0 : 4);
    if ((both & kSteppedAny) != dims * 2 * kStepped || (me.clear >> kRestEmpty & empty))
        return;
    const uint32_t ranks[4] = {r, me.source[0] >> (8 * digit_y) & kSourceRank, me.source[digit_z] & kSourceRank, both & kSourceRank};
    const FastDiv div_y = digit_y == 0 ? me.extent[0] : a.halo[1], div_z = digit_z == 0 ? me.extent[1] : a.halo[2];
    const FastDiv div_x = ends ? a.both_ends : me.units;
    const uint32_t at = local_block * kBlock + thread;
    if (at >= div_y.divisor * div_z.divisor * a.outer * div_x.divisor)
        return;
    const uint32_t row_at = fastdiv(at, div_x);
    uint32_t x = at - row_at * div_x.divisor;
    const uint32_t yz = fastdiv(row_at, div_y), o = fastdiv(yz, div_z);
    const int wy = a.width[1], wz = a.width[2];
    const uint32_t y = row_at - yz * div_y.divisor
                       + (digit_y == 0 ? rest_start(me, 1, wy) : static_cast<uint32_t>(digit_y == 1 ? wy : me.local[1]));
    const uint32_t z = yz - o * div_z.divisor
                       + (digit_z == 0 ? rest_start(me, 2, wz) : static_cast<uint32_t>(digit_z == 1 ? wz : me.local[2]));
    // the halo cell that stands for a lower boundary cell lies behind the lower neighbour's interior, ...
    const uint32_t y_halo = y + (digit_y == 1 ? a.rank[ranks[1]].local[1] : -me.local[1]);
    const uint32_t z_halo = z + (digit_z == 1 ? a.rank[ranks[2]].local[2] : -me.local[2]);
    uint32_t row[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
    {
        const Rank& q = a.rank[ranks[i]];
        row[i] = (o * (q.local[2] + 2 * wz) + (i & 2 ? z_halo : z)) * (q.local[1] + 2 * wy) + (i & 1 ? y_halo : y);
    }
    const uint32_t w = a.width[0], pitch = me.local[0] + 2 * w; // (neighbours along dimensions 1 and 2 have rows as long)
    const auto mine = [&](int i) { return (i & ~dims) == 0; };
    // how many of the strips of a phase cell i lies in, as boundary and in all: what an audit counts
    const auto boundary = [&](int i, int end) { return (dims & ~i & 1) + (dims >> 1 & ~i >> 1 & 1) + end; };
    const int seams = boundary(0, ends);
    if (!ends)
    {
        const uint32_t start = rest_start(me, 0, w);
        uint32_t n = 1;
        if (me.vectors)
        {
            const uint32_t count = (me.clear >> 1 & 1 ? pitch : me.local[0]) - start;
            x *= VEC;
            n = count - x < VEC ? count - x : VEC;
        }
        T* at_cell[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            at_cell[i] = reinterpret_cast<T*>(a.rank[ranks[i]].tensor) + (row[i] * pitch + start + x);
        if (n == VEC)
        {
            W v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (mine(i))
                    v[i] = of_strips(mem, seams).template load<VEC, false>(at_cell[i]);
            fold_outer(dims, [&](int to, int from) {
#pragma unroll
                for (int j = 0; j < VEC; ++j)
                    v[to][j] = op(v[to][j], v[from][j]);
            });
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (mine(i) && boundary(i, 0))
                    of_strips(mem, boundary(i, 0)).template store<VEC, false>(at_cell[i], v[i]);
            return;
        }
        for (uint32_t j = 0; j < n; ++j)
        {
            T v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (mine(i))
                    v[i] = of_strips(mem, seams).load1(at_cell[i] + j);
            fold_outer(dims, [&](int to, int from) { v[to] = op(v[to], v[from]); });
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (mine(i) && boundary(i, 0))
                    of_strips(mem, boundary(i, 0)).store1(at_cell[i] + j, v[i]);
        }
        return;
    }
    // the ends of a row in every rank of the line, side by side with the next row's
    const bool upper = x >= w;
    const uint32_t j = upper ? x - w : x;
    const auto end_of = [&](int k, int i, T** inner_at, T** halo_at) {
        const Rank& q = a.rank[ranks[i] + k];
        const uint64_t lo_from = in_scalar(q.end[0].from), hi_from = in_scalar(q.end[1].from);
        const uint32_t lo_pitch = in_scalar(q.end[0].pitch), hi_pitch = in_scalar(q.end[1].pitch);
        *inner_at = reinterpret_cast<T*>(q.tensor) + (row[i] * (q.local[0] + 2 * w) + (upper ? q.local[0] : w) + j);
        *halo_at = const_cast<T*>(global_place<T>(upper ? hi_from : lo_from)) + (row[i] * (upper ? hi_pitch : lo_pitch) + j);
    };
#pragma unroll 1
    for (int k = 0; k < a.line; ++k)
    {
        if (a.rank[r + k].clear >> (upper ? 1 : 0) & 1)
            continue;
        T inner[4], halo[4];
        T *inner_at[4], *halo_at[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (mine(i))
            {
                end_of(k, i, &inner_at[i], &halo_at[i]);
                inner[i] = of_strips(mem, seams).load1(inner_at[i]);
                halo[i] = of_strips(mem, seams).load1(halo_at[i]);
            }
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (mine(i))
                inner[i] = op(inner[i], halo[i]);
        fold_outer(dims, [&](int to, int from) {
            inner[to] = op(inner[to], inner[from]);
            halo[to] = op(halo[to], halo[from]);
        });
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (mine(i))
            {
                of_strips(mem, boundary(i, 1)).store1(inner_at[i], inner[i]);
                if (boundary(i, 0))
                    of_strips(mem, boundary(i, 0)).store1(halo_at[i], halo[i]);
            }
    }
}

template <typename T, typename Op>
__global__ __launch_bounds__(kBlock, 8) void halo_fold_grid_kernel(const Args a, Op op)
{
    fold_grid_body<T, Op, DeviceMem>(a, blockIdx.x, threadIdx.x, op, DeviceMem());
}

template <typename T, typename Op>
int issue_fold_grid(const Args& a, uint32_t blocks, hipStream_t stream)
{
    if (Audit* const audit = current_audit())
    {
        return play_fold(audit, blocks, [&](uint32_t block, uint32_t thread, const TraceMem& mem) {
            fold_grid_body<T, Op, TraceMem>(a, block, thread, Op(), mem);
        });
    }
    launch(halo_fold_grid_kernel<T, Op>, dim3(blocks), kBlock, stream, a, Op());
    return launch_status();
}

template <typename T>
int issue_fold_grid(int op, const Args& a, uint32_t blocks, hipStream_t stream)
{
    switch (op)
    {
    case H2X_HALO_ID: return issue_fold_grid<T, copy::OpId>(a, blocks, stream);
    case H2X_HALO_SUM: return issue_fold_grid<T, copy::OpSum>(a, blocks, stream);
    case H2X_HALO_MAX: return issue_fold_grid<T, copy::OpMax>(a, blocks, stream);
    default: return issue_fold_grid<T, copy::OpMin>(a, blocks, stream);
    }
}

template <typename T, bool CLEAR>
__global__ __launch_bounds__(kBlock, 8) void halo_grid_kernel(const Args a)
{
    body<T, CLEAR, DeviceMem>(a, blockIdx.x, threadIdx.x, DeviceMem());
}

template <typename T, bool CLEAR>
int issue(const Args& a, uint32_t blocks, hipStream_t stream)
{
    if (Audit* const audit = current_audit())
    {
        const TraceMem mem{audit};
        for (uint32_t block = 0; block < blocks; ++block)
            for (uint32_t thread = 0; thread < kBlock; ++thread)
                body<T, CLEAR, TraceMem>(a, block, thread, mem);
        ++audit->launches;
        audit->workgroups += blocks;
        return H2X_SUCCESS;
    }
    launch(halo_grid_kernel<T, CLEAR>, dim3(blocks), kBlock, stream, a);
    return launch_status();
}

// Everything the kernel relies on: extents that fit, neighbours whose tensors
// lie alike in the other dimensions and hold the strips that are read.
// `cells`: halo widths of interior that a rank with a neighbour has to have.
int make_args(const h2x_halo_grid& h, int cells, int only_unfilled, int elem_size, Args* a)
{
    const int nd = h.num_dims, ns = nd - 2;
    if (nd < 3 || nd > kMaxSpatial + 2 || h.num_ranks < 1 || !h.ranks)
        return H2X_ERR_INVALID_ARGUMENT;
    if (h.num_ranks > kMaxRanks)
        return H2X_ERR_UNSUPPORTED;
    int64_t outer = 1;
    for (int d = ns; d < nd; ++d)
    {
        if (h.overlap[d] != 0)
            return H2X_ERR_UNSUPPORTED;
        outer *= h.ranks[0].local_shape[d];
    }
    a->ranks = make_fastdiv(static_cast<uint32_t>(h.num_ranks));
    for (int d = 0; d < kMaxSpatial; ++d)
    {
        const int64_t w = d < ns ? h.overlap[d] : 0;
        if (w < 0 || w > (1 << 20))
            return H2X_ERR_INVALID_ARGUMENT;
        a->width[d] = static_cast<int32_t>(w);
        a->halo[d] = make_fastdiv(static_cast<uint32_t>(std::max<int64_t>(w, 1)));
    }
    a->both_ends = make_fastdiv(static_cast<uint32_t>(std::max(2 * a->width[0], 1)));
    const int64_t vec = 16 / elem_size;
    for (int r = 0; r < h.num_ranks; ++r)
    {
        const h2x_halo_grid_rank& from = h.ranks[r];
        Rank& k = a->rank[r];
        if (!from.tensor)
            return H2X_ERR_INVALID_ARGUMENT;
        k.tensor = static_cast<char*>(from.tensor);
        int64_t real = 1;
        for (int d = 0; d < nd; ++d)
        {
            if (from.local_shape[d] < 1 || from.local_shape[d] >= (1ll << 31))
                return H2X_ERR_INVALID_ARGUMENT;
            if (d >= ns && from.local_shape[d] != h.ranks[0].local_shape[d])
                return H2X_ERR_UNSUPPORTED; // channels or samples spread unevenly: `outer` is one number
            real *= from.local_shape[d] + 2 * (d < ns ? a->width[d] : 0);
            if (real >= (1ll << 31))
                return H2X_ERR_TOO_LARGE;
        }
        k.clear = 0;
        for (int d = 0; d < kMaxSpatial; ++d)
        {
            k.local[d] = d < ns ? static_cast<int32_t>(from.local_shape[d]) : 1;
            for (int side = 0; side < 2; ++side)
            {
                const int p = d < ns ? from.peer[d][side] : -1;
                if (p >= h.num_ranks || p < -1)
                    return H2X_ERR_INVALID_ARGUMENT;
                k.peer[d][side] = p;
                if (p >= 0)
                {
                    const h2x_halo_grid_rank& q = h.ranks[p];
                    if (q.peer[d][1 - side] != r)
                        return H2X_ERR_INVALID_ARGUMENT;
                    for (int i = 0; i < nd; ++i)
                        if (i != d && q.local_shape[i] != from.local_shape[i])
                            return H2X_ERR_INVALID_ARGUMENT;
                    if (cells > 0 && (q.local_shape[d] < cells * static_cast<int64_t>(a->width[d]) || a->width[d] == 0))
                        return H2X_ERR_INVALID_ARGUMENT;
                }
                if (a->width[d] > 0 && (p < 0 || !only_unfilled))
                    k.clear |= 1u << (2 * d + side);
            }
        }
        k.vectors = k.local[0] >= vec;
        k.units = make_fastdiv(static_cast<uint32_t>(k.vectors ? (k.local[0] + vec - 1) / vec : k.local[0]));
        k.extent[0] = make_fastdiv(static_cast<uint32_t>(k.local[1]));
        k.extent[1] = make_fastdiv(static_cast<uint32_t>(k.local[2]));
    }
    a->outer = static_cast<uint32_t>(outer);
    return H2X_SUCCESS;
}

// Stepping along two dimensions leads to the same rank in either order, and neighbours along one
// dimension have, or lack, neighbours along the others alike.
bool is_grid(const Args& a, int num_ranks)
{
    for (int r = 0; r < num_ranks; ++r)
        for (int d = 0; d < kMaxSpatial; ++d)
            for (int side = 0; side < 2; ++side)
            {
                const int p = a.rank[r].peer[d][side];
                if (p < 0)
                    continue;
                for (int e = 0; e < kMaxSpatial; ++e)
                    for (int s = 0; e != d && s < 2; ++s)
                    {
                        const int q = a.rank[r].peer[e][s], pq = a.rank[p].peer[e][s];
                        if ((q < 0) != (pq < 0) || (q >= 0 && a.rank[q].peer[d][side] != pq))
                            return false;
                    }
            }
    return true;
}

// Renumbers the ranks so that those in a line along dimension 0 follow one another, lower to
// upper; all lines have to be of one length, and a step along another dimension to lead to the
// same place in another line.
bool order_into_lines(Args* a, int num_ranks)
{
    int order[kMaxRanks], place[kMaxRanks], n = 0;
    bool taken[kMaxRanks] = {};
    a->line = 0;
    for (int closed = 0; closed < 2; ++closed) // open lines start where nothing is below, then rings
        for (int r = 0; r < num_ranks; ++r)
        {
            if (taken[r] || (!closed && a->rank[r].peer[0][0] >= 0))
                continue;
            int length = 0;
            for (int q = r; q >= 0 && !taken[q]; q = a->rank[q].peer[0][1], ++length)
            {
                taken[q] = true;
                place[q] = n;
                order[n++] = q;
            }
            if (a->line != 0 && a->line != length)
                return false;
            a->line = length;
        }
    Rank ranks[kMaxRanks];
    for (int i = 0; i < num_ranks; ++i)
    {
        ranks[i] = a->rank[order[i]];
        for (auto& sides : ranks[i].peer)
            for (int32_t& p : sides)
                p = p < 0 ? p : place[p];
        for (int d = 1; d < kMaxSpatial; ++d)
            for (const int32_t p : ranks[i].peer[d])
                if (p >= 0 && p % a->line != i % a->line)
                    return false;
    }
    std::copy(ranks, ranks + num_ranks, a->rank);
    a->lines = make_fastdiv(static_cast<uint32_t>(num_ranks / a->line));
    return true;
}

// Follows the neighbours of ranks that lie in lines: where a region's cells and a row's ends come from.
void resolve_sources(Args* a, int num_ranks, int elem_size)
{
    for (int r = 0; r < num_ranks; ++r)
    {
        Rank& k = a->rank[r];
        for (uint32_t dz = 0; dz < 3; ++dz)
        {
            k.source[dz] = 0;
            for (uint32_t dy = 0; dy < 3; ++dy)
            {
                uint32_t src = static_cast<uint32_t>(r), stepped = 0;
                for (int d = 1; d < kMaxSpatial; ++d)
                {
                    const uint32_t digit = d == 1 ? dy : dz;
                    const int p = digit ? a->rank[src].peer[d][digit - 1] : -1;
                    if (p >= 0)
                    {
                        src = static_cast<uint32_t>(p);
                        stepped |= kStepped << d;
                    }
                }
                k.source[dz] |= (src | stepped) << (8 * dy);
            }
        }
        for (int side = 0; side < 2; ++side)
        {
            const int p = k.peer[0][side];
            const Rank& q = p >= 0 ? a->rank[p] : k;
            // the neighbour's other end, or this end: of {halo, interior, halo}, cells 0, w, local or w + local
            const int64_t cell = side == 0 ? (p >= 0 ? q.local[0] : 0) : a->width[0] + (p >= 0 ? 0 : q.local[0]);
            k.end[side].from = q.tensor + cell * elem_size;
            k.end[side].pitch = static_cast<uint32_t>(q.local[0] + 2 * a->width[0]);
            k.end[side].filled = p >= 0;
        }
    }
}

template <bool CLEAR>
int run(h2x_dtype dtype, const h2x_halo_grid* h, int only_unfilled, h2x_stream_t stream)
{
    const int es = dtype == H2X_F32 ? 4 : dtype == H2X_F64 ? 8 : 0;
    if (es == 0)
        return H2X_ERR_UNSUPPORTED;
    if (!h)
        return H2X_ERR_INVALID_ARGUMENT;
    Args a;
    const int err = make_args(*h, CLEAR ? 0 : 1, only_unfilled, es, &a);
    if (err != 0)
        return err;
    if (!is_grid(a, h->num_ranks))
        return H2X_ERR_INVALID_ARGUMENT;
    if (!order_into_lines(&a, h->num_ranks))
        return H2X_ERR_UNSUPPORTED;
    if constexpr (!CLEAR)
        resolve_sources(&a, h->num_ranks, es);
    // Regions with the same work for every rank: blocks for the largest rank.
    int num_regions = 0;
    uint64_t blocks = 0;
    std::fill(a.first, a.first + kMaxRegions, ~0u);
    for (int ends = 1; ends >= 0; --ends)
        for (int dz = 0; dz < 3; ++dz)
            for (int dy = 0; dy < 3; ++dy)
            {
                if ((ends && a.width[0] == 0) || (dy && a.width[1] == 0) || (dz && a.width[2] == 0)
                    || (!ends && !dy && !dz))
                    continue;
                uint64_t most = 0;
                for (int r = 0; r < h->num_ranks; ++r)
                {
                    const Rank& k = a.rank[r];
                    const int digit[2] = {dy, dz};
                    bool any = false; // something to do for this rank
                    for (int d = 1; d < 3; ++d)
                        if (digit[d - 1])
                            any = any || (CLEAR ? k.clear >> (2 * d + digit[d - 1] - 1) & 1
                                                : k.peer[d][digit[d - 1] - 1] >= 0);
                    if (ends)
                        any = any || (CLEAR ? k.clear & 3 : k.peer[0][0] >= 0 || k.peer[0][1] >= 0);
                    if (!any)
                        continue;
                    const uint64_t rows = static_cast<uint64_t>(dy ? a.width[1] : k.local[1])
                                          * (dz ? a.width[2] : k.local[2]) * a.outer;
                    most = std::max<uint64_t>(
                        most, (rows * (ends ? 2 * a.width[0] : k.units.divisor) + kBlock - 1) / kBlock);
                }
                if (most == 0)
                    continue;
                const int g = num_regions++;
                a.first[g] = static_cast<uint32_t>(blocks);
                a.code[g] = static_cast<uint32_t>(ends + 4 * dy + 16 * dz);
                blocks += most * (ends ? a.lines.divisor : a.ranks.divisor);
                if (most > kMaxRankBlocks || blocks > kMaxBlocks)
                    return H2X_ERR_TOO_LARGE;
            }
    if (blocks == 0)
        return H2X_SUCCESS;
    return es == 4 ? issue<uint32_t, CLEAR>(a, static_cast<uint32_t>(blocks), as_stream(stream))
                   : issue<uint64_t, CLEAR>(a, static_cast<uint32_t>(blocks), as_stream(stream));
}

// Whether a reverse exchange goes in one launch.
bool folds_in_one_launch(const Args& a, int num_ranks, int es)
{
    int dims = 0;
    uint64_t cells = 0;
    for (int d = 0; d < kMaxSpatial; ++d)
    {
        uint64_t strips = 0;
        for (int r = 0; r < num_ranks; ++r)
        {
            const Rank& k = a.rank[r];
            uint64_t strip = static_cast<uint64_t>(a.outer) * a.width[d];
            for (int e = 0; e < kMaxSpatial; ++e)
                strip *= e == d ? 1 : k.local[e] + 2 * a.width[e];
            strips += strip * ((k.peer[d][0] >= 0) + (k.peer[d][1] >= 0));
        }
        dims += strips != 0;
        cells += strips;
    }
    return dims > 1 && cells * es <= (dims == 2 ? kFoldBytes2 : kFoldBytes3) && is_grid(a, num_ranks);
}

int run_fold_grid(Args& a, int num_ranks, int es, int op, hipStream_t stream)
{
    // (4 x 2 grids of 2D samples, 114 x 259: rank by rank 5.7 us, line by line 7.2; 160^3 on 2^3: 8.6 and 6.4)
    const int64_t rows = static_cast<int64_t>(a.rank[0].local[1]) * a.rank[0].local[2] * a.outer;
    if (rows < kLineRows || !order_into_lines(&a, num_ranks))
    {
        a.line = 1;
        a.lines = a.ranks;
    }
    resolve_sources(&a, num_ranks, es);
    const uint32_t vec = 16 / es;
    uint32_t rest[kMaxRanks][kMaxSpatial];
    for (int r = 0; r < num_ranks; ++r)
    {
        Rank& k = a.rank[r];
        for (int d = 0; d < kMaxSpatial; ++d)
        {
            const int seams = (k.peer[d][0] >= 0) + (k.peer[d][1] >= 0);
            rest[r][d] = static_cast<uint32_t>(k.local[d] + 2 * a.width[d] - 2 * seams * a.width[d]);
            k.clear |= static_cast<uint32_t>(rest[r][d] == 0) << (kRestEmpty + d);
        }
        k.vectors = rest[r][0] >= vec;
        k.units = make_fastdiv(std::max(k.vectors ? (rest[r][0] + vec - 1) / vec : rest[r][0], 1u));
        for (int d = 1; d < kMaxSpatial; ++d)
            k.extent[d - 1] = make_fastdiv(std::max(rest[r][d], 1u));
        for (int side = 0; side < 2; ++side)
            if (k.peer[0][side] >= 0)
            {
                const Rank& q = a.rank[k.peer[0][side]]; // its upper halo follows its interior, its lower one comes first
                k.end[side].from = q.tensor + (side == 0 ? static_cast<int64_t>(a.width[0] + q.local[0]) * es : 0);
            }
    }
    int num_regions = 0;
    uint64_t blocks = 0;
    std::fill(a.first, a.first + kMaxRegions, ~0u);
    for (int ends = 1; ends >= 0; --ends)
        for (int dz = 0; dz < 3; ++dz)
            for (int dy = 0; dy < 3; ++dy)
            {
                uint64_t most = 0;
                for (int r = 0; r < num_ranks; ++r)
                {
                    const Rank& k = a.rank[r];
                    if ((!ends && !dy && !dz) || (dy && k.peer[1][dy - 1] < 0) || (dz && k.peer[2][dz - 1] < 0)
                        || (ends && k.peer[0][0] < 0 && k.peer[0][1] < 0))
                        continue;
                    const uint64_t threads = static_cast<uint64_t>(dy ? a.width[1] : rest[r][1]) * (dz ? a.width[2] : rest[r][2])
                                             * a.outer * (ends ? 2 * a.width[0] : rest[r][0] ? k.units.divisor : 0);
                    most = std::max(most, (threads + kBlock - 1) / kBlock);
                }
                if (most == 0)
                    continue;
                const int g = num_regions++;
                a.first[g] = static_cast<uint32_t>(blocks);
                a.code[g] = static_cast<uint32_t>(ends + 4 * dy + 16 * dz);
                blocks += most * (ends ? a.lines.divisor : a.ranks.divisor);
            }
    return es == 4 ? issue_fold_grid<float>(op, a, static_cast<uint32_t>(blocks), stream)
                   : issue_fold_grid<double>(op, a, static_cast<uint32_t>(blocks), stream);
}

int run_fold(h2x_dtype dtype, const h2x_halo_grid* h, int op, h2x_stream_t stream)
{
    const int es = dtype == H2X_F32 ? 4 : dtype == H2X_F64 ? 8 : 0;
    if (es == 0)
        return H2X_ERR_UNSUPPORTED;
    if (!h || op < H2X_HALO_ID || op > H2X_HALO_MIN)
        return H2X_ERR_INVALID_ARGUMENT;
    Args a;
    int err = make_args(*h, 2, 1, es, &a);
    if (err != 0)
        return err;
    if (folds_in_one_launch(a, h->num_ranks, es))
        return run_fold_grid(a, h->num_ranks, es, op, as_stream(stream));
    const int64_t rows = static_cast<int64_t>(a.rank[0].local[1] + 2 * a.width[1])
                         * (a.rank[0].local[2] + 2 * a.width[2]) * a.outer;
    bool lines = rows >= kLineRows && a.width[0] > 0 && order_into_lines(&a, h->num_ranks);
    const bool rings = lines && a.rank[0].peer[0][0] >= 0;
    const int64_t vec = 16 / es;
    FoldArgs f[kMaxSpatial];
    uint64_t blocks[kMaxSpatial] = {};
    for (int dim = 0; dim < kMaxSpatial; ++dim)
    {
        uint32_t seams = 0;
        uint64_t most = 0; // workgroups of the largest rank
        uint64_t longest = 0; // and of the largest line
        for (int r = 0; r < h->num_ranks; ++r)
        {
            const Rank& k = a.rank[r];
            int64_t below = 1, above = a.outer;
            for (int d = 0; d < kMaxSpatial; ++d)
                (d < dim ? below : above) *= d == dim ? 1 : k.local[d] + 2 * a.width[d];
            const int64_t run = a.width[dim] * below;
            const int64_t n = run >= vec ? (run + vec - 1) / vec : std::max<int64_t>(run, 1);
            most = std::max<uint64_t>(most, (n * above + kBlock - 1) / kBlock);
            longest = std::max<uint64_t>(longest, ((rings ? 2 : 1) * run * above + kBlock - 1) / kBlock);
            if (k.peer[dim][1] < 0)
                continue;
            const Rank& u = a.rank[k.peer[dim][1]];
            FoldSeam& seam = f[dim].seam[seams++];
            seam.lower = k.tensor + k.local[dim] * below * es;
            seam.upper = u.tensor;
            seam.lower_pitch = static_cast<uint32_t>((k.local[dim] + 2 * a.width[dim]) * below);
            seam.upper_pitch = static_cast<uint32_t>((u.local[dim] + 2 * a.width[dim]) * below);
            seam.run = static_cast<uint32_t>(run);
            seam.rows = static_cast<uint32_t>(above);
            seam.units = make_fastdiv(static_cast<uint32_t>(n));
            seam.vectors = run >= vec;
        }
        if (seams == 0)
            continue;
        if (most > kMaxRankBlocks || most * h->num_ranks > kMaxBlocks)
            return H2X_ERR_TOO_LARGE;
        f[dim].turns = make_fastdiv(seams);
        blocks[dim] = most * seams;
        // (what can be launched is a matter of the ranks alone)
        // (open lines and rings side by side have no one number of seams)
        if (dim == 0)
            lines = lines && longest <= kMaxRankBlocks && longest * a.lines.divisor <= kMaxBlocks
                    && seams == (rings ? a.line : a.line - 1) * a.lines.divisor;
        if (dim == 0 && lines)
        {
            f[0].turns = a.lines;
            f[0].line = static_cast<int32_t>(seams / a.lines.divisor);
            f[0].cells = rings ? a.both_ends : a.halo[0];
            blocks[0] = longest * a.lines.divisor;
        }
    }
    for (int dim = 0; dim < kMaxSpatial && err == 0; ++dim)
    {
        if (blocks[dim] == 0)
            continue;
        const Fold by = dim > 0 || !lines ? kStrips : rings ? kRings : kOpenLines;
        const uint32_t n = static_cast<uint32_t>(blocks[dim]);
        err = es == 4 ? issue_fold<float>(op, f[dim], n, by, as_stream(stream))
                      : issue_fold<double>(op, f[dim], n, by, as_stream(stream));
    }
    return err;
}

} // namespace
} // namespace grid
} // namespace h2x

extern "C" int h2x_halo_grid_exchange(h2x_dtype dtype, const h2x_halo_grid* grid, h2x_stream_t stream)
{
    return h2x::grid::run<false>(dtype, grid, 0, stream);
}

extern "C" int h2x_halo_grid_clear(h2x_dtype dtype, const h2x_halo_grid* grid, int only_unfilled,
                                   h2x_stream_t stream)
{
    return h2x::grid::run<true>(dtype, grid, only_unfilled, stream);
}

extern "C" int h2x_halo_grid_fold(h2x_dtype dtype, const h2x_halo_grid* grid, int op, h2x_stream_t stream)
{
    return h2x::grid::run_fold(dtype, grid, op, stream);
}
