// CSR x CSR -> CSR product on the device.
//
// The reference declares this product (Includes/Sapphire/compute/sparse/cuda/SparseGemm.cuh:16-100,
// Sparse::Cuda::Gemm over arrays of SparseMatrix, one block per output row, a hash table per
// row, a bitonic sort and a load-distribution pre-pass; helper bodies in
// Sources/Sapphire/compute/cudaUtil/SparseUtil.cu) and defines no host entry for it.  The
// contract kept here is the one its dense leaf gives on the densified operands
// (Sources/Sapphire/compute/dense/naive/NaiveGemm.cpp:12-38): element (i, j) is the sum over
// A's row i, entries in storage order, of a * B[k][j], product and sum rounded separately,
// starting from +0; results that are exactly 0 are not stored (SparseUtil.cu:55-60 deletes
// them as well); a row's entries come out in ascending column order.
//
// One wavefront owns one output row.  Instead of a hash table and a sort it usually keeps a dense
// strip of the row in LDS (up to 4096 columns, 16 KiB; wider matrices are done strip by
// strip): A's entries are taken in order, the entries of the matching row of B are spread
// over the 64 lanes and added into the strip, and because the columns of one row of B are
// distinct no two lanes touch the same element in one step, which makes the sum order fixed
// and the result bit-identical to the CPU loop.  A bit per column records which elements were
// touched.  The strip is then swept in column order, which yields the sorted row without
// sorting: every lane owns a run of consecutive columns (its words of the bit map), counts the
// touched elements of its run that are not zero, a prefix sum over the lanes turns the counts
// into output positions, and the lane writes its entries.  Touched elements are set back to
// zero as they are read, so the strip is cleared once per workgroup and the cost of a strip
// follows the entries it produces, not its width.  The same kernel runs twice: once to count
// the entries of every row (the caller then allocates), once to write them.
//
// Matrices wider than one strip: rows with few products (A's row at most 64 entries, at most
// 512 products) go to SpgemmLightKernel, which sorts a row's products in registers and whose
// cost does not depend on the width; the strip kernel then takes only the remaining rows.  The
// pass that does rows again which overflowed their staging slot takes both kinds.
//
// Requirements on the operands: column indices of B below N and distinct within a row;
// column indices of A below the row count of B.
#include "sph_internal.h"
#include "sph_place_rows.h"
#include "sph_spgemm_plan.h"

#include <algorithm>

#pragma clang fp contract(off)

namespace
{
constexpr uint32_t kStripMax = 4096;  // columns per LDS strip
constexpr uint32_t kAhead = 8;        // rows of B whose first 64 entries are in flight together
constexpr uint32_t kRowsPerTurnMax = 8;  // consecutive output rows a wavefront takes at a time
constexpr uint32_t kWordsPerLaneMax = kStripMax / 32 / 64;  // bit-map words a lane owns
constexpr uint32_t kLightProducts = 512;  // a row with at most this many products is "light"
constexpr uint32_t kPlaceBits = 9;        // a product's place in its row, below its column
constexpr uint32_t kLightWaves = 4;       // wavefronts per workgroup of SpgemmLightKernel
constexpr uint32_t kStripGroups = 64;  // workgroups of a strip pass per compute unit, at most
constexpr uint32_t kMarkedGroups = 18;
constexpr uint32_t kRedoGroups = 2;
constexpr uint32_t kEmpty = 0xffffffffu;
constexpr uint32_t kHeavyMark = 0xffffffffu;  // in place of a count: SpgemmRowKernel's row
static_assert(kLightProducts <= 1u << kPlaceBits, "a key holds column and place");
static_assert(kWordsPerLaneMax <= 4, "the sweep takes a lane's words as two pairs");

struct SpgemmArgs
{
    const float* VA;
    const uint32_t* COLA;
    const uint32_t* ROWA;
    const float* VB;
    const uint32_t* COLB;
    const uint32_t* ROWB;
    uint32_t M, K, N;
    uint32_t strip;  // columns per strip (multiple of 64)
    uint32_t rowsPerTurn;  // 1 .. kRowsPerTurnMax
    uint32_t lightProducts;  // rows with at most this many products are SpgemmLightKernel's (0: none)
    uint32_t heavyOnly;    // strip kernel: leave those rows alone
    // count pass: counts (M + 1 entries, counts[M] = 0).  fill pass: ROWC, VC, COLC.
    // stage pass: counts as in the count pass, and row r's entries into VC / COLC at
    // r * slot .. r * slot + slot - 1 (what does not fit is counted and dropped).
    uint32_t* counts;
    const uint32_t* ROWC;
    float* VC;
    uint32_t* COLC;
    uint32_t slot;      // stage pass: entries per staging slot
    uint32_t skipUpTo;  // fill pass: rows with at most this many entries are left alone
    uint32_t capacity;  // fill pass: nothing is stored at or past this index
    // stage pass: cleared; the move kernel sets it when a row did not fit its slot; the pass over
    // such rows returns at once while it is zero
    uint32_t* overflow;
};

// what a pass of the two product kernels does with a row's entries
constexpr int kCount = 0, kFill = 1, kStage = 2;

__device__ __forceinline__ uint32_t Uniform(uint32_t v, uint32_t lane)
{
    return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), lane));
}

__device__ __forceinline__ float Uniform(float v, uint32_t lane)
{
    return __builtin_bit_cast(
        float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), static_cast<int>(lane)));
}

__device__ __forceinline__ void Touch(uint32_t* bits, uint32_t column)
{
    __hip_atomic_fetch_or(&bits[column >> 5], 1u << (column & 31), __ATOMIC_RELAXED,
                          __HIP_MEMORY_SCOPE_WORKGROUP);
}

__device__ __forceinline__ uint32_t WaveSum(uint32_t v)
{
#pragma unroll
    for (uint32_t d = 1; d < 64; d *= 2)
        v += __shfl_xor(v, d, 64);
    return v;
}

// A row is light when A's row has at most 64 entries and the rows of B they select hold at most
// kLightProducts entries together.  Both kernels decide from these two numbers; a lane counts at
// most kLightProducts + 1 entries of its row of B, so that the sum cannot wrap.
__device__ __forceinline__ uint32_t LightCount(uint32_t begin, uint32_t end)
{
    return end > begin ? min(end - begin, kLightProducts + 1) : 0u;
}

__device__ __forceinline__ bool LightRow(const SpgemmArgs& args, uint32_t entriesOfA,
                                         uint32_t products)
{
    return entriesOfA <= 64 && products <= args.lightProducts;
}

// Lane operations of the vector unit itself (no LDS crossbar, no wait): DPP controls.
constexpr int kDppXor1 = 0xB1, kDppXor2 = 0x4E, kDppXor3 = 0x1B;  // quad permutations
constexpr int kDppXor7 = 0x141, kDppXor15 = 0x140;  // half-row and row mirrored
constexpr int kDppXor8 = 0x128;                     // row rotated by 8
constexpr int kDppShr1 = 0x111, kDppShr2 = 0x112, kDppShr4 = 0x114, kDppShr8 = 0x118;
constexpr int kDppBcast15 = 0x142, kDppBcast31 = 0x143;  // last lane of a row / of two rows
constexpr int kDppWaveShr1 = 0x138;                      // the lane before, across rows

// value that lanes without a source, and rows not in ROWS, get: `none`
template <int CTRL, int ROWS = 0xf>
__device__ __forceinline__ uint32_t Dpp(uint32_t none, uint32_t v)
{
    return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(
        static_cast<int>(none), static_cast<int>(v), CTRL, ROWS, 0xf, false));
}

// a permutation: every lane has a source
template <int CTRL>
__device__ __forceinline__ uint32_t Permute(uint32_t v)
{
    return static_cast<uint32_t>(
        __builtin_amdgcn_update_dpp(0, static_cast<int>(v), CTRL, 0xf, 0xf, true));
}

// inclusive scan over the lanes; combine(0, x) is x
template <typename Combine>
__device__ __forceinline__ uint32_t WaveScan(uint32_t v, Combine combine)
{
    v = combine(v, Dpp<kDppShr1>(0, v));
    v = combine(v, Dpp<kDppShr2>(0, v));
    v = combine(v, Dpp<kDppShr4>(0, v));
    v = combine(v, Dpp<kDppShr8>(0, v));
    v = combine(v, Dpp<kDppBcast15, 0xa>(0, v));
    return combine(v, Dpp<kDppBcast31, 0xc>(0, v));
}

struct LanePair
{
    uint32_t x, y;
};

// MASK 16: odd rows of 16 lanes of x change places with even rows of y; MASK 32: the upper half of
// x with the lower half of y.  Pairs (l, l ^ MASK) of x then stand side by side in the lanes of
// one half and those of y in the others; a second swap undoes it.
template <uint32_t MASK>
__device__ __forceinline__ LanePair SwapLanes(uint32_t x, uint32_t y)
{
    static_assert(MASK == 16 || MASK == 32, "rows of 16 or halves");
    if constexpr (MASK == 16)
    {
        const auto r = __builtin_amdgcn_permlane16_swap(x, y, false, false);
        return { r[0], r[1] };
    }
    else
    {
        const auto r = __builtin_amdgcn_permlane32_swap(x, y, false, false);
        return { r[0], r[1] };
    }
}

// value of lane (lane ^ MASK): a power of two, or one less than a power of two up to 16
template <uint32_t MASK>
__device__ __forceinline__ uint32_t XorLane(uint32_t v)
{
    if constexpr (MASK == 0)
        return v;
    else if constexpr (MASK == 1)
        return Permute<kDppXor1>(v);
    else if constexpr (MASK == 2)
        return Permute<kDppXor2>(v);
    else if constexpr (MASK == 3)
        return Permute<kDppXor3>(v);
    else if constexpr (MASK == 4)
        return Permute<kDppXor3>(Permute<kDppXor7>(v));
    else if constexpr (MASK == 7)
        return Permute<kDppXor7>(v);
    else if constexpr (MASK == 8)
        return Permute<kDppXor8>(v);
    else if constexpr (MASK == 15)
        return Permute<kDppXor15>(v);
    else
    {
        const LanePair p = SwapLanes<MASK>(v, v);
        return (threadIdx.x & MASK) != 0 ? p.x : p.y;
    }
}

// the smaller of x and y where bound is 0, the larger where it is all ones (v_med3_u32)
__device__ __forceinline__ uint32_t Med3(uint32_t x, uint32_t y, uint32_t bound)
{
    return max(min(x, y), min(max(x, y), bound));
}

// all ones in the lanes with that bit set
struct LaneBits
{
    uint32_t bit[6];
    __device__ __forceinline__ explicit LaneBits(uint32_t lane)
    {
#pragma unroll
        for (uint32_t k = 0; k < 6; ++k)
            bit[k] = 0u - ((lane >> k) & 1u);
    }
    // Keeps the compiler from working the bounds of a sort out ahead of the rows, which costs more
    // registers than a row has to spare.
    __device__ __forceinline__ void Pin()
    {
#pragma unroll
        for (uint32_t k = 0; k < 6; ++k)
            asm volatile("" : "+v"(bit[k]));
    }
};

// The one of two keys that a lane keeps: the smaller where `bound` is 0, else the larger.
__device__ __forceinline__ uint32_t Exchange(uint32_t x, uint32_t y, uint32_t bound)
{
    return Med3(x, y, bound);
}

// (keys of 64 bits: 2^23 columns and more, and the pass that does overflowed rows again)
__device__ __forceinline__ uint64_t Exchange(uint64_t x, uint64_t y, uint32_t bound)
{
    return (y < x) == (bound == 0) ? y : x;
}

template <uint32_t MASK>
__device__ __forceinline__ uint64_t XorLane(uint64_t v)
{
    const uint32_t lo = XorLane<MASK>(static_cast<uint32_t>(v));
    const uint32_t hi = XorLane<MASK>(static_cast<uint32_t>(v >> 32));
    return (static_cast<uint64_t>(hi) << 32) | lo;
}

// Bitonic sort of 64 E keys held by one wavefront, E consecutive ones per lane: the exchanges
// from (SIZE, STRIDE) on.  An exchange of 32-bit keys is one lane operation and one v_med3_u32
// against a bound that is 0 in the lanes that keep the smaller key and all ones in the others: no
// condition code, and so no wait between vector and scalar unit.
// Merges inside a row of 16 lanes begin with an exchange between a block and its mirror image,
// which needs no blocks of opposite directions: one bound per stride serves them all.  Odd rows
// then end up descending (`down`), and so does the upper half of the lanes, as the merges
// across rows need it.
template <uint32_t E, typename Key, uint32_t SIZE = 2, uint32_t STRIDE = 1>
__device__ __forceinline__ void SortKeys(Key (&key)[E], const LaneBits& lanes)
{
    constexpr bool kInRow = SIZE <= 16 * E;
    constexpr bool kMirror = kInRow && STRIDE == SIZE / 2;
    const uint32_t down = kInRow ? lanes.bit[4] : SIZE == 32 * E ? lanes.bit[5] : 0u;
    if constexpr (STRIDE < E)
    {
#pragma unroll
        for (uint32_t e = 0; e < E; ++e)
        {
            const uint32_t o = kMirror ? e ^ (SIZE - 1) : e ^ STRIDE;
            if (o < e)
                continue;
            const Key x = key[e], y = key[o];
            key[e] = Exchange(x, y, down);
            key[o] = Exchange(x, y, ~down);
        }
    }
    else if constexpr (STRIDE / E >= 16 && E > 1 && sizeof(Key) == 4)
    {
        // two keys of a lane at once: their pairs side by side, and back
#pragma unroll
        for (uint32_t e = 0; e < E; e += 2)
        {
            const LanePair p = SwapLanes<STRIDE / E>(key[e], key[e + 1]);
            const LanePair q =
                SwapLanes<STRIDE / E>(Med3(p.x, p.y, down), Med3(p.x, p.y, ~down));
            key[e] = q.x;
            key[e + 1] = q.y;
        }
    }
    else
    {
        constexpr uint32_t kLanes = STRIDE / E;  // a power of two
        const uint32_t bound = lanes.bit[__builtin_ctz(kLanes)] ^ down;
        if constexpr (kLanes >= 16 && sizeof(Key) == 4)
        {
            const LanePair p = SwapLanes<kLanes>(key[0], key[0]);
            key[0] = Med3(p.x, p.y, bound);
        }
        else if constexpr (kMirror)
        {
            Key other[E];
#pragma unroll
            for (uint32_t e = 0; e < E; ++e)
                other[e] = XorLane<SIZE / E - 1>(key[E - 1 - e]);
#pragma unroll
            for (uint32_t e = 0; e < E; ++e)
                key[e] = Exchange(key[e], other[e], bound);
        }
        else
        {
#pragma unroll
            for (uint32_t e = 0; e < E; ++e)
                key[e] = Exchange(key[e], XorLane<kLanes>(key[e]), bound);
        }
    }
    if constexpr (STRIDE > 1)
        SortKeys<E, Key, SIZE, STRIDE / 2>(key, lanes);
    else if constexpr (SIZE < 64 * E)
        SortKeys<E, Key, SIZE * 2, SIZE>(key, lanes);
}

// A wavefront's own LDS: nothing is shared between wavefronts, and the LDS operations of one
// wavefront are executed in order.
struct LightScratch
{
    uint32_t column[kLightProducts];  // before the sort: the entry of A that starts here
    float product[kLightProducts];
};

struct LightInput
{
    uint32_t entriesOfA;      // uniform, at most 64
    uint32_t products;        // uniform, at most 64 E
    // of lane j: products of A's entry j, their first entry in B, products of the entries before
    uint32_t mine, bBegin, before;
    float aValue;             // and the value of A's entry j
    uint32_t rowBase, rowLimit;  // uniform: where the entries go
};

// four-byte aligned groups of entries, stored with one access
template <uint32_t E, typename T>
struct EntryGroup
{
    typedef T Type __attribute__((ext_vector_type(E), aligned(4)));
};

// The entries of one light row; returns their number.
template <int MODE, uint32_t E, typename Key>
__device__ __forceinline__ uint32_t LightRowEntries(const SpgemmArgs& args, const LightInput& in,
                                                    LightScratch& lds, uint32_t lane,
                                                    const LaneBits& lanes)
{
    // Product p (in the order in which the sums take them) belongs to lane p % 64.  The entry of A
    // it comes from: every entry that has products leaves its number + 1 at its first one, and
    // the largest number at or before p is the one.
#pragma unroll
    for (uint32_t e = 0; e < E; ++e)
        lds.column[e * 64u + lane] = 0;
    if (in.mine != 0)
        lds.column[in.before] = lane + 1;
    __builtin_amdgcn_wave_barrier();
    const uint32_t from = in.bBegin - in.before;
    uint32_t base[E];
    float a[E];
    uint32_t passed = 0;
#pragma unroll
    for (uint32_t e = 0; e < E; ++e)
    {
        const uint32_t entry =
            max(passed, WaveScan(lds.column[e * 64u + lane],
                                 [](uint32_t x, uint32_t y) { return max(x, y); }));
        passed = Uniform(entry, 63);
        const int source = static_cast<int>(entry * 4u - 4u);
        base[e] = static_cast<uint32_t>(
            __builtin_amdgcn_ds_bpermute(source, static_cast<int>(from)));
        a[e] = __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(
                                             source, __builtin_bit_cast(int, in.aValue)));
    }
    uint32_t col[E];
    float b[E];
#pragma unroll
    for (uint32_t e = 0; e < E; ++e)
    {
        const uint32_t p = e * 64u + lane;
        col[e] = kEmpty;
        b[e] = 0.0f;
        if (p < in.products)
        {
            col[e] = args.COLB[base[e] + p];
            b[e] = args.VB[base[e] + p];
        }
    }
    // keys: column, then place in the order of the sums; where a key starts does not matter
    Key key[E];
#pragma unroll
    for (uint32_t e = 0; e < E; ++e)
    {
        const uint32_t p = e * 64u + lane;
        key[e] = col[e] < args.N ? static_cast<Key>(col[e]) << kPlaceBits | p : ~static_cast<Key>(0);
        lds.product[p] = a[e] * b[e];
    }
    LaneBits bounds = lanes;
    bounds.Pin();
    SortKeys<E, Key>(key, bounds);
    __builtin_amdgcn_wave_barrier();

    // the sorted (column, product) pairs side by side
    const uint32_t place0 = lane * E;
    uint32_t c[E];
    float v[E];
    bool used[E];
    uint32_t valid = 0;  // pairs of the row
#pragma unroll
    for (uint32_t e = 0; e < E; ++e)
    {
        used[e] = key[e] != ~static_cast<Key>(0);
        c[e] = used[e] ? static_cast<uint32_t>(key[e] >> kPlaceBits) : kEmpty;
        v[e] = lds.product[static_cast<uint32_t>(key[e]) & (64u * E - 1)];
        valid += static_cast<uint32_t>(__popcll(__ballot(used[e])));
    }
    // does a pair have the column of the one before it?
    bool repeats[E];
    bool anyRepeats = false;
#pragma unroll
    for (uint32_t e = 0; e < E; ++e)
    {
        const uint32_t left = e != 0 ? c[e == 0 ? 0 : e - 1] : Dpp<kDppWaveShr1>(kEmpty, c[E - 1]);
        repeats[e] = used[e] && c[e] == left;
        anyRepeats = anyRepeats || repeats[e];
    }
    // the first pair of a column sums the column's products, in their order, from +0
    if (__ballot(anyRepeats) == 0)
    {
#pragma unroll
        for (uint32_t e = 0; e < E; ++e)
            v[e] = 0.0f + v[e];
    }
    else
    {
        __builtin_amdgcn_wave_barrier();
        uint32_t place = place0;
        asm volatile("" : "+v"(place));  // (or it is held in E forms through every row)
#pragma unroll
        for (uint32_t e = 0; e < E; ++e)
        {
            lds.column[place + e] = c[e];
            lds.product[place + e] = v[e];
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (uint32_t e = 0; e < E; ++e)
        {
            if (used[e] && !repeats[e])
            {
                float sum = 0.0f + v[e];
                for (uint32_t t = place + e + 1; t < 64u * E && lds.column[t] == c[e]; ++t)
                    sum = sum + lds.product[t];
                v[e] = sum;
            }
        }
    }
    bool keep[E];
    bool dropped = false;
#pragma unroll
    for (uint32_t e = 0; e < E; ++e)
    {
        keep[e] = used[e] && !repeats[e] && v[e] != 0.0f;  // exact zeros are not stored
        dropped = dropped || keep[e] != used[e];
    }
    if (__ballot(dropped) == 0)
    {
        // every pair is an entry: a lane's are neighbours
        if (MODE != kCount)
        {
            const uint32_t at = in.rowBase + place0;
            const uint32_t room = in.rowLimit > in.rowBase ? in.rowLimit - in.rowBase : 0u;
            const uint32_t end = min(valid, room);
            constexpr uint32_t kGroup = E < 4 ? E : 4;
            typedef typename EntryGroup<kGroup, float>::Type Values;
            typedef typename EntryGroup<kGroup, uint32_t>::Type Columns;
#pragma unroll
            for (uint32_t g = 0; g < E; g += kGroup)
            {
                if (place0 + g + kGroup <= end)
                {
                    Values values;
                    Columns columns;
#pragma unroll
                    for (uint32_t e = 0; e < kGroup; ++e)
                    {
                        values[e] = v[g + e];
                        columns[e] = c[g + e];
                    }
                    *reinterpret_cast<Values*>(args.VC + at + g) = values;
                    *reinterpret_cast<Columns*>(args.COLC + at + g) = columns;
                }
                else if (kGroup > 1 && place0 + g < end)
                {
#pragma unroll
                    for (uint32_t e = 0; e < kGroup - 1; ++e)
                        if (place0 + g + e < end)
                        {
                            args.VC[at + g + e] = v[g + e];
                            args.COLC[at + g + e] = c[g + e];
                        }
                }
            }
        }
        return valid;
    }
    const uint64_t below = (1ull << lane) - 1ull;
    uint32_t before = 0, emitted = 0;
#pragma unroll
    for (uint32_t e = 0; e < E; ++e)
    {
        const uint64_t m = __ballot(keep[e]);
        before += static_cast<uint32_t>(__popcll(m & below));
        emitted += static_cast<uint32_t>(__popcll(m));
    }
    if (MODE != kCount)
    {
        uint32_t at = in.rowBase + before;
#pragma unroll
        for (uint32_t e = 0; e < E; ++e)
            if (keep[e])
            {
                if (at < in.rowLimit)
                {
                    args.VC[at] = v[e];
                    args.COLC[at] = c[e];
                }
                ++at;
            }
    }
    return emitted;
}

// Prefix sum of the lanes' numbers of products; true when the row is light.
__device__ __forceinline__ bool CountProducts(const SpgemmArgs& args, LightInput& in, uint32_t mine)
{
    const uint32_t inclusive = WaveScan(mine, [](uint32_t x, uint32_t y) { return x + y; });
    in.mine = mine;
    in.before = inclusive - mine;
    in.products = Uniform(inclusive, 63);
    return LightRow(args, in.entriesOfA, in.products);
}

// The entries of one light row, with as many products per lane as it needs.
template <int MODE, typename Key>
__device__ __forceinline__ uint32_t LightRowOfAnyLength(const SpgemmArgs& args, const LightInput& in,
                                                        LightScratch& lds, uint32_t lane,
                                                        const LaneBits& lanes)
{
    if (in.products <= 64)
        return LightRowEntries<MODE, 1, Key>(args, in, lds, lane, lanes);
    if (in.products <= 128)
        return LightRowEntries<MODE, 2, Key>(args, in, lds, lane, lanes);
    if (in.products <= 256)
        return LightRowEntries<MODE, 4, Key>(args, in, lds, lane, lanes);
    return LightRowEntries<MODE, 8, Key>(args, in, lds, lane, lanes);
}

// Light rows.  The strip kernel walks all products of a row once per strip of 4096 columns, one
// row of B at a time with as many active lanes as that row has entries (8 of 64 on a graph with
// 8 neighbours per node).  Here all products of a row are loaded at once, one per lane and
// register, and sorted in registers by (column, place in the order of the sums); the first
// product of a column then adds the following ones of the same column in that order, sums that
// are exactly zero are dropped, and ballots give the others their output positions.  The cost of
// a row follows its products, not the width of the matrix.
// What bounds it is the issue of vector instructions (about 300 for a row of 64 products) behind a
// chain of four dependent loads; seven wavefronts per SIMD are resident (five left 8192 rows in
// two rounds; eight spill scalars and are level).  Against a sort by compares and selects, shuffles
// through the LDS crossbar and a search of every product's entry of A one entry after the other:
// 65536 rows with 8 entries on both sides 63 -> 35 us for the pass, the whole call 86 -> 59 us;
// 8192 rows 15.8 -> 9.4 us.
template <int MODE, typename Key>
__global__ __launch_bounds__(kLightWaves * 64, 7) void SpgemmLightKernel(const SpgemmArgs args)
{
    __shared__ LightScratch scratch[kLightWaves];
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = threadIdx.x >> 6;
    const LaneBits lanes(lane);
    const uint32_t turn0 = blockIdx.x * kLightWaves + wave;
    const uint64_t step = static_cast<uint64_t>(gridDim.x) * kLightWaves * args.rowsPerTurn;
    // A wavefront takes rowsPerTurn consecutive rows per turn, with the loads that lead to a
    // row's products in a pipeline over the rows of the turn, as in the strip kernel.
    for (uint64_t turn = static_cast<uint64_t>(turn0) * args.rowsPerTurn; turn < args.M; turn += step)
    {
        const uint32_t first = static_cast<uint32_t>(turn);
        const uint32_t rowsHere = min(args.rowsPerTurn, args.M - first);
        uint32_t extentA = 0, extentC = 0;
        if (lane <= rowsHere)
        {
            extentA = args.ROWA[first + lane];
            if (MODE == kFill)
                extentC = args.ROWC[first + lane];
            if (MODE == kStage)
                extentC = (first + lane) * args.slot;
        }
        // a row with more entries than a light row has products is the strip kernel's
        if (MODE == kFill)
        {
            const uint32_t entries = __shfl_down(extentC, 1, 64) - extentC;
            if (__ballot(lane < rowsHere && entries <= kLightProducts) == 0)
                continue;
        }
        // stage 1: this lane's entry of A's row i (rows with more than 64 entries are not ours)
        auto loadStage1 = [&](uint32_t i, uint32_t& k, float& value) {
            k = kEmpty;
            value = 0.0f;
            if (i < rowsHere)
            {
                const uint32_t begin = Uniform(extentA, i), end = Uniform(extentA, i + 1);
                if (end - begin <= 64 && begin + lane < end)
                {
                    k = args.COLA[begin + lane];
                    value = args.VA[begin + lane];
                }
            }
        };
        // stage 2: the extent of the row of B that entry selects
        auto loadStage2 = [&](uint32_t k, uint32_t& begin, uint32_t& end) {
            begin = 0;
            end = 0;
            if (k < args.K)
            {
                begin = args.ROWB[k];
                end = args.ROWB[k + 1];
            }
        };
        uint32_t k1, k2, nextBegin, nextEnd;
        float value1, value2;
        loadStage1(0, k2, value2);
        loadStage2(k2, nextBegin, nextEnd);
        loadStage1(1, k1, value1);

        uint32_t counted = 0;  // of lane i: entries of the turn's row i
        for (uint32_t i = 0; i < rowsHere; ++i)
        {
            LightInput in;
            in.entriesOfA = Uniform(extentA, i + 1) - Uniform(extentA, i);
            in.bBegin = nextBegin;
            in.aValue = value2;
            const uint32_t mine = LightCount(nextBegin, nextEnd);
            k2 = k1;
            value2 = value1;
            loadStage2(k2, nextBegin, nextEnd);
            loadStage1(i + 2, k1, value1);
            if (!CountProducts(args, in, mine))
            {
                counted = lane == i ? kHeavyMark : counted;  // the strip kernel's row
                continue;
            }
            in.rowBase = 0;
            in.rowLimit = 0;
            if (MODE != kCount)
            {
                in.rowBase = Uniform(extentC, i);
                in.rowLimit = Uniform(extentC, i + 1);
                if (MODE == kFill)
                    in.rowLimit = min(in.rowLimit, args.capacity);
            }
            const uint32_t emitted =
                LightRowOfAnyLength<MODE, Key>(args, in, scratch[wave], lane, lanes);
            counted = lane == i ? emitted : counted;
        }
        if (MODE != kFill && lane < rowsHere)
            args.counts[first + lane] = counted;
    }
}

// Which rows a pass of the strip kernel takes.  A pass of its own for each: with the choice made at
// run time the narrow products, which take every row, were 0.3 us slower per launch.
constexpr int kEveryRow = 0;
constexpr int kMarkedRows = 1;    // those that SpgemmLightKernel has marked in `counts`
constexpr int kOverfullRows = 2;  // those with more than skipUpTo entries, if *overflow is set

template <int MODE, int ROWS>
__global__ __launch_bounds__(64) void SpgemmRowKernel(const SpgemmArgs args)
{
    constexpr bool FILL = MODE != kCount;    // entries are stored
    constexpr bool COUNTS = MODE != kFill;   // counts are stored
    extern __shared__ float strip[];
    // one bit per column, after the strip; lane l owns words l*wordsPerLane .. +wordsPerLane-1
    uint32_t* bits = reinterpret_cast<uint32_t*>(strip + args.strip);
    const uint32_t wordsInStrip = args.strip / 32;
    const uint32_t wordsPerLane = (wordsInStrip + 63) / 64;  // at most kStripMax / 2048
    const uint32_t lane = threadIdx.x;
    if (ROWS == kOverfullRows && *args.overflow == 0)
        return;  // every row is in place already
    if (COUNTS && blockIdx.x == 0 && lane == 0)
        args.counts[args.M] = 0;
    if (MODE == kStage && blockIdx.x == 0 && lane == 0)
        *args.overflow = 0;
    // once; every element that is touched is cleared again when it is swept
    auto clear = [&] {
        for (uint32_t x = lane; x < args.strip; x += 64)
            strip[x] = 0.0f;
        for (uint32_t t = lane; t < wordsInStrip; t += 64)
            bits[t] = 0;
    };

    // A wavefront takes rowsPerTurn consecutive rows per turn.  Their extents are read in one
    // go, and the loads that lead to a row's products form a pipeline over the rows of the
    // turn: while row i is multiplied, the first 64 (column, value) pairs of A's row i+2 and
    // the extents of the rows of B that row i+1 needs are already on their way.
    auto multiply = [&](uint32_t turn) {
        const uint32_t rowsHere = min(args.rowsPerTurn, args.M - turn);
        uint32_t extentA = 0, extentC = 0;
        if (lane <= rowsHere)
        {
            extentA = args.ROWA[turn + lane];
            if (MODE == kFill)
                extentC = args.ROWC[turn + lane];
            if (MODE == kStage)
                extentC = (turn + lane) * args.slot;
        }
        // stage 1 (columns and values of A's row) and stage 2 (extents in B) of the pipeline
        auto loadStage1 = [&](uint32_t i, uint32_t& k, float& value) {
            k = 0xffffffffu;
            value = 0.0f;
            if (i < rowsHere)
            {
                const uint32_t begin = Uniform(extentA, i), end = Uniform(extentA, i + 1);
                if (begin + lane < end)
                {
                    k = args.COLA[begin + lane];
                    value = args.VA[begin + lane];
                }
            }
        };
        auto loadStage2 = [&](uint32_t k, uint32_t& bBegin, uint32_t& bEnd) {
            bBegin = 0;
            bEnd = 0;
            if (k < args.K)
            {
                bBegin = args.ROWB[k];
                bEnd = args.ROWB[k + 1];
            }
        };
        uint32_t k1, k2, nextBegin, nextEnd;
        float value1, value2;
        loadStage1(0, k2, value2);
        loadStage2(k2, nextBegin, nextEnd);
        loadStage1(1, k1, value1);

      for (uint32_t i = 0; i < rowsHere; ++i)
      {
        const uint32_t aBegin = Uniform(extentA, i);
        const uint32_t aEnd = Uniform(extentA, i + 1);
        uint32_t emitted = 0;  // entries of this row found so far (all strips)
        const uint32_t rowBase = FILL ? Uniform(extentC, i) : 0u;
        const uint32_t rowEnd = FILL ? Uniform(extentC, i + 1) : 0u;
        const uint32_t rowLimit = MODE == kFill ? min(rowEnd, args.capacity) : rowEnd;
        // this row's first batch comes out of the pipeline, which then moves on
        const uint32_t firstBegin = nextBegin, firstEnd = nextEnd;
        const float firstValue = value2;
        k2 = k1;
        value2 = value1;
        loadStage2(k2, nextBegin, nextEnd);
        loadStage1(i + 2, k1, value1);
        // in a wide product the light rows belong to SpgemmLightKernel
        if (ROWS != kOverfullRows && args.heavyOnly != 0 &&
            LightRow(args, aEnd - aBegin, WaveSum(LightCount(firstBegin, firstEnd))))
            continue;
        if (MODE == kFill && rowEnd - rowBase <= args.skipUpTo)
            continue;  // empty, or already in place
        // Light rows that overflowed are sorted here.  On strips they cost a walk over their
        // products per 4096 columns: capacity of one entry per row, 144 products per row, 65536 rows
        // and columns 6493 us, now 734; 20000 rows, 2^20 columns 27.5 ms, now 0.24 ms.
        if constexpr (ROWS == kOverfullRows)
        {
            __shared__ LightScratch scratch;
            LightInput in;
            in.entriesOfA = aEnd - aBegin;
            in.bBegin = firstBegin;
            in.aValue = firstValue;
            in.rowBase = rowBase;
            in.rowLimit = rowLimit;
            if (CountProducts(args, in, LightCount(firstBegin, firstEnd)))
            {
                LightRowOfAnyLength<kFill, uint64_t>(args, in, scratch, lane, LaneBits(lane));
                continue;
            }
        }

        for (uint32_t c0 = 0; c0 < args.N; c0 += args.strip)
        {
            const uint32_t width = min(args.strip, args.N - c0);

            for (uint32_t pa0 = aBegin; pa0 < aEnd; pa0 += 64)
            {
                // up to 64 entries of A's row, one per lane, with the extent of their rows of B
                const uint32_t have = min(64u, aEnd - pa0);
                uint32_t bBegin = firstBegin, bEnd = firstEnd;
                float aValue = firstValue;
                if (pa0 != aBegin)
                {
                    bBegin = 0;
                    bEnd = 0;
                    aValue = 0.0f;
                    if (lane < have)
                    {
                        const uint32_t k = args.COLA[pa0 + lane];
                        aValue = args.VA[pa0 + lane];
                        if (k < args.K)
                        {
                            bBegin = args.ROWB[k];
                            bEnd = args.ROWB[k + 1];
                        }
                    }
                }
                // the entries are applied in order; the first 64 entries of kAhead rows of B
                // are requested before the first of them is used
                for (uint32_t j0 = 0; j0 < have; j0 += kAhead)
                {
                    uint32_t s[kAhead], e[kAhead], col[kAhead];
                    float a[kAhead], b[kAhead];
#pragma unroll
                    for (uint32_t u = 0; u < kAhead; ++u)
                    {
                        const uint32_t j = min(j0 + u, 63u);
                        s[u] = Uniform(bBegin, j);
                        e[u] = j0 + u < have ? Uniform(bEnd, j) : s[u];
                        a[u] = Uniform(aValue, j);
                    }
#pragma unroll
                    for (uint32_t u = 0; u < kAhead; ++u)
                    {
                        col[u] = 0xffffffffu;
                        b[u] = 0.0f;
                        if (s[u] + lane < e[u])
                        {
                            col[u] = args.COLB[s[u] + lane];
                            b[u] = args.VB[s[u] + lane];
                        }
                    }
#pragma unroll
                    for (uint32_t u = 0; u < kAhead; ++u)
                    {
                        if (col[u] - c0 < width)  // also false for the 0xffffffff of idle lanes
                        {
                            strip[col[u] - c0] = strip[col[u] - c0] + a[u] * b[u];
                            Touch(bits, col[u] - c0);
                        }
                        // rows of B with more than 64 entries: the rest, 64 at a time
                        for (uint32_t pb = s[u] + 64 + lane; pb < e[u]; pb += 64)
                        {
                            const uint32_t c = args.COLB[pb];
                            if (c - c0 < width)
                            {
                                strip[c - c0] = strip[c - c0] + a[u] * args.VB[pb];
                                Touch(bits, c - c0);
                            }
                        }
                    }
                }
            }

            // sweep: this lane's touched columns in ascending order, as two 64-column runs
            // (a pair of bit-map words each)
            auto fetchPair = [&](uint32_t first) {
                uint32_t lo = 0, hi = 0;
                const uint32_t w = lane * wordsPerLane + first;
                if (first < wordsPerLane && w < wordsInStrip)
                {
                    lo = bits[w];
                    if (lo != 0)
                        bits[w] = 0;
                }
                if (first + 1 < wordsPerLane && w + 1 < wordsInStrip)
                {
                    hi = bits[w + 1];
                    if (hi != 0)
                        bits[w + 1] = 0;
                }
                return (static_cast<uint64_t>(hi) << 32) | lo;
            };
            const uint64_t mine0 = fetchPair(0);
            const uint64_t mine1 = fetchPair(2);
            const uint32_t base0 = lane * wordsPerLane * 32;  // first column of run 0
            const uint32_t base1 = base0 + 64;

            // next touched column of this lane's runs, removed from the set
            auto take = [&](uint64_t& set0, uint64_t& set1) {
                if (set0 != 0)
                {
                    const uint32_t b = static_cast<uint32_t>(__builtin_ctzll(set0));
                    set0 &= set0 - 1;
                    return base0 + b;
                }
                const uint32_t b = static_cast<uint32_t>(__builtin_ctzll(set1));
                set1 &= set1 - 1;
                return base1 + b;
            };
            // pass 1: how many of them hold a value that is not zero (the count pass
            // clears them here; the fill pass needs them once more)
            uint32_t kept = 0;
            {
                uint64_t set0 = mine0, set1 = mine1;
                while ((set0 | set1) != 0)
                {
                    const uint32_t x = take(set0, set1);
                    if (strip[x] != 0.0f)
                        ++kept;
                    if (!FILL)
                        strip[x] = 0.0f;  // the storing passes read it once more below
                }
            }
            // positions: exclusive prefix sum of `kept` over the lanes
            uint32_t inclusive = kept;
#pragma unroll
            for (uint32_t d = 1; d < 64; d *= 2)
            {
                const uint32_t other = __shfl_up(inclusive, d, 64);
                if (lane >= d)
                    inclusive += other;
            }
            if (FILL)
            {
                uint32_t at = rowBase + emitted + inclusive - kept;
                uint64_t set0 = mine0, set1 = mine1;
                while ((set0 | set1) != 0)
                {
                    const uint32_t x = take(set0, set1);
                    const float v = strip[x];
                    strip[x] = 0.0f;
                    if (v != 0.0f)
                    {
                        if (at < rowLimit)
                        {
                            args.VC[at] = v;
                            args.COLC[at] = c0 + x;
                        }
                        ++at;
                    }
                }
            }
            emitted += Uniform(inclusive, 63);
        }
        if (COUNTS && lane == 0)
            args.counts[turn + i] = emitted;
      }
    };

    const uint32_t turns = sph::SpgemmTurns(args.M, args.rowsPerTurn);
    if (ROWS == kEveryRow)
    {
        clear();
        for (uint64_t t = blockIdx.x; t < turns; t += gridDim.x)
            multiply(static_cast<uint32_t>(t) * args.rowsPerTurn);
        return;
    }
    // There are usually none or few such rows, so the turns of a wavefront are looked through
    // first, as many at once as 64 lanes have rows for, and only those with one are taken (walking
    // every row for nothing took 28 us on 65536 rows).
    const uint32_t rows = args.rowsPerTurn;
    const uint32_t looked = 64 / rows;  // turns per look
    const uint32_t turnOfLane = lane / rows;
    bool cleared = false;
    for (uint64_t base = blockIdx.x; base < turns; base += static_cast<uint64_t>(looked) * gridDim.x)
    {
        const uint64_t row =
            (base + static_cast<uint64_t>(turnOfLane) * gridDim.x) * rows + lane % rows;
        bool wanted = false;
        if (turnOfLane < looked && row < args.M)
            wanted = COUNTS ? args.counts[row] == kHeavyMark
                            : args.ROWC[row + 1] - args.ROWC[row] > args.skipUpTo;
        uint64_t chosen = __ballot(wanted);
        while (chosen != 0)
        {
            if (!cleared)
                clear();
            cleared = true;
            const uint32_t next = static_cast<uint32_t>(__builtin_ctzll(chosen)) / rows;
            multiply(static_cast<uint32_t>((base + static_cast<uint64_t>(next) * gridDim.x) * rows));
            // the turn's lanes, and those below them, are done
            const uint32_t done = (next + 1) * rows;
            chosen = done < 64 ? chosen >> done << done : 0;
        }
    }
}

// Staged rows move to their place: row r's ROWC[r + 1] - ROWC[r] entries from r * slot.  Rows
// that did not fit their slot are left to a fill pass.  One wavefront per row, 4 per workgroup.
__global__ __launch_bounds__(256) void SpgemmUnstageKernel(float* __restrict__ VC,
                                                           uint32_t* __restrict__ COLC,
                                                           const uint32_t* __restrict__ ROWC,
                                                           const float* __restrict__ stageV,
                                                           const uint32_t* __restrict__ stageCol,
                                                           uint32_t M, uint32_t slot,
                                                           uint32_t capacity, uint32_t* overflow)
{
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t row = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= M)
        return;
    const uint32_t first = ROWC[row];
    const uint32_t count = ROWC[row + 1] - first;
    if (count > slot)
    {
        if (lane == 0)
            *overflow = 1;
        return;
    }
    const size_t from = static_cast<size_t>(row) * slot;
    for (uint32_t i = lane; i < count; i += 64)
        if (first + i < capacity)
        {
            VC[first + i] = stageV[from + i];
            COLC[first + i] = stageCol[from + i];
        }
}

// The scan of the counts and the move in one launch.
__global__ __launch_bounds__(sph::kPlaceThreads) void SpgemmPlaceKernel(
    float* __restrict__ VC, uint32_t* __restrict__ COLC, uint32_t* __restrict__ ROWC,
    const uint32_t* __restrict__ counts, const float* __restrict__ stageV,
    const uint32_t* __restrict__ stageCol, uint32_t M, uint32_t rowsPerGroup, uint32_t slot,
    uint32_t capacity, uint32_t* overflow)
{
    __shared__ sph::PlaceScratch lds;
    sph::PlaceOffsets(ROWC, counts, M, rowsPerGroup, lds);
    sph::MoveStagedRows(VC, COLC, stageV, stageCol, M, rowsPerGroup, slot, capacity, lds,
                        [&](uint32_t, uint32_t, uint32_t) {
                            if ((threadIdx.x & 63u) == 0)
                                *overflow = 1;
                        });
}

// load[p] = entries of the row of B that entry p of A selects (the multiplications entry p
// causes); *total (when given, zero before the launch) receives their sum.
__global__ __launch_bounds__(256) void SpgemmLoadKernel(uint32_t* __restrict__ load,
                                                        const uint32_t* __restrict__ COLA,
                                                        const uint32_t* __restrict__ ROWB,
                                                        uint32_t entries, uint32_t K,
                                                        unsigned long long* total)
{
    unsigned long long sum = 0;
    for (uint64_t p = blockIdx.x * 256ull + threadIdx.x; p < entries; p += 256ull * gridDim.x)
    {
        const uint32_t k = COLA[p];
        const uint32_t n = k < K ? ROWB[k + 1] - ROWB[k] : 0u;
        if (load != nullptr)
            load[p] = n;
        sum += n;
    }
    if (total == nullptr)
        return;
#pragma unroll
    for (int d = 32; d > 0; d >>= 1)
        sum += __shfl_xor(sum, d, 64);
    if ((threadIdx.x & 63u) == 0 && sum != 0)
        atomicAdd(total, sum);
}

__global__ void ClearTotalKernel(unsigned long long* total)
{
    *total = 0;
}

// Most products of a row that SpgemmLightKernel takes; products: the caller's bound on the
// mean products of a row (a capacity is usually that), 0 when there is none.
// One strip: always the strip kernel (4096 columns, 16 / 32 entries per row: 35 / 71 us a call,
// 40 / 80 us with all rows up to 512 products taken; with fewer products the host bounds both).
// Two strips: the strip kernel costs little more than on one, and rows of which only a part is
// light pay both kernels, so nearly all have to be light (6000 columns, 12 / 15 / 16 / 17 entries
// per row 58 / 67 / 72 / 75 us on strips, 32 / 32 / 54 / 61 us here; 4200 columns, 15 / 16 / 17
// entries 46 / 51 / 52 against 46 / 50 / 52; 8192 columns, 17 / 18 / 19 / 22 entries
// 77 / 84 / 87 / 97 against 64 / 82 / 97 / 121: what grows there is a few rows with more than
// 512 products, which the strips then do one by one).  From three strips on always (9000
// columns, 12 / 18 / 21 entries: 110 / 181 / 182 us on strips).
uint32_t LightProductsFor(uint32_t N, uint32_t products)
{
    if (N <= kStripMax)
        return 0;
    if (N <= 2 * kStripMax)
        return products != 0 && products <= 320 ? kLightProducts : 0u;
    return kLightProducts;
}

uint32_t StripFor(uint32_t N)
{
    const uint32_t padded = (N + 63u) / 64u * 64u;
    return std::max<uint32_t>(64u, std::min(padded, kStripMax));
}

// Rows per turn: long turns let the loads of consecutive rows overlap, short ones give a small
// matrix enough workgroups to fill the chip (about eight resident per compute unit).
uint32_t RowsPerTurnFor(uint32_t M)
{
    const uint32_t wanted = static_cast<uint32_t>(sph::ComputeUnits()) * 8;
    return std::max<uint32_t>(1, std::min<uint32_t>(kRowsPerTurnMax, M / std::max<uint32_t>(wanted, 1)));
}

// Light rows: seven workgroups of four wavefronts are resident per compute unit.  Turns are as long
// as if there were eight: enough rows per turn to overlap their loads, with more workgroups than
// places where rows are few, which are handed out as places fall free.
template <int MODE>
void LaunchLight(const SpgemmArgs& args, hipStream_t stream)
{
    SpgemmArgs light = args;
    const uint64_t cus = static_cast<uint64_t>(sph::ComputeUnits());
    light.rowsPerTurn = static_cast<uint32_t>(
        std::max<uint64_t>(1, std::min<uint64_t>(kRowsPerTurnMax, args.M / (cus * 8 * kLightWaves))));
    const uint64_t turns = sph::SpgemmTurns(args.M, light.rowsPerTurn);
    const uint64_t groups = std::min<uint64_t>((turns + kLightWaves - 1) / kLightWaves, cus * 64);
    const dim3 grid(static_cast<uint32_t>(groups)), block(kLightWaves * 64);
    // column and place share 32 bits up to 2^23 columns (all ones stay free for "no product")
    if (args.N < (1u << (32 - kPlaceBits)))
        hipLaunchKernelGGL((SpgemmLightKernel<MODE, uint32_t>), grid, block, 0, stream, light);
    else
        hipLaunchKernelGGL((SpgemmLightKernel<MODE, uint64_t>), grid, block, 0, stream, light);
}

uint32_t GridFor(uint32_t M, uint32_t rowsPerTurn, uint32_t perComputeUnit)
{
    const uint64_t cap = static_cast<uint64_t>(sph::ComputeUnits()) * perComputeUnit;
    const uint64_t turns = sph::SpgemmTurns(M, rowsPerTurn);
    return static_cast<uint32_t>(std::max<uint64_t>(1, std::min<uint64_t>(turns, cap)));
}

template <int MODE, int ROWS>
void LaunchStrips(const SpgemmArgs& args, uint32_t perComputeUnit, hipStream_t stream)
{
    hipLaunchKernelGGL((SpgemmRowKernel<MODE, ROWS>),
                       dim3(GridFor(args.M, args.rowsPerTurn, perComputeUnit)), dim3(64),
                       args.strip * sizeof(float) + args.strip / 8, stream, args);
}

// The passes that count (and stage): the light rows of a wide product first, then the strips.
// A strip pass that looks for marked rows takes at most twice as many workgroups as are resident
// (nine per compute unit, 17 KiB of LDS each): the second half is handed out as places fall
// free, which evens out who got more marked rows.  65536 columns, two calls with a tenth of the
// rows left to the strips: 9 / 18 / 32 / 64 per compute unit 3977 / 3552 / 3494 / 3457 us; with no row
// left (one call, 8 entries per row), where more workgroups only cost their dispatch,
// 86.4 / 87.4 / 88.8 / 88.9 us.
template <int MODE>
void LaunchCounting(const SpgemmArgs& args, hipStream_t stream)
{
    if (args.heavyOnly == 0)
    {
        LaunchStrips<MODE, kEveryRow>(args, kStripGroups, stream);
        return;
    }
    if (args.M != 0)
        LaunchLight<MODE>(args, stream);
    LaunchStrips<MODE, kMarkedRows>(args, kMarkedGroups, stream);
}

// Every row's entries to their place.
void LaunchFill(const SpgemmArgs& args, hipStream_t stream)
{
    if (args.heavyOnly != 0)
        LaunchLight<kFill>(args, stream);
    LaunchStrips<kFill, kEveryRow>(args, kStripGroups, stream);
}
}  // namespace

extern "C" {

int sph_spgemm_row_offsets_f32(uint32_t* ROWC, const float* VA, const uint32_t* COLA,
                               const uint32_t* ROWA, const float* VB, const uint32_t* COLB,
                               const uint32_t* ROWB, uint32_t M, uint32_t K, uint32_t N,
                               uint32_t* nnzHost)
{
    SPH_REQUIRE(ROWC != nullptr && ROWA != nullptr, "null pointer");
    SPH_REQUIRE(M < 0xffffffffu, "too many rows");
    SPH_REQUIRE(K == 0 || ROWB != nullptr, "null pointer");
    if (sph::ScanWaitsOrAllocates(M + 1, nnzHost))
        SPH_REFUSE_WHILE_CAPTURING();  // before anything is enqueued into the graph
    hipStream_t stream = sph::CurrentStream();
    if (stream == nullptr)
        return SPH_ERR_DEVICE;
    SpgemmArgs args{};
    args.VA = VA;
    args.COLA = COLA;
    args.ROWA = ROWA;
    args.VB = VB;
    args.COLB = COLB;
    args.ROWB = ROWB;
    args.M = M;
    args.K = K;
    args.N = N;
    args.strip = StripFor(N);
    args.rowsPerTurn = RowsPerTurnFor(M);
    args.counts = ROWC;
    args.lightProducts = LightProductsFor(N, 0);
    args.heavyOnly = args.lightProducts != 0 ? 1u : 0u;
    LaunchCounting<kCount>(args, stream);
    SPH_CHECK_LAUNCH();
    return sph::ExclusiveScanInPlace(ROWC, M + 1, nnzHost, stream);
}

int sph_spgemm_fill_f32(float* VC, uint32_t* COLC, const uint32_t* ROWC, const float* VA,
                        const uint32_t* COLA, const uint32_t* ROWA, const float* VB,
                        const uint32_t* COLB, const uint32_t* ROWB, uint32_t M, uint32_t K,
                        uint32_t N)
{
    if (M == 0 || N == 0)
        return SPH_OK;
    SPH_REQUIRE(ROWC != nullptr && ROWA != nullptr, "null pointer");
    SPH_REQUIRE(K == 0 || ROWB != nullptr, "null pointer");
    hipStream_t stream = sph::CurrentStream();
    if (stream == nullptr)
        return SPH_ERR_DEVICE;
    SpgemmArgs args{};
    args.VA = VA;
    args.COLA = COLA;
    args.ROWA = ROWA;
    args.VB = VB;
    args.COLB = COLB;
    args.ROWB = ROWB;
    args.M = M;
    args.K = K;
    args.N = N;
    args.strip = StripFor(N);
    args.rowsPerTurn = RowsPerTurnFor(M);
    args.ROWC = ROWC;
    args.VC = VC;
    args.COLC = COLC;
    args.capacity = 0xffffffffu;
    args.lightProducts = LightProductsFor(N, 0);
    args.heavyOnly = args.lightProducts != 0 ? 1u : 0u;
    LaunchFill(args, stream);
    SPH_CHECK_LAUNCH();
    return SPH_OK;
}

int sph_spgemm_load_u32(uint32_t* load, const uint32_t* COLA, const uint32_t* ROWB,
                        uint32_t entries, uint32_t K, uint64_t* productsHost)
{
    SPH_REQUIRE(entries == 0 || COLA != nullptr, "COLA is null");
    SPH_REQUIRE(entries == 0 || K == 0 || ROWB != nullptr, "ROWB is null");
    if (productsHost != nullptr)
        SPH_REFUSE_WHILE_CAPTURING();  // reads back and takes a scratch word
    hipStream_t stream = sph::CurrentStream();
    if (stream == nullptr)
        return SPH_ERR_DEVICE;
    if (entries == 0)
    {
        if (productsHost != nullptr)
            *productsHost = 0;
        return SPH_OK;
    }
    unsigned long long* total = nullptr;
    if (productsHost != nullptr)
    {
        const int taken = sph::AllocScratch(reinterpret_cast<void**>(&total),
                                            sizeof(*total), stream);
        if (taken != SPH_OK)
            return taken;
        hipLaunchKernelGGL(ClearTotalKernel, dim3(1), dim3(1), 0, stream, total);
    }
    const uint32_t blocks = static_cast<uint32_t>(std::min<uint64_t>(
        (static_cast<uint64_t>(entries) + 255) / 256, static_cast<uint64_t>(sph::ComputeUnits()) * 8));
    hipLaunchKernelGGL(SpgemmLoadKernel, dim3(blocks), dim3(256), 0, stream, load, COLA, ROWB,
                       entries, K, total);
    const hipError_t launched = hipGetLastError();
    hipError_t copied = hipSuccess;
    if (launched == hipSuccess && productsHost != nullptr)
    {
        static_assert(sizeof(unsigned long long) == sizeof(uint64_t), "64-bit total");
        copied = hipMemcpyAsync(productsHost, total, sizeof(uint64_t), hipMemcpyDeviceToHost, stream);
        if (copied == hipSuccess)
            copied = hipStreamSynchronize(stream);
    }
    if (total != nullptr)
        SPH_HIP_TRY(hipFreeAsync(total, stream));
    if (launched != hipSuccess)
        return sph::Fail(SPH_ERR_DEVICE, std::string("sph_spgemm_load_u32 - launch failed with ") +
                                             hipGetErrorString(launched));
    SPH_HIP_TRY(copied);
    return SPH_OK;
}

int sph_spgemm_f32(float* VC, uint32_t* COLC, uint32_t* ROWC, uint32_t capacity, const float* VA,
                   const uint32_t* COLA, const uint32_t* ROWA, const float* VB,
                   const uint32_t* COLB, const uint32_t* ROWB, uint32_t M, uint32_t K, uint32_t N,
                   uint32_t* nnzHost)
{
    SPH_REQUIRE(ROWC != nullptr && ROWA != nullptr, "null pointer");
    SPH_REQUIRE(M < 0xffffffffu, "too many rows");
    SPH_REQUIRE(K == 0 || ROWB != nullptr, "null pointer");
    SPH_REQUIRE(capacity == 0 || (VC != nullptr && COLC != nullptr), "VC or COLC is null");
    SPH_REFUSE_WHILE_CAPTURING();  // takes a scratch allocation; before anything is enqueued
    hipStream_t stream = sph::CurrentStream();
    if (stream == nullptr)
        return SPH_ERR_DEVICE;
    SpgemmArgs args{};
    args.VA = VA;
    args.COLA = COLA;
    args.ROWA = ROWA;
    args.VB = VB;
    args.COLB = COLB;
    args.ROWB = ROWB;
    args.M = M;
    args.K = K;
    args.N = N;
    args.strip = StripFor(N);
    args.rowsPerTurn = RowsPerTurnFor(M);
    args.counts = ROWC;
    args.lightProducts = LightProductsFor(N, M != 0 ? capacity / M : 0);
    args.heavyOnly = args.lightProducts != 0 ? 1u : 0u;

    // staging: counts (16-byte aligned, when the move scans them), values, columns, one flag
    const size_t counts = M <= sph::kPlaceMaxRows ? (static_cast<size_t>(M) + 4) / 4 * 4 : 0;
    float* stageV = nullptr;
    int taken = SPH_OK;
    const uint32_t slot = sph::TakeStagingSlot(M, N, capacity, [&](uint32_t entries) {
        taken = sph::TakeStaging(reinterpret_cast<void**>(&stageV),
                                        counts * 4 + static_cast<size_t>(entries) * M * 8 + 4, stream);
        return taken != SPH_OK || stageV != nullptr;  // a full device: with less
    });
    if (taken != SPH_OK)
        return taken;
    const bool staged = slot != 0;
    const bool placed = staged && counts != 0;
    if (staged)
    {
        if (placed)
            args.counts = reinterpret_cast<uint32_t*>(stageV);
        args.VC = stageV + counts;
        args.COLC = reinterpret_cast<uint32_t*>(args.VC + static_cast<size_t>(slot) * M);
        args.overflow = args.COLC + static_cast<size_t>(slot) * M;
        args.slot = slot;
        LaunchCounting<kStage>(args, stream);
    }
    else
    {
        LaunchCounting<kCount>(args, stream);
    }
    hipError_t launched = hipGetLastError();
    int rc = SPH_OK;
    if (launched == hipSuccess && !placed)
        rc = sph::ExclusiveScanInPlace(ROWC, M + 1, nullptr, stream);
    if (launched == hipSuccess && rc == SPH_OK && M != 0 && N != 0 && capacity != 0)
    {
        const uint32_t rowsPerGroup = sph::PlaceRowsPerGroup(M);
        if (placed)
            hipLaunchKernelGGL(SpgemmPlaceKernel, dim3((M + rowsPerGroup - 1) / rowsPerGroup),
                               dim3(sph::kPlaceThreads), 0, stream, VC, COLC, ROWC, args.counts,
                               args.VC, args.COLC, M, rowsPerGroup, args.slot, capacity,
                               args.overflow);
        else if (staged)
            hipLaunchKernelGGL(SpgemmUnstageKernel, dim3((M + 3) / 4), dim3(256), 0, stream, VC,
                               COLC, ROWC, args.VC, args.COLC, M, args.slot, capacity,
                               args.overflow);
        // rows that did not fit their slot (all rows, without staging) are multiplied again
        args.ROWC = ROWC;
        args.VC = VC;
        args.COLC = COLC;
        args.capacity = capacity;
        args.skipUpTo = staged ? args.slot : 0u;
        // after staging this pass usually finds nothing to do (it returns at once then), so it
        // is launched with few workgroups, which walk all rows if they must: dispatching the
        // full grid of empty workgroups alone took 15 us
        if (staged)
            LaunchStrips<kFill, kOverfullRows>(args, kRedoGroups, stream);
        else
            LaunchFill(args, stream);
        launched = hipGetLastError();
    }
    const int given = stageV != nullptr ? sph::GiveStaging(stageV, stream) : SPH_OK;
    if (given != SPH_OK)
        return given;
    if (launched != hipSuccess)
        return sph::Fail(SPH_ERR_DEVICE, std::string("sph_spgemm_f32 - launch failed with ") +
                                             hipGetErrorString(launched));
    if (rc != SPH_OK)
        return rc;
    if (nnzHost != nullptr)
    {
        SPH_HIP_TRY(hipMemcpyAsync(nnzHost, ROWC + M, sizeof(uint32_t), hipMemcpyDeviceToHost,
                                   stream));
        SPH_HIP_TRY(hipStreamSynchronize(stream));
    }
    return SPH_OK;
}

}  // extern "C"
