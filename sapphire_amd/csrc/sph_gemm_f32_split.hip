// fp32 GEMM on the fp16 matrix cores, for products of many tiles.
//
// The fp32 matrix instructions make 64 flops per clock and SIMD, the fp16 ones 1024.  A value is taken
// apart into two fp16 numbers, each rounded to nearest:
//     as = a 2^n,   first = fp16(as),   second = fp16((as - first) 2^11)
// which hold it to 2^-23 of itself, and a product is first first' + 2^-11 (first second' + second first'),
// three fp16 products with fp32 sums in place of one fp32 product; second second', at most 2^-22, is
// left out.  The sums are rounded once per 16 values of k rather than once per value, so the error against
// 64 bits is smaller than that of the fp32 instructions (U(-1, 1), relative 2-norm: K = 333 1.24e-7 / 3.3e-7,
// 1024 2.1e-7 / 5.7e-7, 4096 4.1e-7 / 11.5e-7; with sums in four parts the latter have 2.9e-7 at 1000).
//
// What fp16 lacks is range: 30 binades.  So that no value loses any of its bits
//   * the 32 rows (columns) that a wavefront takes apart share the scale 2^n, which brings the largest of
//     them so far to 2^13 .. 2^15.  When a larger one comes n drops, and the wavefronts that multiply
//     these rows scale their sums down likewise (exactly: powers of two, and by 2^60 at most);
//   * a value below 2^-14 of that scale is left out of the planes; its block of 4 x 4 goes on a list, and
//     what is on it is added to the sums by fp32 multiply-adds at the end (about one tile in a hundred
//     of normally distributed operands has such a value);
//   * a tile whose list overflows, whose scale drops by more than 2^30, or in which a value or a sum is not
//     finite starts again on the fp32 matrix instructions, at the step where that is found out (a NaN
//     shows only in the sums).
//
// One workgroup of 8 wavefronts (2 x 4, 64 x 32 each) per 128 x 128 tile, 32 values of k per step: raw
// values travel global -> registers two steps ahead, are looked over (largest, smallest), taken apart
// and written to one of two LDS stages while the matrix cores work on the other; one barrier per step.
// Every value is taken apart once per tile it takes part in, about 6 vector instructions, and they bound
// the loop beside the LDS: per step and SIMD 232 vector instructions and 24 of the matrix cores, 2000
// clocks (the matrix cores alone 770, everything but the split 940).
//   4096^3 920 -> 545 us (252 TFLOP/s), 2048^3 125 -> 69, 3001 x 2687 x 1000 133 -> 88, 16 x 512^3 36 -> 26.
// Where such tiles leave too many compute units idle, the 8 wavefronts take a 64 x 64 tile as two teams
// (2 x 2, 32 x 32 each): each has 32 values of k of the 64 of a step, and their sums are added up at the
// end.  A step takes 1600 clocks, 12 instructions of the matrix cores per SIMD among as many vector ones.
//   1024^3 18.7 -> 17.3 us (relative error 5.7e-7 -> 1.6e-7), 1024 x 1024 x 4096 63 -> 54; 5 us of these do
//   not depend on K, 3 of them up to the first step: code comes from memory as it is first run.
// Operands that do not fit the planes: 2048^3 125 -> 150 us, 4096^3 920 -> 1110 (exponents spread over 60
// binades, an infinity in every row).
// Tried: 64 x 64 tiles by one team (1024^3 23 us, on the fp32 kernels 19), by three (19.3: spills where the
// operands are stored in two ways, no faster where they are not) and four (83); 4 wavefronts of 64 x 64
// (4096^3 660: one wavefront per SIMD waits out every barrier); three bf16 parts and six products, which need
// no scale (4096^3 780: the energy of twice the products).
#include "sph_gemm_f32.h"

#include <algorithm>
#include <type_traits>

namespace
{
using sph::floatx16;
using sph::floatx4;
using sph::floatx4a4;
using sph::GemmF32Args;
using sph::FinishTile;
using sph::MapTile;
using sph::StoreTile;

typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef _Float16 half8v __attribute__((ext_vector_type(8)));
typedef uint32_t uintx4 __attribute__((ext_vector_type(4)));
typedef uint32_t uintx2 __attribute__((ext_vector_type(2)));

constexpr uint32_t kChunk = 32;      // values of k per step
constexpr uint32_t kGroup = 32;      // rows (columns) that one wavefront splits
constexpr uint32_t kPlane = 2048;    // bytes: 32 rows x 32 halves
constexpr uint32_t kListed = 32;

// A block of 4 rows x 4 k of A, or 4 k x 4 columns of B, with values too small for the planes: those with
// 2 |bits| - 1 < atLeast and k >= from
struct Listed
{
    uint32_t k;      // first
    uint32_t place;  // first row or column within the tile, bit 31: of B
    uint32_t from;
    uint32_t atLeast;
};

// place of 16-byte chunk c (8 halves) of row x of a group
__device__ __forceinline__ uint32_t ChunkAt(uint32_t x, uint32_t c)
{
    const uint32_t q = x / 4, r = x % 4;
    return (8 * r + q) * 64 + ((c ^ r ^ (q >> 2)) & 3u) * 16;
}

__device__ __forceinline__ floatx16 Mul(uintx4 a, uintx4 b, floatx16 c)
{
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8v, a),
                                                  __builtin_bit_cast(half8v, b), c, 0, 0, 0);
}

// max(|a|, |b|, c), in one instruction (fmaxf first quiets a NaN); a NaN counts as nothing
__device__ __forceinline__ float MaxSize(float a, float b, float c)
{
    float r;
    asm("v_max3_f32 %0, |%1|, |%2|, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}

// grows with |a|; a zero is the largest
__device__ __forceinline__ uint32_t Size(float a)
{
    return (__builtin_bit_cast(uint32_t, a) << 1) - 1u;
}

// c - 2048 h
__device__ __forceinline__ float Rest(_Float16 h, float c)
{
    return __builtin_fmaf(static_cast<float>(h), -2048.f, c);
}

// the largest of the 64 lanes' x.  (With six shuffles the first scale of a tile took 430 clocks longer.)
__device__ __forceinline__ uint32_t LargestOfAll(uint32_t x)
{
    x = max(x, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, true)));  // row_shr:1
    x = max(x, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, true)));  // row_shr:2
    x = max(x, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, true)));  // row_shr:4
    x = max(x, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, true)));  // row_shr:8
    // (the last lane of 16 has what is the largest of them)
    return max(max(__builtin_amdgcn_readlane(x, 15), __builtin_amdgcn_readlane(x, 31)),
               max(__builtin_amdgcn_readlane(x, 47), __builtin_amdgcn_readlane(x, 63)));
}

// KS: teams of wavefronts, which take the chunks of k in turn and add up their sums at the end
// DEPTH: steps by which the loads are ahead
template <int BM, int BN, int KS, int WM, int WN, int DEPTH, bool TA, bool TB>
__global__ __launch_bounds__(KS * WM * WN * 64) void GemmF32SplitKernel(
    const GemmF32Args args)
{
    constexpr int PER = WM * WN, NW = KS * PER;
    constexpr int TM = BM / WM / 32, TN = BN / WN / 32;
    constexpr uint32_t kGroupsA = BM / kGroup, kGroupsB = BN / kGroup;
    static_assert(kGroupsA + kGroupsB == PER, "a wavefront splits one group");
    constexpr uint32_t kStage = NW * 2 * kPlane;
    __shared__ __attribute__((aligned(1024))) char lds[2 * kStage];
    struct Scale
    {
        uint32_t step;
        int n;
    };
    __shared__ Scale scaleOf[2][NW];
    __shared__ Listed list[kListed];
    // steps (+ 1) whose planes have another scale, or do not hold what they should
    struct Marks
    {
        uint32_t scale, unfit;
    };
    __shared__ Marks marks[2];
    __shared__ uint32_t listed, notFinite;

    // All that the first loads depend on is asked for at once: a line of the arguments that is first read
    // later is another trip to memory before them (700 clocks; 1024 x 784 x 1024 16.2 -> 16.0 us).  Tiles of 128
    // have no registers for it (2048^3 71.6 -> 72.1).
    if (KS > 1)
        asm volatile("" ::"s"(args.M), "s"(args.N), "s"(args.K), "s"(args.A), "s"(args.B), "s"(args.out),
                     "s"(args.entries), "s"(args.strideOut), "s"(args.strideA), "s"(args.strideB));
    uint32_t tm, tn, unit;
    if (!MapTile(args, tm, tn, unit))
        return;
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t team = wave / PER, member = wave % PER;
    const uint32_t wm = member / WN, wn = member % WN;
    const uint32_t x = lane % 32, h = lane / 32;
    const uint32_t M = args.M, N = args.N, K = args.K;
    if (threadIdx.x < 2 * NW)
        scaleOf[threadIdx.x / NW][threadIdx.x % NW].step = 0;
    if (threadIdx.x == 0)
    {
        listed = 0;
        notFinite = 0;
        marks[0] = marks[1] = { 0, 0 };
    }

    int64_t offOut, offA, offB;
    if (args.entries != nullptr)
    {
        const SphGemmEntry e = args.entries[unit];
        offOut = static_cast<int64_t>(e.outOff);
        offA = static_cast<int64_t>(e.aOff);
        offB = static_cast<int64_t>(e.bOff);
    }
    else
    {
        offOut = unit * args.strideOut;
        offA = unit * args.strideA;
        offB = unit * args.strideB;
    }
    float* __restrict__ out = args.out + offOut;
    const float* __restrict__ srcA = args.A + offA;
    const float* __restrict__ srcB = args.B + offB;
    const uint32_t lda = TA ? M : K, ldb = TB ? K : N;
    const uint32_t baseM = tm * BM, baseN = tn * BN;
    const uint32_t steps = (K + KS * kChunk - 1) / (KS * kChunk);
    // where the chunk of this team begins
    auto chunkOf = [&](uint32_t s) __attribute__((always_inline)) { return (s * KS + team) * kChunk; };

    // ---- what this wavefront splits: rows 4 q .. 4 q + 3, k 4 g .. 4 g + 3 of its group ---------------
    const bool ofA = member < kGroupsA;
    const bool kMajor = ofA ? TA : !TB;
    const uint32_t group = ofA ? member : member - kGroupsA;
    const uint32_t p8 = lane / 8;
    const uint32_t q = kMajor ? lane % 8 : p8;
    const uint32_t g = kMajor ? (p8 & 1) | (p8 & 2) << 1 | (p8 & 4) >> 1 : lane % 8;
    const uint32_t first = (ofA ? baseM : baseN) + group * kGroup, limit = ofA ? M : N;
    const uint32_t ld = ofA ? lda : ldb;
    const size_t perK = kMajor ? static_cast<size_t>(ld) * 4 : 4;
    const char* src;  // of k = 0
    uint32_t off[4];  // bytes
    const uint32_t start = min(first, limit - 4);
    // K-major, a quad that the edge cuts: the last 4 that exist, `cut` earlier.  Each goes to its own row of
    // the planes all the same, and those that another quad has too to the rows past the edge.  (Put in their
    // places in the registers, at every step, 2048 x 2045 x 2048 took 88 us, this 72.)
    uint32_t cut = 0;
    // (of a group with fewer than 4 that exist: the first ones are another group's, and no matter of this scale)
    const uint32_t strays = kMajor && limit < first + 4 ? min(first + 4 - limit, 4u) : 0;
    if (kMajor)
    {
        const uint32_t row = first + 4 * q, from = min(row, limit - 4);
        cut = row < limit ? row - from : 0;
        src = reinterpret_cast<const char*>((ofA ? srcA : srcB) + start);
#pragma unroll
        for (uint32_t e = 0; e < 4; ++e)
            off[e] = ((4 * g + e) * ld + from - start) * 4;
    }
    else
    {
        src = reinterpret_cast<const char*>((ofA ? srcA : srcB) + static_cast<size_t>(start) * ld);
#pragma unroll
        for (uint32_t r = 0; r < 4; ++r)
            off[r] = ((min(first + 4 * q + r, limit - 1) - start) * ld + 4 * g) * 4;
    }
    auto rowOf = [&](uint32_t r) __attribute__((always_inline)) { return 4 * q + ((r - cut) & 3u); };

    auto load = [&](floatx4 (&raw)[4], uint32_t s) __attribute__((always_inline)) {
        // (steps past the last copy it again: a load that may not be there makes every wait one for all)
        const char* base = src + min(chunkOf(s), K - kChunk) * perK;
        // (made opaque, or the compiler adds them up as 64-bit addresses: 2048^3 71.4 -> 69.2 us)
        asm("" : "+v"(off[0]), "+v"(off[1]), "+v"(off[2]), "+v"(off[3]));
#pragma unroll
        for (int n = 0; n < 4; ++n)
            raw[n] = *reinterpret_cast<const floatx4a4*>(base + off[n]);
    };

    // ---- the split ----------------------------------------------------------
    // as = a 2^n, first = fp16(as), second = fp16((as - first) 2^11)
    int n = 0, firstN = 0;
    float s0 = 1.f, s11 = 2048.f;       // 2^n, 2^(n + 11)
    float atMost = 1e-45f;              // |a| below it fits (no scale yet: only zeros)
    uint32_t atLeast = 0;               // 2 |bits| - 1 from it on is held to the last bit
    bool scaled = false;
    using KMajorA = std::integral_constant<bool, TA>;
    using KMajorB = std::integral_constant<bool, !TB>;
    auto at = [](auto kMajorTag, const floatx4 (&raw)[4], int r, int e) __attribute__((always_inline)) -> float {
        return decltype(kMajorTag)::value ? raw[e][r] : raw[r][e];
    };
    auto put = [](auto kMajorTag, floatx4 (&raw)[4], int r, int e, float v) __attribute__((always_inline)) {
        if (decltype(kMajorTag)::value)
            raw[e][r] = v;
        else
            raw[r][e] = v;
    };
    // what a wavefront has is one operand's: one form of it where both are stored alike
    auto stored = [&](auto&& f) __attribute__((always_inline)) {
        if (TA == !TB)
            f(KMajorA{});
        else if (ofA)
            f(KMajorA{});
        else
            f(KMajorB{});
    };
    // whether value r of this lane's is of a row that exists, and no other lane's
    auto exists = [&](auto kMajorTag, uint32_t r) __attribute__((always_inline)) {
        const uint32_t row = first + 4 * q;
        return decltype(kMajorTag)::value ? r >= cut && row < limit : row + r < limit;
    };
    auto rare = [&](auto kMajorTag, floatx4 (&raw)[4], uint32_t s, float most, uint32_t least)
                    __attribute__((always_inline)) {
        if (__ballot(most >= atMost) != 0)
        {
            const int e = static_cast<int>(LargestOfAll(__builtin_bit_cast(uint32_t, most)) >> 23);
            n = min(140 - min(max(e, 1), 254), 110);
            if (!scaled)
                firstN = n;
            scaled = true;
            if ((firstN - n > 30 || e == 255) && first < limit && lane == 0)
                marks[s % 2].unfit = s + 1;
            s0 = __builtin_bit_cast(float, static_cast<uint32_t>(127 + n) << 23);
            s11 = s0 * 2048.f;
            const float inverse = __builtin_bit_cast(float, static_cast<uint32_t>(127 - n) << 23);
            atMost = inverse * 32768.f;
            atLeast = (__builtin_bit_cast(uint32_t, inverse * 0x1p-14f) << 1) - 1u;
            if (lane == 0)
            {
                marks[s % 2].scale = s + 1;
                scaleOf[s % 2][wave] = { s + 1, n };
            }
        }
        if (__ballot(least < atLeast) == 0)
            return;
        bool any = false;
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int e = 0; e < 4; ++e)
            {
                const float a = at(kMajorTag, raw, r, e);
                const bool small = Size(a) < atLeast;
                put(kMajorTag, raw, r, e, small ? 0.f : a);
                any |= small && exists(kMajorTag, r);
            }
        if (any)
        {
            const uint32_t slot = atomicAdd(&listed, 1u);
            if (slot < kListed)
                list[slot] = { min(chunkOf(s), K - kChunk) + 4 * g,
                               group * kGroup + 4 * q + (ofA ? 0u : 1u << 31), chunkOf(s), atLeast };
            else
                marks[s % 2].unfit = s + 1;
        }
    };
    // puts right what is at an edge
    auto mend = [&](auto kMajorTag, floatx4 (&raw)[4], uint32_t s) __attribute__((always_inline)) {
        const uint32_t end = chunkOf(s) + kChunk;
        if (decltype(kMajorTag)::value && strays != 0)
#pragma unroll
            for (uint32_t r = 0; r < 4; ++r)
                if (r < strays)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        raw[e][r] = 0.f;
        if (end <= K)
            return;
        // the last chunk ends with K: what the one before it has had counts as zero (all of one past the last)
        const uint32_t had = end - K;
#pragma unroll
        for (uint32_t e = 0; e < 4; ++e)
            if (4 * g + e < had)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    put(kMajorTag, raw, r, e, 0.f);
    };
    // looks whether the values fit the scale
    auto check = [&](auto kMajorTag, floatx4 (&raw)[4], uint32_t s) __attribute__((always_inline)) {
        mend(kMajorTag, raw, s);
        float mostOf[4];
        uint32_t leastOf[4];
#pragma unroll
        for (int r = 0; r < 4; ++r)
        {
            float v[4];
            uint32_t u[4];
#pragma unroll
            for (int e = 0; e < 4; ++e)
            {
                v[e] = at(kMajorTag, raw, r, e);
                u[e] = Size(v[e]);
            }
            mostOf[r] = MaxSize(v[0], v[1], MaxSize(v[2], v[3], 0.f));
            leastOf[r] = min(min(min(u[0], u[1]), u[2]), u[3]);
        }
        const float most = MaxSize(mostOf[0], mostOf[1], MaxSize(mostOf[2], mostOf[3], 0.f));
        const uint32_t least = min(min(leastOf[0], leastOf[1]), min(leastOf[2], leastOf[3]));
        if (__ballot((most >= atMost) | (least < atLeast)) != 0)
            rare(kMajorTag, raw, s, most, least);
    };
    auto convert = [&](auto kMajorTag, const floatx4 (&raw)[4], uint32_t parity) __attribute__((always_inline)) {
        char* to = lds + parity * kStage + wave * 2 * kPlane;
#pragma unroll
        for (int r = 0; r < 4; ++r)
        {
            uintx2 high, low;
#pragma unroll
            for (int t = 0; t < 2; ++t)
            {
                const float a = at(kMajorTag, raw, r, 2 * t), b = at(kMajorTag, raw, r, 2 * t + 1);
                const half2v pair = __builtin_convertvector((floatx2{ a * s0, b * s0 }), half2v);
                high[t] = __builtin_bit_cast(uint32_t, pair);
                low[t] = __builtin_bit_cast(
                    uint32_t, __builtin_convertvector(
                                  (floatx2{ Rest(pair[0], a * s11), Rest(pair[1], b * s11) }), half2v));
            }
            char* place = to + ChunkAt(rowOf(r), g / 2) + g % 2 * 8;
            *reinterpret_cast<uintx2*>(place) = high;
            *reinterpret_cast<uintx2*>(place + kPlane) = low;
        }
    };
    auto publish = []() __attribute__((always_inline)) { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

    // ---- products -----------------------------------------------------------
    floatx16 acc[TM][TN], low[TM][TN];
    int nA[TM], nB[TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
        {
            acc[i][j] = floatx16{};
            low[i][j] = floatx16{};
        }
#pragma unroll
    for (int i = 0; i < TM; ++i)
        nA[i] = 0;
#pragma unroll
    for (int j = 0; j < TN; ++j)
        nB[j] = 0;
    const uint32_t fragment = ChunkAt(x, h);
    const char* planesA = lds + (team * PER + wm * TM) * 2 * kPlane;
    const char* planesB = lds + (team * PER + kGroupsA + wn * TN) * 2 * kPlane;

    auto rescale = [&](uint32_t s) __attribute__((always_inline)) {
        int a[TM], b[TN];
#pragma unroll
        for (int i = 0; i < TM; ++i)
        {
            const Scale c = scaleOf[s % 2][team * PER + wm * TM + i];
            a[i] = __builtin_amdgcn_readfirstlane(c.step == s + 1 ? c.n : nA[i]);
        }
#pragma unroll
        for (int j = 0; j < TN; ++j)
        {
            const Scale c = scaleOf[s % 2][team * PER + kGroupsA + wn * TN + j];
            b[j] = __builtin_amdgcn_readfirstlane(c.step == s + 1 ? c.n : nB[j]);
        }
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v)
                {
                    const int d = a[i] - nA[i] + b[j] - nB[j];
                    acc[i][j][v] = __builtin_amdgcn_ldexpf(acc[i][j][v], d);
                    low[i][j][v] = __builtin_amdgcn_ldexpf(low[i][j][v], d);
                }
#pragma unroll
        for (int i = 0; i < TM; ++i)
            nA[i] = a[i];
#pragma unroll
        for (int j = 0; j < TN; ++j)
            nB[j] = b[j];
    };
    struct Fragments
    {
        uintx4 a[TM][2], b[TN][2];
    };
    auto read = [&](Fragments& f, uint32_t parity, uint32_t t) __attribute__((always_inline)) {
        const uint32_t at = parity * kStage + (fragment ^ (32 * t));
#pragma unroll
        for (int p = 0; p < 2; ++p)
        {
#pragma unroll
            for (int i = 0; i < TM; ++i)
                f.a[i][p] = *reinterpret_cast<const uintx4*>(planesA + at + (2 * i + p) * kPlane);
#pragma unroll
            for (int j = 0; j < TN; ++j)
                f.b[j][p] = *reinterpret_cast<const uintx4*>(planesB + at + (2 * j + p) * kPlane);
        }
    };
    auto multiply = [&](const Fragments& f) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
                low[i][j] = Mul(f.b[j][1], f.a[i][0], low[i][j]);
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
                acc[i][j] = Mul(f.b[j][0], f.a[i][0], acc[i][j]);
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
                low[i][j] = Mul(f.b[j][0], f.a[i][1], low[i][j]);
    };

    const uint32_t rowBase = baseM + wm * TM * 32, colBase = baseN + wn * TN * 32;
    static_assert(KS > 1 || (TM == DEPTH && TN == 1), "the old values of block i fit raw[i]");
    const bool early = KS == 1 && args.overwrite == 0 && args.bias == nullptr && baseM + BM <= M && baseN + BN <= N;
    const float* oldAt = out + static_cast<size_t>(rowBase + x) * args.ldc + colBase + 4 * h;

    floatx4 raw[DEPTH][4];
#pragma unroll
    for (uint32_t d = 0; d < DEPTH; ++d)
        load(raw[d], d);
    publish();  // listed, marks
    stored([&](auto tag) __attribute__((always_inline)) {
        check(tag, raw[0], 0);
        convert(tag, raw[0], 0);
    });
    load(raw[0], DEPTH);
    publish();
    auto step = [&](auto kMajorTag, uint32_t s, uint32_t parity, floatx4 (&next)[4])
                    __attribute__((always_inline)) {
        Fragments f0, f1;
        read(f0, parity, 0);
        const Marks mark = marks[parity];
        read(f1, parity, 1);
        check(kMajorTag, next, s + 1);
        if (__builtin_amdgcn_readfirstlane(mark.scale) == s + 1)
            rescale(s);
        convert(kMajorTag, next, 1 - parity);
        multiply(f0);
        multiply(f1);
        // (few matrix instructions start later: their operands are under way when the barrier is passed)
        constexpr bool kFew = TM * TN == 1;
        if (kFew)
            __builtin_amdgcn_sched_group_barrier(0x2, 24, 0);
#pragma unroll
        for (int n = 0; n < 6 * TM * TN; ++n)
        {
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x2, kFew ? 8 : 5, 0);
        }
        // The last two of these steps have nothing more to load and ask for what a whole tile is added to:
        // with one workgroup per compute unit nothing else runs beside the round trip (16 x 512^3 26.8 ->
        // 25.8 us, 2048^3 71.4 -> 69.4).
        if (s + 1 + DEPTH < steps || !early)
            load(next, s + 1 + DEPTH);
        else
#pragma unroll
            for (uint32_t q = 0; q < 4; ++q)
                next[q] = *reinterpret_cast<const floatx4a4*>(
                    oldAt + (1 - parity) * 32 * static_cast<size_t>(args.ldc) + 8 * q);
        publish();
        return __builtin_amdgcn_readfirstlane(mark.unfit) == s + 1;
    };
    bool unfit = false;  // the same for all wavefronts, which read it behind the same barrier
    stored([&](auto tag) __attribute__((always_inline)) {
        for (uint32_t s = 0;; s += DEPTH)
#pragma unroll
            for (uint32_t d = 0; d < DEPTH; ++d)
            {
                if (s + d + 1 >= steps)
                    return;
                unfit = step(tag, s + d, d % 2, raw[(d + 1) % DEPTH]);
                if (unfit)
                    return;
            }
    });
    if (!unfit)
    {
        const uint32_t s = steps - 1;
        Fragments f0, f1;
        read(f0, s % 2, 0);
        const Marks mark = marks[s % 2];
        read(f1, s % 2, 1);
        if (__builtin_amdgcn_readfirstlane(mark.scale) == s + 1)
            rescale(s);
        multiply(f0);
        multiply(f1);
        unfit = __builtin_amdgcn_readfirstlane(mark.unfit) == s + 1;
    }

    // ---- what the planes could not hold ----------------------------------------
    float finite = 0.f;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v)
            {
                const float sum = __builtin_fmaf(low[i][j][v], 1.f / 2048.f, acc[i][j][v]);
                finite = __builtin_fmaf(sum, 0.f, finite);
                acc[i][j][v] = __builtin_amdgcn_ldexpf(sum, -(nA[i] + nB[j]));
            }
    if (!unfit)
    {
        if (__ballot(finite != 0.f) != 0 && lane == 0)
            notFinite = 1;
        publish();
        unfit = __builtin_amdgcn_readfirstlane(notFinite) != 0;
    }
    const uint32_t count = __builtin_amdgcn_readfirstlane(listed);
    if (!unfit && count > 1)
    {
        // in an order that does not depend on who came first
        if (threadIdx.x < count)
        {
            const Listed mine = list[threadIdx.x];
            auto key = [](const Listed& e) {
                return static_cast<uint64_t>(e.from) << 32 | e.place;
            };
            uint32_t rank = 0;
            for (uint32_t o = 0; o < count; ++o)
            {
                const Listed e = list[o];
                rank += e.k < mine.k || (e.k == mine.k && key(e) < key(mine));
            }
            list[rank] = mine;  // (one wavefront: all have read)
        }
        publish();
    }
    if (unfit)
    {
        // The same loop with the values as they are, on the fp32 matrix cores.  A stage holds 32 rows of 32
        // floats per group, chunk c of row x at c ^ (x / 2 % 8).
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
                acc[i][j] = floatx16{};
        load(raw[0], 0);
        publish();  // everyone has left the loop above
        stored([&](auto tag) __attribute__((always_inline)) {
            for (uint32_t s = 0; s < steps; ++s)
            {
                char* stage = lds + s % 2 * kStage;
                mend(tag, raw[0], s);
#pragma unroll
                for (int r = 0; r < 4; ++r)
                {
                    const uint32_t row = rowOf(r);
                    *reinterpret_cast<floatx4*>(stage + wave * 2 * kPlane + row * 128 +
                                                (g ^ (row / 2 % 8)) * 16) =
                        floatx4{ at(tag, raw[0], r, 0), at(tag, raw[0], r, 1), at(tag, raw[0], r, 2),
                                 at(tag, raw[0], r, 3) };
                }
                load(raw[0], s + 1);
                publish();
#pragma unroll
                for (uint32_t u = 0; u < 4; ++u)
                {
                    const uint32_t chunk = x * 128 + ((2 * u + h) ^ (x / 2 % 8)) * 16;
                    floatx4 a[TM], b[TN];
#pragma unroll
                    for (int i = 0; i < TM; ++i)
                        a[i] = *reinterpret_cast<const floatx4*>(stage + (team * PER + wm * TM + i) * 2 * kPlane +
                                                                 chunk);
#pragma unroll
                    for (int j = 0; j < TN; ++j)
                        b[j] = *reinterpret_cast<const floatx4*>(
                            stage + (team * PER + kGroupsA + wn * TN + j) * 2 * kPlane + chunk);
#pragma unroll
                    for (int e = 0; e < 4; ++e)
#pragma unroll
                        for (int i = 0; i < TM; ++i)
#pragma unroll
                            for (int j = 0; j < TN; ++j)
                                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(
                                    b[j][e], a[i][e], acc[i][j], 0, 0, 0);
                }
            }
        });
    }
    if (KS > 1)
    {
        // the first team adds up the teams' sums, in their order
        static_assert((KS - 1) * PER * TM * TN * 4096 <= 2 * kStage, "the sums fit the stages");
        auto place = [&](uint32_t t, int block, int q) __attribute__((always_inline)) {
            return reinterpret_cast<floatx4*>(
                lds + (((t - 1) * PER + member) * (TM * TN * 4) + block * 4 + q) * 1024 + lane * 16);
        };
        publish();  // nobody reads the stages any more
        if (team != 0)
        {
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        *place(team, i * TN + j, q) =
                            floatx4{ acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2],
                                     acc[i][j][4 * q + 3] };
        }
        publish();
        if (team != 0)
            return;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (uint32_t t = 1; t < KS; ++t)
                    {
                        const floatx4 sum = *place(t, i * TN + j, q);
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            acc[i][j][4 * q + e] += sum[e];
                    }
    }
    if (!unfit)
        // 16 values of every block, those that were left out
        for (uint32_t n = 0; n < count * 16; ++n)
        {
            const Listed e = list[n / 16];
            const uint32_t k = e.k + n % 4, place = (e.place & 0x7fffffffu) + n / 4 % 4;
            if (k < e.from)
                continue;
            if (e.place >> 31 == 0)
            {
                // + value x row k of B
                const size_t row = baseM + place;
                if (row >= M)
                    continue;
                const float a = srcA[TA ? static_cast<size_t>(k) * lda + row : row * lda + k];
                if (Size(a) >= e.atLeast)
                    continue;
#pragma unroll
                for (int i = 0; i < TM; ++i)
                    if (place == wm * TM * 32 + 32 * i + x)
#pragma unroll
                        for (int j = 0; j < TN; ++j)
#pragma unroll
                            for (uint32_t v = 0; v < 16; ++v)
                            {
                                const size_t col =
                                    min(colBase + 32 * j + 8 * (v / 4) + 4 * h + v % 4, N - 1);
                                const float b =
                                    srcB[TB ? col * ldb + k : static_cast<size_t>(k) * ldb + col];
                                acc[i][j][v] = __builtin_fmaf(a, b, acc[i][j][v]);
                            }
                continue;
            }
            // + column k of A x value, but for the rows where A's value is left out as well
            const size_t col = baseN + place;
            if (col >= N)
                continue;
            const float b = srcB[TB ? col * ldb + k : static_cast<size_t>(k) * ldb + col];
            if (Size(b) >= e.atLeast)
                continue;
#pragma unroll
            for (int i = 0; i < TM; ++i)
            {
                const uint32_t inTile = wm * TM * 32 + 32 * i + x;
                const size_t row = min(baseM + inTile, M - 1);
                float a = srcA[TA ? static_cast<size_t>(k) * lda + row : row * lda + k];
                for (uint32_t o = 0; o < count; ++o)
                    if (inTile - list[o].place < 4 && k - list[o].k < 4 && k >= list[o].from &&
                        Size(a) < list[o].atLeast)
                        a = 0.f;
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (uint32_t v = 0; v < 16; ++v)
                        if (place == wn * TN * 32 + 32 * j + 8 * (v / 4) + 4 * h + v % 4)
                            acc[i][j][v] = __builtin_fmaf(a, b, acc[i][j][v]);
            }
        }
    if (early && !unfit)
    {
        float4 old[TM * TN * 4];
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                old[i * 4 + q] = make_float4(raw[i][q][0], raw[i][q][1], raw[i][q][2], raw[i][q][3]);
        FinishTile<TM, TN>(acc, old, out, rowBase, colBase, M, N, x, h, args);
    }
    else
        StoreTile<TM, TN>(acc, out, rowBase, colBase, M, N, x, h, args);
}

template <int BM, int BN, int KS, int WM, int WN>
void LaunchAs(const GemmF32Args& args, dim3 grid, bool transA, bool transB, hipStream_t stream)
{
    auto launch = [&](auto ta, auto tb) {
        hipLaunchKernelGGL((GemmF32SplitKernel<BM, BN, KS, WM, WN, 2, decltype(ta)::value, decltype(tb)::value>),
                           grid, dim3(KS * WM * WN * 64), 0, stream, args);
    };
    if (transA && transB)
        launch(std::true_type{}, std::true_type{});
    else if (transA)
        launch(std::true_type{}, std::false_type{});
    else if (transB)
        launch(std::false_type{}, std::true_type{});
    else
        launch(std::false_type{}, std::false_type{});
}

uint64_t TilesOf(const GemmF32Args& args, uint32_t units, uint32_t edge)
{
    return static_cast<uint64_t>((args.M + edge - 1) / edge) * ((args.N + edge - 1) / edge) * units;
}

// In the unit of the other kernels' cost (107: 14.5 us per 1000 values of k; a round is one tile per compute
// unit) a round of 128 x 128 tiles costs 210, and 6.8 us that do not depend on K: the first loads, the first
// scale, reading and writing out with nothing beside it.  It replaces three rounds of 64 x 64 tiles
// (1536 x 2048 x 1024 51 -> 38 us; where it would replace two, 1501 x 1203 x 1001, both take 35).
uint64_t Cost128(const GemmF32Args& args, uint32_t units)
{
    const uint64_t cus = static_cast<uint64_t>(sph::ComputeUnits());
    return (TilesOf(args, units, 128) + cus - 1) / cus * (210 + 50000 / args.K);
}

// A round of 64 x 64 tiles by two teams costs 88, and 2.2 us more than on the fp32 matrix cores, whose
// workgroups go on from tile to tile, so that a second round costs these 3.8 us more: 1024^3 18.7 -> 17.4 us,
// 1024 x 1024 x 4096 63 -> 52, K = 900 17.6 -> 16.8, but K = 784 15.0 -> 15.6; in two rounds 1408^3 45 -> 42.6,
// 1280 x 1280 x 4096 117 -> 98, but 1100^3 (both operands transposed) 36.4 -> 37.1.
uint64_t Cost64(const GemmF32Args& args, uint32_t units)
{
    const uint64_t cus = static_cast<uint64_t>(sph::ComputeUnits());
    const uint64_t rounds = (TilesOf(args, units, 64) + cus - 1) / cus;
    return rounds * 88 + (rounds * 28000 - 12000) / args.K;
}
}  // namespace

namespace sph
{
// Below K = 320 the fixed part decides (2048 x 2048 x 320 30 -> 20 us), and a product's bits there do not
// depend on the batch.
bool SplitsF32(const GemmF32Args& args, uint32_t units, uint64_t otherCost, bool transA, bool transB)
{
    // (lane offsets of 32 rows fit 32 bits, and so do the k of chunks past the last)
    if (args.K < 320 || args.K >= (1u << 31) || args.M < 4 || args.N < 4 ||
        std::max(transA ? args.M : args.K, transB ? args.K : args.N) >= (1u << 24))
        return false;
    return std::min(Cost128(args, units), Cost64(args, units)) < otherCost;
}

int LaunchGemmF32Split(GemmF32Args args, uint32_t units, bool transA, bool transB,
                       hipStream_t stream)
{
    const bool small = Cost64(args, units) < Cost128(args, units);
    const uint32_t edge = small ? 64 : 128;
    args.tilesM = (args.M + edge - 1) / edge;
    args.tilesN = (args.N + edge - 1) / edge;
    const uint64_t blocks = TilesOf(args, units, edge);
    if (blocks >= (1ull << 31) - 8)
        return Fail(SPH_ERR_INVALID, "sph_gemm_f32 - too many tiles for one launch");
    args.tilesTotal = static_cast<uint32_t>(blocks);
    args.perXcd = (args.tilesTotal + 7) / 8;
    // one workgroup per compute unit, 32 of them on an XCD: bands of the square root
    const uint32_t together = std::min<uint32_t>(args.perXcd, 32);
    uint32_t band = 1;
    while (band * band * 4 <= together)
        band *= 2;
    args.band = std::min(band, args.tilesM);
    const dim3 grid(args.perXcd * 8);
    if (small)
        LaunchAs<64, 64, 2, 2, 2>(args, grid, transA, transB, stream);
    else
        LaunchAs<128, 128, 1, 2, 4>(args, grid, transA, transB, stream);
    SPH_CHECK_LAUNCH();
    return SPH_OK;
}
}  // namespace sph
