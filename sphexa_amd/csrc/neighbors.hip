// Neighbour search on the cornerstone octree: one wavefront per group of 64 SFC-consecutive
// targets, with the coupled smoothing-length / neighbour-count iteration.
//
// Per group the wave walks the octree once with the group's bounding box grown by the largest
// search radius 2*h_max (exact periodic box-box distance, so no cell holding a neighbour of any
// target is skipped), collecting candidate leaves in LDS; internal nodes live on an LDS stack
// popped 64 at a time, one node per lane, compacted with ballot/mbcnt. The stack is kept in the
// visiting order of the reference's per-target traversal (leaf children in octant order, then
// internal children in reverse octant order, depth first), and found leaves are swept in that
// order, so every list holds its neighbours in the reference's order. Candidate leaves that no
// target's sphere reaches are dropped (one leaf per lane stages its box, moved to the periodic
// image the group sees, in LDS; the wave reads each back as a broadcast, one ballot per leaf).
// The particles of the surviving leaves within reach of the group box are compacted into full
// tiles of 64 in a double-buffered LDS area (coalesced loads of the next window overlap the
// sweep). A tile's 64 x 64 tests are one FP32 matrix product on the matrix cores whose signs are the hits
// (tileMask); where any of them is too close to zero to be certain, and in boxes too small for one periodic
// image per leaf, the tile is tested with the reference predicate
// (domain/include/cstone/findneighbors.hpp:33-60,93,116-140): d2 = dx*dx + dy*dy + dz*dz with
// dx = x_j - x_i, periodic images folded by one box length, unfused FP64 arithmetic, keep if
// d2 < Th(4)*h_i*h_i and j != i. The lists, counts and, past ngmax, the kept first ngmax hits
// are therefore bit-identical to the CPU search; a lane shifts its entries through four registers and
// stores 16 bytes at a time (ListWriter), in the layouts of common.hpp.
//
// Measured (ms; with exact tests of every tile, hits appended tile by tile and statistics by atomics of every group, then
// this): 8M turbulence, mixed 5.2 -> 3.6, 4.1M FP64 3.1 -> 2.2, 1M 0.79 -> 0.51, 4M Evrard sphere 3.7 -> 2.8; vector
// instructions per group 21.2k -> 13.9k. Bound by the vector ALU (0.8 instructions per SIMD and four cycles at 8M) and, at four waves
// per SIMD (16 waves fill a CU's LDS and 128 registers a wave), by latency: the chains of a window's plan, loads and
// filter, and of the appends.
#include <cstring>

#include "pairs.hpp"

namespace sphx
{

namespace
{

// one wave per block: a group's search time varies with its candidates, and a block's LDS is held
// until its slowest wave ends, so single-wave blocks free their share as soon as their group is done
// (8M turbulence 5.29 -> 5.10 ms, 4M Evrard 3.59 -> 3.44 ms against 4-wave blocks)
#ifndef SPHX_SEARCH_WAVES_PER_BLOCK
#define SPHX_SEARCH_WAVES_PER_BLOCK 1
#endif
constexpr int kWavesPerBlock = SPHX_SEARCH_WAVES_PER_BLOCK;
constexpr int kStackCap      = 952;  // LDS node stack per wave (bound argued at searchGroupInto)
constexpr int kLeafCap       = 64;   // leaves per sweep of candidate leaves (one per lane)
constexpr int kBufCap        = 128;  // LDS buffer of found leaves awaiting their turn in visiting order
constexpr int kEachImage     = 64;   // image code of a leaf whose particles each have one image for the whole group
constexpr int kPerPairImage  = 65;   // image code of a leaf swept with the per-pair fold
constexpr int kNoShiftImage  = 13;   // image code of shift (0, 0, 0)

/*! Statistics of one group's search. The groups write them side by side and groupStatsKernel reduces them: with four
 * to six atomics per group on one cache line, which took about 10 ns each, a search could not get below 41 ns
 * per group in any form (8M particles, mixed: 5.16 ms with them, 3.79 without; 1M: 0.75 and 0.54). */
struct alignas(16) GroupStat
{
    double   hMax;
    uint32_t stored, maxCount, swept;
    uint16_t fails, wide, bad, targets;
};
static_assert(sizeof(GroupStat) == 32, "two 16-byte chunks per group");

struct SearchArgs
{
    const double*        x;
    const double*        y;
    const double*        z;
    const TreeNodeIndex* childOffsets;
    const TreeNodeIndex* internalToLeaf;
    const int32_t*       rankLo;    // visiting order of the reference traversal (first leaf of a node)
    const uint32_t*      childPush; // an internal node's children from last to first visited
    const uint32_t*      layout;
    const double*        centers;
    const double*        sizes;
    DevBox               box;
    double               slack; // absolute enlargement of search radii (rounding margin)
    uint32_t             first, last, ng0, ngmax;
    Groups               groups; // target groups, one wavefront each
    int                  iterateH;
    void*                nbrs;
    uint32_t*            owner;      // the targets' groups (null: consecutive groups), kNoGroup before the search
    uint32_t*            table;      // local lists: the groups' tables, tableCap entries each, then `regions` of regionCap ...
    TableInfo*           info;       // ... and where each group's lies
    uint32_t             tableCap, regionCap, region0, regions; // region0: the first region in units of 64 entries
    uint32_t*            regionsTaken;
    uint32_t*            nc;
    GroupStat*           groupStats; // per group, reduced by groupStatsKernel
    double               minLen; // shortest box length
    // fused XMass: masses, kernel table (TabPair of h's type), normalisation, output (xm or rho)
    const void*          m;
    const void*          wh;    // FP64 form: the W table
    float                sincN; // FP32 form: the sinc exponent (W evaluated directly) ...
    int                  sincInt; // ... and that exponent when it is an integer, else -1
    double               K;
    void*                xmOut;
    int                  toRho;
};

/* words from one component of the matrix operand to the next: the 16 rows and 4 components that the lanes
 * read together (tileMask) lie in 64 different banks */
constexpr int kMatStride = 68;

constexpr int kPendingTiles = 4; // swept tiles whose hits are appended together (Pending)

//! per-wave LDS: traversal stack, candidate leaves, and the double-buffered candidate tile (with the
//! candidates' masses for the fused XMass only)
template<bool Mass, bool Local>
struct WaveLds
{
    int32_t  stack[kStackCap];      // pending nodes, the first in visiting order on top
    int32_t  bufNode[kBufCap];      // found leaves ...
    int32_t  bufRank[kBufCap];      // ... and their visiting-order ranks
    double   tx[2][kWave], ty[2][kWave], tz[2][kWave];
    uint32_t tj[2][kWave]; // particle index of each staged candidate
    double   tm[2][Mass ? kWave : 1]; // its mass (fused XMass only)
    uint8_t  self[Local ? kWave : 4]; // local lists: the target's own place in the tile
    uint16_t pos[Local ? kPendingTiles * kWave : 2]; // table positions of the pending tiles' candidates (Pending)
    float    mx[Mass ? 1 : 4 * kMatStride]; // the tile's candidates as matrix operand (tileMask)
};

// sixteen waves of the search share a CU's 160 KB of LDS (the fused search + XMass, with its masses,
// holds three waves per SIMD by its registers)
static_assert(sizeof(WaveLds<false, true>) <= 160 * 1024 / 16, "search LDS must leave room for 16 waves per CU");
static_assert(sizeof(WaveLds<true, false>) <= 160 * 1024 / 12, "fused search LDS must leave room for 12 waves per CU");

//! per-target state of a lane
struct Target
{
    double   x, y, z;
    double   r2;     // exact predicate radius^2 (formed in h's type)
    double   reach2; // (2h + slack)^2, conservative radius for cell tests
    uint32_t i;
    bool     active;
};

//! A lane's appending writer into its neighbour list: entries collect in a register quad that is
//! stored (16 bytes) when full and, for the incomplete last one, by finish(). Local lists pack eight
//! 16-bit table positions into it, global lists four particle indices. Slots past the stored count
//! inside the last 16 bytes repeat the newest entry.
template<bool Local>
struct ListWriter
{
    static constexpr unsigned kRun = Local ? 8 : 4; // entries per 16 bytes

    char*    base; // the lane's slot 0
    uint32_t q0 = 0, q1 = 0, q2 = 0, q3 = 0; // the last entries, oldest first
    uint32_t swept = 0;    // candidates swept by the wave (each tested by all 64 lanes)
    // local lists (the table's members are wave-uniform)
    uint32_t slot    = 0;  // entries put
    uint32_t inTable = 0;  // particles in the group's table
    uint32_t cap     = 0;  // room in it
    uint32_t at      = 0;  // its place (TableInfo)
    bool     asked   = false; // for a region

    //! entry k = e: shifted in behind the previous ones, stored when it completes 16 bytes
    __device__ __forceinline__ void put(unsigned k, uint32_t e)
    {
        if constexpr (Local)
        {
            q0 = __builtin_amdgcn_alignbit(q1, q0, 16), q1 = __builtin_amdgcn_alignbit(q2, q1, 16);
            q2 = __builtin_amdgcn_alignbit(q3, q2, 16), q3 = __builtin_amdgcn_alignbit(e, q3, 16);
        }
        else { q0 = q1, q1 = q2, q2 = q3, q3 = e; }
        if ((k & (kRun - 1)) == kRun - 1)
        {
            // runs of all 64 lanes interleave: run r starts at r * 64 * 16 bytes
            *reinterpret_cast<uint4*>(base + size_t(k / kRun) * (kGroup * 16)) = make_uint4(q0, q1, q2, q3);
        }
    }
    //! flush after `stored` entries
    __device__ __forceinline__ void finish(unsigned stored)
    {
        const uint32_t last = Local ? q3 >> 16 : q3;
        while (stored & (kRun - 1)) { put(stored++, last); }
    }
};

//! what the search does with each stored hit besides listing it: nothing ...
struct ListOnly
{
    static constexpr bool kStageMass = false;
    static constexpr int  kBatch     = 1;
    __device__ __forceinline__ void stage(int, bool, double, double, double, double) {}
    __device__ __forceinline__ void flush() {}
};

//! ... or the XMass sum of xmassJLoop (hydro_ve/xmass_kern.hpp:51-79): m_i + sum_j m_j W(r_ij / h_i)
//! over the stored neighbours in list order, r_ij from the same separation as the pair loop
//! (minimum image, then rounded to h's type), in FP64. Hits are staged
//! kBatch at a time: their kernel values are fetched together, then accumulated in list order,
//! slots without a stored hit leaving the sum untouched (bitwise the one-at-a-time sum).
template<class Th>
struct XMassSum
{
    static constexpr bool kStageMass = true;
    static constexpr int  kBatch     = isMixed<Th> ? 1 : 2; // FP32 evaluates W, no gather to overlap
    SincKernel<Th>        kern;
    Th                    hInv;
    Acc                   rho0;
    double                w[kBatch];
    Th                    mj[kBatch];
    bool                  on[kBatch];

    __device__ __forceinline__ void stage(int u, bool stored, double dx, double dy, double dz, double m)
    {
        Th rx = Th(dx), ry = Th(dy), rz = Th(dz);
        Th d2 = rx * rx + ry * ry + rz * rz;
        on[u] = stored;
        mj[u] = Th(m);
        w[u]  = kern.template w<kAnyIndex>(kern.clamp(kern.arg(d2, kernelScale(hInv)), stored));
    }
    __device__ __forceinline__ void flush()
    {
#pragma unroll
        for (int u = 0; u < kBatch; ++u)
        {
            rho0.addIf(on[u], w[u] * double(mj[u]));
        }
    }
};

__device__ __forceinline__ uint32_t uniform(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }

//! maximum over the wave (uniform result; NaN where no lane has a number): as waveOr
__device__ __forceinline__ double waveMaxD(double v)
{
    auto step = [&](auto ctrl, auto rows) {
        const uint64_t b  = __double_as_longlong(v);
        const uint32_t lo = uint32_t(b), hi = uint32_t(b >> 32);
        const uint32_t l2 = __builtin_amdgcn_update_dpp(lo, lo, decltype(ctrl)::value, decltype(rows)::value, 0xf, false);
        const uint32_t h2 = __builtin_amdgcn_update_dpp(hi, hi, decltype(ctrl)::value, decltype(rows)::value, 0xf, false);
        v                 = fmax(v, __longlong_as_double((long long)((uint64_t(h2) << 32) | l2)));
    };
    step(std::integral_constant<int, 0x111>{}, std::integral_constant<int, 0xf>{});
    step(std::integral_constant<int, 0x112>{}, std::integral_constant<int, 0xf>{});
    step(std::integral_constant<int, 0x114>{}, std::integral_constant<int, 0xf>{});
    step(std::integral_constant<int, 0x118>{}, std::integral_constant<int, 0xf>{});
    step(std::integral_constant<int, 0x142>{}, std::integral_constant<int, 0xa>{});
    step(std::integral_constant<int, 0x143>{}, std::integral_constant<int, 0xc>{});
    const uint64_t b = __double_as_longlong(v);
    return __longlong_as_double((long long)((uint64_t(uint32_t(__builtin_amdgcn_readlane(uint32_t(b >> 32), 63))) << 32) |
                                            uint32_t(__builtin_amdgcn_readlane(uint32_t(b), 63))));
}

//! bitwise or over the wave (uniform result): row steps, then the two row broadcasts, total in lane 63
__device__ __forceinline__ uint32_t waveOr(uint32_t v)
{
    v |= __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true); // row_shr:1
    v |= __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true); // row_shr:2
    v |= __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true); // row_shr:4
    v |= __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true); // row_shr:8
    v |= __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false); // row_bcast:15
    v |= __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false); // row_bcast:31
    return __builtin_amdgcn_readlane(v, 63);
}

enum class Fold
{
    none,    // all pairs of the tile use the direct image (the fused XMass, whose tiles are all tested exactly, without three
             // subtractions a pair: 9.95 -> 9.35 ms at 8M particles, mixed, 12.2 -> 11.8 FP64)
    shifted, // one periodic image (shift a multiple of the box length, or 0) serves all pairs of the tile
    perPair  // box too small for a single image: rint fold per pair, as the reference
};

//! exact hits of the tile's n candidates (n <= 64) against the lane's target, one bit per candidate
template<Fold mode, class Lds>
__device__ __forceinline__ uint64_t exactMask(const SearchArgs& a, const Target& t, const Lds& lds, int buf, uint32_t n,
                                              const double shift[3])
{
#pragma clang fp contract(off)
    const DevBox& b  = a.box;
    const double *tx = lds.tx[buf], *ty = lds.ty[buf], *tz = lds.tz[buf];
    uint64_t      m  = 0;
    for (uint32_t c0 = 0; c0 < n; c0 += 32)
    {
        uint32_t       w  = 0;
        const uint32_t cn = uniform(min(n - c0, 32u));
#pragma unroll 4
        for (uint32_t c = 0; c < cn; ++c)
        {
            double dx = tx[c0 + c] - t.x, dy = ty[c0 + c] - t.y, dz = tz[c0 + c] - t.z;
            if constexpr (mode == Fold::shifted) { dx = dx - shift[0], dy = dy - shift[1], dz = dz - shift[2]; }
            if constexpr (mode == Fold::perPair)
            {
                dx = dx - double(b.pbc[0]) * b.len[0] * rint(dx * b.ilen[0]);
                dy = dy - double(b.pbc[1]) * b.len[1] * rint(dy * b.ilen[1]);
                dz = dz - double(b.pbc[2]) * b.len[2] * rint(dz * b.ilen[2]);
            }
            double d2 = dx * dx + dy * dy + dz * dz;
            w |= d2 < t.r2 ? (1u << c) : 0u;
        }
        m |= uint64_t(w) << c0;
    }
    return m;
}

//! separation v from the group's centre under the nearest image (kEachImage)
__device__ __forceinline__ double groupImage(const DevBox& b, int d, double v)
{
    return b.pbc[d] ? v - b.len[d] * rint(v * b.ilen[d]) : v;
}

/*! The targets of a wave as the right operand of the distance matrix (tileMask). Coordinates are relative to the
 * group's centre and scaled by a power of two so that no separation exceeds 1. */
struct TargetMatrix
{
    double origin[3]; // the group's centre
    double scale;
    bool   each;      // every candidate within reach has one image for all targets (kEachImage)
    bool   usable;    // the group's size allows the scaling
    float  b[4];      // per block of 16 targets: this lane's element, -2 t (component lane / 16) or 1
    float  diff[4];   // per block: |t|^2 - r^2 of this lane's column
};

/*! Hits of the tile's candidates as one matrix product per 16 candidates and 16 targets: with D the matrix of
 * |p - t|^2 - r^2 = [p, |p|^2] . [-2 t, 1] + (|t|^2 - r^2), v_mfma_f32_16x16x4_f32 forms 256 of its elements with K = 4,
 * and a hit is a sign bit. Element (row, column) of a product lies in lane 16 (row / 4) + column, register row % 4; the
 * rows are taken from the candidates so that a lane's 16 elements per target block are consecutive
 * candidates, and two row swaps of the wave bring each lane its own target's four runs of 16 bits.
 *
 * With all coordinates at most 1 in size the product is within 21 * 2^-24 of the exact value (rounding of the
 * coordinates 3, of |p|^2 and |t|^2 - r^2 2, of the sums 16); `close` is set when any element is within 2^-19 of zero,
 * and the tile is then tested exactly. That leaves the reference's FP64 predicate for every pair: a candidate with a
 * coordinate that is not finite, and a target whose coordinates or radius are not numbers, have no hits there and none
 * here, and groups out of the range of the scale are tested exactly throughout (TargetMatrix::usable). About 3% of
 * the tiles on a lattice are tested twice. The vector ALU spends 1.5 instructions per candidate here and 11 in
 * exactMask, where this loop was two fifths of the search. */
template<class Lds>
__device__ __forceinline__ uint64_t tileMask(const DevBox& box, Lds& lds, int buf, uint32_t n, const TargetMatrix& g,
                                             const double shift[3], bool fold, bool& close)
{
    using float4v       = float __attribute__((ext_vector_type(4)));
    const unsigned lane = laneId();
    float          p[4] = {0.0f, 0.0f, 0.0f, 4.0f}; // past the tile: far from every target
    if (lane < n)
    {
        double q[3] = {lds.tx[buf][lane] - (g.origin[0] + shift[0]), lds.ty[buf][lane] - (g.origin[1] + shift[1]),
                       lds.tz[buf][lane] - (g.origin[2] + shift[2])};
        if (fold)
        {
            for (int d = 0; d < 3; ++d)
                q[d] = groupImage(box, d, q[d]);
        }
        p[0] = float(q[0] * g.scale), p[1] = float(q[1] * g.scale), p[2] = float(q[2] * g.scale);
        p[3] = float(double(p[0]) * double(p[0]) + double(p[1]) * double(p[1]) + double(p[2]) * double(p[2]));
        if (!(p[3] < INFINITY)) { p[0] = p[1] = p[2] = 0.0f, p[3] = 4.0f; } // (the sign of a NaN would pass for a hit)
    }
#pragma unroll
    for (int k = 0; k < 4; ++k)
        lds.mx[k * kMatStride + lane] = p[k];
    __builtin_amdgcn_wave_barrier();
    // row 4 q + i of block a is candidate 16 q + 4 a + i
    const float* src = lds.mx + (lane / 16) * kMatStride + 16 * ((lane % 16) / 4) + lane % 4;
    float        m[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
        m[k] = src[4 * k];
    __builtin_amdgcn_wave_barrier();
    uint32_t f[4];
    float    least = 1.0f;
#pragma unroll
    for (int b = 0; b < 4; ++b)
    {
        const float4v c = {g.diff[b], g.diff[b], g.diff[b], g.diff[b]};
        uint32_t      w = 0;
#pragma unroll
        for (int k = 3; k >= 0; --k)
        {
            const float4v d = __builtin_amdgcn_mfma_f32_16x16x4f32(m[k], g.b[b], c, 0, 0, 0);
#pragma unroll
            for (int i = 3; i >= 0; --i)
                w = __builtin_amdgcn_alignbit(w, __float_as_uint(d[i]), 31);
            least = fminf(least, fminf(fabsf(d[0]), fabsf(d[1])));
            least = fminf(least, fminf(fabsf(d[2]), fabsf(d[3])));
        }
        f[b] = w;
    }
    close = ballot(!(least > 0x1p-19f)) != 0;
    // lane row q, run b  <->  lane row b, run q
    auto s0 = __builtin_amdgcn_permlane32_swap(f[0], f[2], false, false);
    auto s1 = __builtin_amdgcn_permlane32_swap(f[1], f[3], false, false);
    auto r0 = __builtin_amdgcn_permlane16_swap(s0[0], s1[0], false, false);
    auto r1 = __builtin_amdgcn_permlane16_swap(s0[1], s1[1], false, false);
    const uint64_t hits = uint64_t(r0[0] | r0[1] << 16) | uint64_t(r1[0] | r1[1] << 16) << 32;
    return n < uint32_t(kWave) ? hits & ((uint64_t(1) << n) - 1) : hits;
}

/*! Hits of up to kPendingTiles swept tiles of a group with local lists, one bit per candidate, waiting to be
 * appended together: the append runs as many rounds as the busiest lane has hits, and over four tiles that is
 * much closer to a lane's share than tile by tile (about 130 rounds for the 91 neighbours of a lattice, against 250). The
 * next entry's table position is read from LDS while the previous one is appended. A round spends about 33
 * instructions of the vector ALU (45 when each asked whether its entry still fits: search of 8M particles
 * 3.79 -> 3.60 ms) and, alone on its SIMD, a few hundred cycles. */
struct Pending
{
    uint32_t w[2 * kPendingTiles] = {}; // word i: candidates 32 i .. of lds.pos
    int      tiles                = 0;  // (uniform)

    __device__ __forceinline__ void push(uint64_t m)
    {
#pragma unroll
        for (int k = 0; k < kPendingTiles; ++k)
        {
            if (tiles == k) { w[2 * k] = uint32_t(m), w[2 * k + 1] = uint32_t(m >> 32); }
        }
        ++tiles;
    }

    //! `count`: the lane's hits so far, of which out.slot are in its list
    template<class Writer>
    __device__ __forceinline__ void drain(const uint16_t* pos, unsigned ngmax, unsigned count, Writer& out)
    {
        uint32_t slot = out.slot, left = min(count, ngmax) - slot;
        auto     next = [&]() {
#pragma unroll
            for (int i = 0; i + 1 < 2 * kPendingTiles; ++i)
                w[i] = w[i + 1];
            w[2 * kPendingTiles - 1] = 0;
            pos += 32;
        };
        auto take = [&]() {
            const uint32_t e = pos[__builtin_ctz(w[0])];
            w[0] &= w[0] - 1;
            return e;
        };
        if (left)
        {
            while (w[0] == 0) { next(); }
            uint32_t e = take(); // on its way from LDS while the one before it is put
            while (--left)
            {
                asm volatile("" : "+v"(w[0])); // (one word per round: the lanes with hits don't wait for the others)
                if (w[0] == 0) { next(); }
                if (w[0] == 0)
                {
                    ++left; // an empty word: the lane sits this round out
                    continue;
                }
                const uint32_t after = take();
                out.put(slot++, e);
                e = after;
            }
            out.put(slot++, e);
        }
        out.slot = slot;
#pragma unroll
        for (int i = 0; i < 2 * kPendingTiles; ++i)
            w[i] = 0;
        tiles = 0;
    }
};

//! a group's table outgrows its place: it moves to a region, if one is left (else the search stores global lists)
template<class Writer>
__device__ __forceinline__ void moveTable(const SearchArgs& a, Writer& out)
{
    uint32_t r = 0;
    if (laneId() == 0) { r = atomicAdd(a.regionsTaken, 1u); }
    r         = uniform(r);
    out.asked = true;
    if (r >= a.regions) { return; }
    const uint32_t  at  = a.region0 + r * (a.regionCap / 64);
    const uint32_t* src = a.table + size_t(out.at) * 64;
    uint32_t*       dst = a.table + size_t(at) * 64;
    __threadfence_block(); // the entries other lanes stored
    for (uint32_t q = laneId(); q < out.inTable; q += kWave)
        dst[q] = src[q];
    out.at = at, out.cap = a.regionCap;
}

/* Sweep the tile's n candidates: their hits as one bit per candidate and target (a tile holds at most 64), appended
 * afterwards in candidate order, so that each list keeps the traversal order while the tests stay free of the
 * divergent append.
 * Local lists: a target's own bit is cleared (a lane finds its place through `self`), the candidates
 * that some target keeps take the next positions of the group's table, and the hits wait in `pending`. A target whose list
 * is full only counts. */
template<bool Local, class Sink, class Lds>
__device__ __forceinline__ void sweepTile(const SearchArgs& a, const Target& t, Lds& lds, const TargetMatrix& g, int buf,
                                          uint32_t n, int code, const double shift[3], unsigned& count,
                                          ListWriter<Local>& out, Pending& pending, double (&next)[3], Sink& sink)
{
    const unsigned ngmax   = a.ngmax;
    const bool     perPair = code >= kEachImage; // the exact tests fold each pair as the reference
    uint32_t*      tj      = lds.tj[buf];
    uint64_t       m       = 0;
    bool           exact   = true;
    if constexpr (!Sink::kStageMass)
    {
        if (code != kPerPairImage && g.usable) { m = tileMask(a.box, lds, buf, n, g, shift, code == kEachImage, exact); }
    }
    if (Sink::kStageMass && code == kNoShiftImage) { m = exactMask<Fold::none>(a, t, lds, buf, n, shift); }
    else if (exact)
    {
        m = perPair ? exactMask<Fold::perPair>(a, t, lds, buf, n, shift)
                    : exactMask<Fold::shifted>(a, t, lds, buf, n, shift);
    }
    if (!t.active) { m = 0; }
    // the next window's particles arrive before the stores below go out: loads and stores return in order, and
    // waiting for them later would wait for the stores too
#pragma unroll
    for (int d = 0; d < 3; ++d)
        asm volatile("" : "+v"(next[d]));
    if constexpr (Local)
    {
        const unsigned lane = laneId();
        const uint32_t j    = lane < n ? tj[lane] : 0xffffffffu;
        // the wave's targets are consecutive particles from lane 0's on
        const uint32_t rel = j - (t.i - lane);
        if (ballot(rel < uint32_t(kWave)))
        {
            lds.self[lane] = uint8_t(kWave);
            __builtin_amdgcn_wave_barrier();
            if (rel < uint32_t(kWave)) { lds.self[rel] = uint8_t(lane); }
            __builtin_amdgcn_wave_barrier();
            const uint32_t own = lds.self[lane];
            if (own < uint32_t(kWave)) { m &= ~(uint64_t(1) << own); }
        }
        const bool full = count >= ngmax;
        count += uint32_t(__popcll(m));
        if (full) { m = 0; }
        const uint64_t used = uint64_t(waveOr(uint32_t(m))) | uint64_t(waveOr(uint32_t(m >> 32))) << 32;
        const uint32_t pos  = out.inTable + laneRank(used);
        const uint32_t size = out.inTable + uint32_t(__popcll(used));
        if (size > out.cap && !out.asked) { moveTable(a, out); }
        if ((used >> lane) & 1u)
        {
            if (pos < out.cap) { a.table[size_t(out.at) * 64 + pos] = j; }
            lds.pos[pending.tiles * kWave + lane] = uint16_t(pos);
        }
        out.inTable = size;
        pending.push(m);
        __builtin_amdgcn_wave_barrier();
        if (pending.tiles == kPendingTiles) { pending.drain(lds.pos, ngmax, count, out); }
        return;
    }
    // (global lists: as many rounds per tile as the busiest lane has hits)
    while (m)
    {
#pragma unroll
        for (int u = 0; u < Sink::kBatch; ++u)
        {
            const bool     have  = m != 0;
            const uint32_t c     = have ? uint32_t(__builtin_ctzll(m)) : 0u;
            const uint32_t j     = tj[c];
            const bool     keep  = have && j != t.i;
            const bool     store = keep && count < ngmax;
            m &= m - 1;
            if (store) { out.put(count, j); }
            count += keep ? 1u : 0u;
            if constexpr (Sink::kStageMass)
            {
#pragma clang fp contract(off)
                const DevBox& b  = a.box;
                double        dx = lds.tx[buf][c] - t.x, dy = lds.ty[buf][c] - t.y, dz = lds.tz[buf][c] - t.z;
                if (perPair)
                {
                    dx = dx - double(b.pbc[0]) * b.len[0] * rint(dx * b.ilen[0]);
                    dy = dy - double(b.pbc[1]) * b.len[1] * rint(dy * b.ilen[1]);
                    dz = dz - double(b.pbc[2]) * b.len[2] * rint(dz * b.ilen[2]);
                }
                else { dx = dx - shift[0], dy = dy - shift[1], dz = dz - shift[2]; }
                sink.stage(u, store, dx, dy, dz, lds.tm[buf][c]);
            }
        }
        sink.flush();
    }
}

//! inclusive prefix sum over the wave: sums within rows of 16, then the rows before
__device__ __forceinline__ uint32_t waveInclusiveSum(uint32_t v)
{
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true); // row_shr:1
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true); // row_shr:2
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true); // row_shr:4
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true); // row_shr:8
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false); // row_bcast:15
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false); // row_bcast:31
    return v;
}

/* Periodic image of a candidate leaf relative to the group centre: the shift by whole box lengths
 * k_d = rint((c_d - g_d) / L_d), k_d in {-1, 0, 1}, coded (k_x+1) + 3 (k_y+1) + 9 (k_z+1), which
 * serves all pairs of the leaf, unless the group, the leaf and the reach together exceed a quarter box in a
 * periodic dimension. Then, while the group and the reach stay within half a box (`each`), every candidate
 * within reach of the group still has one image that serves all targets, the one nearest to the group's centre
 * (kEachImage): a pair closer than the reach under any other would put the candidate within half a box of the centre
 * twice. Else each pair folds by itself as in the reference (kPerPairImage), without the filter by the group's box
 * and without the matrix tests: boxes a few smoothing lengths wide. With one image per candidate where it is
 * possible, the search of a periodic box of 18^3 particles with 100 neighbours takes 181 us instead of 280. */
__device__ __forceinline__ int imageCode(const DevBox& b, const double c[3], const double s[3], const double gc[3],
                                         const double ge[3], double reach, bool each)
{
    int  code    = 0;
    bool perPair = false;
    for (int d = 2; d >= 0; --d)
    {
        int k = 0;
        if (b.pbc[d])
        {
            k       = int(rint((c[d] - gc[d]) * b.ilen[d]));
            perPair = perPair || (ge[d] + s[d] + reach > 0.25 * b.len[d]);
        }
        code = 3 * code + (k + 1);
    }
    return !perPair ? code : each ? kEachImage : kPerPairImage;
}

__device__ __forceinline__ double imageShift(const DevBox& b, int code, int d)
{
    const int k = (d == 0 ? code : d == 1 ? code / 3 : code / 9) % 3 - 1;
    return double(k) * b.len[d];
}

//! sweep the first n candidates of tile buffer `buf`, all of image `code`
template<bool Local, class Sink, class Lds>
__device__ __forceinline__ void sweepBuffer(const SearchArgs& a, const Target& t, Lds& lds, const TargetMatrix& g, int buf,
                                            uint32_t n, int code, unsigned& count, ListWriter<Local>& out,
                                            Pending& pending, double (&next)[3], Sink& sink)
{
    __builtin_amdgcn_wave_barrier(); // a wave's LDS accesses complete in order
    out.swept += n;
    const bool   perPair  = code >= kEachImage;
    const double shift[3] = {perPair ? 0.0 : imageShift(a.box, code, 0), perPair ? 0.0 : imageShift(a.box, code, 1),
                             perPair ? 0.0 : imageShift(a.box, code, 2)};
    sweepTile(a, t, lds, g, buf, n, code, shift, count, out, pending, next, sink);
    __builtin_amdgcn_wave_barrier();
}

/* Sweep the buffered candidate leaves (nLeaf <= 64, traversal order).
 *
 * 1. Lane q takes leaf q: its box, particle range and periodic image load in parallel. The leaf
 *    is kept if some active target's sphere reaches its box (the box is broadcast to the wave
 *    lane by lane). Lane r then holds the r-th kept leaf in traversal order: its first particle, image
 *    and the exclusive prefix of the particle counts.
 * 2. Their particles are read as one stream, 64 per window (a window never spans two images).
 *    Each lane loads one particle and keeps it if it lies within reach of the group box under
 *    its leaf's image. Kept particles are appended, in stream order, to the tile being filled.
 *    A full tile of 64 (or the last one, or one whose image ends) is swept, while the next
 *    window's loads are in flight. The candidate order is therefore the traversal order, as in
 *    the reference. */
template<bool Local, class Sink, class Lds>
__device__ __forceinline__ void flushLeaves(const SearchArgs& a, const Target& t, Lds& lds, const TargetMatrix& g,
                            const int32_t* leaves, int nLeaf,
                            const double gc[3],
                            const double ge[3], double reach, unsigned& count, ListWriter<Local>& out,
                            Pending& pending, Sink& sink)
{
#pragma clang fp contract(off)
    const DevBox&  b    = a.box;
    const unsigned lane = laneId();

    // 1. leaf boxes, ranges and images in parallel; keep test with the box broadcast per leaf
    double   c[3] = {0, 0, 0}, sz[3] = {0, 0, 0};
    uint32_t lo = 0, cnt = 0;
    int      code = kNoShiftImage;
    if (int(lane) < nLeaf)
    {
        const int32_t node = leaves[lane];
        for (int d = 0; d < 3; ++d)
        {
            c[d]  = a.centers[3 * size_t(node) + d];
            sz[d] = a.sizes[3 * size_t(node) + d];
        }
        const uint32_t leaf = uint32_t(a.internalToLeaf[node]);
        lo                  = a.layout[leaf];
        cnt                 = a.layout[leaf + 1] - lo;
        code                = imageCode(b, c, sz, gc, ge, reach, g.each);
    }
    uint64_t keepMask = 0;
    {
        // each leaf's box, its centre moved to its image if it has one for the whole group, goes to the idle
        // tile buffers and is read back as an LDS broadcast
        const double p[3] = {t.x, t.y, t.z};
        if (int(lane) < nLeaf)
        {
            const int one      = code < kEachImage ? code : kNoShiftImage;
            lds.tx[0][lane] = c[0] - imageShift(b, one, 0), lds.tx[1][lane] = sz[0];
            lds.ty[0][lane] = c[1] - imageShift(b, one, 1), lds.ty[1][lane] = sz[1];
            lds.tz[0][lane] = c[2] - imageShift(b, one, 2), lds.tz[1][lane] = sz[2];
        }
        __builtin_amdgcn_wave_barrier();
        auto test = [&](auto fold) {
            for (int q = 0; q < nLeaf; ++q)
            {
                const double cq[3] = {lds.tx[0][q], lds.ty[0][q], lds.tz[0][q]};
                const double sq[3] = {lds.tx[1][q], lds.ty[1][q], lds.tz[1][q]};
                double       d2    = 0.0;
                for (int d = 0; d < 3; ++d)
                {
                    double v = cq[d] - p[d];
                    if constexpr (decltype(fold)::value) { v = groupImage(b, d, v); }
                    v = fabs(v) - sq[d];
                    v = v > 0.0 ? v : 0.0;
                    d2 += v * v;
                }
                keepMask |= ballot(t.active && d2 < t.reach2) ? (uint64_t(1) << q) : uint64_t(0);
            }
        };
        if (ballot(code >= kEachImage)) { test(std::true_type{}); }
        else { test(std::false_type{}); }
        __builtin_amdgcn_wave_barrier();
    }
    if (keepMask == 0) { return; }
    // lane r takes the r-th kept leaf (the others' lanes follow, empty)
    const uint64_t kept  = uint64_t(1) << lane & keepMask;
    const int      nKept = __popcll(keepMask);
    const unsigned r     = laneRank(keepMask);
    const int      to    = 4 * int(kept ? r : unsigned(nKept) + lane - r);
    lo                   = __builtin_amdgcn_ds_permute(to, int(lo));
    code                 = __builtin_amdgcn_ds_permute(to, code);
    cnt                  = __builtin_amdgcn_ds_permute(to, int(kept ? cnt : 0u));
    const uint32_t incl  = waveInclusiveSum(cnt);
    const uint32_t pre   = incl - cnt; // stream position of the leaf's first particle
    const uint32_t off   = lo - pre;
    const bool     leaf  = int(lane) < nKept;
    const uint32_t total = __builtin_amdgcn_readlane(incl, kWave - 1);
    if (total == 0) { return; }

    // 2. the kept leaves' particles as one stream of windows, compacted into full tiles
    const double reach2 = reach * reach;
    uint32_t     S      = 0;  // stream position of the current window
    uint32_t     runEnd = 0;  // stream end of the run of leaves with the current window's image
    int          runImg = kNoShiftImage;
    // plan the window at S: its end, and this lane's particle (valid, index)
    auto plan = [&](uint32_t& E, bool& valid, uint32_t& idx) {
        int q = __popcll(ballot(leaf && pre <= S)) - 1; // kept leaf holding S
        if (S >= runEnd)
        {
            runImg              = __builtin_amdgcn_readlane(code, q);
            const uint64_t past = ballot(leaf && int(lane) > q && code != runImg);
            runEnd              = past ? uint32_t(__builtin_amdgcn_readlane(pre, __builtin_ctzll(past))) : total;
        }
        E                = min(S + uint32_t(kWave), runEnd);
        const uint32_t p = S + lane;
        valid            = p < E;
        idx              = p + uint32_t(__builtin_amdgcn_readlane(off, q));
        while (++q < nKept)
        {
            const uint32_t start = __builtin_amdgcn_readlane(pre, q), o = __builtin_amdgcn_readlane(off, q);
            if (start >= E) { break; }
            idx = p >= start ? p + o : idx;
        }
    };
    double   pn[3] = {0, 0, 0}, pm = 0;
    auto     load = [&](bool valid, uint32_t idx) {
        if (valid)
        {
            pn[0] = a.x[idx], pn[1] = a.y[idx], pn[2] = a.z[idx];
            if constexpr (Sink::kStageMass) { pm = double(static_cast<const decltype(sink.hInv)*>(a.m)[idx]); }
        }
    };

    uint32_t E;
    bool     valid;
    uint32_t idx;
    plan(E, valid, idx);
    load(valid, idx);
    int      cur     = 0;             // tile buffer being filled
    uint32_t acc     = 0;             // candidates in it
    int      tileImg = runImg;        // their image
    bool     more    = true;          // a window is loaded
    while (true)
    {
        // take the loaded window, unless its image ends the tile (a tile holds one image)
        if (more && (acc == 0 || runImg == tileImg))
        {
            tileImg = runImg;
            // keep the window's particles within reach of the group box under its image
            bool keep = valid;
            if (keep && tileImg != kPerPairImage)
            {
                const int one  = tileImg < kEachImage ? tileImg : kNoShiftImage;
                double    q[3] = {pn[0] - imageShift(b, one, 0) - gc[0], pn[1] - imageShift(b, one, 1) - gc[1],
                                  pn[2] - imageShift(b, one, 2) - gc[2]};
                double    d2   = 0.0;
                if (tileImg == kEachImage)
                {
                    for (int d = 0; d < 3; ++d)
                        q[d] = groupImage(b, d, q[d]);
                }
                for (int d = 0; d < 3; ++d)
                {
                    double v = fabs(q[d]) - ge[d];
                    v        = v > 0.0 ? v : 0.0;
                    d2 += v * v;
                }
                keep = d2 < reach2;
            }
            const uint64_t kmask = ballot(keep);
            if (keep)
            {
                const uint32_t slot = acc + laneRank(kmask);
                const int      bb   = slot < uint32_t(kWave) ? cur : cur ^ 1;
                const uint32_t sl   = slot < uint32_t(kWave) ? slot : slot - kWave;
                lds.tx[bb][sl] = pn[0], lds.ty[bb][sl] = pn[1], lds.tz[bb][sl] = pn[2];
                lds.tj[bb][sl] = idx;
                if constexpr (Sink::kStageMass) { lds.tm[bb][sl] = pm; }
            }
            acc += uint32_t(__popcll(kmask));
            // next window's loads go out before the sweep
            S    = E;
            more = S < total;
            if (more)
            {
                plan(E, valid, idx);
                load(valid, idx);
            }
        }
        // a full tile, or the last one of its image
        if (acc >= uint32_t(kWave) || (acc > 0 && (!more || runImg != tileImg)))
        {
            const uint32_t n = min(acc, uint32_t(kWave));
            sweepBuffer(a, t, lds, g, cur, n, tileImg, count, out, pending, pn, sink);
            acc -= n, cur ^= 1;
        }
        if (!more && acc == 0) { break; }
    }
}

/*! Sort the first n <= 128 entries of the found-leaf buffer by rank: an entry's place is the number of smaller
 * ranks (the ranks of distinct leaves are distinct). Eight ranks at a time, past n the largest: a group whose box spans a
 * dense cluster sorts some 300 buffers on an otherwise idle SIMD, where half of a plain loop is its branch (std pass
 * over 250k particles, 90% in a ball of a thousandth of the box, mixed: 11.75 -> 11.42 ms; one over a lattice is unchanged). */
template<class Lds>
__device__ __forceinline__ void sortFoundLeaves(Lds& lds, int n)
{
    static_assert(kBufCap == 2 * kWave, "two entries per lane");
    const int  lane = int(laneId());
    const bool on0 = lane < n, on1 = lane + kWave < n;
    const int  r0 = on0 ? lds.bufRank[lane] : INT32_MAX, r1 = on1 ? lds.bufRank[lane + kWave] : INT32_MAX;
    // leaves found in one pop arrive in order: often there is nothing to sort
    const bool inversion = (lane + 1 < n && r0 > lds.bufRank[lane + 1]) ||
                           (lane + kWave + 1 < n && r1 > lds.bufRank[lane + kWave + 1]);
    if (!ballot(inversion)) { return; }
    const int node0 = on0 ? lds.bufNode[lane] : 0, node1 = on1 ? lds.bufNode[lane + kWave] : 0;
    int       at0 = 0, at1 = 0;
    auto below = [&](int mine, int count) {
        for (int q = 0; q < count; q += 8)
        {
#pragma unroll
            for (int u = 0; u < 8; ++u)
            {
                const int r = __builtin_amdgcn_readlane(mine, q + u);
                at0 += r < r0 ? 1 : 0, at1 += r < r1 ? 1 : 0;
            }
        }
    };
    below(r0, min(n, kWave));
    below(r1, n - kWave);
    __builtin_amdgcn_wave_barrier();
    if (on0) { lds.bufRank[at0] = r0, lds.bufNode[at0] = node0; }
    if (on1) { lds.bufRank[at1] = r1, lds.bufNode[at1] = node1; }
    __builtin_amdgcn_wave_barrier();
}

/* Collect all leaves whose (periodic) distance to the active targets' bounding box is below the
 * largest active search radius and sweep them in the reference's visiting order
 * (singleTraversal, traversal/traversal.hpp:52-93: at each node its leaf children in octant
 * order, then its internal children in reverse octant order, depth first), which is the order
 * of each target's list. Returns each lane's neighbour count.
 *
 * Every node carries the rank of its first leaf in that order (rankLo), and the leaves of a
 * subtree have consecutive ranks. The stack holds pending nodes sorted by rank, the first on top:
 * a pop takes the up to 64 first pending nodes (lane 0 the first), whose subtrees all precede the
 * rest of the stack, and pushes the children of the overlapping internal ones back on top in the
 * same order (childPush). Found leaves wait in an LDS buffer with their ranks; once no pending
 * node can hold an earlier leaf (rank below the top node's), they are final and are swept in rank
 * order, 64 at a time.
 *
 * Bounds: nodes are popped 64 at a time only while top + 7*64 <= kStackCap - 160 and the buffer
 * can take 64 more leaves with 8 to spare, else one at a time. A single pop takes the first
 * pending node and replaces it by at most 8 children, the next pop taking the first of them,
 * i.e. it proceeds depth first and adds at most 7 entries per tree level below the popped node
 * (<= 7*20 = 140 < 160) on top of the stack it started from. A single pop adds at most one leaf,
 * the first in order of all, and the buffer is swept whenever it reaches its spare slots. */
template<bool Local, class Sink, class Lds>
__device__ __forceinline__ unsigned searchGroupInto(const SearchArgs& a, const Target& t, double radius, Lds& lds,
                                                    ListWriter<Local>& out, Sink& sink)
{
#pragma clang fp contract(off)
    const unsigned lane = laneId();
    const DevBox&  b    = a.box;

    double gc[3], ge[3];
    double p[3] = {t.x, t.y, t.z};
    for (int d = 0; d < 3; ++d)
    {
        const double gmin = -waveMaxD(t.active ? -p[d] : -INFINITY), gmax = waveMaxD(t.active ? p[d] : -INFINITY);
        gc[d]             = 0.5 * (gmin + gmax);
        ge[d]             = 0.5 * (gmax - gmin);
    }
    double reach  = waveMaxD(t.active ? radius : 0.0) + a.slack;
    double reach2 = reach * reach;
    if (ballot(t.active) == 0) { return 0; }

    TargetMatrix g;
    g.each = true;
    for (int d = 0; d < 3; ++d)
    {
        // (below 2^-20 of the box the rounding of a coordinate would count in the matrix tests)
        const double w = ge[d] + reach;
        if (b.pbc[d]) { g.each = g.each && w * (1.0 + 1e-6) <= 0.5 * b.len[d] && w >= 0x1p-20 * b.len[d]; }
    }
    if constexpr (!Sink::kStageMass)
    {
        // every kept candidate and every target within 1 of the centre after scaling, and every separation
        const double size = 2.0 * sqrt(ge[0] * ge[0] + ge[1] * ge[1] + ge[2] * ge[2]) + reach;
        g.usable          = size > 1e-150 && size < 1e150; // (the squares of the scale and the size stay in range)
        g.scale           = g.usable ? ldexp(1.0, -(ilogb(size) + 1)) : 1.0;
        float q[3], diff;
        for (int d = 0; d < 3; ++d)
        {
            g.origin[d] = gc[d];
            q[d]        = t.active ? float((p[d] - gc[d]) * g.scale) : 0.0f;
        }
        diff = t.active ? float(double(q[0]) * double(q[0]) + double(q[1]) * double(q[1]) + double(q[2]) * double(q[2]) -
                                t.r2 * (g.scale * g.scale))
                        : 4.0f; // no hits
        if (!(fabsf(q[0]) + fabsf(q[1]) + fabsf(q[2]) < 4.0f) || diff != diff) { q[0] = q[1] = q[2] = 0.0f, diff = 4.0f; } // NaN: none
        for (int b4 = 0; b4 < 4; ++b4)
        {
            const int   col = 16 * b4 + int(lane % 16);
            const float bx = __shfl(q[0], col, kWave), by = __shfl(q[1], col, kWave), bz = __shfl(q[2], col, kWave);
            g.b[b4]        = lane < 16 ? -2.0f * bx : lane < 32 ? -2.0f * by : lane < 48 ? -2.0f * bz : 1.0f;
            g.diff[b4]     = __shfl(diff, col, kWave);
        }
    }

    unsigned count = 0;
    out.slot       = 0;
    Pending  pending;
    int      top   = 1;
    int      nBuf  = 0;
    if (lane == 0) { lds.stack[0] = 0; }
    __builtin_amdgcn_wave_barrier();

    // sweep the buffered leaves ranked below `limit`, in rank order, and keep the others
    auto sweepFound = [&](int32_t limit) {
        sortFoundLeaves(lds, nBuf);
        int final = 0;
        for (int q = 0; q < nBuf; q += kWave)
        {
            const int i = q + int(lane);
            final += __popcll(ballot(i < nBuf && lds.bufRank[i] < limit));
        }
        for (int done = 0; done < final; done += kLeafCap)
        {
            flushLeaves(a, t, lds, g, lds.bufNode + done, min(kLeafCap, final - done), gc, ge, reach, count, out,
                        pending, sink);
        }
        // move the rest to the front
        const int rest = nBuf - final;
        int32_t   n0 = 0, r0 = 0, n1 = 0, r1 = 0;
        if (int(lane) < rest) { n0 = lds.bufNode[final + lane], r0 = lds.bufRank[final + lane]; }
        if (int(lane) + kWave < rest) { n1 = lds.bufNode[final + kWave + lane], r1 = lds.bufRank[final + kWave + lane]; }
        __builtin_amdgcn_wave_barrier();
        if (int(lane) < rest) { lds.bufNode[lane] = n0, lds.bufRank[lane] = r0; }
        if (int(lane) + kWave < rest) { lds.bufNode[kWave + lane] = n1, lds.bufRank[kWave + lane] = r1; }
        __builtin_amdgcn_wave_barrier();
        nBuf = rest;
    };

    for (bool done = false; !done;)
    {
        const bool batch = top + 7 * kWave <= kStackCap - 160 && nBuf + kWave <= kBufCap - 8;
        const int  k     = batch ? min(kWave, top) : 1;
        int        node  = -1;
        if (int(lane) < k) { node = lds.stack[top - 1 - int(lane)]; }
        top -= k;
        __builtin_amdgcn_wave_barrier();

        bool     ov = false, isLeaf = false;
        int      child = 0;
        int32_t  rank  = 0;
        uint32_t push  = 0;
        if (node >= 0)
        {
            // the node's rank and child order load with its box (childPush is read for leaves too,
            // unused there)
            rank = a.rankLo[node];
            push = a.childPush[node];
            double d2 = 0.0;
            for (int d = 0; d < 3; ++d)
            {
                double v = a.centers[3 * size_t(node) + d] - gc[d];
                if (b.pbc[d]) { v = v - b.len[d] * rint(v * b.ilen[d]); }
                v = fabs(v) - a.sizes[3 * size_t(node) + d] - ge[d];
                v = v > 0.0 ? v : 0.0;
                d2 += v * v;
            }
            ov     = d2 < reach2;
            child  = a.childOffsets[node];
            isLeaf = child == 0;
        }
        const uint64_t mLeaf = ballot(ov && isLeaf);
        const uint64_t mInt  = ballot(ov && !isLeaf);
        if (ov && isLeaf)
        {
            const int pos  = nBuf + int(laneRank(mLeaf));
            lds.bufNode[pos] = node;
            lds.bufRank[pos] = rank;
        }
        if (ov && !isLeaf)
        {
            // the children of later lanes go deeper: lane 0's, the first in order, end on top
            const int later = __popcll(lane + 1 < kWave ? mInt >> (lane + 1) : uint64_t(0));
            const int pos   = top + 8 * later;
            for (int c = 0; c < 8; ++c)
                lds.stack[pos + c] = child + int((push >> (3 * c)) & 7u);
        }
        nBuf += __popcll(mLeaf);
        top += 8 * __popcll(mInt);
        __builtin_amdgcn_wave_barrier();

        // leaves ranked below the first pending node are final; all are when none is pending
        done         = top == 0;
        bool  sweep  = done;
        int32_t limit = INT32_MAX;
        if (!done && nBuf >= kLeafCap)
        {
            // the first pending node: the first visited child of the first pushed node, whose rank
            // is its parent's, or else the node left below the popped ones
            if (mInt) { limit = __builtin_amdgcn_readlane(rank, __builtin_ctzll(mInt)); }
            else { limit = a.rankLo[lds.stack[top - 1]]; }
            int           final = 0;
            for (int q = 0; q < nBuf; q += kWave)
            {
                const int i = q + int(lane);
                final += __popcll(ballot(i < nBuf && lds.bufRank[i] < limit));
            }
            sweep = final >= kLeafCap || (nBuf > kBufCap - 8 && final > 0);
        }
        if (sweep) { sweepFound(limit); }
    }
    if constexpr (Local)
    {
        if (pending.tiles) { pending.drain(lds.pos, a.ngmax, count, out); }
    }
    return count;
}

//! search of the active lanes' targets into their lists (`out` at slot 0); returns the counts
template<bool Local, class Sink, class Lds>
__device__ __forceinline__ unsigned searchGroup(const SearchArgs& a, const Target& t, double radius, Lds& lds,
                                                ListWriter<Local>& out, Sink& sink)
{
    unsigned count = searchGroupInto(a, t, radius, lds, out, sink);
    if (t.active) { out.finish(min(count, a.ngmax)); }
    return count;
}

//! updateH (sph/include/sph/kernels.hpp:27-32)
template<class Th>
__device__ __forceinline__ Th updateH(unsigned ng0, unsigned nc, Th h)
{
#pragma clang fp contract(off)
    constexpr Th c0 = 1023.0;
    constexpr Th ex = 1.0 / 10.0;
    return h * Th(0.5) * pow(Th(1) + c0 * ng0 / Th(nc), ex);
}

template<class Th>
__device__ __forceinline__ void setRadius(Target& t, Th hi, double slack)
{
#pragma clang fp contract(off)
    Th r2      = Th(4.0) * hi * hi; // radius in h's type, as the reference
    t.r2       = double(r2);
    double rr  = 2.0 * double(hi) + slack;
    t.reach2   = rr * rr;
}

/* One wave per group: search, h/nc iteration, and with XMass the fused density sum of the final
 * search, stored as xm = m / rho0 (xmassJLoop) or rho = m / xm (computeDensity,
 * hydro_std/density.hpp:42-53), with the per-target epilogue of the XMass kernel. */
// waves per SIMD the search kernel's register allocation must leave room for, per form (the
// fused XMass variant is left to the compiler)
#ifndef SPHX_WAVES_SEARCH_F32
#define SPHX_WAVES_SEARCH_F32 4
#endif
#ifndef SPHX_WAVES_SEARCH_F64
#define SPHX_WAVES_SEARCH_F64 4
#endif

template<class Th, bool XMass, bool Local>
__global__ void __launch_bounds__(kWavesPerBlock * kWave)
__attribute__((amdgpu_waves_per_eu(XMass ? 1 : isMixed<Th> ? SPHX_WAVES_SEARCH_F32 : SPHX_WAVES_SEARCH_F64)))
searchKernel(SearchArgs a, Th* __restrict__ h)
{
    static_assert(!(XMass && Local), "the fused XMass stores global lists");
    __shared__ WaveLds<XMass, Local> ldsMem[kWavesPerBlock];

    const unsigned wid  = threadIdx.x / kWave;
    const unsigned lane = laneId();
    const uint32_t g    = uniform(xcdBlock(blockIdx.x, gridDim.x) * kWavesPerBlock + wid);
    if (g >= a.groups.num) { return; }
    uint32_t base, end;
    bool     oversized;
    groupRange(a.groups, g, base, end, oversized);
    base = uniform(base), end = uniform(end);
    WaveLds<XMass, Local>& lds = ldsMem[wid];

    Target t;
    t.i      = base + lane;
    t.active = t.i < end;
    Th hi    = t.active ? h[t.i] : Th(0);
    t.x      = t.active ? a.x[t.i] : 0.0;
    t.y      = t.active ? a.y[t.i] : 0.0;
    t.z      = t.active ? a.z[t.i] : 0.0;
    // a target of two groups is the first one's alone: its list refers to one table
    if (a.owner && t.active) { t.active = atomicCAS(&a.owner[t.i - a.first], NeighborLists::kNoGroup, g) == NeighborLists::kNoGroup; }
    setRadius(t, hi, a.slack);
    // lists are indexed by particle: target i at group (i - first) / 64, lane (i - first) % 64
    const uint32_t    r = t.active ? t.i - a.first : 0u;
    ListWriter<Local> out;
    if constexpr (Local)
    {
        out.base  = static_cast<char*>(a.nbrs) + 2 * localOffset(r / kGroup, paddedNgmax8(a.ngmax), 0, r % kGroup);
        out.cap = a.tableCap, out.at = g * (a.tableCap / 64);
    }
    else { out.base = static_cast<char*>(a.nbrs) + 4 * listOffset(r / kGroup, paddedNgmax(a.ngmax), 0, r % kGroup); }

    using Sink = std::conditional_t<XMass, XMassSum<Th>, ListOnly>;
    Sink      sink;
    const Th  mi = XMass && t.active ? static_cast<const Th*>(a.m)[t.i] : Th(0);
    auto      resetSink = [&]()
    {
        if constexpr (XMass)
        {
            if constexpr (isMixed<Th>) { sink.kern.n = a.sincN, sink.kern.ni = a.sincInt; }
            else { sink.kern.wTab = static_cast<const TabPair<double>*>(a.wh); }
            sink.hInv = Th(1) / hi;
            sink.rho0 = Acc(double(mi));
        }
    };
    resetSink();

    const bool     valid   = t.active;
    unsigned       ncSph   = 1;
    int            updates = 0;
    const unsigned ngmin   = a.ng0 / 4;
    while (true)
    {
        const unsigned count = searchGroup(a, t, double(2) * double(hi), lds, out, sink);
        if (t.active) { ncSph = 1 + count; }
        if (!a.iterateH) { break; }
        const bool repeat = valid && (ngmin > ncSph || (ncSph - 1) > a.ngmax) && updates < 10;
        if (!ballot(repeat)) { break; }
        // no list refers to the table yet when every target is searched again
        if (Local && !ballot(valid && !repeat)) { out.inTable = 0; }
        if (repeat)
        {
            updates++;
            hi = updateH(a.ng0, ncSph, hi);
            setRadius(t, hi, a.slack);
            resetSink();
        }
        t.active = repeat;
    }
    if (valid)
    {
        if (updates > 0) { h[t.i] = hi; }
        a.nc[t.i] = ncSph;
        if constexpr (XMass)
        {
            // epilogue of xmassKernel: FP64 normalisation with h^-3 rounded in h's type
            const Th hInv    = Th(1) / hi;
            const Th h3Inv   = hInv * hInv * hInv;
            double   rhoZero = sink.rho0.value() * a.K * double(h3Inv);
            Th       xmi     = Th(double(mi) / rhoZero);
            static_cast<Th*>(a.xmOut)[t.i] = a.toRho ? Th(mi / xmi) : xmi;
        }
    }

    const unsigned stored = waveSum(valid ? min(ncSph - 1, a.ngmax) : 0u);
    const unsigned mx     = waveMax(valid ? ncSph : 0u);
    const unsigned fails  = __popcll(ballot(valid && updates >= 10));
    // support 2h reaching half a box length: the FP32 pair loops then take exact separations
    const unsigned wide  = __popcll(ballot(valid && 4.0 * double(hi) * (1.0 + 1e-6) >= a.minLen));
    const unsigned taken = __popcll(ballot(valid));
    // largest h: sets the fixed-point period of the FP32 pair loops
    const double hMax = waveMaxD(valid ? double(hi) : 0.0);
    if (lane == 0)
    {
        a.groupStats[g] = {hMax, stored, mx, out.swept, uint16_t(fails), uint16_t(wide), uint16_t(oversized ? 1 : 0),
                           uint16_t(taken)};
        if constexpr (Local) { a.info[g] = {out.inTable <= out.cap ? out.inTable : TableInfo::kFailed, out.at}; }
    }
}

/*! Statistics of the search from its groups': stats[0] stored pairs, [1] max count, [2] non-converged particles,
 * [kStatWide] wide support, [kStatTests] candidate distance tests (swept candidates x 64 lanes),
 * [kStatBadGroups], [kStatHMax], [kStatTargets]; with `info` also the histogram of the groups' table sizes. One
 * block's atomics per slot. */
__global__ void __launch_bounds__(256)
    groupStatsKernel(const GroupStat* __restrict__ groupStats, const TableInfo* __restrict__ info, uint32_t groups,
                     unsigned long long* __restrict__ stats)
{
    __shared__ uint32_t           part[kTableBins + 2];
    __shared__ unsigned long long sum[6], hBits;
    __shared__ uint32_t           most;
    if (threadIdx.x < kTableBins + 2) { part[threadIdx.x] = 0; }
    if (threadIdx.x < 6) { sum[threadIdx.x] = 0; }
    if (threadIdx.x == 0) { hBits = 0, most = 0; }
    __syncthreads();
    unsigned long long v[6] = {};
    double             hMax = 0.0;
    uint32_t           mx   = 0;
    for (uint32_t g = blockIdx.x * blockDim.x + threadIdx.x; g < groups; g += gridDim.x * blockDim.x)
    {
        const GroupStat q = groupStats[g];
        v[0] += q.stored, v[1] += q.fails, v[2] += q.wide, v[3] += q.swept, v[4] += q.bad, v[5] += q.targets;
        mx   = max(mx, q.maxCount);
        hMax = fmax(hMax, q.hMax);
        if (info != nullptr)
        {
            const uint32_t s = info[g].count;
            atomicAdd(&part[s == TableInfo::kFailed ? kFailedTable : min(s == 0 ? 0u : (s - 1) / kTableBin, kLargeTable)], 1u);
        }
    }
    for (int k = 0; k < 6; ++k)
        v[k] = waveSum(v[k]);
    mx   = waveMax(mx);
    hMax = waveMaxD(hMax);
    if (laneId() == 0)
    {
        for (int k = 0; k < 6; ++k)
            atomicAdd(&sum[k], v[k]);
        atomicMax(&most, mx);
        // positive doubles order as their bit patterns
        atomicMax(&hBits, (unsigned long long)__double_as_longlong(hMax));
    }
    __syncthreads();
    if (threadIdx.x == 0)
    {
        atomicMax(&stats[kStatHMax], hBits);
        atomicAdd(&stats[0], sum[0]);
        atomicMax(&stats[1], (unsigned long long)most);
        if (sum[1]) { atomicAdd(&stats[2], sum[1]); }
        if (sum[2]) { atomicAdd(&stats[kStatWide], sum[2]); }
        atomicAdd(&stats[kStatTests], sum[3] * kWave);
        if (sum[4]) { atomicAdd(&stats[kStatBadGroups], sum[4]); }
        atomicAdd(&stats[kStatTargets], sum[5]);
    }
    uint32_t* hist = reinterpret_cast<uint32_t*>(stats + kStatHist);
    if (threadIdx.x < kTableBins + 2 && part[threadIdx.x]) { atomicAdd(&hist[threadIdx.x], part[threadIdx.x]); }
}

//! clears the search's slots of the counters (those between are the time step's)
constexpr unsigned kClearThreads = 128;
__global__ void __launch_bounds__(kClearThreads) clearStatsKernel(unsigned long long* stats)
{
    static_assert(kCounterSlots <= kClearThreads, "one slot per thread");
    if (threadIdx.x < 3 || (threadIdx.x >= kStatWide && threadIdx.x < kCounterSlots)) { stats[threadIdx.x] = 0; }
}

constexpr unsigned kCopyWaves = 4;
constexpr unsigned kCopyRun   = 32; // entries of each row per round

/*! row i - first of `out` = stored list of target i. A wave takes the 64 targets of one list block: it reads kCopyRun
 * entries of each (16-byte runs of the 64 lists lie side by side), turns the tile in LDS and writes 128 bytes per row and
 * half wave. One thread per row, each writing its own 4 bytes, took 349 us for 250k particles and 25M
 * entries; this takes 62, and one row alone 23 us with its call (24 when each quad of a round waited for the last). Bound by the table lookups and the writes (105 MB). */
__global__ void __launch_bounds__(kCopyWaves* kWave)
    copyListsKernel(NeighborLists lists, const uint32_t* __restrict__ nc, uint32_t* __restrict__ out,
                    uint32_t searchFirst, uint32_t first, uint32_t last)
{
    __shared__ uint32_t tile[kCopyWaves][kWave][kCopyRun + 1];
    const unsigned      w = threadIdx.x / kWave, lane = laneId();
    const uint32_t      block = (first - searchFirst) / kGroup + blockIdx.x * kCopyWaves + w;
    const uint64_t      i     = uint64_t(searchFirst) + uint64_t(block) * kGroup + lane;
    const bool          on    = i >= first && i < last && lists.searched(uint32_t(i - searchFirst));
    const uint32_t      n     = on ? min(nc[i] - 1, lists.ngmax) : 0u;
    const TargetList    list  = lists.list(on ? uint32_t(i - searchFirst) : 0u);
    const uint32_t      most  = waveMax(n);
    for (uint32_t k0 = 0; k0 < most; k0 += kCopyRun)
    {
        if (k0 < n)
        {
            // (past the last quad it again, so that the round's loads go out together)
            uint32_t j[kCopyRun / 4][4];
#pragma unroll
            for (uint32_t q = 0; q < kCopyRun / 4; ++q)
                list.quad(min(k0 + 4 * q, (n - 1) & ~3u), j[q]);
#pragma unroll
            for (uint32_t k = 0; k < kCopyRun; ++k)
                tile[w][lane][k] = j[k / 4][k % 4];
        }
        __builtin_amdgcn_wave_barrier(); // a wave's LDS accesses complete in order
        const uint32_t k = lane % kCopyRun;
        for (uint32_t row = lane / kCopyRun; row < kWave; row += kWave / kCopyRun)
        {
            const uint32_t rowN = __shfl(n, int(row), kWave);
            const uint64_t to   = uint64_t(searchFirst) + uint64_t(block) * kGroup + row - first;
            if (k0 + k < rowN) { out[to * lists.ngmax + k0 + k] = tile[w][row][k]; }
        }
        __builtin_amdgcn_wave_barrier();
    }
}

} // namespace

int findNeighbors(sphx_workspace* ws, const DevBox& box, const sphx_fields_t* f, const sphx_params_t* p,
                  uint32_t first, uint32_t last, bool iterateH, int xmassOut)
{
    SPHX_REQUIRE(ws->tree.valid, SPHX_ERR_STATE, "find_neighbors called before the tree was built");
    SPHX_REQUIRE(f->x && f->y && f->z && f->h && f->nc, SPHX_ERR_ARG, "find_neighbors needs x, y, z, h and nc");
    SPHX_REQUIRE(first <= last && last <= ws->tree.numParticles, SPHX_ERR_ARG, "invalid target range");
    SPHX_REQUIRE(p->ng0 <= p->ngmax, SPHX_ERR_ARG, "ng0 should be smaller than ngmax");
    SPHX_REQUIRE(p->ngmax > 0, SPHX_ERR_ARG, "ngmax must be positive");

    SPHX_REQUIRE(xmassOut == kSearchOnly || ws->tablesValid, SPHX_ERR_STATE,
                 "kernel tables not set (sphx_workspace_set_kernel)");
    SPHX_REQUIRE(xmassOut == kSearchOnly || (f->m && (xmassOut == kSearchRho ? f->rho : f->xm)), SPHX_ERR_ARG,
                 "the fused XMass needs m and its output field (xm or rho)");
    // from here on the former lists are overwritten: they are gone unless this search completes
    ws->nbValid = false;

    const Tree&  t      = ws->tree;
    const Groups grp    = groupsFor(ws, first, last);
    const uint32_t groups = grp.num;
    // list blocks of 64 consecutive particles from first, whatever the target groups. Local lists take 2 bytes
    // a slot and 8 KB of table per group (more for large ngmax); with more than twice as many groups as blocks the
    // tables would outgrow the lists, and the search stores global lists (4 bytes a slot)
    const size_t blocks64    = std::max<size_t>(1, ceilDiv(last - first, kGroup));
    bool         tryLocal    = xmassOut == kSearchOnly && groups <= 2 * blocks64 + 64;
    if (tryLocal && ws->nbGlobalNext > 0 && ws->nbGlobalNgmax == p->ngmax) { tryLocal = false, --ws->nbGlobalNext; }
    // regions for the few groups whose table outgrows its place: one in 64 groups at first (a tenth of the tables' memory at
    // ngmax = 150), as many as a former search asked for, at most as much memory as the tables themselves
    const uint32_t tableCap = tableCapacity(p->ngmax), regionCap = tableRegion(p->ngmax);
    const size_t   tables      = std::max<size_t>(1, groups) * tableCap;
    const uint32_t mostRegions = std::max<uint32_t>(groups / 64 + 4, uint32_t(tables / regionCap));
    const bool   owned       = grp.start != nullptr;
    const size_t localWords  = blocks64 * paddedNgmax8(p->ngmax) * kGroup / 2;
    const size_t globalWords = blocks64 * paddedNgmax(p->ngmax) * kGroup;
    ws->nbrs.reserve(tryLocal ? localWords : globalWords);
    ws->counters.reserve(2 * kCounterSlots);

    double scale = 0;
    for (int d = 0; d < 3; ++d)
        scale = std::max(scale, std::max(std::abs(box.lo[d]), std::abs(box.hi[d])));

    SearchArgs a;
    a.x = f->x, a.y = f->y, a.z = f->z;
    a.childOffsets   = t.childOffsets.get();
    a.internalToLeaf = t.internalToLeaf.get();
    a.rankLo         = t.rankLo.get();
    a.childPush      = t.childPush.get();
    a.layout         = t.layout.get();
    a.centers        = t.centers.get();
    a.sizes          = t.sizes.get();
    a.box            = box;
    a.slack          = 1e-12 * scale;
    a.first = first, a.last = last, a.ng0 = p->ng0, a.ngmax = p->ngmax;
    a.groups = grp;
    a.iterateH = iterateH ? 1 : 0;
    a.nbrs       = ws->nbrs.get();
    a.tableCap = tableCap, a.regionCap = regionCap, a.region0 = uint32_t(tables / 64);
    a.regionsTaken = reinterpret_cast<uint32_t*>(ws->counters.get()) + 2 * kStatRegions;
    // nbSide: statistics (8 words a group), places (2), owners (with room for them also where this search has no view), then
    // the tables and regions of local lists
    static_assert(sizeof(GroupStat) == 32 && sizeof(TableInfo) == 8, "words per group");
    const size_t statWords = 8 * std::max<size_t>(1, groups), infoWords = 2 * std::max<size_t>(1, groups);
    const size_t ownerWords = (size_t(last - first) + 1) / 2 * 2, sideWords = (statWords + infoWords + ownerWords + 63) / 64 * 64;
    auto         reserveSide = [&](bool local, uint32_t wanted)
    {
        a.regions = std::min(std::max(groups / 64 + 4, wanted), mostRegions);
        ws->nbSide.reserve(sideWords + (local ? tables + size_t(a.regions) * regionCap : 0));
        uint32_t* words = ws->nbSide.get();
        a.groupStats    = reinterpret_cast<GroupStat*>(words);
        a.info = ws->nbTableInfo = reinterpret_cast<TableInfo*>(words + statWords);
        ws->nbOwner              = words + statWords + infoWords;
        a.owner                  = owned ? ws->nbOwner : nullptr;
        a.table = ws->nbTable = words + sideWords;
    };
    reserveSide(tryLocal, ws->nbRegions);
    a.nc         = f->nc;
    a.minLen   = std::min(box.len[0], std::min(box.len[1], box.len[2]));
    a.m = nullptr, a.wh = nullptr, a.sincN = 0, a.sincInt = -1, a.K = 0, a.xmOut = nullptr, a.toRho = 0;
    const bool f32 = p->hydro_type == SPHX_F32;
    if (xmassOut != kSearchOnly)
    {
        a.m     = f->m;
        a.wh    = ws->wh64.get();
        a.sincN   = sincKernel<float>(ws).n;
        a.sincInt = sincKernel<float>(ws).ni;
        a.K     = p->K;
        a.xmOut = xmassOut == kSearchRho ? f->rho : f->xm;
        a.toRho = xmassOut == kSearchRho;
    }

    unsigned long long stats[kCounterSlots];
    uint32_t           hist[kTableBins + 2];
    auto               run = [&](bool local)
    {
        clearStatsKernel<<<1, kClearThreads, 0, ws->stream>>>(reinterpret_cast<unsigned long long*>(ws->counters.get()));
        SPHX_CHECK_LAUNCH();
        static_assert(NeighborLists::kNoGroup == 0xffffffffu, "the fill value");
        if (owned && ownerWords) { fill64(ws, reinterpret_cast<uint64_t*>(ws->nbOwner), ~uint64_t(0), ownerWords / 2); }
        if (groups > 0)
        {
            unsigned    blocks = ceilDiv(groups, kWavesPerBlock);
            KernelScope timer(ws, "search");
            const dim3  grid(blocks), block(kWavesPerBlock * kWave);
            if (local)
            {
                if (f32) searchKernel<float, false, true><<<grid, block, 0, ws->stream>>>(a, static_cast<float*>(f->h));
                else searchKernel<double, false, true><<<grid, block, 0, ws->stream>>>(a, static_cast<double*>(f->h));
            }
            else if (xmassOut == kSearchOnly)
            {
                if (f32) searchKernel<float, false, false><<<grid, block, 0, ws->stream>>>(a, static_cast<float*>(f->h));
                else searchKernel<double, false, false><<<grid, block, 0, ws->stream>>>(a, static_cast<double*>(f->h));
            }
            else
            {
                if (f32) searchKernel<float, true, false><<<grid, block, 0, ws->stream>>>(a, static_cast<float*>(f->h));
                else searchKernel<double, true, false><<<grid, block, 0, ws->stream>>>(a, static_cast<double*>(f->h));
            }
            SPHX_CHECK_LAUNCH();
            groupStatsKernel<<<std::min(ceilDiv(groups, 256), 64u), 256, 0, ws->stream>>>(
                a.groupStats, local ? a.info : nullptr, groups,
                reinterpret_cast<unsigned long long*>(ws->counters.get()));
            SPHX_CHECK_LAUNCH();
        }
        SPHX_HIP(hipMemcpyAsync(stats, ws->counters.get(), sizeof(stats), hipMemcpyDeviceToHost, ws->stream));
        SPHX_HIP(hipStreamSynchronize(ws->stream));
        std::memcpy(hist, &stats[kStatHist], sizeof(hist));
    };
    run(tryLocal);
    bool                     local = tryLocal;
    const unsigned long long fails = stats[2];
    if (local && hist[kFailedTable] > 0)
    {
        // tables that fit neither their place nor a region: again, at the h the first run converged to (without the
        // rounds of the iteration the tables are smaller), with as many regions as were asked for ...
        const uint64_t asked = stats[kStatRegions];
        if (a.iterateH || (asked > a.regions && asked <= mostRegions))
        {
            ws->nbRegions = std::min(uint32_t(asked + asked / 4), mostRegions);
            reserveSide(true, ws->nbRegions);
            a.iterateH = 0;
            run(true);
        }
        // ... or, and then the next 15 searches too, in the global layout
        if (hist[kFailedTable] > 0)
        {
            local            = false;
            ws->nbGlobalNext = 15, ws->nbGlobalNgmax = p->ngmax;
            ws->nbrs.reserve(globalWords);
            a.nbrs = ws->nbrs.get();
            run(false);
        }
    }

    ws->nbFirst      = first;
    ws->nbLast       = last;
    ws->nbNgmax      = p->ngmax;
    ws->nbNc         = f->nc;
    ws->nbLocal      = local;
    ws->nbOwned      = owned;
    ws->nbPartial    = owned && stats[kStatTargets] < uint64_t(last - first);
    std::memcpy(ws->nbTableHist, hist, sizeof(hist));
    ++ws->searchSerial;
    ws->statSumPairs = stats[0];
    ws->statMaxCount = uint32_t(stats[1]);
    ws->nbWide       = stats[kStatWide] > 0;
    ws->statTests    = stats[kStatTests];
    std::memcpy(&ws->nbHMax, &stats[kStatHMax], sizeof(double));
    if (stats[kStatBadGroups] > 0)
    {
        throw Error{SPHX_ERR_ARG, std::to_string(stats[kStatBadGroups]) + " target groups hold more than 64 particles"};
    }
    ws->nbValid = true;
    return fails > 0 ? SPHX_ERR_NOT_CONVERGED : SPHX_OK;
}

void copyNeighbors(sphx_workspace* ws, uint32_t* out, uint32_t first, uint32_t last)
{
    SPHX_REQUIRE(ws->nbValid, SPHX_ERR_STATE, "no neighbour lists: call find_neighbors first");
    SPHX_REQUIRE(ws->nbFirst <= first && first <= last && last <= ws->nbLast, SPHX_ERR_ARG,
                 "copy range must lie inside the searched range");
    SPHX_REQUIRE(out != nullptr, SPHX_ERR_ARG, "null output");
    if (last == first) { return; }
    size_t             len = size_t(last - first) * ws->nbNgmax;
    hipPointerAttribute_t attr{};
    bool               onDevice = hipPointerGetAttributes(&attr, out) == hipSuccess && attr.type == hipMemoryTypeDevice;
    (void)hipGetLastError();
    uint32_t* dst = out;
    DevBuf<uint32_t> staging;
    if (!onDevice)
    {
        staging.reserve(len);
        dst = staging.get();
        // the rows of targets without a list stay as they are
        if (ws->nbPartial) { SPHX_HIP(hipMemcpyAsync(dst, out, len * sizeof(uint32_t), hipMemcpyHostToDevice, ws->stream)); }
    }
    // the list blocks that hold [first, last)
    const uint32_t blocks = (last - 1 - ws->nbFirst) / kGroup - (first - ws->nbFirst) / kGroup + 1;
    copyListsKernel<<<ceilDiv(blocks, kCopyWaves), kCopyWaves * kWave, 0, ws->stream>>>(
        neighborLists(ws), ws->nbNc, dst, ws->nbFirst, first, last);
    SPHX_CHECK_LAUNCH();
    if (!onDevice)
    {
        SPHX_HIP(hipMemcpyAsync(out, dst, len * sizeof(uint32_t), hipMemcpyDeviceToHost, ws->stream));
        SPHX_HIP(hipStreamSynchronize(ws->stream));
        staging.release();
    }
}

} // namespace sphx
