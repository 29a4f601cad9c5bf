// Helpers shared by the SPH pair-loop kernels (std and VE).
//
// Launch shape: one block of W waves (4, or 8 to 12 where the records fill a CU's LDS) per group of 64 consecutive
// targets (the neighbour-search group), blocks renumbered per XCD (xcdBlock) so that neighbouring groups share an L2. Lane l of
// every wave owns target first + 64 g + l; wave w takes the quads w, w + W, .. of its list, and the
// waves' partial sums are added at the end in a fixed order (waveSums), so a target's result does
// not depend on the grouping of the call.
//
// The targets of a group share most of their neighbours: about 600 distinct particles against
// 64 x 91 list entries on a lattice. Read from global memory, each entry costs one tag lookup of the
// vector cache per lane and 16-byte chunk of its record, about 50 cycles of a CU per chunk, which
// bound the loops. With local lists (common.hpp) the block first copies the records of the group's
// table to LDS, chunk c of all records side by side, and every neighbour is read from there
// (PairWalk). Groups whose table does not fit the launch's LDS, and global lists,
// read the records from global memory in the same order, two or four neighbours at a time with the next list entries
// on their way (one at a time, the loops took up to 1.7 times as long there; 1M particles after a
// fused search, ms, with that and with this: mixed AV switches 0.61 -> 0.35, momentum-energy 0.97 -> 0.56, FP64
// 0.88 -> 0.63 and 1.64 -> 1.43). Measured (ms; gathers from global memory, then this):
// mixed VE at 8M particles, XMass 1.27 -> 0.79, grad-h 2.13 -> 1.30, IAD 2.17 -> 1.49, AV switches 2.84 -> 1.42,
// momentum-energy 4.92 -> 3.24; FP64 VE at 4.1M, 2.35 -> 1.02, 2.90 -> 1.70, 3.26 -> 1.74, 4.06 -> 1.77, 6.76 ->
// 5.1-5.4 (with the kernel evaluated instead of gathered from its table; a card at its power limit runs
// momentum slower when the loops before it are faster). What bounds them now: the FP32 form
// the vector ALU (0.9 to 1.1 instructions per SIMD and four cycles; FP32 and FP64 multiply-adds by turns reach 1.1), the FP64
// form (0.6 to 0.85) the latency of a block's phases at 2-3 waves per SIMD.
//
// Two arithmetic forms share each kernel template:
//  * T = double ("plain" FP64): the reference JLoop formulas in FP64.
//  * T = float ("mixed"): HydroType fields in float (the reference's SphTypes layout); pair
//    separations from 32-bit fixed point, gradients and pair terms in FP32; kernel values and the
//    density, grad-h and energy sums in FP64; the IAD 3x3 inversion in FP64.
#pragma once

#include <algorithm>
#include <cmath>
#include <tuple>
#include <type_traits>

#include "common.hpp"

namespace sphx
{

template<class T>
constexpr bool isMixed = std::is_same_v<T, float>;

/*! Waves per block. The light loops (XMass, grad-h, IAD, AV switches) take four. The FP64 momentum records of a
 * group take 92-112 KB of LDS, one block per CU, so the block has to bring the CU's waves: twelve (three per SIMD,
 * 168 registers each), or eight with AV cleaning, whose FP64 loop needs more registers. FP64 VE momentum at 4.1M
 * particles: four waves 8.85 ms, eight 5.25, twelve 5.11. */
constexpr int kLightWaves = 4;
template<class T, bool avClean = false>
constexpr int kMomWaves = isMixed<T> ? 4 : avClean ? 8 : 12;

//! waves per SIMD that a light loop's registers must leave room for: five in the FP32 form, three in the FP64 form
//! (its LDS holds three blocks or more); without the bound some take a few registers too many for that
template<class T>
constexpr int kLightPerSimd = isMixed<T> ? 5 : 3;
#define SPHX_LIGHT_WAVES(T) __attribute__((amdgpu_waves_per_eu(kLightPerSimd<T>, isMixed<T> ? 8 : 3)))

//! waves per SIMD that the momentum loop's registers leave room for
template<class T, bool avClean = false>
constexpr int kMomPerSimd = isMixed<T> ? 4 : kMomWaves<T, avClean> / 4;

//! waves per block of the adjoint loops, which take one group per wave
constexpr int kVjpWaves = 4;

struct Lists
{
    static constexpr uint32_t kNoBlock = 0xffffffffu;

    NeighborLists   lists;
    const uint32_t* nc;
    uint32_t        first, last, ngmax; // [first, last): the searched targets
    uint32_t        stage;              // records the launch's LDS holds
    uint32_t        block0;             // list block of the call's first group, whose targets are whole blocks; or kNoBlock
    bool            partial;            // the search left targets of its range out
    Groups          groups;             // the call's target groups
};

//! a lane's target
struct Lane
{
    uint32_t i;     // target index (a lane without a target: the first searched particle)
    uint32_t r;     // its place in the searched range
    unsigned n;     // neighbours to visit (0 without a target)
    bool     valid; // lane holds a target
};

/*! lane l takes the l-th target of group g; its list is that of the (i - first)-th searched target,
 * whatever the grouping. Targets outside the searched range [first, last), and those that the search's view
 * left out, are not taken: a call leaves their results as they were. */
__device__ __forceinline__ Lane groupTarget(const Lists& L, uint32_t g)
{
    Lane     t;
    uint32_t i0 = 0, i1 = 0;
    bool     oversized;
    if (g < L.groups.num) { groupRange(L.groups, g, i0, i1, oversized); }
    t.i     = i0 + threadIdx.x % kWave;
    t.valid = t.i < i1 && t.i >= L.first && t.i < L.last;
    t.i     = t.valid ? t.i : L.first;
    t.r     = t.i - L.first;
    // (both loads go out together)
    const bool     searched = L.lists.searched(t.r);
    const uint32_t nc       = L.nc[t.i];
    t.valid                 = t.valid && searched;
    t.n                     = t.valid ? min(nc - 1, L.ngmax) : 0u;
    return t;
}

//! group of a pair-loop block
__device__ __forceinline__ uint32_t blockGroup() { return xcdBlock(blockIdx.x, gridDim.x); }

//! target of a lane of the adjoint loops (one group per wave)
__device__ __forceinline__ Lane vjpTarget(const Lists& L)
{
    return groupTarget(L, __builtin_amdgcn_readfirstlane(xcdBlock(blockIdx.x, gridDim.x) * kVjpWaves + threadIdx.x / kWave));
}

inline unsigned vjpBlocks(const Lists& L) { return ceilDiv(L.groups.num, kVjpWaves); }

//! lt::lookup (sph/include/sph/table_lookup.hpp:10-26): linear interpolation of a 20000-point
//! table on [0,2], zero beyond the support. The table is stored per interval (both end values
//! adjacent), so one lookup is one vector gather instead of two scalar ones. Interval 19999, one
//! past the last, holds zeros: arguments at or beyond the support clamp onto it and interpolate
//! to +0, the reference's value there, without a branch around the load. Arguments are >= 0.
template<class T>
__device__ __forceinline__ T interpolate(T t0, T t1, T v, int idx)
{
    constexpr T dx         = T(2.0) / (kTableSize - 1);
    constexpr T invDx      = T(1) / dx;
    T           derivative = (t1 - t0) * invDx;
    return t0 + derivative * (v - T(idx) * dx);
}

template<class T>
__device__ __forceinline__ int tableInterval(T v)
{
    constexpr int numIntervals = kTableSize - 1;
    constexpr T   dx           = T(2.0) / numIntervals;
    constexpr T   invDx        = T(1) / dx;
    T             vc           = v < T(4) ? v : T(4); // keeps the conversion in range
    return min(int(vc * invDx), numIntervals);
}

template<class T>
__device__ __forceinline__ T lookup(const TabPair<T>* __restrict__ table, T v)
{
    int              idx = tableInterval(v);
    const TabPair<T> e   = table[idx];
    return interpolate(e.t0, e.t1, v, idx);
}

//! W(v) and dW/dv(v) from one interval record
template<class T>
__device__ __forceinline__ void lookupBoth(const TabQuad<T>* __restrict__ table, T v, T& w, T& dw)
{
    int              idx = tableInterval(v);
    const TabQuad<T> e   = table[idx];
    w                    = interpolate(e.w0, e.w1, v, idx);
    dw                   = interpolate(e.d0, e.d1, v, idx);
}

//! fast reciprocal / square root for the FP32 form, IEEE operations for FP64
template<class T>
__device__ __forceinline__ T fastDiv(T a, T b)
{
    if constexpr (isMixed<T>) { return a * __builtin_amdgcn_rcpf(b); }
    else { return a / b; }
}

template<class T>
__device__ __forceinline__ T fastSqrt(T a)
{
    if constexpr (isMixed<T>) { return __builtin_amdgcn_sqrtf(a); }
    else { return sqrt(a); }
}

//! a / sqrt(d2). FP64: the hardware's reciprocal root (2^-24) and two Newton steps, to about an ulp
template<class T>
__device__ __forceinline__ T overDistance(T a, T d2)
{
    if constexpr (isMixed<T>) { return a * __builtin_amdgcn_rsqf(d2); }
    else
    {
        double r = __builtin_amdgcn_rsq(d2);
        r        = r + r * (0.5 - 0.5 * (d2 * r) * r);
        r        = r + r * (0.5 - 0.5 * (d2 * r) * r);
        return a * r;
    }
}

//! LDS of a pair-loop block: the staged records, then the partial sums
extern __shared__ Chunk16 pairLds[];

//! bytes of a staged neighbour of `bytes` of records: an odd number of 16-byte chunks, so that the records of
//! different neighbours start in all sixteen 16-byte bank groups. The 64 lanes of a read still meet in them by chance:
//! conflicts take 12 to 36% of a CU's cycles in the loops at 8M particles.
__host__ __device__ constexpr uint32_t stagedBytes(uint32_t bytes) { return 16u * ((bytes / 16u) | 1u); }

/*! copy the records of the group's table to LDS (all waves), record e at dst + e * stride. Each thread has B
 * chunks in flight: their table entries, then their records, load together, so a block pays two memory
 * latencies per B * blockDim chunks rather than per chunk. */
template<class R>
__device__ __forceinline__ void stageRecords(const uint32_t* __restrict__ table, uint32_t count, const R* __restrict__ rec,
                                             char* dst, uint32_t stride)
{
    constexpr uint32_t NC = sizeof(R) / 16;
    constexpr uint32_t B  = NC < 3 ? 4 : 8;
    static_assert(sizeof(R) % 16 == 0, "records are whole 16-byte chunks");
    const Chunk16* src   = reinterpret_cast<const Chunk16*>(rec);
    const uint32_t total = count * NC;
    for (uint32_t q0 = threadIdx.x; q0 < total; q0 += B * blockDim.x)
    {
        uint32_t j[B];
        Chunk16  v[B];
#pragma unroll
        for (uint32_t u = 0; u < B; ++u)
            j[u] = table[min(q0 + u * blockDim.x, total - 1) / NC];
#pragma unroll
        for (uint32_t u = 0; u < B; ++u)
            v[u] = src[size_t(j[u]) * NC + min(q0 + u * blockDim.x, total - 1) % NC];
#pragma unroll
        for (uint32_t u = 0; u < B; ++u)
        {
            // past the end: the last chunk again, the same value at the same place
            const uint32_t q = min(q0 + u * blockDim.x, total - 1);
            *reinterpret_cast<Chunk16*>(dst + (q / NC) * stride + 16 * (q % NC)) = v[u];
        }
    }
}

template<class R>
__device__ __forceinline__ R stagedRecord(const char* src)
{
    constexpr uint32_t NC = sizeof(R) / 16;
    Chunk16            c[NC];
#pragma unroll
    for (uint32_t k = 0; k < NC; ++k)
        c[k] = reinterpret_cast<const Chunk16*>(src)[k];
    R r;
    __builtin_memcpy(&r, c, sizeof(R));
    return r;
}

/*! Walk over the neighbours of a block's targets, wave w taking the quads w, w + W, .. of each list:
 * pair(live, records...) for every slot, with the neighbour's record of each of Rs. Slots past a lane's count
 * (the rest of its last quad) hold the list's last neighbour again, with live = false. U of a quad's
 * staged records are in flight at a time, or G gathered ones, and the next quad of the list. */
template<int W, int U, int G, class... Rs>
struct PairWalk
{
    static_assert((U == 1 || U == 2 || U == 4) && (G <= 2 || G == 4), "whole parts of a quad");
    static constexpr uint32_t kChunks = uint32_t((sizeof(Rs) + ...)) / 16;
    static constexpr uint32_t kStride = stagedBytes(16 * kChunks);

    const Lists& L;
    const Lane&  t;
    bool         staged;
    uint64_t     next; // local lists: the wave's first quad

    //! stages the group's records, unless they do not fit or are not one group's. Where the call's groups are the
    //! search's, the table and the first quad of the lists load without waiting for the targets' counts.
    __device__ __forceinline__ PairWalk(const Lists& lists, const Lane& lane, const Rs*... rec)
        : L(lists)
        , t(lane)
        , staged(false)
        , next(0)
    {
        if (L.lists.info != nullptr)
        {
            bool     one;
            uint32_t b0;
            if (L.block0 != Lists::kNoBlock)
            {
                b0  = L.block0 + blockGroup();
                one = true;
            }
            else
            {
                const bool     some = t.n > 0;
                const uint32_t b    = some ? L.lists.group(t.r) : 0u;
                const uint64_t mask = ballot(some);
                b0                  = mask ? __builtin_amdgcn_readlane(b, __builtin_ctzll(mask)) : 0u;
                one                 = ballot(some && b != b0) == 0 && mask != 0;
            }
            const TableInfo info = L.lists.info[b0];
            if (one && info.count <= L.stage)
            {
                staged = true;
                if (firstSlot() < paddedNgmax8(L.ngmax)) { next = *reinterpret_cast<const uint64_t*>(listStart()); }
                const uint32_t* tb = L.lists.tableAt(info);
                uint32_t        at = 0;
                ((stageRecords(tb, info.count, rec, ldsBytes() + at, kStride), at += uint32_t(sizeof(Rs))), ...);
            }
        }
        __syncthreads();
    }

    __device__ __forceinline__ static uint32_t firstSlot() { return 4 * (threadIdx.x / kWave); }
    __device__ __forceinline__ const uint16_t* listStart() const
    {
        return static_cast<const uint16_t*>(L.lists.nbrs) +
               localOffset(t.r / kGroup, paddedNgmax8(L.ngmax), firstSlot(), t.r % kGroup);
    }
    __device__ __forceinline__ static char* ldsBytes() { return reinterpret_cast<char*>(pairLds); }

    template<class F>
    __device__ __forceinline__ void operator()(F&& pair, const Rs*... rec)
    {
        const uint32_t k0 = firstSlot();
        if (staged)
        {
            static_assert(W % 2 == 0, "a wave's quads lie at one place of their octets");
            constexpr size_t step = size_t(4 * W) * kGroup; // list words from a quad to the wave's next
            const uint16_t*  list = listStart();
            for (uint32_t k = k0; k < t.n; k += 4 * W)
            {
                uint64_t q = next;
                list += k + 4 * W < t.n ? step : 0;
                next = *reinterpret_cast<const uint64_t*>(list);
                asm volatile("" : "+v"(next)); // the load stays here, ahead of its use
#pragma unroll 1
                for (int u0 = 0; u0 < 4; u0 += U)
                {
#pragma unroll
                    for (int u = 0; u < U; ++u)
                    {
                        const char* from = ldsBytes() + (uint32_t(q >> (16 * u)) & 0xffffu) * kStride;
                        uint32_t    at   = 0;
                        auto        load = [&](auto* p)
                        {
                            using R    = std::remove_const_t<std::remove_pointer_t<decltype(p)>>;
                            const R rj = stagedRecord<R>(from + at);
                            at += uint32_t(sizeof(R));
                            return rj;
                        };
                        const std::tuple<Rs...> r{load(rec)...};
                        std::apply([&](const Rs&... rj) { pair(k + u0 + u < t.n, rj...); }, r);
                    }
                    q >>= 16 * (U % 4);
                }
            }
        }
        else
        {
            constexpr int    B    = G ? G : 1;
            const TargetList list = L.lists.list(t.r);
            uint32_t         ahead[4] = {};
            if (G && k0 < t.n) { list.quad(k0, ahead); }
#pragma unroll
            for (int u = 0; u < 4; ++u)
                asm volatile("" : "+v"(ahead[u])); // (else this load and the loop's become one at the top of each round)
            for (uint32_t k = k0; k < t.n; k += 4 * W)
            {
                uint32_t j[4] = {ahead[0], ahead[1], ahead[2], ahead[3]};
                if constexpr (G)
                {
                    // the next quad's entries (the last one's again) load while this one's records do
                    list.quad(k + 4 * W < t.n ? k + 4 * W : k, ahead);
                }
                else { list.quad(k, j); }
#pragma unroll 1
                for (int u0 = 0; u0 < 4; u0 += B)
                {
                    Chunk16 w[B][kChunks];
#pragma unroll
                    for (int u = 0; u < B; ++u)
                    {
                        uint32_t at   = 0;
                        auto     load = [&](auto* p)
                        {
                            const Chunk16* src = reinterpret_cast<const Chunk16*>(p + j[u]);
#pragma unroll
                            for (uint32_t c = 0; c < sizeof(*p) / 16; ++c)
                                w[u][at + c] = src[c];
                            at += sizeof(*p) / 16;
                        };
                        (load(rec), ...);
                    }
#pragma unroll
                    for (int u = 0; u < B; ++u)
                    {
                        uint32_t at    = 0;
                        auto     taken = [&](auto* p)
                        {
                            std::remove_const_t<std::remove_pointer_t<decltype(p)>> rj;
                            __builtin_memcpy(&rj, &w[u][at], sizeof(rj));
                            at += sizeof(rj) / 16;
                            return rj;
                        };
                        const std::tuple<Rs...> r{taken(rec)...};
                        std::apply([&](const Rs&... rj) { pair(k + u0 + u < t.n, rj...); }, r);
                    }
#pragma unroll
                    for (int u = 0; u + B < 4; ++u)
                        j[u] = j[u + B];
                }
            }
        }
    }
};

/*! Add the waves' partial sums v[0..N) of each lane's target in wave order; the first M are combined by maximum
 * instead. True on the first wave, which then holds the totals. */
template<int W, int N, int M = 0>
__device__ __forceinline__ bool waveSums(double (&v)[N])
{
    double*        part = reinterpret_cast<double*>(pairLds);
    const unsigned lane = threadIdx.x % kWave, w = threadIdx.x / kWave;
    __syncthreads(); // every wave has read its records
    if (w > 0)
    {
#pragma unroll
        for (int q = 0; q < N; ++q)
            part[((w - 1) * N + q) * kWave + lane] = v[q];
    }
    __syncthreads();
    if (w > 0) { return false; }
#pragma unroll
    for (int q = 0; q < N; ++q)
    {
#pragma unroll
        for (int p = 0; p < W - 1; ++p)
        {
            const double x = part[(p * N + q) * kWave + lane];
            if (q < M) { v[q] = x > v[q] ? x : v[q]; }
            else { v[q] += x; }
        }
    }
    return true;
}

/*! host: the records a launch stages and its dynamic LDS, for records of `recBytes`, N partial sums and a kernel whose
 * registers leave room for `perSimd` waves on a SIMD. A block whose table does not fit the stage reads its
 * neighbours from global memory, 1.2 (FP64) to 1.7 times as long; a smaller stage leaves room for more blocks on a CU, and the
 * loops' time goes with about the power -0.4 of the waves per SIMD. The number of blocks per CU is the one with the
 * least product of both, the stage what its share of the 160 KB holds. Measured against a stage for 99.5% of the
 * tables (ms): mixed std momentum of the 4M Evrard sphere 2.15 -> 1.69 (three blocks instead of two, 8% of the
 * blocks gathering), FP64 AV switches and IAD at 4.1M 2.04 -> 1.77 and 2.07 -> 1.74, mixed IAD at 2M 0.42 -> 0.38. */
struct PairLaunch
{
    uint32_t stage;
    size_t   lds;
};
inline PairLaunch pairLaunch(const sphx_workspace* ws, size_t recBytes, int waves, int sums, int perSimd)
{
    constexpr double kGathered = 1.6;
    constexpr size_t kLds = 160 * 1024, kLdsUnit = 1280; // of a CU, and what it is given out in
    const size_t     part      = size_t(waves - 1) * sums * kWave * sizeof(double);
    uint64_t         blocks    = 0;
    for (uint32_t b = 0; b <= kLargeTable; ++b)
        blocks += ws->nbTableHist[b];
    if (!ws->nbLocal || blocks == 0) { return {0, part}; }
    const uint32_t each = stagedBytes(uint32_t(recBytes));
    PairLaunch     best{0, part};
    double         least = INFINITY;
    for (int perCu = 1; perCu == 1 || perCu * waves <= 4 * perSimd; ++perCu)
    {
        const size_t room = kLds / kLdsUnit / perCu * kLdsUnit;
        if (part > room) { break; }
        const uint32_t fit    = std::min(uint32_t(room / each), kTableBins * kTableBin);
        uint64_t       staged = 0;
        uint32_t       stage  = 0; // the largest table among those that fit
        for (uint32_t b = 0; (b + 1) * kTableBin <= fit; ++b)
        {
            staged += ws->nbTableHist[b];
            if (ws->nbTableHist[b]) { stage = (b + 1) * kTableBin; }
        }
        const double share = double(staged) / double(blocks);
        const double time  = (share + (1.0 - share) * kGathered) / std::pow(double(perCu), 0.4);
        if (time < least) { least = time, best = {stage, std::max(part, size_t(stage) * each)}; }
    }
    return best;
}

/*! The SPH kernel W(v) = sinc(pi v / 2)^n and dW/dv on [0, 2), zero from v = 2 on.
 *
 * Both forms evaluate the kernel as a function of z = v^2, without a square root, a reciprocal or a
 * table: sinc(pi v / 2) = (1 - z/4) P(z), whose first factor carries the zero at the edge of the
 * support exactly (so sinc keeps its relative accuracy up to there) and whose second is a polynomial
 * fitted at Chebyshev nodes of [0, 4]; d sinc/dz is a polynomial of its own. A table lookup is a
 * 64-lane gather that touches about one cache line per lane, and a separate sine, cosine and
 * reciprocal cost three times the arithmetic of the polynomial. W = sinc^n by multiplication for an
 * integer n (the reference's sinc indices); for other n the FP32 form takes FP32 log2 / exp2 and the
 * FP64 form its tables.
 *
 * FP32 form: sinc and z d sinc/dz as polynomials of y = 1 - z/4 (degree 6 and 7, errors below 6e-11), in
 * FP64 arithmetic (which on this GPU issues at the FP32 rate, since FP32 ops are not packed here), so W is exact
 * to its final rounding. y is one fused multiply-add of the squared distance.
 *
 * FP64 form: the reference interpolates W linearly in a 20000-point table, up to 6e-9 off the function
 * for n = 6, and the FP64 results are held to that interpolant. With t = the fraction of v / dx,
 * the interpolant differs from W(v) by
 *     L(v) - W(v) = 1/2 dx^2 t (1 - t) W''(v + dx (1 - 2t) / 3) + O(dx^4),
 * so it is formed as W(v) plus that term, with P of degree 9 (2e-17) and d sinc/dz in the
 * correction of degree 5 (5e-9 of a term below 6e-9). It equals the interpolated table entries to
 * 2e-15 of W(0) for n = 3, 5, 6 and 9. W'' follows from Y = d sinc/dv = 2 v sinc_z and the equation of the
 * sinc function, Y' = -(pi/2)^2 sinc - 4 sinc_z. */
constexpr double kHalfPiSq = 2.4674011002723396547; // (pi/2)^2

/*! The loops are compiled per variant, chosen on the host for a launch (launchVariant):
 * kCommon: the default sinc index 6, its powers unrolled; in the FP32 form the wrapping fixed-point
 * separation as well, in units of the fixed point (DevBox::raw). kWide (FP32 form): the exact separations of
 * boxes a few smoothing lengths wide, any index. kAnyIndex: any other index, or (FP32 form) periodic
 * dimensions of different lengths. */
enum Variant
{
    kCommon,
    kWide,
    kAnyIndex
};

//! x^k for a small integer k >= 0 (wave-uniform loop)
__device__ __forceinline__ double sincPower(double x, int k)
{
    double r = 1.0, b = x;
    for (int e = k; e > 0; e >>= 1)
    {
        if (e & 1) { r *= b; }
        b *= b;
    }
    return r;
}

//! sinc(pi v / 2) at y = 1 - v^2 / 4 in [0, 1], relative error 6e-11 (FP32 form)
__device__ __forceinline__ double sincOfY(double y)
{
    double p = 5.919975391732741e-06;
    p        = p * y + 0.00010508787551814265;
    p        = p * y + 0.0015894063856577154;
    p        = p * y + 0.016416305415662014;
    p        = p * y + 0.10688328287516924;
    p        = p * y + 0.3749999974191315;
    p        = p * y + 0.5000000000263431;
    return p * y;
}

//! z d sinc(pi v / 2) / dz = v/2 d sinc/dv at y = 1 - v^2 / 4, absolute error 6e-11
__device__ __forceinline__ double sincSlopeOfY(double y)
{
    double q = 4.132672691073703e-05;
    q        = q * y + 0.0005894009530895289;
    q        = q * y + 0.007316207227363674;
    q        = q * y + 0.05771828331287214;
    q        = q * y + 0.25498464086819245;
    q        = q * y + 0.42935013419273005;
    q        = q * y - 0.24999999328291864;
    return q * y - 0.5000000000524906;
}

//! d sinc(pi v / 2) / dz, absolute error 6e-11
__device__ __forceinline__ double sincSlope6(double z)
{
    double q = -2.5764109465564327e-09;
    q        = q * z + 2.152531546520502e-07;
    q        = q * z - 1.1449615339245935e-05;
    q        = q * z + 0.00040855196998758054;
    q        = q * z - 0.0089414863396859;
    q        = q * z + 0.10146780180875682;
    return q * z - 0.4112335166569054;
}

//! sinc(pi v / 2) at z = v^2 in [0, 4] to FP64 rounding
__device__ __forceinline__ double sincOfZ9(double z)
{
    double p = -5.823067516159113e-16;
    p        = p * z + 1.0839061254289035e-13;
    p        = p * z - 1.501141501734521e-11;
    p        = p * z + 1.643032500260312e-09;
    p        = p * z - 1.3837782504438124e-07;
    p        = p * z + 8.610867685597616e-06;
    p        = p * z - 0.0003741166513510571;
    p        = p * z + 0.010425522402193063;
    p        = p * z - 0.16123351671205632;
    p        = p * z + 1.0;
    return p - 0.25 * z * p;
}

//! d sinc(pi v / 2) / dz to FP64 rounding
__device__ __forceinline__ double sincSlope9(double z)
{
    double q = 1.4701693771604546e-15;
    q        = q * z - 2.4939334615094517e-13;
    q        = q * z + 3.0892145129869457e-11;
    q        = q * z - 2.9803963653457545e-09;
    q        = q * z + 2.174249574964597e-07;
    q        = q * z - 1.1455473771406392e-05;
    q        = q * z + 0.00040856012212963613;
    q        = q * z - 0.008941491755716072;
    q        = q * z + 0.1014678031604184;
    return q * z - 0.4112335167120566;
}

//! d sinc(pi v / 2) / dz, absolute error 5e-9 (the interpolation term)
__device__ __forceinline__ double sincSlope5(double z)
{
    double q = 1.843090979760722e-07;
    q        = q * z - 1.1310217672036537e-05;
    q        = q * z + 0.0004082624607906118;
    q        = q * z - 0.00894121445580337;
    q        = q * z + 0.10146770837624979;
    return q * z - 0.4112335114493841;
}

/*! The point where the linear interpolation between table nodes differs from W by weight * W'':
 * weight = 1/2 dx^2 t (1 - t), at z1 = (v + dx (1 - 2t) / 3)^2 and sinc s1 there. Only t's value to about
 * 1e-9 matters, so v = sqrt(z) takes one Newton step from the hardware reciprocal root. */
struct InterpolationPoint
{
    double weight, z1, s1, slope;
    double back; // v over the shifted v
};
__device__ __forceinline__ InterpolationPoint interpolationPoint(double z, double s)
{
    constexpr double   dx = 2.0 / (kTableSize - 1);
    const double       zc = z > 1e-280 ? z : 1e-280;
    const double       rs = __builtin_amdgcn_rsq(zc);
    double             v  = zc * rs;
    v                     = v + 0.5 * rs * (zc - v * v);
    const double       t  = __builtin_amdgcn_fract(v * (1.0 / dx));
    InterpolationPoint i;
    i.weight       = (0.5 * dx * dx) * (t - t * t);
    const double shift = dx / 3.0 - (2.0 / 3.0) * dx * t;
    const double u     = 2.0 * v * shift; // z1 - z
    i.z1               = z + u;
    i.back             = 1.0 - shift * rs;
    i.slope        = sincSlope5(i.z1);
    i.s1           = s + u * i.slope;
    return i;
}

//! length of a separation's unit (DevBox::unit)
template<class T>
__device__ __forceinline__ T unitOf(const DevBox& b)
{
    return isMixed<T> ? T(b.unit) : T(1);
}

//! what the records and targets hold of 1/h for the kernel argument of a squared distance in units of the
//! separations: (unit / h)^2, times -1/4 in the FP32 form
template<class T>
__device__ __forceinline__ T kernelScale(T unitOverH)
{
    return isMixed<T> ? T(-0.25) * unitOverH * unitOverH : unitOverH * unitOverH;
}
template<class T>
__device__ __forceinline__ T kernelScale(const DevBox& b, T hInv)
{
    return kernelScale(hInv * unitOf<T>(b));
}

template<class T>
struct SincKernel;

//! FP64: the reference's interpolant for the default index (see above), its tables for any other
template<>
struct SincKernel<double>
{
    const TabPair<double>* wTab;
    const TabQuad<double>* wqTab;

    //! the loops' kernel argument of a pair at squared distance d2, kernelScale(1/h) = scale: z = v^2
    __device__ __forceinline__ static double arg(double d2, double scale) { return d2 * scale; }
    //! the argument held to [0, 4], and to the edge of the support for a slot that is not live: every pair term
    //! is proportional to a kernel value, so such a slot contributes exactly zero without a branch
    __device__ __forceinline__ static double clamp(double z, bool live)
    {
        return fmin(fmax(z, live ? 0.0 : 4.0), 4.0);
    }

    //! W at z in [0, 4]
    template<int V>
    __device__ __forceinline__ double w(double z) const
    {
        if constexpr (V != kCommon) { return lookup(wTab, sqrt(z)); }
        else
        {
            constexpr double n         = kDefaultIndex;
            const double             s = sincOfZ9(z);
            const InterpolationPoint i = interpolationPoint(z, s);
            const double             q = i.s1 * i.s1; // s1^(n-2) = q^2
            const double yp            = -kHalfPiSq * i.s1 - 4.0 * i.slope;
            const double w2            = (q * q) * ((n - 1.0) * 4.0 * i.z1 * (i.slope * i.slope) + i.s1 * yp);
            const double c             = s * s * s;
            return c * c + (n * i.weight) * w2;
        }
    }

    //! W and v dW/dv at z in [0, 4]
    template<int V>
    __device__ __forceinline__ void wAndVdw(double z, double& w, double& vdw) const
    {
        if constexpr (V != kCommon)
        {
            const double v = sqrt(z);
            double       dw;
            lookupBoth(wqTab, v, w, dw);
            vdw = v * dw;
        }
        else
        {
            constexpr double n          = kDefaultIndex;
            const double             s  = sincOfZ9(z);
            const InterpolationPoint i  = interpolationPoint(z, s);
            const double             q  = i.s1 * i.s1, p3 = q * i.s1, p2 = q * q; // s1^(n-3), s1^(n-2)
            const double             yp = -kHalfPiSq * i.s1 - 4.0 * i.slope;
            const double             vy = 2.0 * i.z1 * i.slope;
            const double w2  = p2 * (2.0 * (n - 1.0) * vy * i.slope + i.s1 * yp);
            const double vw3 = p3 * (2.0 * (n - 1.0) * (n - 2.0)) * (vy * vy) * i.slope +
                               p2 * (3.0 * (n - 1.0) * vy * yp + i.s1 * (4.0 * i.slope - 2.0 * yp - kHalfPiSq * vy));
            const double c   = s * s, pm1 = c * c * s;
            w                = pm1 * s + (n * i.weight) * w2;
            vdw              = 2.0 * n * z * pm1 * sincSlope9(z) + (n * i.weight * i.back) * vw3;
            // the reference forms its dW/dv table from cot x - 1/x, whose cancellation leaves an error of
            // 1e-16 / v in the entries: below v = 1/4 the entries themselves are taken
            if (z < 1.0 / 16.0)
            {
                const double     v = sqrt(z);
                const int        k = tableInterval(v);
                const TabQuad<double>* e = wqTab + k;
                vdw = v * interpolate(e->d0, e->d1, v, k);
            }
        }
    }

    //! W and dW/dv at v from the tables (the adjoints)
    __device__ __forceinline__ void wAndDw(double v, double& w, double& dw) const { lookupBoth(wqTab, v, w, dw); }
};

//! FP32: the kernel function itself, in FP64 arithmetic
template<>
struct SincKernel<float>
{
    float n;
    int   ni; // n when it is an integer >= 2, else -1

    template<int V>
    __device__ __forceinline__ double index() const
    {
        return V == kCommon ? double(kDefaultIndex) : double(n);
    }
    //! s^(n-1), 0 at the edge of the support
    template<int V>
    __device__ __forceinline__ double power(double s) const
    {
        if constexpr (V == kCommon)
        {
            const double c = s * s;
            return c * c * s;
        }
        else
        {
            if (ni > 0) { return sincPower(s, ni - 1); }
            return s > 0.0 ? double(__builtin_amdgcn_exp2f((n - 1.0f) * __builtin_amdgcn_logf(float(s)))) : 0.0;
        }
    }
    //! the loops' kernel argument of a pair at squared distance d2, kernelScale(1/h) = scale: y = 1 - v^2 / 4
    __device__ __forceinline__ static float arg(float d2, float scale) { return d2 * scale + 1.0f; }
    //! the argument held to [0, 1], and to the edge of the support for a slot that is not live: every pair term
    //! is proportional to a kernel value, so such a slot contributes exactly zero without a branch
    __device__ __forceinline__ static float clamp(float y, bool live)
    {
        return __builtin_amdgcn_fmed3f(y, 0.0f, live ? 1.0f : 0.0f);
    }

    //! W at y in [0, 1]
    template<int V>
    __device__ __forceinline__ double w(float y) const
    {
        const double s = sincOfY(double(y));
        return power<V>(s) * s;
    }
    //! W and v dW/dv
    template<int V>
    __device__ __forceinline__ void wAndVdw(float yf, double& w, double& vdw) const
    {
        const double y = double(yf);
        const double s = sincOfY(y), p = power<V>(s);
        w              = p * s;
        vdw            = (2.0 * index<V>()) * p * sincSlopeOfY(y);
    }
    __device__ __forceinline__ void wAndDw(float vf, float& w, float& dw) const
    {
        const double v = double(fminf(vf, 2.0f)), z = v * v;
        const double s = sincOfY(1.0 - 0.25 * z), p = power<kAnyIndex>(s);
        w              = float(p * s);
        dw             = float((2.0 * double(n)) * v * p * sincSlope6(z));
    }
};

/*! Whether a wave must apply the legacy fold (sfc/box.hpp:218-238). The fold changes a separation
 * only when |x_i - x_j| exceeds the cut-off 2h_i. For a listed neighbour (minimum-image distance
 * below 2h_i) that needs the raw difference to wrap across a periodic face, which puts the target
 * within 2h_i of that face. Waves without such a target run the loop without the fold. */
__device__ __forceinline__ bool waveNeedsFold(const DevBox& b, double x, double y, double z, double r2h)
{
    const double p[3] = {x, y, z};
    const double r    = r2h * (1.0 + 1e-6);
    bool         near = false;
    for (int d = 0; d < 3; ++d)
        near |= b.pbc[d] && (p[d] - b.lo[d] <= r || b.hi[d] - p[d] <= r);
    return ballot(near) != 0;
}

/*! separation x_i - x_j in the pair type, formed in FP64 (exact for T = double, then rounded for
 * float). With Fold, the legacy minimum image with cut-off r (sfc/box.hpp:218-238): per periodic
 * dimension subtract L if d > r, add L if d < -r. Written with selects, d - 0 == d exactly, so the
 * result is that of the reference's branches. */
template<bool Fold, class T>
__device__ __forceinline__ void separation(const DevBox& b, double r, double xi, double yi, double zi, double xj,
                                           double yj, double zj, T& rx, T& ry, T& rz)
{
    double d[3] = {xi - xj, yi - yj, zi - zj};
    if constexpr (Fold)
    {
        for (int q = 0; q < 3; ++q)
        {
            bool   up   = b.pbc[q] && d[q] > r;
            bool   down = b.pbc[q] && d[q] < -r;
            double s    = up ? b.len[q] : (down ? -b.len[q] : 0.0);
            d[q]        = d[q] - s;
        }
    }
    rx = T(d[0]), ry = T(d[1]), rz = T(d[2]);
}

//! separation of a pair and its squared length
template<class T>
struct Sep
{
    T x, y, z, d2;
};

/*! Position of a particle in the neighbour records: FP64 in the plain form; in the FP32 form
 * 32-bit fixed point over a period P = L / 2^s of the box length L, u = rint((x - lo) 2^32 / P)
 * mod 2^32 per dimension. The shift s is set after each search from its largest h: the largest
 * s <= 16 with P >= 8 h_max (fixedPointShift), so a listed pair, closer than 2h_max in each
 * dimension, is closer than P/4. A record position is 12 bytes instead of 24; coordinates are
 * quantized to P / 2^32, about 2e-9 h_max whatever the box size (an open box much larger than the
 * particles' extent, or a wide range of h, keeps the resolution of the smoothing lengths, as FP32
 * offsets from a nearby cell would). The separation is converted to FP32 and scaled by P / 2^32
 * (about one ulp in all). Which integer difference stands for x_i - x_j:
 *  - while every target has 2h < L/2 in every dimension, the wrapping difference u_i - u_j read as
 *    a signed 32-bit integer. A listed pair is closer than 2h < P/2 in each dimension, so this is
 *    the raw difference in an open dimension, and in a periodic one (P divides L) the minimum
 *    image, which equals the reference's fold with cut-off 2h (sfc/box.hpp:218-238) for any pair
 *    closer than 2h < L/2;
 *  - otherwise (2h >= L/2: a box a few smoothing lengths wide, as for a few hundred particles or
 *    fewer; then s = 0, P = L), the exact difference u_i - u_j in 64 bits, the raw difference of
 *    coordinates that lie in [lo, hi] (the box update of the domain sync keeps open dimensions
 *    there), folded in a periodic dimension with cut-off 2h as the reference does. */
template<class T>
using Coord = std::conditional_t<isMixed<T>, uint32_t, double>;

__device__ __forceinline__ uint32_t fixedCoord(const DevBox& b, int d, double x)
{
    return uint32_t(uint64_t(int64_t(rint((x - b.lo[d]) * b.fixScale[d]))));
}

template<class T>
__device__ __forceinline__ Coord<T> coordOf(const DevBox& b, int d, double x)
{
    if constexpr (isMixed<T>) { return fixedCoord(b, d, x); }
    else { return x; }
}

/*! exact fixed-point separation of one dimension for boxes a few smoothing lengths wide: the 64-bit
 * difference, then the legacy fold with cut-off r in a periodic dimension (see Coord above) */
__device__ __forceinline__ float wideFixedSeparation(const DevBox& b, int q, double r, uint32_t ui, uint32_t uj)
{
    double d = double(int64_t(ui) - int64_t(uj)); // exact: |d| < 2^33
    if (b.pbc[q])
    {
        double dx = d * b.fixStepD[q];
        d         = dx > r ? d - 4294967296.0 : (dx < -r ? d + 4294967296.0 : d);
    }
    return float(d) * b.fixStep[q];
}

/*! separation x_i - x_j of a pair (DevBox::unit is its unit) */
template<bool Fold, int V, class T, class Ri, class Rj>
__device__ __forceinline__ Sep<T> pairSeparation(const DevBox& b, double r2h, const Ri& ri, const Rj& rj)
{
    Sep<T> s;
    if constexpr (isMixed<T> && Fold)
    {
        s.x = wideFixedSeparation(b, 0, r2h, ri.x, rj.x);
        s.y = wideFixedSeparation(b, 1, r2h, ri.y, rj.y);
        s.z = wideFixedSeparation(b, 2, r2h, ri.z, rj.z);
    }
    else if constexpr (isMixed<T> && V == kCommon)
    {
        s.x = float(int32_t(ri.x - rj.x));
        s.y = float(int32_t(ri.y - rj.y));
        s.z = float(int32_t(ri.z - rj.z));
    }
    else if constexpr (isMixed<T>)
    {
        s.x = float(int32_t(ri.x - rj.x)) * b.fixStep[0];
        s.y = float(int32_t(ri.y - rj.y)) * b.fixStep[1];
        s.z = float(int32_t(ri.z - rj.z)) * b.fixStep[2];
    }
    else { separation<Fold>(b, r2h, ri.x, ri.y, ri.z, rj.x, rj.y, rj.z, s.x, s.y, s.z); }
    s.d2 = s.x * s.x + s.y * s.y + s.z * s.z;
    return s;
}

/*! whether the wave of target record ri must fold its FP64 separations; in the FP32 form, kWide: the
 * last search met a target whose support 2h reaches half a box length, where the wrapping 32-bit
 * difference stops standing for the reference's separation (see Coord above), so the loop takes the
 * exact 64-bit difference. The variant is a kernel template argument, chosen on the host
 * (launchVariant), so that the common loop carries none of the registers of the others. */
template<class T, int V, class R>
__device__ __forceinline__ bool recordNeedsFold(const DevBox& b, const Lane& t, const R& ri, double r2h)
{
    if constexpr (isMixed<T>) { return V == kWide; }
    else { return waveNeedsFold(b, ri.x, ri.y, ri.z, t.valid ? r2h : -INFINITY); }
}

//! host: launch(std::integral_constant<int, V>) with the loop variant V of this search, box and sinc index
template<class T, class F>
inline void launchVariant(const sphx_workspace* ws, const DevBox& box, F&& launch)
{
    const bool common = isMixed<T> ? box.raw : ws->sincIndex == double(kDefaultIndex);
    if (common) { launch(std::integral_constant<int, kCommon>{}); }
    else if (isMixed<T> && ws->nbWide) { launch(std::integral_constant<int, kWide>{}); }
    else { launch(std::integral_constant<int, kAnyIndex>{}); }
}

/*! Neighbours in flight where a walk reads staged records, and where it gathers them (0: one, and its quad of list entries
 * not ahead of time). The loops other than the common ones gather one at a time: more spill registers, in their staged
 * blocks as well. */
template<class T>
constexpr int kLightBatch = isMixed<T> ? 4 : 2;
template<class T, int V>
constexpr int kLightGather = V == kCommon ? kLightBatch<T> : 1;
template<class T>
constexpr int kMomBatch = isMixed<T> ? 2 : 1;
template<class T, int V, bool avClean = false>
constexpr int kMomGather = V == kCommon && !avClean ? kMomBatch<T> : 0;

//! run `loop` with the fold compiled in or out, chosen once per wave
template<class F>
__device__ __forceinline__ void withFold(bool fold, F&& loop)
{
    if (fold) { loop(std::true_type{}); }
    else { loop(std::false_type{}); }
}

//! FP64 accumulator of both forms. The FP32 form's density, grad-h and energy sums add their terms in
//! FP64 (the kernel values come in FP64 anyway): two instructions a term where a compensated FP32 sum
//! takes four, and no larger error.
struct Acc
{
    double s;
    __device__ __forceinline__ explicit Acc(double init = 0.0) : s(init) {}
    __device__ __forceinline__ void add(double v) { s += v; }
    //! add(v) where p holds
    __device__ __forceinline__ void addIf(bool p, double v) { s = p ? s + v : s; }
    __device__ __forceinline__ double value() const { return s; }
};

//! positive-double minimum through the integer order of their bit patterns
__device__ __forceinline__ void atomicMinPositive(unsigned long long* dst, double v)
{
    atomicMin(dst, (unsigned long long)__double_as_longlong(v));
}

template<class T>
__device__ __forceinline__ T ld(const void* p, size_t i)
{
    return static_cast<const T*>(p)[i];
}

template<class T>
__device__ __forceinline__ void st(void* p, size_t i, T v)
{
    static_cast<T*>(p)[i] = v;
}

//! IAD: scale tau by 2^-mean(ilogb) and invert through the adjugate (hydro_std/iad_kern.hpp:52-76),
//! computed in FP64 for both forms; returns c11, c12, c13, c22, c23, c33
__device__ __forceinline__ void iadInvert(double t11, double t12, double t13, double t22, double t23, double t33,
                                          double hi, double K, double out[6])
{
    auto getExp   = [](double v) { return v == 0.0 ? 0 : ilogb(v); };
    int  expSum   = getExp(t11) + getExp(t12) + getExp(t13) + getExp(t22) + getExp(t23) + getExp(t33);
    double norm   = ldexp(1.0, -expSum / 6);
    t11 *= norm, t12 *= norm, t13 *= norm, t22 *= norm, t23 *= norm, t33 *= norm;
    double det    = t11 * t22 * t33 + 2.0 * t12 * t23 * t13 - t11 * t23 * t23 - t22 * t13 * t13 - t33 * t12 * t12;
    double factor = norm * (hi * hi * hi) / (det * K);
    out[0]        = (t22 * t33 - t23 * t23) * factor;
    out[1]        = (t13 * t23 - t33 * t12) * factor;
    out[2]        = (t12 * t23 - t22 * t13) * factor;
    out[3]        = (t11 * t33 - t13 * t13) * factor;
    out[4]        = (t13 * t12 - t11 * t23) * factor;
    out[5]        = (t11 * t22 - t12 * t12) * factor;
}

//! tsKCourant (sph/include/sph/kernels.hpp:11-16); Kcour is passed as float like the reference
template<class T>
__device__ __forceinline__ double courantDt(T maxvs, T h, T c, float Kcour)
{
    T v = maxvs > T(0) ? maxvs : c;
    return double(T(Kcour * h / v));
}

//! artificial_viscosity (kernels.hpp:71-84), beta = 2: -vsig w for approaching particles, else 0, without a
//! branch (a NaN of coincident particles gives 0, as the comparison would)
template<class T>
__device__ __forceinline__ T artificialViscosity(T alpha_i, T alpha_j, T c_sum, T w_ij)
{
    constexpr T beta = 2.0;
    const T     w    = w_ij < T(0) ? w_ij : T(0);
    return (beta * w - (alpha_i + alpha_j) * T(0.25) * c_sum) * w;
}

//! arguments shared by all pair kernels
struct PairArgs
{
    const double* x;
    const double* y;
    const double* z;
    DevBox        box;
    double        K;
    Lists         L;
    uint32_t      numParticles; // all particles that can appear as neighbours
};

inline PairArgs makePairArgs(sphx_workspace* ws, const DevBox& box, const sphx_fields_t* f, const sphx_params_t* p,
                             uint32_t first, uint32_t last)
{
    SPHX_REQUIRE(ws->nbValid, SPHX_ERR_STATE, "pair loop called before find_neighbors");
    SPHX_REQUIRE(ws->nbFirst <= first && first <= last && last <= ws->nbLast, SPHX_ERR_ARG,
                 "target range must stay inside the searched range");
    SPHX_REQUIRE(p->ngmax == ws->nbNgmax, SPHX_ERR_ARG, "ngmax differs from the one used by find_neighbors");
    SPHX_REQUIRE(ws->tablesValid, SPHX_ERR_STATE, "kernel tables not set (sphx_workspace_set_kernel)");
    SPHX_REQUIRE(f->x && f->y && f->z && f->nc, SPHX_ERR_ARG, "x, y, z and nc are required");
    PairArgs c;
    c.x = f->x, c.y = f->y, c.z = f->z, c.box = box, c.K = p->K;
    const Groups G = groupsFor(ws, first, last);
    const bool   whole = !ws->nbOwned && G.start == nullptr && (first - ws->nbFirst) % kGroup == 0;
    c.L = Lists{neighborLists(ws), f->nc,    ws->nbFirst, ws->nbLast, p->ngmax, 0,
                whole ? (first - ws->nbFirst) / kGroup : Lists::kNoBlock, ws->nbPartial, G};
    c.numParticles = uint32_t(ws->tree.numParticles);
    return c;
}

//! the kernel function of form T for the device (the workspace's tables, or its sinc index)
template<class T>
inline SincKernel<T> sincKernel(sphx_workspace* ws)
{
    SincKernel<T> k;
    if constexpr (isMixed<T>)
    {
        const double n = ws->sincIndex;
        k.n            = float(n);
        k.ni           = n == double(int(n)) && n >= 2 && n < 64 ? int(n) : -1;
    }
    else
    {
        k.wTab  = ws->wh64.get();
        k.wqTab = ws->whq64.get();
    }
    return k;
}

/*! block minimum (its first wave's lanes) then one atomic per block; with per-group steps (block time steps), also
 * groupDt[g] = min(groupDt[g], the group's minimum) as a float (hydro_ve/momentum_energy_gpu.cu:96-104) */
__device__ __forceinline__ void reduceMinDt(unsigned long long* dst, double dt, const Groups& G)
{
    double m = waveMin(dt);
    if (threadIdx.x == 0)
    {
        atomicMinPositive(dst, m);
        const uint32_t g = blockGroup();
        if (G.dt != nullptr && g < G.num) { G.dt[g] = fminf(G.dt[g], float(m)); }
    }
}

} // namespace sphx
