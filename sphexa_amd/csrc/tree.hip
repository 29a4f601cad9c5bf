// Cornerstone leaf array + linked octree + layout + geometric node centres, built from the sorted keys at once.
//
// The reference converges a leaf array by repeated count/split/merge sweeps (computeOctree,
// domain/include/cstone/tree/csarray.hpp:409-440) and then derives the internal tree by sorting
// placeholder-bit prefixes (buildOctreeGpu, tree/octree_gpu.cu:137-157). Its fixed point is
// unique: a node is internal iff it holds more than `bucket` particles and lies above the
// deepest level. That can be read off the sorted keys without descending level by level: the node of level l whose
// first particle is i is internal iff key i - 1 lies outside it and key i + bucket inside. So
//  1. every key counts the levels at which it opens an internal node (planCountKernel), per block and level;
//  2. a scan gives each internal node its rank in the reference's node order, which is level by level and
//     along the curve within a level, and its place in depth-first order (planScanKernel, planEmitKernel);
//  3. eight threads per internal node link its children (childKernel): the r-th internal node's children are nodes
//     1 + 8 r .. 8 + 8 r; a leaf's place in the leaf array and the leaves below a node follow from
//     depth-first places, each split adding seven leaves;
//  4. every node adds up its place in the search's visiting order along its ancestors (visitKernel).
// Five launches and one host read of the internal nodes per level, where a level-by-level descent took about forty
// launches and a read per level. What bounds it: launch latency up to about a million particles, then reading the
// keys twice and the chains of searches in childKernel (33 us at 1M particles by halves, 19 with seven probes
// at a time). Measured, a whole std step with
// the former descent and with this: 0.65 -> 0.51 ms at 1728 particles (FP64), 1.98 -> 1.77 ms at 1M (mixed); a mixed VE
// step at 8M 15.2 -> 14.8 ms.
#include <cstring> // rocprim uses memset without including it
#include <rocprim/rocprim.hpp>

#include "common.hpp"

namespace sphx
{

namespace
{

/*! first index in [lo, hi) whose key is at least v, else hi. Seven probes at a time: what a search costs is its chain of
 * dependent loads, a third as long as by halves. */
__device__ __forceinline__ uint32_t lowerBound(const Key* __restrict__ keys, uint32_t lo, uint32_t hi, Key v)
{
    while (hi - lo >= 8)
    {
        const uint32_t step  = (hi - lo) / 8;
        uint32_t       below = 0;
#pragma unroll
        for (uint32_t i = 1; i < 8; ++i)
            below += keys[lo + i * step] < v ? 1u : 0u;
        hi = below < 7 ? lo + (below + 1) * step : hi;
        lo = below > 0 ? lo + below * step + 1 : lo;
    }
    if (lo == hi) { return lo; }
    uint32_t below = 0;
#pragma unroll
    for (uint32_t i = 0; i < 7; ++i)
    {
        const Key k = keys[min(lo + i, hi - 1)]; // (all loads go out together)
        below += lo + i < hi && k < v ? 1u : 0u;
    }
    return lo + below;
}

//! the same in [lo, n), for searches that end soon: eight probes at doubling distances bracket the end
__device__ __forceinline__ uint32_t lowerBoundFrom(const Key* __restrict__ keys, uint32_t lo, uint32_t n, Key v)
{
    if (lo >= n) { return n; }
    uint32_t a = lo;
    for (uint64_t step = 16;; step <<= 8)
    {
        uint32_t below = 0;
#pragma unroll
        for (int k = 0; k < 8; ++k)
        {
            const uint64_t q = lo + (step << k);
            below += keys[q < n ? q : n - 1] < v && q < n ? 1u : 0u;
        }
        if (below > 0) { a = uint32_t(lo + (step << (below - 1))) + 1; }
        if (below < 8)
        {
            const uint64_t end = lo + (step << below);
            return lowerBound(keys, a, uint32_t(end < n ? end : n), v);
        }
    }
}

constexpr unsigned kPlanWaves = 4;
constexpr unsigned kPlanTiles = 8; // tiles of 64 keys per wave
constexpr unsigned kPlanKeys  = kPlanWaves * kPlanTiles * kWave;
constexpr unsigned kPlanRows  = kMaxLevel + 1; // internal nodes per level, then keys out of order

//! keys past the curve (removed particles) count as its last one
__device__ __forceinline__ Key onCurve(Key k)
{
    constexpr Key last = (Key(1) << 63) - 1;
    return k < last ? k : last;
}

//! deepest level whose node holds both keys
__device__ __forceinline__ int commonLevel(Key a, Key b)
{
    a = onCurve(a), b = onCurve(b);
    return a == b ? int(kMaxLevel) : (__builtin_clzll(a ^ b) - 1) / 3;
}

//! key i is the first of the internal nodes of levels (p, l] (none when l <= p)
__device__ __forceinline__ void openedLevels(const Key* __restrict__ keys, uint32_t n, unsigned bucket, uint32_t i, int& p,
                                             int& l)
{
    p = 0, l = -1;
    if (i >= n) { return; }
    const Key      k = keys[i];
    const uint64_t j = uint64_t(i) + bucket;
    if (j < n) { l = min(commonLevel(k, keys[j]), int(kMaxLevel) - 1); }
    p = i == 0 ? -1 : commonLevel(keys[i - 1], k);
}

//! internal nodes per level (row) that the keys of each block open: counts[level * gridDim.x + block]; the last row
//! counts the keys below their predecessor, from which no tree can be linked
__global__ void __launch_bounds__(kPlanWaves* kWave)
    planCountKernel(const Key* __restrict__ keys, uint32_t n, unsigned bucket, uint32_t* __restrict__ counts)
{
    __shared__ uint32_t cnt[kPlanRows];
    if (threadIdx.x < kPlanRows) { cnt[threadIdx.x] = 0; }
    __syncthreads();
    for (unsigned t = 0; t < kPlanTiles; ++t)
    {
        const uint32_t i = blockIdx.x * kPlanKeys + t * kPlanWaves * kWave + threadIdx.x;
        int            p, l;
        openedLevels(keys, n, bucket, i, p, l);
        for (int v = p + 1; v <= l; ++v)
            atomicAdd(&cnt[v], 1u);
        if (i > 0 && i < n && keys[i] < keys[i - 1]) { atomicAdd(&cnt[kMaxLevel], 1u); }
    }
    __syncthreads();
    if (threadIdx.x < kPlanRows) { counts[size_t(threadIdx.x) * gridDim.x + blockIdx.x] = cnt[threadIdx.x]; }
}

//! block l: exclusive scan of row l of `counts` in place, and its total
__global__ void __launch_bounds__(256) planScanKernel(uint32_t* __restrict__ counts, uint32_t blocks,
                                                      uint32_t* __restrict__ totals)
{
    __shared__ uint32_t part[256 / kWave];
    uint32_t*           row  = counts + size_t(blockIdx.x) * blocks;
    const unsigned      lane = laneId(), w = threadIdx.x / kWave;
    uint32_t            run  = 0;
    for (uint32_t b0 = 0; b0 < blocks; b0 += 256)
    {
        const uint32_t b    = b0 + threadIdx.x;
        const uint32_t v    = b < blocks ? row[b] : 0u;
        uint32_t       incl = v;
        for (int o = 1; o < kWave; o <<= 1)
        {
            const uint32_t x = __shfl_up(incl, o, kWave);
            incl += lane >= unsigned(o) ? x : 0u;
        }
        if (lane == kWave - 1) { part[w] = incl; }
        __syncthreads();
        uint32_t before = run, all = 0;
        for (unsigned q = 0; q < 256 / kWave; ++q)
        {
            before += q < w ? part[q] : 0u;
            all += part[q];
        }
        if (b < blocks) { row[b] = before + incl - v; }
        run += all;
        __syncthreads();
    }
    if (threadIdx.x == 0) { totals[blockIdx.x] = run; }
}

//! internal nodes of the shallower levels, per level (kernel argument; [kMaxLevel]: all of them)
struct LevelBase
{
    uint32_t base[kMaxLevel + 1];
};

//! the internal nodes by rank (level by level) and in depth-first order
struct InternalNodes
{
    Key*      key;   // by rank: first key of the node ...
    uint32_t* lo;    // ... first particle ...
    uint32_t* place; // ... and its place in depth-first order
    Key*      dfKey; // by place: first key ...
    uint32_t* rank;  // ... and rank
    uint32_t* push;  // by rank: children from last to first visited (childPush)
};

//! writes the internal nodes; the waves of a block take consecutive runs of its keys
__global__ void __launch_bounds__(kPlanWaves* kWave)
    planEmitKernel(const Key* __restrict__ keys, uint32_t n, unsigned bucket, const uint32_t* __restrict__ counts,
                   LevelBase levels, InternalNodes out)
{
    __shared__ uint32_t next[kPlanWaves][kMaxLevel]; // count, then rank of the wave's first node, per level
    __shared__ uint32_t place[kPlanWaves];           // depth-first place of its first node
    const unsigned      w = threadIdx.x / kWave, lane = laneId();
    const uint32_t      first = blockIdx.x * kPlanKeys + w * kPlanTiles * kWave;
    if (lane < kMaxLevel) { next[w][lane] = 0; }
    __syncthreads();
    int p[kPlanTiles], l[kPlanTiles];
#pragma unroll
    for (unsigned t = 0; t < kPlanTiles; ++t)
    {
        openedLevels(keys, n, bucket, first + t * kWave + lane, p[t], l[t]);
        for (int v = p[t] + 1; v <= l[t]; ++v)
            atomicAdd(&next[w][v], 1u);
    }
    __syncthreads();
    if (w == 0)
    {
        uint32_t before = lane < kMaxLevel ? counts[size_t(lane) * gridDim.x + blockIdx.x] : 0u;
        for (unsigned q = 0; q < kPlanWaves; ++q)
        {
            const uint32_t all = waveSum(before);
            if (lane == 0) { place[q] = all; }
            if (lane < kMaxLevel)
            {
                const uint32_t c = next[q][lane];
                next[q][lane]    = levels.base[lane] + before;
                before += c;
            }
        }
    }
    __syncthreads();
    uint32_t at = place[w], r = lane < kMaxLevel ? next[w][lane] : 0u; // lane v holds the next rank of level v
#pragma unroll
    for (unsigned t = 0; t < kPlanTiles; ++t)
    {
        uint64_t open = ballot(l[t] > p[t]);
        while (open)
        {
            const int s = __builtin_ctzll(open);
            open &= open - 1;
            const int      from = __builtin_amdgcn_readlane(p[t], s) + 1, to = __builtin_amdgcn_readlane(l[t], s);
            const uint32_t i    = first + t * kWave + uint32_t(s);
            if (int(lane) >= from && int(lane) <= to)
            {
                const Key      k = onCurve(keys[i]) & ~(nodeRange(lane) - 1);
                const uint32_t q = at + lane - uint32_t(from); // outermost first
                out.key[r] = k, out.lo[r] = i, out.place[r] = q;
                out.dfKey[q] = k, out.rank[q] = r;
                ++r;
            }
            at += uint32_t(to - from + 1);
        }
    }
}

//! arrays of the linked tree (Tree) as kernel arguments
struct TreeArrays
{
    Key *          prefixes, *leaves;
    TreeNodeIndex *childOffsets, *parents, *internalToLeaf, *levelRange;
    uint32_t *     counts, *layout, *childPush;
    int32_t *      rankLo, *offset; // offset: leaves visited between a node's parent's first leaf and its own
    double *       centers, *sizes;
};

//! geometric centre and half size of the node of key k and level l: hilbertIBox + centerAndSize
//! (sfc/hilbert.hpp:259-274, sfc/box.hpp:318-334)
__device__ __forceinline__ void nodeBox(const DevBox& box, Key k, unsigned l, size_t i, double* centers, double* sizes)
{
#pragma clang fp contract(off)
    unsigned ix, iy, iz;
    hilbertDecode(k, ix, iy, iz);
    unsigned     cube = (1u << kMaxLevel) >> l;
    unsigned     mask = ~(cube - 1);
    unsigned     ic[3] = {ix & mask, iy & mask, iz & mask};
    const double uL    = 1.0 / double(1u << kMaxLevel);
    for (int d = 0; d < 3; ++d)
    {
        int    imin = int(ic[d]), imax = int(ic[d] + cube);
        double half = 0.5 * uL * box.len[d];
        centers[3 * i + d] = box.lo[d] + double(imax + imin) * half;
        sizes[3 * i + d]   = double(imax - imin) * half;
    }
}

/*! Eight threads per internal node, thread c its c-th child: the child's particles, links, box, its place in the leaf
 * array or its rank, and the visiting order among its siblings. singleTraversal (traversal/traversal.hpp:52-93) handles
 * a node's leaf children in octant order as it meets them, pushes its internal children in octant order and pops
 * the last pushed first. */
__global__ void __launch_bounds__(256) childKernel(const Key* __restrict__ keys, uint32_t n, unsigned bucket,
                                                   LevelBase levels, InternalNodes in, DevBox box, TreeArrays t)
{
    const uint32_t id = blockIdx.x * blockDim.x + threadIdx.x, total = levels.base[kMaxLevel];
    const uint32_t r = id / 8;
    const int      c = int(id % 8);
    if (r >= total) { return; } // uniform over the node's 8 threads
    unsigned l = 0;
    while (levels.base[l + 1] <= r) { ++l; }
    const Key      range = nodeRange(l + 1), k = in.key[r] + Key(c) * range;
    const uint32_t place = in.place[r];
    const bool     atEnd = in.key[r] + 8 * range == nodeRange(0);

    // particles and depth-first places of the child: its own first (the first child's are the node's), and the next
    // child's; thread 0 finds the node's end
    const uint32_t lo0 = in.lo[r];
    const Key      sought = c == 0 ? k + 8 * range : k;
    uint32_t       first = lowerBoundFrom(keys, lo0, n, sought), q0 = lowerBoundFrom(in.dfKey, place + 1, total, sought);
    const uint32_t end = atEnd ? n : __shfl(first, 0, 8), qEnd = atEnd ? total : __shfl(q0, 0, 8);
    if (c == 0) { first = lo0, q0 = place + 1; }
    uint32_t last = __shfl_down(first, 1, 8), q1 = __shfl_down(q0, 1, 8);
    if (c == 7) { last = end, q1 = qEnd; }
    const uint32_t node   = 1 + id;
    const bool     leaf   = last - first <= bucket || l + 1 >= kMaxLevel;
    const int32_t  leaves = leaf ? 1 : 1 + 7 * int32_t(q1 - q0);
    t.prefixes[node]      = encodePlaceholder(k, 3 * (l + 1));
    nodeBox(box, k, l + 1, node, t.centers, t.sizes);
    if (leaf)
    {
        // leaves before it: its preceding siblings on the way down as one each, and seven per internal
        // node that ended before (those before it in depth-first order without its l + 1 ancestors)
        uint32_t digits = 0;
        for (unsigned v = 1; v <= l + 1; ++v)
            digits += unsigned(k >> (3 * (kMaxLevel - v))) & 7u;
        const uint32_t at      = digits + 7 * (q0 - (l + 1));
        t.childOffsets[node]   = 0;
        t.internalToLeaf[node] = TreeNodeIndex(at);
        t.leaves[at] = k, t.counts[at] = last - first, t.layout[at] = first;
    }
    else
    {
        const uint32_t rank    = in.rank[q0];
        t.childOffsets[node]   = TreeNodeIndex(1 + 8 * rank);
        t.parents[rank]        = TreeNodeIndex(node);
        t.internalToLeaf[node] = -1;
    }
    // visiting order among the siblings
    const unsigned mask   = unsigned(ballot(leaf) >> (laneId() & ~7u)) & 0xffu;
    const int      nLeaf  = __popc(mask);
    int32_t        offset = leaf ? __popc(mask & ((1u << c) - 1u)) : nLeaf;
    int            pos    = leaf ? offset : nLeaf;
    for (int o = 1; o < 8; ++o)
    {
        const int32_t other = __shfl(leaves, o, 8);
        if (!leaf && o > c && !((mask >> o) & 1u)) { offset += other, ++pos; }
    }
    uint32_t push = uint32_t(c) << (3 * (7 - pos));
    push |= __shfl_xor(push, 1, 8), push |= __shfl_xor(push, 2, 8), push |= __shfl_xor(push, 4, 8);
    t.offset[node] = offset;
    if (c == 0) { in.push[r] = push; }
    if (id == 0)
    {
        t.prefixes[0] = encodePlaceholder(0, 0), t.childOffsets[0] = 1, t.parents[0] = 0, t.internalToLeaf[0] = -1;
        t.offset[0] = 0;
        nodeBox(box, 0, 0, 0, t.centers, t.sizes);
        const uint32_t L = 1 + 7 * total;
        t.leaves[L] = nodeRange(0), t.layout[L] = n;
    }
}

//! a node's place in the visiting order, along its ancestors; children's order of internal nodes; level ranges
__global__ void __launch_bounds__(256) visitKernel(LevelBase levels, InternalNodes in, TreeArrays t)
{
    const uint32_t node = blockIdx.x * blockDim.x + threadIdx.x, numNodes = 1 + 8 * levels.base[kMaxLevel];
    if (node <= kMaxLevel + 1)
    {
        // level l + 1 holds the children of level l; the levels below the deepest start at the end
        t.levelRange[node] = node == 0 ? 0 : TreeNodeIndex(node <= kMaxLevel ? 1 + 8 * levels.base[node - 1] : numNodes);
    }
    if (node >= numNodes) { return; }
    int32_t rank = 0;
    for (TreeNodeIndex a = TreeNodeIndex(node); a > 0; a = t.parents[(a - 1) / 8])
        rank += t.offset[a];
    t.rankLo[node]            = rank;
    const TreeNodeIndex child = t.childOffsets[node];
    t.childPush[node]         = child ? in.push[(child - 1) / 8] : 0u;
}

//! the tree of at most `bucket` keys: the root as its only leaf
__global__ void rootLeafKernel(uint32_t n, DevBox box, TreeArrays t)
{
    if (threadIdx.x <= kMaxLevel + 1) { t.levelRange[threadIdx.x] = threadIdx.x == 0 ? 0 : 1; }
    if (threadIdx.x > 0) { return; }
    t.prefixes[0] = encodePlaceholder(0, 0), t.childOffsets[0] = 0, t.internalToLeaf[0] = 0;
    t.leaves[0] = 0, t.leaves[1] = nodeRange(0);
    t.counts[0] = n, t.layout[0] = 0, t.layout[1] = n;
    t.parents[0] = 0, t.rankLo[0] = 0, t.childPush[0] = 0;
    nodeBox(box, 0, 0, 0, t.centers, t.sizes);
}

/* The linked tree whose nodes are exactly the octree nodes holding more than `bucket` of the sorted
 * keys `keys` (and their children): the converged cornerstone tree of particle keys with the bucket
 * size, or, with bucket 1 and the leaf starts of a cornerstone array as keys, the octree of that leaf
 * array (a node is internal iff more than one leaf starts inside it). Leaf counts and layout come out
 * in units of keys. */
void buildLinked(sphx_workspace* ws, const Key* keys, size_t nParticles, unsigned bucket, const DevBox& box)
{
    hipStream_t    st     = ws->stream;
    const uint32_t n      = uint32_t(nParticles);
    auto&          s      = ws->tree.build;
    const uint32_t blocks = std::max(1u, ceilDiv(n, kPlanKeys));
    ws->tree.valid        = false; // until it is linked: no search over the former tree, or half of this one, after an error
    s.planCounts.reserve(size_t(blocks) * kPlanRows + kPlanRows);
    uint32_t* counts = s.planCounts.get();
    uint32_t* totals = counts + size_t(blocks) * kPlanRows;
    planCountKernel<<<blocks, kPlanWaves * kWave, 0, st>>>(keys, n, bucket, counts);
    SPHX_CHECK_LAUNCH();
    planScanKernel<<<kPlanRows, 256, 0, st>>>(counts, blocks, totals);
    SPHX_CHECK_LAUNCH();
    uint32_t perLevel[kPlanRows];
    SPHX_HIP(hipMemcpyAsync(perLevel, totals, sizeof(perLevel), hipMemcpyDeviceToHost, st));
    SPHX_HIP(hipStreamSynchronize(st));
    SPHX_REQUIRE(perLevel[kMaxLevel] == 0, SPHX_ERR_ARG, "the keys of a tree must be sorted");
    LevelBase levels;
    levels.base[0] = 0;
    for (unsigned l = 0; l < kMaxLevel; ++l)
        levels.base[l + 1] = levels.base[l] + perLevel[l];
    const uint32_t numInternal = levels.base[kMaxLevel], numNodes = 1 + 8 * numInternal, L = 1 + 7 * numInternal;

    Tree& t = ws->tree;
    t.prefixes.reserve(numNodes), t.childOffsets.reserve(numNodes + 1), t.internalToLeaf.reserve(numNodes);
    t.parents.reserve(std::max(1u, numInternal)), t.levelRange.reserve(kMaxLevel + 2);
    t.centers.reserve(3 * size_t(numNodes)), t.sizes.reserve(3 * size_t(numNodes));
    t.leaves.reserve(L + 1), t.counts.reserve(L), t.layout.reserve(L + 1);
    t.rankLo.reserve(numNodes), t.offset.reserve(numNodes), t.childPush.reserve(numNodes);
    const TreeArrays arrays{t.prefixes.get(), t.leaves.get(),  t.childOffsets.get(), t.parents.get(), t.internalToLeaf.get(),
                            t.levelRange.get(), t.counts.get(), t.layout.get(),      t.childPush.get(), t.rankLo.get(),
                            t.offset.get(),   t.centers.get(), t.sizes.get()};
    if (numInternal == 0)
    {
        rootLeafKernel<<<1, kWave, 0, st>>>(n, box, arrays);
        SPHX_CHECK_LAUNCH();
    }
    else
    {
        s.intKey.reserve(numInternal), s.intLo.reserve(numInternal), s.intPlace.reserve(numInternal);
        s.dfKey.reserve(numInternal), s.dfRank.reserve(numInternal), s.intPush.reserve(numInternal);
        const InternalNodes in{s.intKey.get(), s.intLo.get(),  s.intPlace.get(),
                               s.dfKey.get(),  s.dfRank.get(), s.intPush.get()};
        planEmitKernel<<<blocks, kPlanWaves * kWave, 0, st>>>(keys, n, bucket, counts, levels, in);
        SPHX_CHECK_LAUNCH();
        childKernel<<<ceilDiv(8 * size_t(numInternal), 256), 256, 0, st>>>(keys, n, bucket, levels, in, box, arrays);
        SPHX_CHECK_LAUNCH();
        visitKernel<<<ceilDiv(numNodes, 256), 256, 0, st>>>(levels, in, arrays);
        SPHX_CHECK_LAUNCH();
    }
    t.numLeafNodes     = int32_t(L);
    t.numInternalNodes = int32_t(numInternal);
    t.numNodes         = int32_t(numNodes);
    t.numParticles     = nParticles;
    t.valid            = true;
}

//! particle count of every node of the tree: a leaf's from its count, an internal node's from the layout
//! of the leaves it spans
__global__ void nodeCountKernel(const Key* __restrict__ prefixes, const TreeNodeIndex* __restrict__ childOffsets,
                                const TreeNodeIndex* __restrict__ internalToLeaf, const Key* __restrict__ leaves,
                                const uint32_t* __restrict__ layout, const uint32_t* __restrict__ counts, uint32_t L,
                                uint32_t N, uint32_t* __restrict__ nodeCnt, int32_t* __restrict__ leafOp)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) { return; }
    if (i == 0) { leafOp[L] = 0, leafOp[L + 1] = 0; } // the scan's end, and no change so far
    if (childOffsets[i] == 0)
    {
        nodeCnt[i] = counts[internalToLeaf[i]];
        return;
    }
    const Key      p     = prefixes[i];
    const Key      start = decodePlaceholder(p);
    const Key      end   = start + nodeRange(decodePrefixLength(p) / 3u);
    const uint32_t a     = lowerBound(leaves, 0, L, start);
    const uint32_t b     = lowerBound(leaves, a, L + 1, end);
    nodeCnt[i]           = layout[b] - layout[a];
}

/* mergeCountAndMacOp (focus/rebalance.hpp:31-68) on one rank, the focus spanning every key: node i > 0
 * merges (0) when its parent holds at most `bucket` particles; a leaf above the deepest level holding
 * more splits in 8; else 1 */
__global__ void nodeOpKernel(const Key* __restrict__ prefixes, const TreeNodeIndex* __restrict__ childOffsets,
                             const TreeNodeIndex* __restrict__ parents, const uint32_t* __restrict__ nodeCnt,
                             uint32_t N, unsigned bucket, int32_t* __restrict__ op)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) { return; }
    if (i > 0 && nodeCnt[parents[(i - 1) / 8]] <= bucket)
    {
        op[i] = 0;
        return;
    }
    const unsigned level = decodePrefixLength(prefixes[i]) / 3u;
    op[i]                = (childOffsets[i] == 0 && level < kMaxLevel && nodeCnt[i] > bucket) ? 8 : 1;
}

/* protectAncestors / nzAncestorOp (focus/rebalance.hpp:88-107,219-233) for every node, reading the ops
 * before protection: a node marked 0 takes the op of its closest ancestor not marked 0 when it is that
 * ancestor's first descendant, else stays 0. An ancestor marked 0 that protection would turn to 1 is the
 * first descendant of its own closest unmarked ancestor, so walking past it gives the same answer as the
 * reference's in-place loop. Leaves store their final op by leaf index; any node left != 1 marks a change. */
__global__ void protectKernel(const Key* __restrict__ prefixes, const TreeNodeIndex* __restrict__ parents,
                              const TreeNodeIndex* __restrict__ internalToLeaf, const int32_t* __restrict__ op,
                              uint32_t N, int32_t* __restrict__ leafOp, int32_t* __restrict__ changed)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) { return; }
    int32_t o = op[i];
    if (o == 0) // never the root
    {
        TreeNodeIndex a = TreeNodeIndex(i);
        while (op[a] == 0) { a = parents[(a - 1) / 8]; }
        o = decodePlaceholder(prefixes[i]) == decodePlaceholder(prefixes[a]) ? op[a] : 0;
    }
    if (o != 1) { *changed = 1; }
    const TreeNodeIndex leaf = internalToLeaf[i];
    if (leaf >= 0) { leafOp[leaf] = o; }
}

//! rebalanceTree / processNode (tree/csarray.hpp:340-389) with ops 0, 1 and 8 at offsets `offs`
__global__ void rebalanceKernel(const Key* __restrict__ leaves, const int32_t* __restrict__ offs, uint32_t L,
                                Key* __restrict__ next)
{
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s > L) { return; }
    if (s == L)
    {
        next[offs[L]] = leaves[L];
        return;
    }
    const Key      node = leaves[s];
    const int32_t  k    = offs[s + 1] - offs[s];
    if (k == 1) { next[offs[s]] = node; }
    else if (k == 8)
    {
        const Key r = nodeRange(treeLevel(leaves[s + 1] - node) + 1u);
        for (int c = 0; c < 8; ++c)
            next[offs[s] + c] = node + Key(c) * r;
    }
}

//! first particle and count of every leaf of the linked leaf array (computeNodeCounts)
__global__ void leafLayoutKernel(const Key* __restrict__ leaves, uint32_t L, const Key* __restrict__ keys, uint32_t n,
                                 uint32_t* __restrict__ layout, uint32_t* __restrict__ counts)
{
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s > L) { return; }
    const uint32_t lo   = s == L ? n : lowerBound(keys, 0, n, leaves[s]);
    uint32_t       next = __shfl_down(lo, 1, kWave); // the next leaf's, by the lane beside
    if (s < L && laneId() == kWave - 1) { next = s + 1 == L ? n : lowerBoundFrom(keys, lo, n, leaves[s + 1]); }
    layout[s] = lo;
    if (s < L) { counts[s] = next - lo; }
}

} // namespace

void buildTree(sphx_workspace* ws, const Key* keys, size_t nParticles, unsigned bucket, const DevBox& box)
{
    SPHX_REQUIRE(nParticles < (size_t(1) << 32), SPHX_ERR_ARG, "particle count must fit 32-bit indices");
    SPHX_REQUIRE(bucket >= 1, SPHX_ERR_ARG, "bucket size must be positive");
    buildLinked(ws, keys, nParticles, bucket, box);
}

bool updateTree(sphx_workspace* ws, const Key* keys, size_t nParticles, unsigned bucket, const DevBox& box)
{
    SPHX_REQUIRE(nParticles < (size_t(1) << 32), SPHX_ERR_ARG, "particle count must fit 32-bit indices");
    SPHX_REQUIRE(bucket >= 1, SPHX_ERR_ARG, "bucket size must be positive");
    Tree& t = ws->tree;
    SPHX_REQUIRE(t.valid, SPHX_ERR_STATE, "no tree to update");
    hipStream_t    st = ws->stream;
    auto&          s  = t.build;
    const uint32_t N = uint32_t(t.numNodes), L = uint32_t(t.numLeafNodes);
    s.nodeCnt.reserve(N), s.nodeOp.reserve(N), s.leafOp.reserve(size_t(L) + 2);
    int32_t* changed = s.leafOp.get() + L + 1; // behind the leaves' ops and their end, so one read takes both
    nodeCountKernel<<<ceilDiv(N, 256), 256, 0, st>>>(t.prefixes.get(), t.childOffsets.get(), t.internalToLeaf.get(),
                                                      t.leaves.get(), t.layout.get(), t.counts.get(), L, N,
                                                      s.nodeCnt.get(), s.leafOp.get());
    SPHX_CHECK_LAUNCH();
    nodeOpKernel<<<ceilDiv(N, 256), 256, 0, st>>>(t.prefixes.get(), t.childOffsets.get(), t.parents.get(),
                                                   s.nodeCnt.get(), N, bucket, s.nodeOp.get());
    SPHX_CHECK_LAUNCH();
    protectKernel<<<ceilDiv(N, 256), 256, 0, st>>>(t.prefixes.get(), t.parents.get(), t.internalToLeaf.get(),
                                                    s.nodeOp.get(), N, s.leafOp.get(), changed);
    SPHX_CHECK_LAUNCH();
    size_t bytes = 0;
    SPHX_HIP(rocprim::exclusive_scan(nullptr, bytes, s.leafOp.get(), s.leafOp.get(), 0, size_t(L) + 1,
                                     rocprim::plus<int32_t>(), st));
    SPHX_HIP(rocprim::exclusive_scan(scratchBytes(ws, bytes), bytes, s.leafOp.get(), s.leafOp.get(), 0,
                                     size_t(L) + 1, rocprim::plus<int32_t>(), st));
    int32_t read[2]; // leaves of the new array, whether any node changed
    SPHX_HIP(hipMemcpyAsync(read, s.leafOp.get() + L, sizeof(read), hipMemcpyDeviceToHost, st));
    SPHX_HIP(hipStreamSynchronize(st));
    const int32_t newL      = read[0];
    const bool    unchanged = read[1] == 0;
    SPHX_REQUIRE(newL >= 1, SPHX_ERR_STATE, "tree update left no leaf");
    s.nextLeaves.reserve(size_t(newL) + 1);
    rebalanceKernel<<<ceilDiv(size_t(L) + 1, 256), 256, 0, st>>>(t.leaves.get(), s.leafOp.get(), L,
                                                                 s.nextLeaves.get());
    SPHX_CHECK_LAUNCH();

    // link the new leaf array (its leaf starts as the keys, one per leaf), then count the particles
    buildLinked(ws, s.nextLeaves.get(), size_t(newL), 1, box);
    t.valid = false; // its layout is of leaves until the particles are counted
    SPHX_REQUIRE(t.numLeafNodes == newL, SPHX_ERR_STATE, "linking the updated leaves changed their number");
    const uint32_t n = uint32_t(nParticles);
    leafLayoutKernel<<<ceilDiv(size_t(newL) + 1, 256), 256, 0, st>>>(t.leaves.get(), uint32_t(newL), keys, n,
                                                                     t.layout.get(), t.counts.get());
    SPHX_CHECK_LAUNCH();
    t.numParticles = nParticles;
    t.valid        = true;
    return unchanged;
}

} // namespace sphx
