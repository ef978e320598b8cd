// sphx_neighbors.hip - wave64 target-group neighbor search.
//
// A target group is up to 64 SFC-consecutive particles.
//   nsGroupRanges : one wave per group: breadth-first walk of the octree with the group's
//                   search box (union of the targets' 2h spheres, minimum image in periodic
//                   dimensions); overlapping leaves are collected in LDS, put in order
//                   (leaf order = SFC order = particle order) and merged into
//                   contiguous particle ranges, in pieces of at most 64 particles.
//   nsCandidates  : one workgroup of four waves per group streams the pieces and finds hits with
//                   FP32 tests on the matrix cores; a pair that FP32 cannot decide
//                   follows the reference predicate d^2 < (2h)^2 in FP64 with separately
//                   rounded operations (findneighbors.hpp:33-60,115-140), so the neighbor sets are bit-identical to the CPU path; hits are
//                   appended in ascending j, which is also the CPU's depth-first
//                   order, so truncation at ngmax keeps the same entries.
//   nsCandidatesExact : the same result with FP64 tests only, for groups with a list to be cut at
//                   ngmax (targets that stay beyond it after the h iteration), whose search box
//                   has no single nearest image, with candidates outside a periodic domain, with
//                   extreme units, or with too many pieces.
// The smoothing-length iteration of findNeighborsSph (sph/find_neighbors.hpp:10-41)
// re-runs only the groups that still have particles outside [ng0/4, ngmax + 1].
#include <algorithm>
#include <climits>
#include <cstddef>
#include <type_traits>

#include "sphx_internal.hpp"

namespace sphx
{

// traversal capacities: every group is first walked with the small ones (LDS for more
// waves per CU); the groups that exceed them are walked again with the large ones
constexpr int NS_FCAP_SMALL = 512;  // BFS frontier capacity (per buffer)
constexpr int NS_LCAP_SMALL = 512;  // candidate leaves per group
constexpr int NS_FCAP       = 2048;
constexpr int NS_LCAP       = 1024; // also the stride of the per-group range lists

struct NsFlags
{
    uint32_t           redoCount;  // groups appended to the redo list
    uint32_t           overflow;   // traversal capacity exceeded
    uint32_t           badGroup;   // a group with more than 64 particles
    uint32_t           retryCount; // groups that exceeded the small traversal capacities
    uint32_t           hfacMiss;   // a count to update h from lies beyond the factor table
    unsigned long long tests;      // (target, candidate) distance tests of this pass
    unsigned long long listTests;  // after the first pass: those of every group's last pass
    uint32_t           overCount;  // groups that nsCandidates leaves to nsCandidatesExact
};

// minimum and maximum over the wave's numbers, the same in every lane: a NaN (of a particle without a
// usable position or h) is left out
__device__ inline double waveMinNumber(double v)
{
    for (int o = 32; o > 0; o >>= 1)
        v = fmin(v, __shfl_xor(v, o, 64));
    return v;
}
__device__ inline double waveMaxNumber(double v)
{
    for (int o = 32; o > 0; o >>= 1)
        v = fmax(v, __shfl_xor(v, o, 64));
    return v;
}

__device__ inline bool nodeOverlapsBox(const double* __restrict__ centers, const double* __restrict__ sizes, int node,
                                       const double gc[3], const double gh[3], const DBox& box)
{
    // all six loads are issued at once: one memory round trip per level, not one per dimension
    // (the walk waits for memory: 0.60 -> 0.50 ms at 256^3)
    double c[3], w[3];
#pragma unroll
    for (int d = 0; d < 3; ++d)
        c[d] = centers[3 * node + d], w[d] = sizes[3 * node + d];
    bool ov = true;
#pragma unroll
    for (int d = 0; d < 3; ++d)
    {
        double dx = c[d] - gc[d];
        if (box.pbc[d]) dx -= box.len[d] * rint(dx * box.ilen[d]);
        ov = ov & (fabs(dx) <= w[d] + gh[d]);
    }
    return ov;
}

// What nsCandidates needs of a group's search box
struct GroupSearch
{
    double   cx, cy, cz, inv;  // its centre, and the scale of the FP32 coordinates: 1 over its largest half-width
    float    hwx, hwy, hwz;    // half-widths of the targets' bounding box, scaled and widened
    float    lim;              // a candidate farther than sqrt(lim) from that box has no hits
    float    undecided;        // width of the shell in which FP32 results are not trusted
    uint32_t fold, exact;      // candidates take the image nearest the centre; left to nsCandidatesExact
    uint32_t pad;
};
__device__ inline GroupSearch groupSearch(const double gc[3], const double gh[3], double rmin, double rmax, const DBox& box,
                                          bool exact)
{
    // Candidates are folded to the image nearest the centre where a target's sphere may leave the box,
    // the condition of the exact predicate; a search box over half the domain's length has no single
    // nearest image.  Folding rounds at 2^-53 of the domain's length: below 2^-24 of it, that is no
    // longer small beside the rounding that `undecided` covers.
    GroupSearch  b{};
    const double S    = fmax(fmax(gh[0], gh[1]), gh[2]);
    bool         fold = false;
    exact             = exact || !(S > 0x1p-100 && S < 0x1p100);
    for (int d = 0; d < 3; ++d)
    {
        fold  = fold || gc[d] - gh[d] < box.lo[d] || gc[d] + gh[d] > box.hi[d];
        exact = exact || (box.pbc[d] && gh[d] >= 0.4999 * box.len[d]);
    }
    fold = fold && box.anyPbc;
    for (int d = 0; d < 3; ++d)
        exact = exact || (fold && box.pbc[d] && S < 0x1p-24 * box.len[d]);
    b.cx = gc[0], b.cy = gc[1], b.cz = gc[2], b.inv = 1.0 / S;
    // 2^-20 covers the rounding of the half-widths, 2^-17 that of the distances
    b.hwx = fmaxf(float((gh[0] - rmin) * b.inv), 0.f) + 0x1p-20f;
    b.hwy = fmaxf(float((gh[1] - rmin) * b.inv), 0.f) + 0x1p-20f;
    b.hwz = fmaxf(float((gh[2] - rmin) * b.inv), 0.f) + 0x1p-20f;
    const float rf = float(rmax * b.inv);
    b.lim          = rf * rf + 0x1p-17f;
    // Half-width of the shell around d^2 = (2h)^2 in which the FP32 result is not trusted.  With
    // Q = max |e|^2 and T = max |t|^2 over the box: three roundings (2^-24 each) of a coordinate
    // move d^2 by at most 2^-24 * 18 (Q + T) near the sphere; |e|^2, |t|^2 and (2h)^2 are off by
    // 2^-24 of 3 Q, 3 T and 1; the products and sums, none over 2 (Q + T), by 8 roundings in any
    // order: together below 2^-24 * (37 (Q + T) + 1).  Half as much again is used.
    const float ux = b.hwx + rf, uy = b.hwy + rf, uz = b.hwz + rf;
    const float QT = ux * ux + uy * uy + uz * uz + b.hwx * b.hwx + b.hwy * b.hwy + b.hwz * b.hwz;
    b.undecided    = 2.f * (0x1p-24f * (56.f * QT + 2.f));
    b.fold = fold, b.exact = exact;
    return b;
}

// The ranges of one group g (all 64 lanes of the wave call this).  A group whose walk
// exceeds the capacities gets no ranges and is appended to retryList, or, without a
// retry list, raises the overflow flag.
template<class Th, int FCAP, int LCAP>
__device__ void groupRangesOf(uint32_t g, GroupsDev G, const double* __restrict__ x, const double* __restrict__ y,
                              const double* __restrict__ z, const Th* __restrict__ h,
                              const int32_t* __restrict__ childOffsets, const int32_t* __restrict__ internalToLeaf,
                              const uint32_t* __restrict__ layout, const double* __restrict__ centers,
                              const double* __restrict__ sizes, const DBox& box, uint2* __restrict__ ranges,
                              uint32_t* __restrict__ rangeCount, GroupSearch* __restrict__ search,
                              uint32_t* __restrict__ retryList, NsFlags* __restrict__ flags)
{
    static_assert((LCAP & (LCAP - 1)) == 0 && LCAP <= NS_LCAP, "leaf capacity: a power of two within the range stride");
    static_assert(2 * FCAP >= LCAP, "the sorted leaves take the place of the walk's fronts");
    __shared__ int32_t front[2][FCAP];
    __shared__ int32_t leafList[LCAP];
    __shared__ int32_t segEnd[kMaxLevel + 1]; // ends in leafList of the levels that have leaves

    const unsigned lane = threadIdx.x;
    uint32_t       s, e;
    groupRange(G, g, s, e);
    if (e - s > 64)
    {
        if (lane == 0) atomicOr(&flags->badGroup, 1u);
        e = s + 64;
    }
    uint32_t i   = s + lane;
    bool     act = i < e;

    double lo[3], hi[3], rmin, rmax;
    {
        double px[3] = {0, 0, 0};
        double r     = 0;
        if (act)
        {
            px[0] = x[i], px[1] = y[i], px[2] = z[i];
            r     = 2.0 * double(h[i]);
        }
#pragma unroll
        for (int d = 0; d < 3; ++d)
        {
            lo[d] = waveMinNumber(act ? px[d] - r : INFINITY);
            hi[d] = waveMaxNumber(act ? px[d] + r : -INFINITY);
        }
        rmin = waveMinNumber(act ? r : INFINITY);
        rmax = waveMaxNumber(act ? r : -INFINITY);
    }
    if (!(lo[0] <= hi[0]))
    {
        if (lane == 0) rangeCount[g] = 0;
        return;
    }
    double gc[3], gh[3];
#pragma unroll
    for (int d = 0; d < 3; ++d)
    {
        gc[d] = 0.5 * (lo[d] + hi[d]);
        gh[d] = 0.5 * (hi[d] - lo[d]);
        gh[d] += 1e-12 * (fabs(gc[d]) + gh[d]); // never under-cover the union of spheres
    }

    // ---- breadth-first traversal
    int  lcount   = 0;
    bool overflow = false;
    int  fcount   = 0;
    int  cur      = 0;
    int  nseg     = 0;
    if (childOffsets[0] == 0)
    {
        if (lane == 0) leafList[0] = internalToLeaf[0];
        lcount = nseg = 1;
    }
    else
    {
        if (lane < 8) front[0][lane] = childOffsets[0] + int(lane);
        fcount = 8;
    }
    __syncthreads();
    const uint64_t lt = lanemaskLt();
    while (fcount > 0 && !overflow)
    {
        int ncount = 0;
        int nxt    = cur ^ 1;
        int first  = lcount;
        for (int b = 0; b < fcount; b += 64)
        {
            int idx  = b + int(lane);
            int node = front[cur][idx < fcount ? idx : 0];
            // the node's child offset and leaf index are loaded with its box (one memory
            // round trip per level), whether or not the box overlaps
            const int childOf = childOffsets[node], leafOf = internalToLeaf[node];
            bool      ov      = (idx < fcount) & nodeOverlapsBox(centers, sizes, node, gc, gh, box);
            int  child = ov ? childOf : 0;
            bool leaf  = ov && child == 0;
            bool inner = ov && child != 0;

            uint64_t mL   = ballot(leaf);
            int      posL = lcount + int(popc64(mL & lt));
            if (leaf && posL < LCAP) leafList[posL] = leafOf;
            lcount += int(popc64(mL));

            uint64_t mI   = ballot(inner);
            int      posI = ncount + 8 * int(popc64(mI & lt));
            if (inner && posI + 8 <= FCAP)
            {
#pragma unroll
                for (int c = 0; c < 8; ++c)
                    front[nxt][posI + c] = child + c;
            }
            ncount += 8 * int(popc64(mI));
        }
        if (lcount > first)
        {
            if (lane == 0) segEnd[nseg] = lcount;
            ++nseg;
        }
        __syncthreads();
        if (lcount > LCAP || ncount > FCAP) overflow = true;
        cur    = nxt;
        fcount = ncount;
    }
    if (overflow)
    {
        if (lane == 0)
        {
            rangeCount[g] = 0;
            if (retryList) retryList[atomicAdd(&flags->retryCount, 1u)] = g;
            else atomicOr(&flags->overflow, 1u);
        }
        return;
    }

    // ---- the candidate leaves in ascending order.  The walk keeps the order of the nodes, so the
    // leaves of one level are ascending: a leaf's place is the sum of its lower bounds in the
    // levels' segments (2 or 3 of them as a rule).  With a bitonic sort of the whole list in LDS the
    // kernel took 0.74 ms at 256^3 and 0.31 ms on a 4 M Evrard sphere, so 0.60 and 0.22.
    const int32_t* leaves = leafList;
    if (nseg > 1)
    {
        int32_t* sorted = front[0]; // the walk is done with it
        for (int k = int(lane); k < lcount; k += 64)
        {
            const int32_t v   = leafList[k];
            int           pos = 0;
            for (int t = 0, a = 0; t < nseg; ++t)
            {
                const int b = __builtin_amdgcn_readfirstlane(segEnd[t]);
                int       p = a;
                for (int len = b - a; len > 1;)
                {
                    const int half = len >> 1;
                    p += leafList[p + half - 1] < v ? half : 0;
                    len -= half;
                }
                pos += p - a + (leafList[p] < v ? 1 : 0);
                a = b;
            }
            sorted[pos] = v;
        }
        __syncthreads();
        leaves = sorted;
    }

    // ---- merge consecutive leaves into particle ranges, in pieces of at most 64 particles (the
    // chunks of nsCandidates); more pieces than there is room for stay whole ranges
    auto writeRanges = [&](uint32_t piece) {
        int rcount = 0;
        for (int b = 0; b < lcount; b += 64)
        {
            const int  k       = b + int(lane);
            const bool inRange = k < lcount;
            const int  leaf    = inRange ? leaves[k] : 0;
            const bool isStart = inRange && (k == 0 || leaf != leaves[k - 1] + 1);
            uint32_t   ps = 0, pe = 0;
            // the end of a run: before the next start of these 64 leaves, or on in the next 64
            const uint64_t after = (ballot(isStart) >> lane) >> 1;
            if (isStart)
            {
                int kk = after ? k + __builtin_ctzll(after) : min(b + 63, lcount - 1);
                while (!after && kk + 1 < lcount && leaves[kk + 1] == leaves[kk] + 1)
                    ++kk;
                ps = layout[leaf];
                pe = layout[leaves[kk] + 1];
            }
            const int np  = pe > ps ? int((pe - ps - 1u) / piece + 1u) : 0;
            int       sum = np;
            for (int o = 1; o < 64; o <<= 1)
            {
                const int v = __shfl_up(sum, o, 64);
                if (int(lane) >= o) sum += v;
            }
            int r = rcount + sum - np;
            for (uint32_t c = ps; c < pe; ++r, c = pe - c > piece ? c + piece : pe)
                if (r < NS_LCAP) ranges[size_t(g) * NS_LCAP + r] = make_uint2(c, pe - c > piece ? c + piece : pe);
            rcount += __shfl(sum, 63, 64);
        }
        return rcount;
    };
    int  rcount = writeRanges(64u);
    bool exact  = rcount > NS_LCAP;
    if (exact) rcount = writeRanges(~0u);
    if (lane == 0)
    {
        rangeCount[g] = uint32_t(rcount);
        search[g]     = groupSearch(gc, gh, rmin, rmax, box, exact);
    }
}

// all groups (or those of groupList) with the small capacities
template<class Th>
__global__ __launch_bounds__(64) void nsGroupRanges(GroupsDev G, const uint32_t* __restrict__ groupList,
                                                    const double* __restrict__ x, const double* __restrict__ y,
                                                    const double* __restrict__ z, const Th* __restrict__ h,
                                                    const int32_t* __restrict__ childOffsets,
                                                    const int32_t* __restrict__ internalToLeaf,
                                                    const uint32_t* __restrict__ layout,
                                                    const double* __restrict__ centers,
                                                    const double* __restrict__ sizes, DBox box,
                                                    uint2* __restrict__ ranges, uint32_t* __restrict__ rangeCount,
                                                    GroupSearch* __restrict__ search,
                                                    uint32_t* __restrict__ retryList, NsFlags* __restrict__ flags)
{
    const uint32_t blk = xcdContiguous(blockIdx.x, gridDim.x);
    const uint32_t g   = groupList ? groupList[blk] : blk;
    groupRangesOf<Th, NS_FCAP_SMALL, NS_LCAP_SMALL>(g, G, x, y, z, h, childOffsets, internalToLeaf, layout, centers,
                                                    sizes, box, ranges, rangeCount, search, retryList, flags);
}

// the groups of the retry list with the large capacities (grid-stride over the list,
// whose length the first walk left in flags->retryCount)
template<class Th>
__global__ __launch_bounds__(64) void nsGroupRangesRetry(GroupsDev G, const double* __restrict__ x,
                                                         const double* __restrict__ y, const double* __restrict__ z,
                                                         const Th* __restrict__ h,
                                                         const int32_t* __restrict__ childOffsets,
                                                         const int32_t* __restrict__ internalToLeaf,
                                                         const uint32_t* __restrict__ layout,
                                                         const double* __restrict__ centers,
                                                         const double* __restrict__ sizes, DBox box,
                                                         uint2* __restrict__ ranges, uint32_t* __restrict__ rangeCount,
                                                         GroupSearch* __restrict__ search,
                                                         const uint32_t* __restrict__ retryList,
                                                         NsFlags* __restrict__ flags)
{
    const uint32_t n = flags->retryCount;
    for (uint32_t k = blockIdx.x; k < n; k += gridDim.x)
    {
        groupRangesOf<Th, NS_FCAP, NS_LCAP>(retryList[k], G, x, y, z, h, childOffsets, internalToLeaf, layout,
                                             centers, sizes, box, ranges, rangeCount, search, nullptr, flags);
        __syncthreads(); // the next group reuses the LDS lists
    }
}

// Candidate test with the predicate in FP64 for all pairs, of the groups that nsCandidates
// leaves to it.  Sph = true: findNeighborsSph semantics (nc counts self, h updates,
// redo flags) and the SPH list format below; Sph = false: findNeighbors semantics
// (count without self, u32 lists in the reference CPU layout).
//
// SPH list format, per sub-group of 16 consecutive targets (quarter q of the wave,
// sg = 4 g + q): the sorted union of the stored neighbors of its 16 targets
// (unions[sg][0..usize)) and per target a bitmask over that union
// (masks[sg][w][t]).
//
// Thread mapping (transposed test).  The group's candidate ranges are streamed in
// chunks of 64 particles, lane = candidate; every chunk is filtered against the
// regions of the four quarters (16 targets each) and the survivors are appended, in
// ascending j, to per-quarter LDS queues.  A queue holding 64 candidates
// (or the rest, at the end) is tested as one batch: lane = candidate, and the wave
// walks the quarter's 16 targets, one target per step, so a step costs a handful of
// FP64 instructions for 64 tests and its ballot is the target's hit mask over the
// batch.  The hit masks give the batch's union entries (candidates stored by some
// target, in lane order = ascending j); a lane permutation compacts the entries and
// one ballot per target turns the compacted bits into that target's mask bits, which
// the target's lane appends to its mask word stream.
constexpr uint32_t NS_QCAP = 128; // per-quarter queue capacity (ring buffer)

// v_writelane_b32: `old` with lane `lane` replaced by the wave-uniform value v
__device__ int writeLane(int v, int lane, int old) __asm("llvm.amdgcn.writelane.i32");

template<class Th, bool Sph>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(6))) void nsCandidatesExact(GroupsDev G, const uint32_t* __restrict__ groupList,
                                                   const double* __restrict__ x, const double* __restrict__ y,
                                                   const double* __restrict__ z, Th* __restrict__ h,
                                                   uint8_t* __restrict__ iter, const uint2* __restrict__ ranges,
                                                   const uint32_t* __restrict__ rangeCount, DBox box, uint32_t ngmax,
                                                   uint32_t ng0, HFactors hfac, uint32_t* __restrict__ nbrs, SphLists out,
                                                   uint32_t* __restrict__ nc, uint32_t* __restrict__ redoList,
                                                   NsFlags* __restrict__ flags,
                                                   unsigned long long* __restrict__ groupTests)
{
#pragma clang fp contract(off)
    __shared__ uint32_t qj[4][NS_QCAP]; // queued candidate indices per quarter
    __shared__ double   tgt[64][4];     // target of lane l: x, y, z, (2h)^2
    __shared__ uint32_t tid[64];        // its particle index
    __shared__ double   qbox[4][7];     // quarter: box centre xyz, half-widths xyz, (radius)^2

    const uint32_t blk  = xcdContiguous(blockIdx.x, gridDim.x);
    const uint32_t g    = groupList ? groupList[blk] : blk;
    const unsigned lane = threadIdx.x;
    uint32_t       s, e;
    groupRange(G, g, s, e);
    if (e - s > 64) e = s + 64;
    const uint32_t i   = s + lane;
    const bool     act = i < e;

    double xi = 0, yi = 0, zi = 0, hi = 0;
    if (act) xi = x[i], yi = y[i], zi = z[i], hi = double(h[i]);
    const double radiusSq = 4.0 * hi * hi;
    bool         inside   = true;
    {
        double p[3] = {xi, yi, zi};
#pragma unroll
        for (int d = 0; d < 3; ++d)
            inside = inside && (p[d] - 2.0 * hi >= box.lo[d]) && (p[d] + 2.0 * hi <= box.hi[d]);
    }
    const bool   usePbc = box.anyPbc && !inside;
    const double px     = box.pbc[0] ? box.len[0] : 0.0;
    const double py     = box.pbc[1] ? box.len[1] : 0.0;
    const double pz     = box.pbc[2] ? box.len[2] : 0.0;

    // quarter regions: the bounding box of the 16 targets' positions (centre, half-widths
    // widened by a relative 1e-12) and the largest search radius 2h of the quarter.  A
    // neighbor of any target of the quarter lies within that radius of the box (its image
    // nearest the box centre, when the quarter uses periodic images), so the filter keeps
    // candidates whose distance to the box is at most the radius, with a relative slack of
    // 1e-9 on the squared radius; a quarter without targets keeps nothing.
    const unsigned q = lane >> 4, t = lane & 15u;
    const uint64_t actMask = ballot(act);
    const uint64_t pbcMask = ballot(usePbc);
    {
        double pp[3] = {xi, yi, zi};
        double lo[3], hh[3];
#pragma unroll
        for (int d = 0; d < 3; ++d)
        {
            double a = act ? pp[d] : INFINITY, b = act ? pp[d] : -INFINITY;
#pragma unroll
            for (int o = 1; o < 16; o <<= 1)
            {
                a = fmin(a, __shfl_xor(a, o, 64));
                b = fmax(b, __shfl_xor(b, o, 64));
            }
            lo[d] = a, hh[d] = b;
        }
        double rmax = act ? 2.0 * hi : -1.0;
#pragma unroll
        for (int o = 1; o < 16; o <<= 1)
            rmax = fmax(rmax, __shfl_xor(rmax, o, 64));
        if (t == 0)
        {
#pragma unroll
            for (int d = 0; d < 3; ++d)
            {
                double c = 0.5 * (lo[d] + hh[d]), w = 0.5 * (hh[d] - lo[d]);
                qbox[q][d]     = c;
                qbox[q][3 + d] = w + 1e-12 * (fabs(c) + w + box.len[d]);
            }
            qbox[q][6] = rmax < 0.0 ? -1.0 : rmax * rmax * (1.0 + 1e-9);
        }
        tgt[lane][0] = xi, tgt[lane][1] = yi, tgt[lane][2] = zi, tgt[lane][3] = radiusSq;
        tid[lane]    = act ? i : 0xFFFFFFFFu;
    }
    __syncthreads();

    const uint64_t lt = lanemaskLt();
    // per-target state, in the target's lane
    uint32_t count = 0; // hits so far (stored or not)
    uint32_t word  = 0; // SPH: mask bits of union entries 32 * (usz / 32) ...
    uint32_t extra = 0; // hits of the current batch beyond the per-target cap (SPH)
    uint32_t delta = 0; // hits of the current batch (non-SPH)
    // per-quarter state (wave-uniform; indexed by compile-time quarter numbers only)
    uint32_t qhead[4] = {0, 0, 0, 0}, qlen[4] = {0, 0, 0, 0}, usz[4] = {0, 0, 0, 0};
    unsigned long long tests = 0;

    // test the first nb queued candidates of quarter Q: lane = candidate
    auto batch = [&](auto Qc, uint32_t nb) {
        constexpr uint32_t Q  = decltype(Qc)::value;
        constexpr uint32_t qb = 16u * Q;
        const bool         valid = lane < nb;
        uint32_t           jc    = 0;
        double             xc = 0, yc = 0, zc = 0;
        if (valid)
        {
            jc = qj[Q][(qhead[Q] + lane) & (NS_QCAP - 1)];
            xc = x[jc], yc = y[jc], zc = z[jc];
        }
        tests += (unsigned long long)nb * popc64((actMask >> qb) & 0xFFFFu);
        uint32_t hb = 0; // bit tt: target tt of the quarter hits this candidate
        // straight-line steps; an inactive target has (2h)^2 = 0 and never hits
        if (((pbcMask >> qb) & 0xFFFFu) == 0)
        {
#pragma unroll
            for (uint32_t tt = 0; tt < 16; ++tt)
            {
                const double dx = xc - tgt[qb + tt][0];
                const double dy = yc - tgt[qb + tt][1];
                const double dz = zc - tgt[qb + tt][2];
                const double d2 = dx * dx + dy * dy + dz * dz;
                hb |= (valid & (d2 < tgt[qb + tt][3])) ? (1u << tt) : 0u;
            }
        }
        else
        {
            // quarters with periodic targets (near the box faces): the targets that use
            // periodic images fold the offsets (volatile reads keep this rare path's loads
            // from being merged with the common path)
            const volatile double* tv = &tgt[qb][0];
#pragma unroll 4
            for (uint32_t tt = 0; tt < 16; ++tt)
            {
                double dx = xc - tv[4 * tt + 0];
                double dy = yc - tv[4 * tt + 1];
                double dz = zc - tv[4 * tt + 2];
                if ((pbcMask >> (qb + tt)) & 1u)
                {
                    dx -= px * rint(dx * box.ilen[0]);
                    dy -= py * rint(dy * box.ilen[1]);
                    dz -= pz * rint(dz * box.ilen[2]);
                }
                const double d2 = dx * dx + dy * dy + dz * dz;
                hb |= (valid & (d2 < tv[4 * tt + 3])) ? (1u << tt) : 0u;
            }
        }
        // a target is not its own neighbor
        {
            const uint32_t self = jc - (s + qb);
            if (valid & (self < 16u)) hb &= ~(1u << self);
        }

        const bool mine = q == Q;
        if constexpr (Sph)
        {
            // union entries of the batch (candidates stored by some target) compacted into
            // lanes 0..nU-1 by a lane permutation; target lane qb + tt receives its mask
            // bits over them in (cmHi:cmLo)
            uint32_t nU = 0, jp = 0, cmLo = 0, cmHi = 0;
            for (int pass = 0; pass < 2; ++pass)
            {
                const uint64_t U = ballot(hb != 0);
                nU               = popc64(U);
                cmLo = cmHi = 0;
                if (nU)
                {
                    const uint32_t dst = hb ? rankIn(U) : nU + rankIn(~U);
                    const uint32_t hp  = uint32_t(__builtin_amdgcn_ds_permute(int(4u * dst), int(hb)));
                    jp                 = uint32_t(__builtin_amdgcn_ds_permute(int(4u * dst), int(jc)));
#pragma unroll
                    for (uint32_t tt = 0; tt < 16; ++tt)
                    {
                        const uint64_t cm = ballot((hp >> tt) & 1u);
                        cmLo = uint32_t(writeLane(int(uint32_t(cm)), int(qb + tt), int(cmLo)));
                        cmHi = uint32_t(writeLane(int(uint32_t(cm >> 32)), int(qb + tt), int(cmHi)));
                    }
                }
                const uint32_t gain = uint32_t(__builtin_popcount(cmLo)) + uint32_t(__builtin_popcount(cmHi));
                if (pass == 1 || ballot(mine && count + gain > ngmax) == 0) break;
                // a target reaches its cap in this batch: keep only its first hits, count
                // the others, and compact again
#pragma unroll 1
                for (uint32_t tt = 0; tt < 16; ++tt)
                {
                    const bool     hit  = (hb >> tt) & 1u;
                    const uint64_t mh   = ballot(hit);
                    const uint32_t pc   = popc64(mh);
                    const uint32_t ct   = uint32_t(__builtin_amdgcn_readlane(int(count), int(qb + tt)));
                    const uint32_t room = ct < ngmax ? ngmax - ct : 0u;
                    if (pc > room)
                    {
                        if (hit && rankIn(mh) >= room) hb &= ~(1u << tt);
                        extra = uint32_t(writeLane(int(pc - room), int(qb + tt), int(extra)));
                    }
                }
            }
            if (lane < nU) out.unions[size_t(4u * g + Q) * out.capU + usz[Q] + lane] = jp;
            if (mine)
            {
                count += uint32_t(__builtin_popcount(cmLo)) + uint32_t(__builtin_popcount(cmHi)) + extra;
                extra = 0;
                if (nU)
                {
                    // append nU mask bits at bit offset usz of the target's word stream
                    const uint32_t u0 = usz[Q], o = u0 & 31u, end = o + nU;
                    const uint64_t cm64 = (uint64_t(cmHi) << 32) | cmLo;
                    const uint64_t lo64 = uint64_t(word) | (cm64 << o);
                    const uint32_t w2   = o ? uint32_t(cm64 >> (64u - o)) : 0u;
                    uint32_t* wp = out.masks + (size_t(4u * g + Q) * out.words + (u0 >> 5)) * 16 + t;
                    if (end >= 32) wp[0] = uint32_t(lo64);
                    if (end >= 64) wp[16] = uint32_t(lo64 >> 32);
                    word = end >= 64 ? w2 : (end >= 32 ? uint32_t(lo64 >> 32) : uint32_t(lo64));
                }
            }
            usz[Q] += nU;
        }
        else
        {
            // reference CPU layout: the k-th hit of target i goes to nbrs[(i - first) * ngmax + k]
#pragma unroll 1
            for (uint32_t tt = 0; tt < 16; ++tt)
            {
                const bool     hit = (hb >> tt) & 1u;
                const uint64_t mh  = ballot(hit);
                if (mh == 0) continue;
                const uint32_t ct  = uint32_t(__builtin_amdgcn_readlane(int(count), int(qb + tt)));
                const uint32_t pos = ct + rankIn(mh);
                if (hit && nbrs && pos < ngmax) nbrs[size_t(s + qb + tt - G.first) * ngmax + pos] = jc;
                delta = uint32_t(writeLane(int(popc64(mh)), int(qb + tt), int(delta)));
            }
            if (mine) count += delta;
            delta = 0;
        }
        qhead[Q] += nb;
        qlen[Q] -= nb;
    };

    // Stream the candidates in chunks of 64 (lane = candidate): filter each chunk against
    // the 4 quarter boxes and queue the survivors; then every quarter whose queue holds
    // 64 candidates tests one batch (a chunk adds at most 64, so queues stay below 128).
    // After the last chunk the remaining partial queues are tested.
    const uint32_t R   = rangeCount[g];
    uint32_t       r   = 0;
    uint2          rg  = R ? ranges[size_t(g) * NS_LCAP] : make_uint2(0u, 0u);
    uint32_t       cur = rg.x;
    for (;;)
    {
        const bool done = r >= R;
        if (!done)
        {
            const uint32_t m  = min(64u, rg.y - cur);
            const bool     in = lane < m;
            const uint32_t j  = cur + lane;
            double         ax = 0, ay = 0, az = 0;
            if (in) ax = x[j], ay = y[j], az = z[j];
#pragma unroll
            for (uint32_t qq = 0; qq < 4; ++qq)
            {
                double dx = ax - qbox[qq][0], dy = ay - qbox[qq][1], dz = az - qbox[qq][2];
                if ((pbcMask >> (16u * qq)) & 0xFFFFu)
                {
                    dx -= px * rint(dx * box.ilen[0]);
                    dy -= py * rint(dy * box.ilen[1]);
                    dz -= pz * rint(dz * box.ilen[2]);
                }
                const double ex   = fmax(fabs(dx) - qbox[qq][3], 0.0);
                const double ey   = fmax(fabs(dy) - qbox[qq][4], 0.0);
                const double ez   = fmax(fabs(dz) - qbox[qq][5], 0.0);
                const bool   pass = in & (ex * ex + ey * ey + ez * ez <= qbox[qq][6]);
                const uint64_t mk = ballot(pass);
                if (pass) qj[qq][(qhead[qq] + qlen[qq] + rankIn(mk)) & (NS_QCAP - 1)] = j;
                qlen[qq] += popc64(mk);
            }
            cur += m;
            if (cur >= rg.y && ++r < R)
            {
                rg  = ranges[size_t(g) * NS_LCAP + r];
                cur = rg.x;
            }
            __syncthreads();
        }
        if (qlen[0] >= 64 || (done && qlen[0])) batch(std::integral_constant<uint32_t, 0>{}, min(qlen[0], 64u));
        if (qlen[1] >= 64 || (done && qlen[1])) batch(std::integral_constant<uint32_t, 1>{}, min(qlen[1], 64u));
        if (qlen[2] >= 64 || (done && qlen[2])) batch(std::integral_constant<uint32_t, 2>{}, min(qlen[2], 64u));
        if (qlen[3] >= 64 || (done && qlen[3])) batch(std::integral_constant<uint32_t, 3>{}, min(qlen[3], 64u));
        if (done) break;
    }
    // exact pair tests of this pass
    // (stored per group and summed by nsSumTests: one atomic per group on a single counter
    // would serialize)
    if (lane == 0) groupTests[g] = tests;

    if constexpr (Sph)
    {
        const uint32_t sg    = 4u * g + q;
        const uint32_t myUsz = q == 0 ? usz[0] : q == 1 ? usz[1] : q == 2 ? usz[2] : usz[3];
        if (t == 0) out.usize[sg] = myUsz;
        if (myUsz & 31u) out.masks[(size_t(sg) * out.words + myUsz / 32u) * 16 + t] = word;
        bool redo = false;
        if (act)
        {
            uint32_t ncSph = count + 1;
            uint32_t ngmin = ng0 / 4;
            bool     outR  = (ngmin > ncSph) || (ncSph - 1 > ngmax);
            nc[i] = ncSph; // dataset counts are indexed by particle (sph/find_neighbors.hpp:51)
            if (outR && iter[i] < 10)
            {
                // updateH (sph/kernels.hpp:27-33) in the precision of h, factor from the table
                Th hn = Th(hi);
                if (updateHTab(hfac, ncSph, hn))
                {
                    h[i] = hn;
                    iter[i] += 1;
                    redo = true;
                }
                else
                    flags->hfacMiss = 1;
            }
        }
        uint64_t anyRedo = ballot(redo);
        if (anyRedo && lane == 0)
        {
            uint32_t pos  = atomicAdd(&flags->redoCount, 1u);
            redoList[pos] = g;
        }
    }
    else
    {
        if (act) nc[i - G.first] = count;
    }
}

// The neighbor search proper.  One workgroup of 4 waves per target group, wave q for the 16
// targets of quarter q.
//
//   filter : the group's candidate ranges are streamed in chunks of 64 particles, lane =
//            candidate, 8 chunks at a time (two per wave).  A candidate within the group's
//            largest 2h of the targets' bounding box is put, in ascending j, into an LDS ring:
//            its position relative to the group's centre, in units of the search box's
//            half-width, in FP32, and |e|^2.
//   union  : every wave tests the ring's entries, 64 at a time, against its 16 targets with four
//            MFMA (16x16x4 FP32): rows = targets (-2x, -2y, -2z, 1), columns = entries
//            (x, y, z, |e|^2), C = |t|^2 - (2h)^2, so that the result is d^2 - (2h)^2.  Its
//            minimum over the targets says whether the entry joins the quarter's union; the
//            members are appended to a queue of the wave.
//   masks  : 64 members of the queue at a time go through the MFMA again, rows = entries, columns =
//            targets: a lane receives the results of 16 consecutive members for one target, whose
//            sign bits are 16 bits of that target's mask, stored as they are.
//
// FP32 error bounds leave a shell around the sphere (about one pair in 30,000) where the
// reference predicate d^2 < (2h)^2 is evaluated in FP64 with separately rounded operations
// (findneighbors.hpp:33-60,115-140), so the neighbor sets are bit-identical to the CPU path.
//
// Groups without a single nearest periodic image, with a candidate outside a periodic domain, without
// a usable search box, or with a target beyond ngmax neighbors (whose lists keep the first ngmax) are
// left to nsCandidatesExact by overList; the last not while a target of the group is still to be
// searched again, where only the counts matter (1 M particles, h for 300 neighbors at first, ngmax 150:
// 7.2 ms with the exact kernel in each of the iterations, now 2.7).
//
// One wave per group with the predicate in FP64 for all pairs (nsCandidatesExact) took 4.66 ms at
// 256^3 and 0.185 ms for 4,096 particles, where it leaves most of the chip idle; this takes 3.51
// and 0.027 ms.  Bound by instruction issue: 1,250 VALU and 700 SALU instructions per wave, 60 %
// of the time with VALU work, the rest waits for the first chunks and the barriers of a step.
// candidate chunks per wave and step: 2 (1: 3.6 ms at 256^3, more steps; 3: 4.1, registers)
constexpr uint32_t NS_PER_WAVE = 2;
constexpr uint32_t NS_CHUNKS   = 4 * NS_PER_WAVE;     // per step
constexpr uint32_t NS_RING     = 64 + 64 * NS_CHUNKS; // 63 entries carried over + a step's, whole batches
// a wave's queue: two batches of 64 members (float4), 64 bytes of padding after each 16 of them
// so that the masks' operand reads (members 16 apart) meet different banks
constexpr uint32_t NS_QHALF = 64 * 4 + 4 * 16; // floats per batch
static_assert(NS_QHALF % 4 == 0, "every wave's queue and both of its batches start at 16 bytes");

using floatx4 = __attribute__((ext_vector_type(4))) float;

// LDS written by other lanes of the same wave (whose LDS operations execute in order)
__device__ inline void waveFence()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// min(a, b) after exchanging the upper half of every 2 * Rows lanes of a with the lower half of
// b's: the lower half then holds a's minima over both halves, the upper half b's
template<int Rows>
__device__ inline int swapMin(int a, int b)
{
    if constexpr (Rows == 32)
    {
        const auto v = __builtin_amdgcn_permlane32_swap(uint32_t(a), uint32_t(b), false, false);
        return min(int(v[0]), int(v[1]));
    }
    else
    {
        const auto v = __builtin_amdgcn_permlane16_swap(uint32_t(a), uint32_t(b), false, false);
        return min(int(v[0]), int(v[1]));
    }
}

template<class Th, bool Sph>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(6))) void nsCandidates(
    GroupsDev G, const uint32_t* __restrict__ groupList, const double* __restrict__ x, const double* __restrict__ y,
    const double* __restrict__ z, Th* __restrict__ h, uint8_t* __restrict__ iter, const uint2* __restrict__ ranges,
    const uint32_t* __restrict__ rangeCount, const GroupSearch* __restrict__ search, DBox box, uint32_t ngmax,
    uint32_t ng0, HFactors hfac, uint32_t* __restrict__ nbrs, SphLists out, uint32_t* __restrict__ nc, uint32_t* __restrict__ redoList,
    uint32_t* __restrict__ overList, NsFlags* __restrict__ flags, unsigned long long* __restrict__ groupTests)
{
#pragma clang fp contract(off)
    __shared__ float4   ent[NS_RING];
    __shared__ uint32_t entJ[NS_RING];
    __shared__ alignas(16) float queAll[4][2 * NS_QHALF]; // (written 16 bytes at a time)
    __shared__ uint32_t queJAll[4][128];
    __shared__ uint32_t selfAll[4][16]; // the union index of each target
    __shared__ uint32_t wcnt[4], wflag[4];

    const uint32_t blk  = xcdContiguous(blockIdx.x, gridDim.x);
    const uint32_t g    = groupList ? groupList[blk] : blk;
    const uint32_t q    = uint32_t(__builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6)));
    const unsigned lane = threadIdx.x & 63u, part = lane >> 4, n = lane & 15u;
    float*         que  = queAll[q];
    uint32_t*      queJ = queJAll[q];
    uint32_t       s, e;
    groupRange(G, g, s, e);
    if (e - s > 64) e = s + 64;
    const uint32_t R = rangeCount[g];

    if (R == 0 || search[g].exact)
    {
        if (threadIdx.x == 0)
        {
            overList[atomicAdd(&flags->overCount, 1u)] = g;
            groupTests[g]                              = 0;
        }
        return;
    }
    const GroupSearch sb   = search[g];
    const float       invF = float(sb.inv);

    // the wave's targets: lane 16 p + n holds target n (four copies)
    const uint32_t i   = s + 16u * q + n;
    const bool     act = i < e;
    const double   px  = box.pbc[0] ? box.len[0] : 0.0;
    const double   py  = box.pbc[1] ? box.len[1] : 0.0;
    const double   pz  = box.pbc[2] ? box.len[2] : 0.0;
    // the reference predicate for target ii; its fields are loaded anew (the empty asm keeps the
    // loads and what follows from them here, off the common path's registers)
    auto exactHit = [&](uint32_t ii, uint32_t j) {
        asm volatile("" : "+v"(ii));
        const double p[3] = {x[ii], y[ii], z[ii]}, hi = double(h[ii]);
        double       dx = x[j] - p[0], dy = y[j] - p[1], dz = z[j] - p[2];
        bool         inside = true;
#pragma unroll
        for (int d = 0; d < 3; ++d)
            inside = inside && (p[d] - 2.0 * hi >= box.lo[d]) && (p[d] + 2.0 * hi <= box.hi[d]);
        if (box.anyPbc && !inside)
        {
            dx -= px * rint(dx * box.ilen[0]);
            dy -= py * rint(dy * box.ilen[1]);
            dz -= pz * rint(dz * box.ilen[2]);
        }
        return dx * dx + dy * dy + dz * dz < 4.0 * hi * hi;
    };

    // MFMA operand of the targets and C; a target without neighbors (none, or a position or h that
    // is no number) gets +1e30 for every distance
    float tx = 4.f, ty = 4.f, tz = 4.f, r2 = 0.f;
    if (act)
    {
        const double rs = 2.0 * double(h[i]) * sb.inv;
        tx = float(x[i] - sb.cx) * invF, ty = float(y[i] - sb.cy) * invF, tz = float(z[i] - sb.cz) * invF;
        r2 = float(rs * rs);
    }
    const float undecided = sb.undecided;
    const bool  usable = fabsf(tx) <= 2.f && fabsf(ty) <= 2.f && fabsf(tz) <= 2.f && r2 == r2; // (false for NaN)
    const float tval   = part == 3 ? 1.f : !usable ? 0.f : -2.f * (part == 0 ? tx : part == 1 ? ty : tz);
    const float c0     = usable ? tx * tx + ty * ty + tz * tz - r2 + 0.5f * undecided : 1e30f;
    const floatx4 cCol = {c0, c0, c0, c0};
    floatx4       cRow; // of targets 4 part + k
#pragma unroll
    for (int k = 0; k < 4; ++k)
        cRow[k] = __shfl(c0, int(4u * part) + k, 64);
    const bool anyTarget = 16u * q < e - s; // whole waves

    if (lane < 16) selfAll[q][lane] = ~0u;
    uint32_t  queued = 0, masked = 0; // members appended to the queue, and those of them with masks
    uint32_t  count  = 0;             // this lane's hits
    uint32_t  listed[Sph ? 1 : 16] = {}; // !Sph: each target's neighbors so far
    const uint32_t sg     = 4u * g + q;
    uint32_t*      unions = Sph ? out.unions + size_t(sg) * out.capU : nullptr;
    // this lane's 16 bits of the masks of a batch
    uint16_t*      maskAt = Sph ? reinterpret_cast<uint16_t*>(out.masks + (size_t(sg) * out.words + (part >> 1)) * 16 + n) + (part & 1u)
                                : nullptr;

    // the masks of the next 64 members of the queue (nb of them)
    auto masks = [&](uint32_t nb) {
        const uint32_t half = masked & 64u;
        const float*   A    = que + (half ? NS_QHALF : 0u) + 80u * (n >> 2) + 4u * (n & 3u) + part;
        floatx4        d[4];
#pragma unroll
        for (int m = 0; m < 4; ++m)
            d[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(A[16 * m], tval, cCol, 0, 0, 0);
        const uint32_t j = queJ[half + lane];
        const uint32_t o = selfAll[q][n] - masked;
        __builtin_amdgcn_sched_barrier(0); // all four in flight before the first result is used
        // result (m, k): member 16 part + 4 m + k
        uint32_t P = 0, mn = ~0u;
#pragma unroll
        for (int k = 15; k >= 0; --k)
        {
            const uint32_t a = __float_as_uint(d[k >> 2][k & 3]);
            P                = __builtin_amdgcn_alignbit(P, a, 31);
            mn               = min(mn, a);
        }
        if (__builtin_expect(ballot(mn < __float_as_uint(undecided)) != 0, 0))
        {
            // the pairs whose FP32 result does not decide, exactly
            uint32_t amb = 0;
#pragma unroll
            for (int k = 15; k >= 0; --k)
                amb = (amb << 1) | (__float_as_uint(d[k >> 2][k & 3]) < __float_as_uint(undecided) ? 1u : 0u);
            while (amb)
            {
                const uint32_t b = uint32_t(__builtin_ctz(amb));
                amb &= amb - 1u;
                if (act && 16u * part + b < nb && exactHit(i, queJ[half + 16u * part + b])) P |= 1u << b;
            }
        }
        // a target is not its own neighbor
        if ((o >> 4) == part) P &= ~(1u << (o & 15u));
        count += uint32_t(__builtin_popcount(P));
        if constexpr (Sph)
        {
            if (masked + 64u <= out.capU)
            {
                *maskAt = uint16_t(P);
                if (lane < nb) unions[masked + lane] = j;
            }
            maskAt += 64; // two words of 16 targets
        }
        else
        {
            // reference CPU layout: the k-th hit of target i goes to nbrs[(i - first) * ngmax + k]
#pragma unroll
            for (int t = 0; t < 16; ++t)
            {
                const uint32_t lo = uint32_t(__builtin_amdgcn_readlane(int(P), t)) |
                                    (uint32_t(__builtin_amdgcn_readlane(int(P), 16 + t)) << 16);
                const uint32_t hw = uint32_t(__builtin_amdgcn_readlane(int(P), 32 + t)) |
                                    (uint32_t(__builtin_amdgcn_readlane(int(P), 48 + t)) << 16);
                const uint64_t mt = (uint64_t(hw) << 32) | lo;
                if (mt == 0) continue;
                const uint32_t pos = listed[t] + rankIn(mt);
                if (((mt >> lane) & 1u) && nbrs && pos < ngmax)
                    nbrs[size_t(s + 16u * q + uint32_t(t) - G.first) * ngmax + pos] = j;
                listed[t] += popc64(mt);
            }
        }
        masked += 64u;
    };

    // this wave's chunks of the next NS_CHUNKS (their bounds are scalars), loaded a step ahead
    const uint2* pieces = ranges + size_t(g) * NS_LCAP + NS_PER_WAVE * q;
    uint32_t     st[NS_PER_WAVE], len[NS_PER_WAVE];
    double       ax[NS_PER_WAVE], ay[NS_PER_WAVE], az[NS_PER_WAVE];
    auto         loadChunks = [&](uint32_t k) {
#pragma unroll
        for (uint32_t c = 0; c < NS_PER_WAVE; ++c)
        {
            const bool  in = k + NS_PER_WAVE * q + c < R;
            const uint2 v  = in ? pieces[k + c] : make_uint2(0u, 0u);
            st[c] = v.x, len[c] = v.y - v.x;
            ax[c] = ay[c] = az[c] = 0.0;
            if (lane < len[c]) ax[c] = x[st[c] + lane], ay[c] = y[st[c] + lane], az[c] = z[st[c] + lane];
        }
    };
    loadChunks(0u);
    uint64_t leave = 0;               // nonzero: the group is left to nsCandidatesExact
    uint32_t avail = 0, proc = 0;     // entries put into the ring, entries tested
    uint32_t ringIn = 0, ringOut = 0; // avail and proc modulo the ring's size
    for (uint32_t fill = 0;; fill += NS_CHUNKS)
    {
        const bool last = fill + NS_CHUNKS >= R;
        float4     ev[NS_PER_WAVE];
        uint32_t   jv[NS_PER_WAVE];
        uint64_t   mk[NS_PER_WAVE];
#pragma unroll
        for (uint32_t c = 0; c < NS_PER_WAVE; ++c)
        {
            double dx = ax[c] - sb.cx, dy = ay[c] - sb.cy, dz = az[c] - sb.cz;
            if (sb.fold)
            {
                // a candidate outside the domain: the predicate folds it for some targets only
                bool away = false;
                if (box.pbc[0]) away = away | (ax[c] < box.lo[0]) | (ax[c] > box.hi[0]);
                if (box.pbc[1]) away = away | (ay[c] < box.lo[1]) | (ay[c] > box.hi[1]);
                if (box.pbc[2]) away = away | (az[c] < box.lo[2]) | (az[c] > box.hi[2]);
                leave |= ballot(away & (lane < len[c]));
                dx -= px * rint(dx * box.ilen[0]);
                dy -= py * rint(dy * box.ilen[1]);
                dz -= pz * rint(dz * box.ilen[2]);
            }
            const float fx = float(dx) * invF, fy = float(dy) * invF, fz = float(dz) * invF;
            // the distance from the box; |f| - min(|f|, hw) stays NaN for a NaN coordinate, which is no
            // neighbor (max(|f| - hw, 0) would be 0)
            const float ex = fabsf(fx) - fminf(fabsf(fx), sb.hwx), ey = fabsf(fy) - fminf(fabsf(fy), sb.hwy),
                        ez = fabsf(fz) - fminf(fabsf(fz), sb.hwz);
            mk[c] = ballot(__builtin_fmaf(ez, ez, __builtin_fmaf(ey, ey, ex * ex)) <= sb.lim) &
                    (len[c] ? ~uint64_t(0) >> (64u - len[c]) : 0u);
            ev[c]   = make_float4(fx, fy, fz, __builtin_fmaf(fz, fz, __builtin_fmaf(fy, fy, fx * fx)));
            jv[c]   = st[c] + lane;
        }
        if (!last) loadChunks(fill + NS_CHUNKS);
        uint32_t mine = 0;
#pragma unroll
        for (uint32_t c = 0; c < NS_PER_WAVE; ++c)
            mine += popc64(mk[c]);
        if (lane == 0) wcnt[q] = mine;
        __syncthreads(); // the counts; the previous step's batches are tested
        uint32_t before = 0, total = 0;
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k)
        {
            const uint32_t v = uint32_t(__builtin_amdgcn_readfirstlane(int(wcnt[k])));
            before += k < q ? v : 0u;
            total += v;
        }
#pragma unroll
        for (uint32_t c = 0; c < NS_PER_WAVE; ++c)
        {
            if (__builtin_amdgcn_inverse_ballot_w64(mk[c]))
            {
                const uint32_t k = before + rankIn(mk[c]);
                uint32_t       p = ringIn + k;
                p                = min(p, p - NS_RING);
                ent[p]           = ev[c];
                entJ[p]          = jv[c];
            }
            before += popc64(mk[c]);
        }
        avail += total;
        ringIn += total;
        ringIn = ringIn >= NS_RING ? ringIn - NS_RING : ringIn;
        if (last && q == 3 && lane < ((64u - (avail & 63u)) & 63u))
        {
            // pad the last batch
            uint32_t p = ringIn + lane;
            p          = min(p, p - NS_RING);
            ent[p]     = make_float4(0.f, 0.f, 0.f, 1e30f);
            entJ[p]    = ~0u;
        }
        __syncthreads(); // the new entries

        const uint32_t goal = last ? (avail + 63u) & ~63u : avail & ~63u;
        while (proc < goal && anyTarget)
        {
            // 16 targets x 64 entries
            const float* B = reinterpret_cast<const float*>(ent + ringOut + n) + part;
            floatx4      d[4];
#pragma unroll
            for (int m = 0; m < 4; ++m)
                d[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(tval, B[64 * m], cRow, 0, 0, 0);
            const float4   own = ent[ringOut + lane];
            const uint32_t j = entJ[ringOut + lane], o = j - (s + 16u * q);
            __builtin_amdgcn_sched_barrier(0);
            // entry 16 m + n's minimum over the lane's four targets, then over the four parts: the
            // first swap leaves the lower half with entries of m = 0 and 1, the second each row
            // of 16 lanes with those of its own m
            // (as integers: a negative result is below any positive one, and those keep their order)
            int mn[4];
#pragma unroll
            for (int m = 0; m < 4; ++m)
            {
                auto bits = [&](int k) { return int(__float_as_uint(d[m][k])); };
                mn[m]     = min(min(min(bits(0), bits(1)), bits(2)), bits(3));
            }
            if (ballot(o < 16u))
            {
                // targets among the entries: without their own results
#pragma unroll
                for (int m = 0; m < 4; ++m)
                {
                    const uint32_t om = entJ[ringOut + 16u * uint32_t(m) + n] - (s + 16u * q) - 4u * part;
                    mn[m]             = INT_MAX;
#pragma unroll
                    for (uint32_t k = 0; k < 4; ++k)
                        mn[m] = min(mn[m], om == k ? INT_MAX : int(__float_as_uint(d[m][k])));
                }
            }
            const int  a = swapMin<32>(mn[0], mn[2]), b = swapMin<32>(mn[1], mn[3]);
            const int  v = swapMin<16>(a, b);
            uint64_t   U = ballot(v < 0);
            const uint64_t V = ballot(v < int(__float_as_uint(undecided)));
            if (__builtin_expect(U != V, 0))
            {
                // entries whose nearest results do not decide
                for (uint64_t W = V & ~U; W; W &= W - 1u)
                {
                    const uint32_t b  = uint32_t(__builtin_ctzll(W));
                    const uint32_t jb = uint32_t(__builtin_amdgcn_readlane(int(j), int(b)));
                    if (ballot(act && i != jb && exactHit(i, jb))) U |= uint64_t(1) << b;
                }
            }
            if (__builtin_amdgcn_inverse_ballot_w64(U))
            {
                const uint32_t u = queued + rankIn(U), p = u & 127u;
                float*         f = que + 4u * (p + 4u * (p >> 4));
                *reinterpret_cast<float4*>(f) = own;
                queJ[p]                       = j;
                if (o < 16u) selfAll[q][o] = u;
            }
            queued += popc64(U);
            proc += 64u;
            ringOut += 64u;
            ringOut = ringOut == NS_RING ? 0u : ringOut;
            waveFence();
            if (queued - masked >= 64u) masks(64u);
            waveFence();
        }
        proc = goal;
        if (last) break;
    }
    if (masked < queued)
    {
        // the rest, padded with members that no target hits
        const uint32_t nb = queued - masked, p = (masked & 64u) + lane;
        if (lane >= nb) *reinterpret_cast<float4*>(que + 4u * (p + 4u * (p >> 4))) = make_float4(0.f, 0.f, 0.f, 1e30f);
        waveFence();
        masks(nb);
    }
    // pair tests of this pass (stored per group and summed by nsSumTests: one atomic per group on
    // a single counter would serialize)
    if (threadIdx.x == 0) groupTests[g] = (unsigned long long)avail * (e - s);

    count += uint32_t(__shfl_xor(int(count), 16, 64));
    count += uint32_t(__shfl_xor(int(count), 32, 64));
    // A target beyond ngmax neighbors, whose list keeps the first ngmax, needs the exact kernel.  Where a
    // target of the group is going to be searched again with another h, the whole group is, and the
    // counts are all that this pass is for.
    bool redo = false;
    if constexpr (Sph)
    {
        if (act && part == 0)
        {
            const uint32_t ncSph = count + 1, ngmin = ng0 / 4;
            redo = ((ngmin > ncSph) || (ncSph - 1 > ngmax)) && iter[i] < 10;
        }
    }
    uint32_t state = 0; // 1: searched again, 2: a list too long, 4: not decided by the FP32 tests
    if (Sph || sb.fold)
    {
        uint32_t mine = leave ? 4u : 0u;
        if constexpr (Sph) mine |= (ballot(redo) ? 1u : 0u) | (ballot(count > ngmax || queued + 64u > out.capU) ? 2u : 0u);
        if (lane == 0) wflag[q] = mine;
        __syncthreads();
        state = wflag[0] | wflag[1] | wflag[2] | wflag[3];
        if (state == 2u || (state & 4u))
        {
            if (threadIdx.x == 0)
            {
                overList[atomicAdd(&flags->overCount, 1u)] = g;
                groupTests[g]                              = 0;
            }
            return;
        }
    }
    if constexpr (Sph)
    {
        if (lane == 0) out.usize[sg] = queued;
        if (act && part == 0) nc[i] = count + 1; // dataset counts are indexed by particle (sph/find_neighbors.hpp:51)
        if (redo)
        {
            // updateH (sph/kernels.hpp:27-33) in the precision of h, factor from the table
            Th hn = h[i];
            if (updateHTab(hfac, count + 1, hn))
            {
                h[i] = hn;
                iter[i] += 1;
            }
            else
                flags->hfacMiss = 1;
        }
        if (threadIdx.x == 0 && (state & 1u)) redoList[atomicAdd(&flags->redoCount, 1u)] = g;
    }
    else
    {
        if (act && part == 0) nc[i - G.first] = count;
    }
}

__global__ __launch_bounds__(256) void nsInitState(uint8_t* iter, uint32_t first, uint32_t last)
{
    uint32_t i = first + blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= last) return;
    iter[i] = 0;
}

__global__ void nsResetFlags(NsFlags* f, int clearErrors)
{
    if (threadIdx.x == 0)
    {
        f->redoCount  = 0;
        f->retryCount = 0;
        f->overCount  = 0;
        f->tests      = 0;
        f->listTests  = 0;
        if (clearErrors)
        {
            f->overflow = 0;
            f->badGroup = 0;
            f->hfacMiss = 0;
        }
    }
}

// *sum += the test counts of the n groups of list (nullptr: the first n), one atomic per block
__global__ __launch_bounds__(256) void nsSumTests(const unsigned long long* __restrict__ groupTests,
                                                  const uint32_t* __restrict__ list, uint32_t n,
                                                  unsigned long long* __restrict__ sum)
{
    __shared__ unsigned long long part[4];
    unsigned long long            v = 0;
    for (uint32_t k = blockIdx.x * 256u + threadIdx.x; k < n; k += gridDim.x * 256u)
        v += groupTests[list ? list[k] : k];
    v = waveSum(v);
    if ((threadIdx.x & 63u) == 0) part[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0)
    {
        unsigned long long tot = part[0] + part[1] + part[2] + part[3];
        if (tot) atomicAdd(sum, tot);
    }
}

// export the SPH lists into the reference CPU layout [i - first][k]
__global__ __launch_bounds__(256) void nsExport(GroupsDev G, SphLists L, uint32_t ngmax,
                                                const uint32_t* __restrict__ nc, uint32_t* __restrict__ out)
{
    uint32_t g    = blockIdx.x * 4 + (threadIdx.x >> 6);
    uint32_t lane = threadIdx.x & 63u;
    if (g >= G.numGroups) return;
    uint32_t s, e;
    groupRange(G, g, s, e);
    uint32_t i = s + lane;
    if (i >= e || lane >= 64) return;
    uint32_t        sg   = 4u * g + (lane >> 4);
    const uint32_t* M    = maskRow(L, sg, lane & 15u);
    const uint32_t* uni  = L.unions + size_t(sg) * L.capU;
    const uint32_t  nw   = (L.usize[sg] + 31u) / 32u;
    uint32_t        k    = 0;
    for (uint32_t w = 0; w < nw; ++w)
    {
        uint32_t m = M[size_t(w) * 16];
        while (m)
        {
            uint32_t b = uint32_t(__builtin_ctz(m));
            m &= m - 1u;
            out[size_t(i - G.first) * ngmax + k++] = uni[32u * w + b];
        }
    }
}


// ---------------------------------------------------------------------------
// target groups: computeGroupSplits (domain/include/cstone/traversal/groups_gpu.cu:108-137,
// groups_gpu.cuh:37-77,148-216).  Fixed 64-particle groups are split after particle p
// when |X(p+1) - X(p)|^2 > min(distCrit^2, (2 h_p / minExtent)^2) in box-length units,
// distCrit = tolFactor * cbrt(volume of the smallest leaf holding a particle of the group).
//
// One wave per fixed group.  The leaves holding the group's particles p0..p1 are the
// non-empty leaves from leaf(p0) (the last leaf with layout <= p0; layout[0] = 0) through
// leaf(p1): the wave finds leaf(p0) with a 64-way search (four dependent probes for 2^24
// leaves) and then walks the leaves after it 64 at a time until one starts beyond p1,
// which for a group of 64 particles is nearly always one step.
template<class Th>
__global__ __launch_bounds__(256) void grpSplitMasks(uint32_t first, uint32_t last, uint32_t numFixed,
                                                     const double* __restrict__ x, const double* __restrict__ y,
                                                     const double* __restrict__ z, const Th* __restrict__ h,
                                                     const uint64_t* __restrict__ leaves, int numLeaves,
                                                     const uint32_t* __restrict__ layout, DBox box, float tolFactor,
                                                     uint64_t* __restrict__ masks, uint32_t* __restrict__ numSegments)
{
#pragma clang fp contract(off)
    const uint32_t g    = blockIdx.x * 4u + (threadIdx.x >> 6);
    const unsigned lane = threadIdx.x & 63u;
    if (g >= numFixed) return; // whole waves
    const uint32_t p0 = first + 64u * g;
    const uint32_t p1 = min(p0 + 63u, last - 1);
    const uint32_t bi = min(p0 + lane, p1);
    // the particle's fields load while the leaf search below runs (they do not depend on it)
    const double xb = x[bi], yb = y[bi], zb = z[bi];
    const double hb = h ? double(h[bi]) : 0.0;

    int lo = 0, hi = numLeaves; // layout[lo] <= p0; leaf(p0) in [lo, hi)
    while (hi - lo > 1)
    {
        const int  stride = (hi - lo + 63) / 64;
        const int  m      = lo + int(lane) * stride;
        const bool le     = m < hi && layout[m] <= p0;
        const int  k      = 63 - int(clz64(ballot(le))); // lane 0 always holds
        hi                = min(hi, lo + (k + 1) * stride);
        lo                = lo + k * stride;
    }
    unsigned level = 0;
    for (int c = lo;; c += 64)
    {
        const int  m  = c + int(lane);
        const bool in = m < numLeaves && layout[m] <= p1; // m <= leaf(p1)
        if (in && layout[m + 1] > layout[m]) level = max(level, treeLevel(leaves[m + 1] - leaves[m]));
        if (ballot(in) != ~uint64_t(0)) break;
    }
    // unit-box leaf volume 2^(-3 level); its cube root 2^(-level) is exact
    int      maxLevel = int(waveMax(int(level)));
    double   distCrit = ldexp(1.0, -maxLevel) * double(tolFactor);
    double   minExt   = fmin(fmin(box.len[0], box.len[1]), box.len[2]);
    double   px = xb * box.ilen[0], py = yb * box.ilen[1], pz = zb * box.ilen[2];
    double   pw = h ? 2.0 * hb / minExt : 1.0;
    double   qx = __shfl_down(px, 1, 64), qy = __shfl_down(py, 1, 64), qz = __shfl_down(pz, 1, 64);
    if (lane == 63) qx = px, qy = py, qz = pz;
    double   dx = qx - px, dy = qy - py, dz = qz - pz;
    double   d2 = dx * dx + dy * dy + dz * dz;
    double   crit2 = distCrit * distCrit;
    bool     split = d2 > fmin(crit2, pw * pw);
    uint64_t m     = ballot(split);
    if (lane == 0)
    {
        masks[g]       = m;
        numSegments[g] = 1u + popc64(m);
    }
}

// group boundaries from the split masks (makeSplits, groups_gpu.cuh:91-114)
__global__ __launch_bounds__(256) void grpBoundaries(uint32_t first, uint32_t last, uint32_t numFixed,
                                                     const uint64_t* __restrict__ masks,
                                                     const uint32_t* __restrict__ segOfs,
                                                     uint32_t* __restrict__ bounds)
{
    uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= numFixed) return;
    uint32_t base = first + 64u * g;
    uint32_t o    = segOfs[g];
    uint64_t m    = masks[g];
    bounds[o++]   = base;
    while (m)
    {
        uint32_t b  = uint32_t(__ffsll((unsigned long long)m) - 1);
        bounds[o++] = base + b + 1;
        m &= m - 1;
    }
    if (g + 1 == numFixed) bounds[o] = last;
}

// ---------------------------------------------------------------------------
// host driver shared by both entry points
static int sumTests(sphx_ctx* ctx, const unsigned long long* gtests, const uint32_t* list, uint32_t n,
                    unsigned long long* sum)
{
    nsSumTests<<<std::min<uint32_t>(256u, (n + 1023u) / 1024u), 256, 0, ctx->stream>>>(gtests, list, n, sum);
    SPHX_LAUNCH_CHECK(ctx, "nsSumTests");
    return SPHX_OK;
}

template<class Th, bool Sph>
static int runSearch(sphx_ctx* ctx, const GroupsDev& G, const double* x, const double* y, const double* z, Th* h,
                     const sphx_box* box, const sphx_octree* t, uint32_t ngmax, uint32_t ng0, uint32_t* nbrs,
                     SphLists lists, uint32_t* nc, double* listTests)
{
    ctx->nsTests = 0;
    *listTests   = 0;
    if (G.numGroups == 0) return SPHX_OK;
    uint32_t  numG   = G.numGroups;
    uint2*    ranges = scratchT<uint2>(ctx, S_NS_RANGES, size_t(numG) * NS_LCAP);
    uint32_t* rcnt   = scratchT<uint32_t>(ctx, S_NS_RCOUNT, numG);
    uint8_t*  iter   = scratchT<uint8_t>(ctx, S_NS_STATE, size_t(G.last));
    uint32_t* redo   = scratchT<uint32_t>(ctx, S_NS_REDO, 2 * size_t(numG));
    uint32_t* retry  = scratchT<uint32_t>(ctx, S_NS_RETRY, numG);
    auto*     gtests = scratchT<unsigned long long>(ctx, S_NS_TESTS, numG);
    auto*     gbox   = scratchT<GroupSearch>(ctx, S_NS_BOX, numG);
    uint32_t* over   = scratchT<uint32_t>(ctx, S_NS_OVER, numG);
    NsFlags*  flags  = scratchT<NsFlags>(ctx, S_SMALL, 1);
    if (!ranges || !rcnt || !iter || !redo || !retry || !gtests || !gbox || !over || !flags)
        return SPHX_ERR_NOMEM;
    DBox     db = makeDBox(box);
    HFactors hfac;
    if (Sph) SPHX_TRY(hFactors(ctx, ng0, hfac));

    if (G.last > G.first)
    {
        nsInitState<<<gridFor(G.last - G.first, 256), 256, 0, ctx->stream>>>(iter, G.first, G.last);
        SPHX_LAUNCH_CHECK(ctx, "nsInitState");
    }
    nsResetFlags<<<1, 64, 0, ctx->stream>>>(flags, 1);
    SPHX_LAUNCH_CHECK(ctx, "nsResetFlags");

    const uint32_t* list      = nullptr; // nullptr: all groups
    uint32_t        numLaunch = numG;
    int             pingpong  = 0;
    for (int pass = 0; pass < 12 && numLaunch > 0; ++pass)
    {
        uint32_t* outList = redo + size_t(pingpong) * numG;
        {
            KTimer kt_(ctx, "nsGroupRanges");
            nsGroupRanges<Th><<<numLaunch, 64, 0, ctx->stream>>>(G, list, x, y, z, h, t->childOffsets,
                                                                t->internalToLeaf, t->layout, t->centers, t->sizes,
                                                                db, ranges, rcnt, gbox, retry, flags);
        }
        SPHX_LAUNCH_CHECK(ctx, "nsGroupRanges");
        {
            KTimer   kt_(ctx, "nsGroupRangesRetry");
            uint32_t grid = std::min<uint32_t>(numLaunch, uint32_t(ctx->numCU) * 4u);
            nsGroupRangesRetry<Th><<<grid, 64, 0, ctx->stream>>>(G, x, y, z, h, t->childOffsets, t->internalToLeaf,
                                                                 t->layout, t->centers, t->sizes, db, ranges, rcnt,
                                                                 gbox, retry, flags);
        }
        SPHX_LAUNCH_CHECK(ctx, "nsGroupRangesRetry");
        {
            KTimer kt_(ctx, "nsCandidates", true);
            nsCandidates<Th, Sph><<<numLaunch, 256, 0, ctx->stream>>>(G, list, x, y, z, h, iter, ranges, rcnt, gbox, db,
                                                                      ngmax, ng0, hfac, nbrs, lists, nc, outList, over,
                                                                      flags, gtests);
        }
        SPHX_LAUNCH_CHECK(ctx, "nsCandidates");
        // the tests of this pass, and those behind the lists as they are now: every group's last pass
        SPHX_TRY(sumTests(ctx, gtests, list, numLaunch, &flags->tests));
        if (pass) SPHX_TRY(sumTests(ctx, gtests, nullptr, numG, &flags->listTests));
        NsFlags hf;
        SPHX_TRY(readBack(ctx, flags, &hf, sizeof(NsFlags)));
        if (hf.overCount && !hf.overflow && !hf.badGroup)
        {
            {
                KTimer kt_(ctx, "nsCandidatesExact", true);
                nsCandidatesExact<Th, Sph><<<hf.overCount, 64, 0, ctx->stream>>>(G, over, x, y, z, h, iter, ranges, rcnt,
                                                                                 db, ngmax, ng0, hfac, nbrs, lists, nc,
                                                                                 outList, flags, gtests);
            }
            SPHX_LAUNCH_CHECK(ctx, "nsCandidatesExact");
            // (nsCandidates left 0 for these groups)
            SPHX_TRY(sumTests(ctx, gtests, over, hf.overCount, &flags->tests));
            if (pass) SPHX_TRY(sumTests(ctx, gtests, over, hf.overCount, &flags->listTests));
            SPHX_TRY(readBack(ctx, flags, &hf, sizeof(NsFlags)));
        }
        ctx->nsTests += double(hf.tests);
        *listTests = double(pass ? hf.listTests : hf.tests);
        if (hf.overflow) return fail(ctx, SPHX_ERR_STACK, "neighbor search: traversal capacity exceeded");
        if (hf.badGroup) return argError(ctx, "neighbor search: a target group holds more than 64 particles");
        if (hf.hfacMiss)
            return fail(ctx, SPHX_ERR_STACK,
                        "neighbor search: a neighbor count to update h from exceeds the factor table (" +
                            std::to_string(kHFactorCap) + ")");
        if (!Sph || hf.redoCount == 0) break;
        numLaunch = hf.redoCount;
        list      = outList;
        pingpong ^= 1;
        nsResetFlags<<<1, 64, 0, ctx->stream>>>(flags, 0);
        SPHX_LAUNCH_CHECK(ctx, "nsResetFlags");
    }
    return SPHX_OK;
}

int groupsFromArgs(sphx_ctx* ctx, const sphx_groups* groups, uint32_t first, uint32_t last, GroupsDev& G)
{
    if (groups && groups->groupStart)
    {
        if (!groups->groupEnd) return argError(ctx, "groups: groupEnd is null");
        G.first     = groups->firstBody;
        G.last      = groups->lastBody;
        G.numGroups = groups->numGroups;
        G.start     = groups->groupStart;
        G.end       = groups->groupEnd;
    }
    else
    {
        G.first     = groups ? groups->firstBody : first;
        G.last      = groups ? groups->lastBody : last;
        G.numGroups = (G.last - G.first + 63) / 64;
        G.start     = nullptr;
        G.end       = nullptr;
    }
    if (G.last < G.first) return argError(ctx, "groups: lastBody < firstBody");
    return SPHX_OK;
}

static bool validTree(const sphx_octree* t)
{
    return t && t->numNodes > 0 && t->childOffsets && t->internalToLeaf && t->layout && t->centers && t->sizes;
}

} // namespace sphx

using namespace sphx;

extern "C"
{

int sphx_compute_groups(sphx_ctx* ctx, uint32_t first, uint32_t last, const double* x, const double* y,
                        const double* z, const void* h, int32_t precision, const sphx_octree* tree,
                        const sphx_box* box, float tolFactor, sphx_groups* groups)
{
    if (!ctx) return SPHX_ERR_ARG;
    if (!groups) return argError(ctx, "compute_groups: null output");
    if (last < first) return argError(ctx, "compute_groups: last < first");
    if (!validBox(box)) return argError(ctx, "compute_groups: invalid box");
    if (!tree || tree->numLeafNodes < 1 || !tree->leaves || !tree->layout)
        return argError(ctx, "compute_groups: tree needs numLeafNodes, leaves and layout");
    if (precision != SPHX_FP64 && precision != SPHX_MIXED) return argError(ctx, "compute_groups: unknown precision");
    uint32_t numFixed = (last - first + 63) / 64;
    *groups           = sphx_groups{first, last, 0, nullptr, nullptr};
    if (numFixed == 0) return SPHX_OK;
    if (!x || !y || !z) return argError(ctx, "compute_groups: null coordinates");
    uint64_t* masks = scratchT<uint64_t>(ctx, S_GROUPS_TMP, numFixed);
    uint32_t* segs  = scratchT<uint32_t>(ctx, S_NS_RCOUNT, size_t(numFixed) + 1);
    if (!masks || !segs) return SPHX_ERR_NOMEM;
    DBox db = makeDBox(box);
    {
        KTimer   kt_(ctx, "grpSplitMasks");
        uint32_t grid = (numFixed + 3u) / 4u;
        if (precision == SPHX_FP64)
            grpSplitMasks<double><<<grid, 256, 0, ctx->stream>>>(first, last, numFixed, x, y, z,
                                                                 static_cast<const double*>(h), tree->leaves,
                                                                 tree->numLeafNodes, tree->layout, db, tolFactor,
                                                                 masks, segs);
        else
            grpSplitMasks<float><<<grid, 256, 0, ctx->stream>>>(first, last, numFixed, x, y, z,
                                                                static_cast<const float*>(h), tree->leaves,
                                                                tree->numLeafNodes, tree->layout, db, tolFactor,
                                                                masks, segs);
    }
    SPHX_LAUNCH_CHECK(ctx, "grpSplitMasks");
    SPHX_TRY(exclusiveScanU32(ctx, segs, segs, numFixed));
    uint32_t numGroups = 0;
    SPHX_TRY(readBack(ctx, segs + numFixed, &numGroups, sizeof(uint32_t)));
    uint32_t* bounds = scratchT<uint32_t>(ctx, S_GROUPS, size_t(numGroups) + 1);
    if (!bounds) return SPHX_ERR_NOMEM;
    grpBoundaries<<<gridFor(numFixed, 256), 256, 0, ctx->stream>>>(first, last, numFixed, masks, segs, bounds);
    SPHX_LAUNCH_CHECK(ctx, "grpBoundaries");
    groups->numGroups  = numGroups;
    groups->groupStart = bounds;
    groups->groupEnd   = bounds + 1;
    return SPHX_OK;
}

int sphx_find_neighbors(sphx_ctx* ctx, const double* x, const double* y, const double* z, const double* h,
                        uint32_t first, uint32_t last, const sphx_box* box, const sphx_octree* tree, uint32_t ngmax,
                        uint32_t* nbrs, uint32_t* nc)
{
    if (!ctx) return SPHX_ERR_ARG;
    if (last < first) return argError(ctx, "find_neighbors: last < first");
    if (last == first) return SPHX_OK;
    if (!x || !y || !z || !h || !nc) return argError(ctx, "find_neighbors: null pointer");
    if (!validBox(box)) return argError(ctx, "find_neighbors: invalid box");
    if (!validTree(tree)) return argError(ctx, "find_neighbors: incomplete tree view");
    GroupsDev G;
    SPHX_TRY(groupsFromArgs(ctx, nullptr, first, last, G));
    double listTests; // (of no interest: the lists go to the caller)
    return runSearch<double, false>(ctx, G, x, y, z, const_cast<double*>(h), box, tree, ngmax, 0, nbrs, SphLists{},
                                    nc, &listTests);
}

int sphx_find_neighbors_sph(sphx_ctx* ctx, const sphx_groups* groups, sphx_particles* d, const sphx_box* box,
                            const sphx_octree* tree)
{
    if (!ctx) return SPHX_ERR_ARG;
    if (!d || !d->x || !d->y || !d->z || !d->h || !d->nc) return argError(ctx, "find_neighbors_sph: null field");
    if (!validBox(box)) return argError(ctx, "find_neighbors_sph: invalid box");
    if (!validTree(tree)) return argError(ctx, "find_neighbors_sph: incomplete tree view");
    if (d->ng0 > d->ngmax) return fail(ctx, SPHX_ERR_NGMAX, "ng0 should be smaller than ngmax");
    if (d->ngmax == 0) return argError(ctx, "find_neighbors_sph: ngmax must be > 0");
    GroupsDev G;
    SPHX_TRY(groupsFromArgs(ctx, groups, 0, uint32_t(d->n), G));
    if (G.last > d->n) return argError(ctx, "find_neighbors_sph: group range exceeds n");
    if (d->ngmax > 4096) return argError(ctx, "find_neighbors_sph: ngmax must be <= 4096");
    ctx->nsValid = false;
    size_t   numSub = size_t(G.numGroups) * 4;
    SphLists L;
    L.capU   = 32u * ((16u * d->ngmax + 31u) / 32u);
    L.words  = L.capU / 32u;
    L.masks  = scratchT<uint32_t>(ctx, S_NS_LISTS, numSub * L.words * 16);
    L.unions = scratchT<uint32_t>(ctx, S_NS_UNION, numSub * L.capU);
    L.usize  = scratchT<uint32_t>(ctx, S_NS_USIZE, numSub);
    if (!L.masks || !L.unions || !L.usize) return SPHX_ERR_NOMEM;
    int    st;
    double listTests;
    if (d->precision == SPHX_FP64)
        st = runSearch<double, true>(ctx, G, d->x, d->y, d->z, static_cast<double*>(d->h), box, tree, d->ngmax,
                                     d->ng0, nullptr, L, d->nc, &listTests);
    else if (d->precision == SPHX_MIXED)
        st = runSearch<float, true>(ctx, G, d->x, d->y, d->z, static_cast<float*>(d->h), box, tree, d->ngmax,
                                    d->ng0, nullptr, L, d->nc, &listTests);
    else
        return argError(ctx, "find_neighbors_sph: unknown precision");
    if (st != SPHX_OK) return st;
    ctx->nsLists  = L;
    ctx->nsValid  = true;
    ctx->nsGroups = G;
    ctx->nsNgmax  = d->ngmax;
    ctx->nsListTests = listTests;
    ctx->nsNc     = d->nc;
    return SPHX_OK;
}

int sphx_export_neighbors(sphx_ctx* ctx, uint32_t* nbrs)
{
    if (!ctx) return SPHX_ERR_ARG;
    if (!ctx->nsValid) return fail(ctx, SPHX_ERR_STATE, "export_neighbors: no neighbor lists in context");
    if (!nbrs) return argError(ctx, "export_neighbors: null pointer");
    const GroupsDev& G = ctx->nsGroups;
    if (G.numGroups == 0) return SPHX_OK;
    nsExport<<<gridFor(G.numGroups, 4), 256, 0, ctx->stream>>>(G, ctx->nsLists, ctx->nsNgmax, ctx->nsNc, nbrs);
    SPHX_LAUNCH_CHECK(ctx, "nsExport");
    return SPHX_OK;
}

} // extern "C"
