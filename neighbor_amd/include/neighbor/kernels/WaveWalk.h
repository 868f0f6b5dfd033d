// WaveWalk.h -- exact counts and pair rows by one rope path per wave.
//
// 64 consecutive queries of the traversal order (one per lane) walk the bucket records together:
// node indices are wave-uniform (node records are scalar loads) and the wave descends where any
// lane's padded box test passes.  One image after the other.  Against the walk by node fronts
// (FrontWalk.h) it takes more dependent loads per wave, but 64 registers and 16 KB of LDS per block
// instead of 128 and 28-39, so twice the waves: it is the faster one where a launch has many times
// more waves than the chip holds and few leaves per query (LBVHTraverser::sparseLimit has the lines
// and the figures of both sides), and it serves unusual queries, whose box tests may pass everywhere,
// 64 leaves at a time.
#ifndef NEIGHBOR_KERNELS_WAVE_WALK_H_
#define NEIGHBOR_KERNELS_WAVE_WALK_H_

#include "LBVHTraverse.h"

namespace neighbor
{
namespace gpu
{
namespace kernel
{
namespace wave
{
//! The library's pair rows: at positions their thread data holds (pos, end), written by the walks.
template<class O>
struct pair_rows
    : std::integral_constant<bool, std::is_same<O, PairListOp>::value || std::is_same<O, RowPairOp>::value
                                       || std::is_same<O, PlacedRowPairOp>::value>
    {};
//! Output ops of this walk.
template<class O>
struct walks : std::integral_constant<bool, pair_rows<O>::value || std::is_same<O, CountNeighborsOp>::value> {};

//! Per-wave LDS of the buckets.  The per-rank records share one 16-byte stride, so a round reaches
//! all of a rank's data from one 32-bit offset (immediate offsets in the LDS instructions, no
//! per-array address arithmetic).
struct CompactWave
    {
    float4 leaf[64];                 //!< bucket leaves (x, y, z, bits(primitive))
    float4 qc[64];                   //!< per rank: float center, t_lo
    uint4 qx[64];                    //!< per rank: bits(t_hi), lane, unused, unused
    ulonglong2 row[64];              //!< per rank: (next row position, row end); the count op uses .x only
    };

//! Orders the wave's LDS accesses before and after it (one wave: no instruction).
__device__ __forceinline__ void lds_order()
    {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }

//! Element of an array member of the wave's CompactWave at byte offset `off` (16-byte records).
template<class T>
__device__ __forceinline__ T& compact_at(CompactWave& cw, const unsigned int member, const unsigned int off)
    {
    return *reinterpret_cast<T*>(reinterpret_cast<char*>(&cw) + member + off);
    }

//! Leaves per lane in a round (a divisor of 64).  Measured on the N=10^6 exact fill: 1 leaf 0.688
//! ms, 2 leaves 0.659 ms, 4 leaves 0.725 ms (fewer instructions per candidate, but more tests of
//! padding and of the last partial round of each bucket).
constexpr unsigned int kCompactLeaves = 2;

//! Leaf tests of the bucket [first, end) for the lanes set in A (wave-uniform).
/*!
 * Only the lanes whose box test passed (a of 64) have work, so the wave enumerates the a x n (query,
 * leaf) pairs instead of n leaves for 64 lanes, two leaves per lane: slot t is query rank r = t / n2
 * (r-th active lane, n2 = ceil(n / 2)) and leaves 2 (t % n2) and the next, 128 pairs per round.  A
 * query's slots sit in consecutive lanes in leaf order, so its hits of a round are numbered by two
 * lane-mask counts and written as one contiguous run of its row; ranks, leaves and running counts
 * are exchanged through LDS, within the wave only.  Each query's hits come in bucket order, then in
 * leaf order.  Leaves are decided by ExactSphereQueryOp's banded float test, the band in FP64.
 */
template<class OutputOpT, class TransformOpT>
__device__ __forceinline__ void bucket_compact(const OutputOpT& out, typename OutputOpT::ThreadData& result,
                                               const TransformOpT& transform, const unsigned long long A, CompactWave& cw,
                                               const ExactSphere& v, const float4* __restrict__ points,
                                               const unsigned int first, const unsigned int end)
    {
    constexpr bool kPairs = pair_rows<OutputOpT>::value;
    const unsigned int lane = threadIdx.x & 63u;
    const bool hit = lane_in(A);
    const unsigned int a = static_cast<unsigned int>(__popcll(A));
    const unsigned int n = end - first;                   // 1..64 leaves
    const unsigned int rank = count_below(A);
    unsigned long long pos0 = 0ull;
    // The last slot of a bucket whose size K does not divide pairs its leaves with padding
    // leaves, which only need x = NaN: so is then their squared distance, which no comparison
    // accepts (stale y, z; an infinite one would be within an infinite radius).  Leaf j sits at (j % K) 64/K + j / K: the lanes of a round
    // read their k-th leaves from consecutive 16-byte records (no LDS bank conflicts).
    constexpr unsigned int K = kCompactLeaves;
    const unsigned int lpos = (lane % K) * (64u / K) + lane / K;
    if (lane < n) cw.leaf[lpos] = points[first + lane];
    else if (lane < (n + K - 1u) / K * K) cw.leaf[lpos].x = __builtin_nanf("");
    if (hit)
        {
        cw.qc[rank] = make_float4(v.c.x, v.c.y, v.c.z, v.t_lo);
        cw.qx[rank] = make_uint4(__float_as_uint(v.t_hi), lane, 0u, 0u);
        unsigned long long row_end = 0ull;
        if constexpr (kPairs)
            {
            pos0 = result.pos;
            row_end = result.end;
            }
        cw.row[rank] = make_ulonglong2(pos0, row_end);
        }
    lds_order();

    // slots of K consecutive leaves: slot (r, k) tests query rank r against leaves K k ..
    // K k + K - 1 (padding past n), so one pair index serves K leaf tests
    const unsigned int nK = (n + K - 1u) / K;
    const unsigned int total = a * nK;
    // hardware reciprocal (1 ulp): r = t / nK below needs (t + 1/2) * inv_n within 1/(2 nK) of
    // (t + 1/2) / nK, and the error here is below 64 * 2^-22 for t < 4096, nK <= 64
    const float inv_n = __builtin_amdgcn_rcpf(static_cast<float>(nK));
    for (unsigned int t0 = 0; t0 < total; t0 += 64u)
        {
        const unsigned int left = total - t0;
        const unsigned long long validm = left >= 64u ? ~0ull : ((1ull << left) - 1ull);
        const unsigned int t = t0 + lane;
        // r = t / nK exactly: (t + 1/2) / nK is at least 1/(2 nK) away from an integer and the
        // float product errs by far less for t < 4096; lanes past the end take the last slot
        const unsigned int tc = min(t, total - 1u);
        const unsigned int r = static_cast<unsigned int>((static_cast<float>(tc) + 0.5f) * inv_n);
        const unsigned int rn = __umul24(r, nK);
        const unsigned int k0 = tc - rn;                 // slot in the query's row: leaves K k0 ..
        const unsigned int ro = r << 4;                  // byte offset of rank r's records
        const float4 q = compact_at<float4>(cw, offsetof(CompactWave, qc), ro);
        const uint4 qx = compact_at<uint4>(cw, offsetof(CompactWave, qx), ro);
        const float T_hi = __uint_as_float(qx.x);
        float4 p[K];
        unsigned long long m[K], bm[K];
        unsigned long long band = 0ull;
        #pragma unroll
        for (unsigned int k = 0; k < K; ++k)
            {
            p[k] = compact_at<float4>(cw, offsetof(CompactWave, leaf), (k * (64u / K) + k0) << 4);
            const float ex = q.x - p[k].x;
            const float ey = q.y - p[k].y;
            const float ez = q.z - p[k].z;
            const float d = fmaf(ex, ex, fmaf(ey, ey, ez * ez));     // NaN for padding
            m[k] = vote(d <= q.w) & validm;
            bm[k] = vote(d <= T_hi) & ~m[k] & validm;
            band |= bm[k];
            }
        if (band)
            {
            // the FP64 definition for the pairs in the float band; the query's FP64 center
            // and R^2 come from the lane that owns it (every lane takes part in the shuffles)
            const int src = static_cast<int>(qx.y);
            const double cx = __shfl(v.cd.x, src, 64);
            const double cy = __shfl(v.cd.y, src, 64);
            const double cz = __shfl(v.cd.z, src, 64);
            const double R2 = __shfl(v.R2, src, 64);
            #pragma unroll
            for (unsigned int k = 0; k < K; ++k)
                {
                bool e = false;
                if (lane_in(bm[k]))
                    {
                    const double dx = cx - static_cast<double>(p[k].x);
                    const double dy = cy - static_cast<double>(p[k].y);
                    const double dz = cz - static_cast<double>(p[k].z);
                    e = (dx * dx + dy * dy) + dz * dz <= R2;
                    }
                m[k] |= vote(e);
                }
            }
        // lanes of query r in this round: [lo, hi); its hits below this lane are the hits of
        // the lanes from lo up (per-lane masks of the wave-uniform hit masks), K per lane
        const unsigned int lo = rn > t0 ? rn - t0 : 0u;
        const unsigned int hi = min(min(rn + nK - t0, 64u), left);
        const unsigned long long from_lo = ~0ull << lo;
        unsigned int before = 0u;
        #pragma unroll
        for (unsigned int k = 0; k < K; ++k) before += count_below(m[k] & from_lo);
        // one read of the rank's row record serves the hits' stores and the cursor update
        ulonglong2& rowref = compact_at<ulonglong2>(cw, offsetof(CompactWave, row), ro);
        const ulonglong2 row = rowref;
        unsigned long long at = row.x + before;
        #pragma unroll
        for (unsigned int k = 0; k < K; ++k)
            {
            const bool in = lane_in(m[k]);
            // the image bytes are written per image walk (image_run)
            if constexpr (kPairs)
                if (in && at < row.y) out.neigh[at] = transform(__float_as_uint(p[k].w));
            at += in ? 1u : 0u;
            }
        if (lane + 1u == hi) rowref.x = at;
        lds_order();
        }
    if (hit)
        {
        const unsigned int c = static_cast<unsigned int>(cw.row[rank].x - pos0);
        result.num_neigh += c;
        if constexpr (kPairs) result.pos += c;
        }
    lds_order();
    }

//! False for a query that has no hit whatever the points: no distance from a center that is not finite
//! is within a finite radius, and none within or from a NaN (box tests let such centers through
//! everywhere).
__device__ __forceinline__ bool can_hit(const float4& q)
    {
    const float inf = __builtin_huge_valf();
    const bool finite = fabsf(q.x) < inf && fabsf(q.y) < inf && fabsf(q.z) < inf;
    return finite ? q.w == q.w : fabsf(q.w) == inf && q.x == q.x && q.y == q.y && q.z == q.z;
    }

//! The walk of one wave over the subtree [root, stop) for one query per valid lane.
/*!
 * Image bits come from each query's own test against root_box; the wave visits the images any lane
 * needs, in ascending order.  Hits come out image by image, then in Morton order, as from the other
 * walks; the emitted value is transform(primitive).  Output ops that relocate overflowed rows get a
 * second pass for the moved lanes.
 */
template<class OutputOpT, class TranslateOpT, class TransformOpT>
__device__ __forceinline__ void walk(const OutputOpT& out, const float4* __restrict__ nodes, const float4* __restrict__ points,
                                     const BoundingBox& root_box, const int root, const int stop, const ExactSphereQueryOp& query,
                                     const TranslateOpT& images, const TransformOpT& transform, const bool valid,
                                     const unsigned int idx, const float4& q, const unsigned int n_internal,
                                     const unsigned int n_nodes, CompactWave& compact)
    {
    static_assert(walks<OutputOpT>::value, "counts and the library's pair rows");
    constexpr bool kPairs = pair_rows<OutputOpT>::value;
    typename OutputOpT::ThreadData result = out.setup(idx, q);

    uint32_t image_flags = 0;
    const unsigned int nimg = images.size() < 32u ? images.size() : 32u;
    for (unsigned int k = 0; k < nimg; ++k)
        if (valid && can_hit(q) && query.overlap(query.get(q, images.get(k)), root_box)) image_flags |= 1u << k;

    // pass 1 walks every lane; pass 2 (output ops that relocate overflowed rows) only the moved lanes
    uint32_t flags = image_flags;
    for (int pass = 0; pass < 2; ++pass)
        {
        uint32_t wave_flags = 0;
        for (unsigned int k = 0; k < nimg; ++k)
            if (vote((flags >> k) & 1u)) wave_flags |= 1u << k;

        while (wave_flags)
            {
            const unsigned int k = __builtin_ctz(wave_flags);
            wave_flags &= wave_flags - 1u;
            const unsigned long long activem = vote((flags >> k) & 1u);
            const ExactSphere v = query.get(q, images.get(k));
            unsigned long long run0 = 0ull;
            if constexpr (kPairs) run0 = result.pos;
            int node = root;
            for (int budget = 2 * static_cast<int>(n_nodes); node != stop && budget > 0; --budget)
                {
                node = __builtin_amdgcn_readfirstlane(node);
                const float4 a = uniform_load(nodes, 2u * node);
                const float4 b = uniform_load(nodes, 2u * node + 1u);
                // every lane tests (no divergent branch); inactive lanes are masked out
                const unsigned long long hitm = vote(box_distance2(center(v), a, b) <= threshold(v)) & activem;
                int next = __float_as_int(b.w);
                if (hitm)
                    {
                    const int lf = __float_as_int(a.w);
                    if (lf < 0) bucket_compact(out, result, transform, hitm, compact, v, points, ~static_cast<unsigned int>(lf), bucket_end(next, n_internal));
                    else next = lf;
                    }
                node = next;
                }
            if constexpr (kPairs)
                if (out.image) image_run(out.image, run0, result.pos < result.end ? result.pos : result.end, k);
            }
        if constexpr (!detail::relocates<OutputOpT>::value) break;
        else
            {
            const bool again = valid && out.relocate(result);
            if (!vote(again)) break;
            flags = again ? image_flags : 0u;
            }
        }
    if (valid) out.finalize(result);
    }
} // end namespace wave
} // end namespace kernel
} // end namespace gpu
} // end namespace neighbor

#endif // NEIGHBOR_KERNELS_WAVE_WALK_H_
