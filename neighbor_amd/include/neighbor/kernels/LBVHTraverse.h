// LBVHTraverse.h -- compression and stackless rope traversal kernels.
//
// Reference semantics kept (include/neighbor/kernels/LBVHTraverser.cuh):
//   lbvh_compress  node boxes quantized to 10 bits per axis against the root box,
//                  lower bins rounded down from the root's lower corner, upper bins
//                  rounded down from the root's upper corner, with the HIP-path
//                  directed rounding (:45-125).  The rope comes from the build.
//   lbvh_traverse  per query: image bits from the unquantized root box, then for
//                  each image in ascending order a rope walk from the root that
//                  descends left on overlap and follows the rope otherwise; a leaf
//                  overlap goes through refine and the output op (:155-252).
// Additions: a float rope record (no decode work in the hot loop), an optional
// query order (thread t serves query order[t]; with the LBVH's primitive order a
// self-query walks neighboring paths in neighboring lanes), and the image index
// handed to output ops that accept it.
#ifndef NEIGHBOR_KERNELS_LBVH_TRAVERSE_H_
#define NEIGHBOR_KERNELS_LBVH_TRAVERSE_H_

#include "../BoundingVolumes.h"
#include "../LBVHData.h"
#include "../LBVHTraverserData.h"

#include <cstddef>
#include <type_traits>
#include <utility>

namespace neighbor
{
namespace gpu
{
namespace detail
{
// prefer refine(ThreadData, Volume, prim) when the query op has it
template<class Q>
__device__ __forceinline__ auto refine_hit(const Q& q, const typename Q::ThreadData& t, const typename Q::Volume& v, int p, int)
    -> decltype(q.refine(t, v, p))
    {
    return q.refine(t, v, p);
    }
template<class Q>
__device__ __forceinline__ bool refine_hit(const Q& q, const typename Q::ThreadData& t, const typename Q::Volume&, int p, long)
    {
    return q.refine(t, p);
    }
// prefer process(ThreadData&, prim, image) when the output op has it
template<class O>
__device__ __forceinline__ auto emit_hit(const O& o, typename O::ThreadData& t, int p, unsigned int k, int)
    -> decltype(o.process(t, p, k))
    {
    o.process(t, p, k);
    }
template<class O>
__device__ __forceinline__ void emit_hit(const O& o, typename O::ThreadData& t, int p, unsigned int, long)
    {
    o.process(t, p);
    }

// output ops whose rows can overflow and be moved provide bool relocate(ThreadData&): true when
// the query's row was moved (the query is then walked again into its new row)
template<class O, class = void>
struct relocates : std::false_type {};
template<class O>
struct relocates<O, decltype(void(std::declval<const O&>().relocate(std::declval<typename O::ThreadData&>())))>
    : std::true_type {};

//! Root quantization scales (kernels/LBVHTraverser.cuh:64-74).
__device__ __forceinline__ float bin_scale(float lo, float hi)
    {
    float L = approx::fsub_ru(hi, lo);
    if (L <= 0.0f) L = 1.0f;
    return approx::fdiv_rd(1023.0f, L);
    }

__device__ __forceinline__ uint32_t quantize(float offset, float scale)
    {
    return approx::sat_f2u(floorf(approx::fmul_rd(offset, scale)));
    }

//! Decompressed (outward) box of a quantized record (kernels/LBVHTraverser.cuh:218-226).
__device__ __forceinline__ BoundingBox decode_box(uint32_t lo3, uint32_t hi3, const float3& rlo, const float3& rhi, const float3& bins)
    {
    BoundingBox b;
    b.lo.x = approx::fadd_rd(rlo.x, approx::fmul_rd(static_cast<float>((lo3 >> 20) & 0x3ffu), bins.x));
    b.lo.y = approx::fadd_rd(rlo.y, approx::fmul_rd(static_cast<float>((lo3 >> 10) & 0x3ffu), bins.y));
    b.lo.z = approx::fadd_rd(rlo.z, approx::fmul_rd(static_cast<float>(lo3 & 0x3ffu), bins.z));
    b.hi.x = approx::fsub_ru(rhi.x, approx::fmul_rd(static_cast<float>((hi3 >> 20) & 0x3ffu), bins.x));
    b.hi.y = approx::fsub_ru(rhi.y, approx::fmul_rd(static_cast<float>((hi3 >> 10) & 0x3ffu), bins.y));
    b.hi.z = approx::fsub_ru(rhi.z, approx::fmul_rd(static_cast<float>(hi3 & 0x3ffu), bins.z));
    return b;
    }
} // end namespace detail

namespace kernel
{

//! Quantized records for all nodes; node 0's thread also writes the root box and bin sizes.
template<class TransformOpT>
__global__ void __launch_bounds__(1024) lbvh_compress(const LBVHCompressedData ctree,
                                                      const TransformOpT transform,
                                                      const ConstLBVHData tree,
                                                      const uint32_t n_internal,
                                                      const uint32_t n_nodes)
    {
    const uint32_t idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= n_nodes) return;
    const float3 rlo = tree.lo[tree.root];
    const float3 rhi = tree.hi[tree.root];
    const float3 scale = make_float3(detail::bin_scale(rlo.x, rhi.x), detail::bin_scale(rlo.y, rhi.y), detail::bin_scale(rlo.z, rhi.z));

    const float3 lo = tree.lo[idx];
    const float3 hi = tree.hi[idx];
    const uint32_t lo3 = (detail::quantize(approx::fsub_rd(lo.x, rlo.x), scale.x) << 20)
                       + (detail::quantize(approx::fsub_rd(lo.y, rlo.y), scale.y) << 10)
                       + detail::quantize(approx::fsub_rd(lo.z, rlo.z), scale.z);
    const uint32_t hi3 = (detail::quantize(approx::fsub_rd(rhi.x, hi.x), scale.x) << 20)
                       + (detail::quantize(approx::fsub_rd(rhi.y, hi.y), scale.y) << 10)
                       + detail::quantize(approx::fsub_rd(rhi.z, hi.z), scale.z);
    const int lf = (idx < n_internal) ? tree.left[idx] : static_cast<int>(~transform(tree.primitive[idx - n_internal]));
    ctree.data[idx] = make_int4(static_cast<int>(lo3), static_cast<int>(hi3), lf, tree.rope[idx]);

    if (idx == 0)
        {
        *ctree.lo = rlo;
        *ctree.hi = rhi;
        *ctree.bins = make_float3(approx::frcp_rd(scale.x), approx::frcp_rd(scale.y), approx::frcp_rd(scale.z));
        }
    }

//! Float rope records.  DECODED: store the decompressed quantized boxes (results
//! identical to the quantized walk); otherwise store the exact node boxes.
template<bool DECODED>
__global__ void __launch_bounds__(1024) lbvh_float_ropes(float4* __restrict__ out,
                                                         const LBVHCompressedData ctree,
                                                         const ConstLBVHData tree,
                                                         const uint32_t n_nodes)
    {
    const uint32_t idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= n_nodes) return;
    const int4 r = ctree.data[idx];
    BoundingBox b;
    if (DECODED)
        b = detail::decode_box(static_cast<uint32_t>(r.x), static_cast<uint32_t>(r.y), tree.lo[tree.root], tree.hi[tree.root], *ctree.bins);
    else
        b = BoundingBox(tree.lo[idx], tree.hi[idx]);
    out[2 * idx] = make_float4(b.lo.x, b.lo.y, b.lo.z, __int_as_float(r.z));
    out[2 * idx + 1] = make_float4(b.hi.x, b.hi.y, b.hi.z, __int_as_float(r.w));
    }

//! Quantized rope traversal, one query per thread.
template<class OutputOpT, class QueryOpT, class TranslateOpT>
__global__ void __launch_bounds__(1024) lbvh_traverse_ropes(const OutputOpT out,
                                                            const LBVHCompressedData lbvh,
                                                            const QueryOpT query,
                                                            const TranslateOpT images,
                                                            const unsigned int* __restrict__ order,
                                                            const unsigned int query_budget)
    {
    const unsigned int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= query.size()) return;
    const unsigned int idx = order ? order[t] : t;

    const BoundingBox root_box(*lbvh.lo, *lbvh.hi);
    const float3 rlo = root_box.lo, rhi = root_box.hi;
    const float3 bins = *lbvh.bins;

    const typename QueryOpT::ThreadData qdata = query.setup(idx);
    typename OutputOpT::ThreadData result = out.setup(idx, qdata);

    uint32_t image_flags = 0;
    const unsigned int nimg = images.size() < 32u ? images.size() : 32u;
    for (unsigned int k = 0; k < nimg; ++k)
        if (query.overlap(query.get(qdata, images.get(k)), root_box)) image_flags |= 1u << k;

    for (int pass = 0; pass < 2; ++pass)
        {
        uint32_t flags = image_flags;
        while (flags)
            {
            const unsigned int k = __builtin_ctz(flags);
            flags &= flags - 1u;
            const typename QueryOpT::Volume v = query.get(qdata, images.get(k));
            int node = lbvh.root;
            // ropes and left children only move forward in preorder: a walk visits each node at most once
            for (int budget = 2 * static_cast<int>(query_budget); node != LBVHSentinel && budget > 0; --budget)
                {
                const int4 rec = lbvh.data[node];
                const BoundingBox box = detail::decode_box(static_cast<uint32_t>(rec.x), static_cast<uint32_t>(rec.y), rlo, rhi, bins);
                node = rec.w;
                if (query.overlap(v, box))
                    {
                    if (rec.z < 0)
                        {
                        const int prim = ~rec.z;
                        if (detail::refine_hit(query, qdata, v, prim, 0)) detail::emit_hit(out, result, prim, k, 0);
                        }
                    else
                        {
                        node = rec.z;
                        }
                    }
                }
            }
        if constexpr (!detail::relocates<OutputOpT>::value) break;
        else if (!out.relocate(result)) break;
        }
    out.finalize(result);
    }

//! Float rope traversal (no decode work per node), one query per thread.
template<class OutputOpT, class QueryOpT, class TranslateOpT>
__global__ void __launch_bounds__(1024) lbvh_traverse_float_ropes(const OutputOpT out,
                                                                  const LBVHFloatRopeData lbvh,
                                                                  const float3* __restrict__ root_lo,
                                                                  const float3* __restrict__ root_hi,
                                                                  const QueryOpT query,
                                                                  const TranslateOpT images,
                                                                  const unsigned int* __restrict__ order,
                                                                  const unsigned int query_budget)
    {
    const unsigned int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= query.size()) return;
    const unsigned int idx = order ? order[t] : t;
    const BoundingBox root_box(*root_lo, *root_hi);

    const typename QueryOpT::ThreadData qdata = query.setup(idx);
    typename OutputOpT::ThreadData result = out.setup(idx, qdata);

    uint32_t image_flags = 0;
    const unsigned int nimg = images.size() < 32u ? images.size() : 32u;
    for (unsigned int k = 0; k < nimg; ++k)
        if (query.overlap(query.get(qdata, images.get(k)), root_box)) image_flags |= 1u << k;

    for (int pass = 0; pass < 2; ++pass)
        {
        uint32_t flags = image_flags;
        while (flags)
            {
            const unsigned int k = __builtin_ctz(flags);
            flags &= flags - 1u;
            const typename QueryOpT::Volume v = query.get(qdata, images.get(k));
            int node = lbvh.root;
            for (int budget = 2 * static_cast<int>(query_budget); node != LBVHSentinel && budget > 0; --budget)
                {
                const float4 a = lbvh.data[2 * node];
                const float4 b = lbvh.data[2 * node + 1];
                const int lf = __float_as_int(a.w);
                node = __float_as_int(b.w);
                if (query.overlap(v, BoundingBox(make_float3(a.x, a.y, a.z), make_float3(b.x, b.y, b.z))))
                    {
                    if (lf < 0)
                        {
                        const int prim = ~lf;
                        if (detail::refine_hit(query, qdata, v, prim, 0)) detail::emit_hit(out, result, prim, k, 0);
                        }
                    else
                        {
                        node = lf;
                        }
                    }
                }
            }
        if constexpr (!detail::relocates<OutputOpT>::value) break;
        else if (!out.relocate(result)) break;
        }
    out.finalize(result);
    }

//! One past the last sorted leaf of a subtree, read off its rope.
/*!
 * A subtree ending at sorted leaf r has as rope the internal node r+1, the leaf
 * N-1+(r+1), or the sentinel when r = N-1 (see rope_after in LBVHBuild.h).
 */
__device__ __forceinline__ unsigned int bucket_end(int rope, unsigned int n_internal)
    {
    if (rope == LBVHSentinel) return n_internal + 1u;
    const unsigned int v = static_cast<unsigned int>(rope);
    return (v < n_internal) ? v : v - n_internal;
    }

//! Bucket rope records for the wave walk: float4(lo, bits(a)), float4(hi, bits(rope)).
/*!
 * a >= 0: internal node, descend to left child a.  a < 0: the node's subtree holds at
 * most `bucket` leaves and is handled as one bucket of the consecutive sorted leaves
 * [~a, bucket_end(rope)).  Nodes below a bucket are never reached (a bucket's rope
 * skips its subtree).  DECODED selects the decoded quantized boxes instead of the
 * exact ones.  TOP_ONLY (walks that start at the root only): the records of nodes below
 * a bucket are not written.
 */
template<bool DECODED, bool TOP_ONLY = false>
__global__ void __launch_bounds__(1024) lbvh_bucket_records(float4* __restrict__ out,
                                                            const LBVHCompressedData ctree,
                                                            const ConstLBVHData tree,
                                                            const uint32_t n_internal,
                                                            const uint32_t n_nodes,
                                                            const uint32_t bucket)
    {
    const uint32_t idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= n_nodes) return;
    int first, count;
    if (idx < n_internal)
        {
        const int j = tree.range_end[idx];
        first = min(static_cast<int>(idx), j);
        count = abs(j - static_cast<int>(idx)) + 1;
        }
    else
        {
        first = static_cast<int>(idx - n_internal);
        count = 1;
        }
    if constexpr (TOP_ONLY)
        {
        const int p = tree.parent[idx];
        if (p != LBVHSentinel && abs(tree.range_end[p] - p) + 1 <= static_cast<int>(bucket)) return;   // below a bucket
        }
    const int a = (count <= static_cast<int>(bucket)) ? ~first : tree.left[idx];
    BoundingBox b;
    if (DECODED)
        {
        const int4 r = ctree.data[idx];
        b = detail::decode_box(static_cast<uint32_t>(r.x), static_cast<uint32_t>(r.y), tree.lo[tree.root], tree.hi[tree.root], *ctree.bins);
        }
    else
        {
        b = BoundingBox(tree.lo[idx], tree.hi[idx]);
        }
    out[2 * idx] = make_float4(b.lo.x, b.lo.y, b.lo.z, __int_as_float(a));
    out[2 * idx + 1] = make_float4(b.hi.x, b.hi.y, b.hi.z, __int_as_float(tree.rope[idx]));
    if (!DECODED && idx == 0 && ctree.lo && ctree.hi)
        {
        // the exact root box (the quantized compression, which otherwise writes it, is skipped)
        *ctree.lo = tree.lo[tree.root];
        *ctree.hi = tree.hi[tree.root];
        }
    }

//! Read-only data addressed through the constant address space: a wave-uniform
//! index then compiles to scalar loads (SMEM) instead of 64 vector lanes.
typedef float native_float4 __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(4))) native_float4 uniform_native_float4;

__device__ __forceinline__ float4 uniform_load(const float4* base, unsigned int i)
    {
    const native_float4 v = ((uniform_native_float4*)(base))[i];
    return make_float4(v.x, v.y, v.z, v.w);
    }

namespace wave
{
//! Lanes of the wave (64 bits) whose predicate holds: the compare mask itself, with no
//! detour through a VGPR.
__device__ __forceinline__ unsigned long long vote(bool p)
    {
    return __builtin_amdgcn_ballot_w64(p);
    }

//! Number of XCDs (accelerator complex dies, each with its own L2) on gfx950.
constexpr unsigned int kXcds = 8;

//! Logical block index under the round-robin dispatch of workgroups over the XCDs.
/*!
 * Workgroup b runs on XCD b % 8.  Renumbering so that XCD x owns the contiguous
 * logical range [x*q + min(x, r), ...) (q = G/8, r = G%8) gives each XCD's L2 one
 * contiguous stretch of the (Morton-ordered) queries instead of every 8th block.
 */
__device__ __forceinline__ unsigned int xcd_block(unsigned int b, unsigned int G)
    {
    const unsigned int x = b % kXcds;
    const unsigned int j = b / kXcds;
    const unsigned int q = G / kXcds;
    const unsigned int r = G % kXcds;
    return x * q + (x < r ? x : r) + j;
    }

//! Queries of one 256-thread block (tail-split launch map).
struct BlockSpan
    {
    unsigned int first;      //!< first query position of the block
    unsigned int lead;       //!< positions of the block's group of 256 before `first`
    unsigned int per_wave;   //!< queries per wave (lanes below it serve one each)
    bool live;               //!< false: a block past its XCD's share (exits at once)
    };

//! Map of workgroup b of a tail-split launch over G groups of 256 query positions.
/*!
 * XCD x owns the contiguous groups [x*q + min(x, r), ...) as in xcd_block.  Its first groups
 * run as one block each (64 queries per wave); its last T groups are each split into S
 * blocks of 256/S positions (64/S queries per wave, the other lanes idle).  A launch of
 * about two waves per wave slot ends with waves that started late and run with few others
 * beside them, at the latency of their own dependent loads: split, those last waves are
 * shorter.  The grid is 8 * (blocks of XCD 0); blocks past an XCD's own count are not live.
 * T = 0 is the plain map of xcd_block (grid G, every block live).
 */
__host__ __device__ __forceinline__ BlockSpan tail_block(const unsigned int b, const unsigned int G,
                                                         const unsigned int T, const unsigned int S)
    {
    const unsigned int x = b % kXcds;
    const unsigned int j = b / kXcds;
    const unsigned int q = G / kXcds;
    const unsigned int r = G % kXcds;
    const unsigned int gx = q + (x < r ? 1u : 0u);
    const unsigned int g0 = x * q + (x < r ? x : r);
    const unsigned int tb = gx < T ? gx : T;
    const unsigned int head = gx - tb;
    if (j < head) return BlockSpan{256u * (g0 + j), 0u, 64u, true};
    const unsigned int k = j - head;
    if (k >= S * tb) return BlockSpan{0u, 0u, 0u, false};
    const unsigned int lead = (k % S) * (256u / S);
    return BlockSpan{256u * (g0 + head + k / S) + lead, lead, 64u / S, true};
    }

//! Node test of the wave walk: float distance from the RN center to the box against a
//! threshold that is never tighter than the query's own test (so no hit is pruned).
__device__ __forceinline__ float box_distance2(const float3& c, const float4& lo, const float4& hi)
    {
    const float dx = fmaxf(fmaxf(lo.x - c.x, c.x - hi.x), 0.0f);
    const float dy = fmaxf(fmaxf(lo.y - c.y, c.y - hi.y), 0.0f);
    const float dz = fmaxf(fmaxf(lo.z - c.z, c.z - hi.z), 0.0f);
    return fmaf(dx, dx, fmaf(dy, dy, dz * dz));
    }

//! Exact query: ExactSphere's own box test is already this padded float test.
__device__ __forceinline__ float3 center(const ExactSphere& v) { return v.c; }
__device__ __forceinline__ float threshold(const ExactSphere& v) { return v.T; }

//! Reference query: the directed-rounding test satisfies dr2 >= d2 (1 - 15u) (u = 2^-24)
//! for the exact distance d2 from the float origin, and the RN float distance is at most
//! d2 (1 + 5u); Rsq (1 + 2^-18) therefore admits every box the reference test admits.
__device__ __forceinline__ float3 center(const BoundingSphere& v) { return v.origin; }
__device__ __forceinline__ float threshold(const BoundingSphere& v) { return approx::fmul_ru(v.Rsq, 1.0f + 0x1p-18f); }

//! Output ops whose rows the wave kernels place before the walk (kPlacedRows: PlacedRowPairOp;
//! every thread of the 256-thread block takes part).
template<class O, class = void>
struct places_rows : std::false_type {};
template<class O>
struct places_rows<O, typename std::enable_if<O::kPlacedRows>::type> : std::true_type {};

template<class OutputOpT>
__device__ __forceinline__ void place_rows(const OutputOpT& out, const unsigned int t, const unsigned int idx, const bool valid)
    {
    if constexpr (places_rows<OutputOpT>::value) out.place(t, idx, valid);
    }

//! True in the lanes set in the wave-uniform mask m.
__device__ __forceinline__ bool lane_in(unsigned long long m)
    {
    return __builtin_amdgcn_inverse_ballot_w64(m);
    }

//! Image bytes of the run [a, b) of one row: the image of one walk is the same for all of a
//! query's pairs found in it, so the walks write the image array once per image
//! walk and row, as a run (16-byte stores in the aligned middle), not one byte per pair: the
//! bytes of a wave's rows are then written within a short time and leave L2 as whole lines.
__device__ __forceinline__ void image_run(unsigned char* __restrict__ img, unsigned long long a, const unsigned long long b,
                                          const unsigned int k)
    {
    const unsigned char kb = static_cast<unsigned char>(k);
    const unsigned int k4 = (k & 0xffu) * 0x01010101u;
    const uint4 k16 = make_uint4(k4, k4, k4, k4);
    // bytes up to a 4-byte boundary, dwords up to a 16-byte boundary, 16-byte stores, then the tail
    for (; a < b && (reinterpret_cast<uintptr_t>(img + a) & 3u); ++a) img[a] = kb;
    for (; a + 4u <= b && (reinterpret_cast<uintptr_t>(img + a) & 15u); a += 4u) *reinterpret_cast<unsigned int*>(img + a) = k4;
    for (; a + 16u <= b; a += 16u) *reinterpret_cast<uint4*>(img + a) = k16;
    for (; a + 4u <= b; a += 4u) *reinterpret_cast<unsigned int*>(img + a) = k4;
    for (; a < b; ++a) img[a] = kb;
    }

//! Set bits of the wave-uniform mask m in the lanes below this one.
__device__ __forceinline__ unsigned int count_below(unsigned long long m)
    {
    return __builtin_amdgcn_mbcnt_hi(static_cast<unsigned int>(m >> 32),
                                     __builtin_amdgcn_mbcnt_lo(static_cast<unsigned int>(m), 0u));
    }

} // end namespace wave

//! Counts with a log of the walk: one rope path per wave for 64 consecutive queries (thread t
//! serves query order[t]), the least that a walk of single paths over bucket records loads.
/*!
 * Image bits come from each query's own test against the root box; the wave visits the images any
 * lane needs, in ascending order, and descends where any lane's box test passes.  Node indices are
 * wave-uniform: node records are scalar loads.  At a bucket the lanes whose box test passed apply
 * the query's leaf test to each leaf.  Each wave writes its node records loaded, buckets tested
 * and leaves in them to visits[3w .. 3w+2] (w: the launched wave).
 */
template<class QueryOpT, class TranslateOpT>
__global__ void __launch_bounds__(256) lbvh_visit_log(const CountNeighborsOp out,
                                                      const float4* __restrict__ nodes,
                                                      const float4* __restrict__ points,
                                                      const float3* __restrict__ root_lo,
                                                      const float3* __restrict__ root_hi,
                                                      const int root,
                                                      const QueryOpT query,
                                                      const TranslateOpT images,
                                                      const unsigned int* __restrict__ order,
                                                      const unsigned int n_nodes,
                                                      unsigned int* __restrict__ visits)
    {
    const unsigned int t = wave::xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
    const unsigned int n_internal = (n_nodes - 1u) / 2u;
    const bool valid = t < query.size();
    const unsigned int idx = valid ? (order ? order[t] : t) : 0u;
    const BoundingBox root_box(*root_lo, *root_hi);
    const typename QueryOpT::ThreadData q = valid ? query.setup(idx) : typename QueryOpT::ThreadData();
    typename CountNeighborsOp::ThreadData result = out.setup(idx, q);
    unsigned int n_node = 0, n_bucket = 0, n_leaf = 0;     // wave-uniform
    const unsigned int nimg = images.size() < 32u ? images.size() : 32u;
    for (unsigned int k = 0; k < nimg; ++k)
        {
        const typename QueryOpT::Volume v = query.get(q, images.get(k));
        const unsigned long long active = wave::vote(valid && query.overlap(v, root_box));
        if (!active) continue;
        const float3 c = wave::center(v);
        const float T = wave::threshold(v);
        int node = root;
        for (int budget = 2 * static_cast<int>(n_nodes); node != LBVHSentinel && budget > 0; --budget)
            {
            node = __builtin_amdgcn_readfirstlane(node);
            const float4 a = uniform_load(nodes, 2u * node);
            const float4 b = uniform_load(nodes, 2u * node + 1u);
            const unsigned long long hitm = wave::vote(wave::box_distance2(c, a, b) <= T) & active;
            int next = __float_as_int(b.w);
            ++n_node;
            if (hitm)
                {
                const int lf = __float_as_int(a.w);
                if (lf < 0)
                    {
                    const unsigned int first = ~static_cast<unsigned int>(lf), end = bucket_end(next, n_internal);
                    ++n_bucket;
                    n_leaf += end - first;
                    for (unsigned int leaf = first; leaf < end; ++leaf)
                        {
                        if (!wave::lane_in(hitm)) continue;
                        bool in;
                        if constexpr (std::is_same<QueryOpT, ExactSphereQueryOp>::value) in = query.refine_point(v, points[leaf]);
                        else
                            {
                            const float4 lo = nodes[2u * (n_internal + leaf)], hi = nodes[2u * (n_internal + leaf) + 1u];
                            in = query.overlap(v, BoundingBox(make_float3(lo.x, lo.y, lo.z), make_float3(hi.x, hi.y, hi.z)));
                            }
                        if (in) ++result.num_neigh;
                        }
                    }
                else
                    {
                    next = lf;
                    }
                }
            node = next;
            }
        }
    if ((threadIdx.x & 63u) == 0u)
        {
        unsigned int* slot = visits + 3u * (t >> 6);
        slot[0] = n_node;
        slot[1] = n_bucket;
        slot[2] = n_leaf;
        }
    if (valid) out.finalize(result);
    }

} // end namespace kernel
} // end namespace gpu
} // end namespace neighbor

#endif // NEIGHBOR_KERNELS_LBVH_TRAVERSE_H_
