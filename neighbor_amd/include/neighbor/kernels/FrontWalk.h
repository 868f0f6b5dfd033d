// FrontWalk.h -- walk of the tree by node fronts, with matrix leaf tests.
//
// One wave serves up to 64 consecutive queries of the traversal order, with the roles of lanes
// and nodes exchanged against a rope walk:
//  * The walk down the tree tests up to 64 nodes at once, one per lane, against the boxes
//    around the wave's four groups of 16 queries.  All periodic images start together (the
//    front begins with one root entry per image), so the chain of dependent record loads is
//    about the depth of the tree, where a rope walk loads one record after the other (245 of
//    them for a wave of the N = 10^6 uniform workload, and again for every image).
//  * A run of leaves is tested against the queries as a matrix product:
//    |p|^2 - 2 p.q + (|q|^2 - R^2) of 16 leaves x 16 queries is one v_mfma_f32_16x16x4_f32
//    (K = x, y, z, 1), about origins local to the wave.  Its sign decides; values within the
//    error bound of zero are decided by the query's own definition.  For the float sphere query
//    p is the center of the leaf's box and the bound includes the box's half diagonal.
//
// Hits come out image by image, then in Morton order, as in the rope walks.
#ifndef NEIGHBOR_KERNELS_FRONT_WALK_H_
#define NEIGHBOR_KERNELS_FRONT_WALK_H_

#include "WaveWalk.h"

#include <new>
#include <stdint.h>

namespace neighbor
{
namespace gpu
{
namespace kernel
{
namespace front
{
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr unsigned int kStack = 192;        //!< entries of the wave's front
//! Front entries kept free for single-entry steps: the levels below any node (30 code bits and
//! 31 position bits at most) each add one entry there.
constexpr unsigned int kReserve = 64;
constexpr unsigned int kList = 128;         //!< buckets found and not yet tested
//! Hits written at once: the most that leaves four workgroups of lbvh_traverse_front their LDS (exact
//! fill of 10^6 points, 78 neighbors each, 595 us against 610 with 512; of clustered rows 2895 against
//! 2952).  Of lbvh_traverse_team, whose blocks hold the team's words, too, three fit (42 KB each).
constexpr unsigned int kHits = 1024;
constexpr unsigned int kLeafStride = 68;    //!< floats between a batch's component rows (bank spread)
constexpr unsigned int kRun = 32;           //!< leaves from which a node is walked into (sources with kFirst)
//! A group's (quad's) box is taken to be mostly empty, and tested by its quads (queries), when a
//! side is longer than this many radii and this many sides of the tree's mean cell per leaf.
constexpr float kSpreadRadii = 3.0f, kSpreadCells = 6.3f;
//! Eighths of a wave's queries in wide quads above which its queries take one rope path each.
constexpr unsigned int kScattered = 5;
//! Tree nodes up to which fronts of scattered queries are still the shorter walk: measured with
//! queries in random order (count, radius 2.5, density 0.85, 27 images), fronts against rope
//! paths: 8000 points 179 against 1816 us, 16,000 points 221 against 2074, 40,000 points 2323
//! against 2169.
constexpr unsigned int kSmallTree = 60000;
constexpr unsigned int kTeam = 4;           //!< waves of a team (one block)

//! Magnitude up to which coordinates, radii and image vectors take this walk (others, and
//! infinities and NaN, take lane_walk): squares and their sums stay finite in float.
constexpr float kMaxCoordinate = 0x1p46f;
//! Leaves whose squared distance from the wave's origin is not below this are out of every
//! query's reach (at most (sqrt(3) 2 + 1) 2^46 < 10^15 away).
constexpr float kFarLeaf = 1e30f;
constexpr float kNever = 3e38f;             //!< added to a distance: never a hit

//! LDS of one wave.  Pair ops also use the second part.
struct FrontWave
    {
    uint32_t node[kStack];          //!< front, last entry first in the traversal order
    uint32_t first[kStack];         //!< first leaf of the entry's node (sources with kFirst)
    uint8_t img[kStack];            //!< image of each entry
    uint2 list[kList];              //!< first leaf; leaves | image << 8 | groups << 16
    float4 image[32];               //!< image vectors in float
    float4 lo[20];                  //!< lower corner of the box around each group's (16) queries and, from
                                    //!< 4 on, each quad's (4); padded squared radius
    float4 hi[20];                  //!< upper corners
    float4 sphere[64];              //!< query center, padded squared radius (negative: no query)
    float leaf[4 * kLeafStride];    //!< batch leaves about the origin: x, y, z, x^2 + y^2 + z^2
    float4 local[64];               //!< queries: -2 x, -2 y, -2 z about the origin, |q|^2 - R^2
    };
struct FrontPairs
    {
    unsigned long long row[64];     //!< next row position less the query's first hit slot
    uint32_t prim[64];              //!< the batch leaves' values for the output op
    uint16_t hit[kHits];            //!< query << 6 | leaf
    };

//! LDS shared by the waves of a team: each wave's hits per query in a round of batches (two
//! rounds in turn); the rows of queries that overflowed.
struct Team
    {
    uint32_t count[2][kTeam][64];
    unsigned long long pos[64];
    unsigned long long end[64];
    };

// ------------------------------------------------------------------------- tree records
//! A node record: box, left child (inner nodes) or a leaf's or bucket's negative word, rope.
struct Node
    {
    float3 lo, hi;
    int lf;
    int rope;
    };

//! Bucket records (lbvh_bucket_records): a negative word is a bucket's first leaf.
template<class TransformOpT>
struct BucketSource
    {
    static constexpr bool kFirst = false;       //!< nodes' first leaves come from the records
    const float4* __restrict__ nodes;
    const float4* __restrict__ points;          //!< sorted points
    const unsigned int* __restrict__ primitive;
    TransformOpT transform;
    unsigned int n_internal;

    __device__ __forceinline__ Node node(const uint32_t i) const
        {
        const float4 a = nodes[2u * i], b = nodes[2u * i + 1u];
        return Node{make_float3(a.x, a.y, a.z), make_float3(b.x, b.y, b.z), __float_as_int(a.w), __float_as_int(b.w)};
        }
    //! Box test of the reference query: as walked and as defined (decoded boxes are stored).
    __device__ __forceinline__ Node leaf(const unsigned int l) const { return node(n_internal + l); }
    __device__ __forceinline__ BoundingBox box(const uint32_t i) const
        {
        const Node r = node(i);
        return BoundingBox(r.lo, r.hi);
        }
    __device__ __forceinline__ uint32_t value(const unsigned int l, const Node&) const { return transform(primitive[l]); }
    //! Point of a leaf and its value for the output op (exact query).
    __device__ __forceinline__ float4 point(const ExactSphereQueryOp&, const unsigned int l) const { return points[l]; }
    __device__ __forceinline__ float4 point(const ExactSphereQueryOp&, const unsigned int l, const BoundingBox&, bool& inside) const
        {
        inside = true;
        return points[l];
        }
    __device__ __forceinline__ uint32_t point_value(const float4& p) const { return transform(__float_as_uint(p.w)); }
    __device__ __forceinline__ float error() const { return 0.0f; }
    };

//! The point that an exact query holds for a leaf's value (w: the value), and whether it lies in
//! the leaf's box and the root's.
__device__ __forceinline__ float4 value_point(const ExactSphereQueryOp& query, const uint32_t value)
    {
    const float* p = query.points + static_cast<size_t>(query.stride) * value;
    return make_float4(p[0], p[1], p[2], __uint_as_float(value));
    }
__device__ __forceinline__ bool holds(const BoundingBox& b, const float4& p)
    {
    return p.x >= b.lo.x && p.x <= b.hi.x && p.y >= b.lo.y && p.y <= b.hi.y && p.z >= b.lo.z && p.z <= b.hi.z;
    }

//! Float rope records: a negative word is a leaf's value.
struct RopeSource
    {
    static constexpr bool kFirst = true;
    const float4* __restrict__ nodes;
    unsigned int n_internal;

    __device__ __forceinline__ Node node(const uint32_t i) const
        {
        const float4 a = nodes[2u * i], b = nodes[2u * i + 1u];
        return Node{make_float3(a.x, a.y, a.z), make_float3(b.x, b.y, b.z), __float_as_int(a.w), __float_as_int(b.w)};
        }
    __device__ __forceinline__ Node leaf(const unsigned int l) const { return node(n_internal + l); }
    __device__ __forceinline__ BoundingBox box(const uint32_t i) const
        {
        const Node r = node(i);
        return BoundingBox(r.lo, r.hi);
        }
    __device__ __forceinline__ uint32_t value(const unsigned int, const Node& r) const { return ~static_cast<uint32_t>(r.lf); }
    __device__ __forceinline__ float4 point(const ExactSphereQueryOp& query, const unsigned int l) const
        {
        return value_point(query, ~__float_as_uint(nodes[2u * (n_internal + l)].w));
        }
    __device__ __forceinline__ float4 point(const ExactSphereQueryOp& query, const unsigned int l, const BoundingBox& root_box, bool& inside) const
        {
        const float4 p = point(query, l);
        inside = holds(box(n_internal + l), p) && holds(root_box, p);
        return p;
        }
    __device__ __forceinline__ uint32_t point_value(const float4& p) const { return __float_as_uint(p.w); }
    __device__ __forceinline__ float error() const { return 0.0f; }
    };

//! Quantized records (lbvh_compress).  node(): boxes decoded with plain roundings, within
//! error() of the defined ones on each side; box(): as defined.
struct QuantizedSource
    {
    static constexpr bool kFirst = true;
    const int4* __restrict__ data;
    float3 rlo, rhi, bins;
    unsigned int n_internal;

    __device__ __forceinline__ Node node(const uint32_t i) const
        {
        const int4 r = data[i];
        const uint32_t l = static_cast<uint32_t>(r.x), h = static_cast<uint32_t>(r.y);
        return Node{make_float3(fmaf(static_cast<float>((l >> 20) & 0x3ffu), bins.x, rlo.x),
                                fmaf(static_cast<float>((l >> 10) & 0x3ffu), bins.y, rlo.y),
                                fmaf(static_cast<float>(l & 0x3ffu), bins.z, rlo.z)),
                    make_float3(fmaf(-static_cast<float>((h >> 20) & 0x3ffu), bins.x, rhi.x),
                                fmaf(-static_cast<float>((h >> 10) & 0x3ffu), bins.y, rhi.y),
                                fmaf(-static_cast<float>(h & 0x3ffu), bins.z, rhi.z)),
                    r.z, r.w};
        }
    __device__ __forceinline__ Node leaf(const unsigned int l) const { return node(n_internal + l); }
    __device__ __forceinline__ BoundingBox box(const uint32_t i) const
        {
        const int4 r = data[i];
        return detail::decode_box(static_cast<uint32_t>(r.x), static_cast<uint32_t>(r.y), rlo, rhi, bins);
        }
    __device__ __forceinline__ uint32_t value(const unsigned int, const Node& r) const { return ~static_cast<uint32_t>(r.lf); }
    __device__ __forceinline__ float4 point(const ExactSphereQueryOp& query, const unsigned int l) const
        {
        return value_point(query, ~static_cast<uint32_t>(data[n_internal + l].z));
        }
    __device__ __forceinline__ float4 point(const ExactSphereQueryOp& query, const unsigned int l, const BoundingBox& root_box, bool& inside) const
        {
        const float4 p = point(query, l);
        inside = holds(box(n_internal + l), p) && holds(root_box, p);
        return p;
        }
    __device__ __forceinline__ uint32_t point_value(const float4& p) const { return __float_as_uint(p.w); }
    //! The defined decoding rounds the product (at most 1023 bins, within an ulp of the box's
    //! side) and the sum down or up by an ulp each, the plain one the sum to nearest: together
    //! below 4 2^-23 of (largest corner + side).
    __device__ __forceinline__ float error() const
        {
        const float c = fmaxf(fmaxf(fmaxf(fabsf(rlo.x), fabsf(rhi.x)), fmaxf(fabsf(rlo.y), fabsf(rhi.y))), fmaxf(fabsf(rlo.z), fabsf(rhi.z)));
        const float side = fmaxf(fmaxf(rhi.x - rlo.x, rhi.y - rlo.y), rhi.z - rlo.z);
        return 0x1p-21f * (c + side) + 0x1p-120f;
        }
    };

//! Completes a source with the root box and bin sizes kept on the device.
template<class SrcT>
__device__ __forceinline__ void bind(SrcT&, const BoundingBox&, const float3*) {}
__device__ __forceinline__ void bind(QuantizedSource& src, const BoundingBox& root_box, const float3* bins)
    {
    src.rlo = root_box.lo;
    src.rhi = root_box.hi;
    src.bins = *bins;
    }

__device__ __forceinline__ double3 as_double3(const double3& v) { return v; }
__device__ __forceinline__ double3 as_double3(const float3& v) { return make_double3(v.x, v.y, v.z); }

//! The value, computed anew from here on: keeps what depends on it out of the registers held
//! across the walk's loops (hoisted addresses and conversions cost two waves per SIMD).
__device__ __forceinline__ unsigned int anew(unsigned int v)
    {
    asm volatile("" : "+v"(v));
    return v;
    }
__device__ __forceinline__ float4 anew(float4 v)
    {
    asm volatile("" : "+v"(v.x), "+v"(v.y), "+v"(v.z), "+v"(v.w));
    return v;
    }

__device__ __forceinline__ float lane_value(const float v, const unsigned int l)
    {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), static_cast<int>(l)));
    }
__device__ __forceinline__ float uniform(const float v)
    {
    return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
    }

template<int CTRL>
__device__ __forceinline__ float row_move(const float v)
    {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
    }

//! Minimum over each quad of lanes, in all of its lanes; and over a row's quads of such a value.
__device__ __forceinline__ float quad_min(float v)
    {
    v = fminf(v, row_move<0xb1>(v));    // quad_perm:[1,0,3,2]
    return fminf(v, row_move<0x4e>(v)); // quad_perm:[2,3,0,1]
    }
__device__ __forceinline__ float over_quads_min(float v)
    {
    v = fminf(v, row_move<0x128>(v));   // row_ror:8, 4
    return fminf(v, row_move<0x124>(v));
    }
//! Minimum over the four rows of a value that is the same in all lanes of a row (wave-uniform).
__device__ __forceinline__ float over_rows_min(const float v)
    {
    return fminf(fminf(lane_value(v, 0), lane_value(v, 16)), fminf(lane_value(v, 32), lane_value(v, 48)));
    }

//! Inclusive sum over the lanes of the wave.
__device__ __forceinline__ uint32_t wave_sum_inclusive(uint32_t v)
    {
    v += static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x111, 0xf, 0xf, false));   // row_shr:1
    v += static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x112, 0xf, 0xf, false));
    v += static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x114, 0xf, 0xf, false));
    v += static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x118, 0xf, 0xf, false));
    v += static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x142, 0xa, 0xf, false));   // row_bcast:15
    v += static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x143, 0xc, 0xf, false));   // row_bcast:31
    return v;
    }

//! Groups (bits) that may have hits in the box [lo, hi] shifted by an image vector already.
/*!
 * active: groups with queries.  spread: groups (bits 0-3) whose box is mostly empty, tested quad
 * by quad, and quads (bits 4-19) whose box is, tested query by query.
 */
__device__ __forceinline__ unsigned int groups_in_reach(const FrontWave& W, const unsigned int active, const unsigned int spread,
                                                        const float3& lo, const float3& hi)
    {
    const auto reaches = [&](const float4& a, const float4& b) {
        const float dx = fmaxf(fmaxf(lo.x - b.x, a.x - hi.x), 0.0f);
        const float dy = fmaxf(fmaxf(lo.y - b.y, a.y - hi.y), 0.0f);
        const float dz = fmaxf(fmaxf(lo.z - b.z, a.z - hi.z), 0.0f);
        return fmaf(dx, dx, fmaf(dy, dy, dz * dz)) <= a.w;
    };
    unsigned int hit = 0u;
    #pragma unroll
    for (unsigned int g = 0; g < 4; ++g)
        {
        if (!((active >> g) & 1u)) continue;
        bool any = false;
        if (!((spread >> g) & 1u)) any = reaches(W.lo[g], W.hi[g]);
        else
            {
            #pragma unroll 2
            for (unsigned int c = 4u + 4u * g; c < 8u + 4u * g; ++c)
                {
                if (!((spread >> c) & 1u)) any |= reaches(W.lo[c], W.hi[c]);
                else
                    {
                    #pragma unroll 1
                    for (unsigned int j = 4u * c - 16u; j < 4u * c - 12u; ++j) any |= reaches(W.sphere[j], W.sphere[j]);
                    }
                }
            }
        if (any) hit |= 1u << g;
        }
    return hit;
    }

//! Sign bits of one batch of NT tiles of 16 leaves against the groups set in `groups`: bit 4t + v
//! of acc[g] is the sign of the test value of query 16g + j and leaf 4NT kq + 4t + v (lane =
//! 16 kq + j).  Returns the smallest |value| of the lane's tests, or, BAND, sets am's bits where
//! |value| is below band.
/*!
 * Leaves are dealt to the tiles so that the values a lane gets from them are those of 4NT
 * consecutive leaves: row 4r + v of tile t holds leaf 4NT r + 4t + v.  A value costs one
 * instruction for its sign (alignbit shifts it into the mask) and half a one for the minimum.
 */
template<unsigned int NT, bool BAND>
__device__ __forceinline__ float batch_signs(const FrontWave& W, const float B[4], const floatx4 C[4], const unsigned int groups,
                                             const float band, uint32_t acc[4], uint32_t am[4])
    {
    const unsigned int lane = threadIdx.x & 63u;
    const float* a = W.leaf + (lane >> 4) * kLeafStride + ((lane >> 2) & 3u) * (4u * NT) + (lane & 3u);
    float A[NT];
    #pragma unroll
    for (unsigned int t = 0; t < NT; ++t) A[t] = a[4u * t];
    float least = kNever;
    #pragma unroll
    for (unsigned int g = 0; g < 4; ++g)
        {
        acc[g] = 0u;
        if constexpr (BAND) am[g] = 0u;
        if (!((groups >> g) & 1u)) continue;
        floatx4 d[NT];
        #pragma unroll
        for (unsigned int t = 0; t < NT; ++t) d[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(A[t], B[g], C[g], 0, 0, 0);
        #pragma unroll
        for (unsigned int u = 4u * NT; u-- > 0u;)
            {
            const float s = d[u / 4u][u % 4u];
            acc[g] = __builtin_amdgcn_alignbit(acc[g], __float_as_uint(s), 31u);     // acc << 1 | sign
            if constexpr (BAND) am[g] = __builtin_amdgcn_alignbit(am[g], __float_as_uint(fabsf(s) - band), 31u);
            else least = fminf(least, fabsf(s));
            }
        }
    return least;
    }

template<bool BAND>
__device__ __forceinline__ float batch_signs(const FrontWave& W, const float B[4], const floatx4 C[4], const unsigned int nt,
                                             const unsigned int groups, const float band, uint32_t acc[4], uint32_t am[4])
    {
    switch (nt)
        {
        case 1: return batch_signs<1, BAND>(W, B, C, groups, band, acc, am);
        case 2: return batch_signs<2, BAND>(W, B, C, groups, band, acc, am);
        case 3: return batch_signs<3, BAND>(W, B, C, groups, band, acc, am);
        default: return batch_signs<4, BAND>(W, B, C, groups, band, acc, am);
        }
    }

//! The lanes' bits of one batch (nt tiles) by query: bit s of the result is the bit of batch leaf
//! s and of this lane's query (a 4 x 4 transpose of the rows of 16 lanes and the registers).
__device__ __forceinline__ unsigned long long by_query(const uint32_t acc[4], const unsigned int nt)
    {
    typedef unsigned int uint2_t __attribute__((ext_vector_type(2)));
    const uint2_t s02 = __builtin_amdgcn_permlane32_swap(acc[0], acc[2], false, false);
    const uint2_t s13 = __builtin_amdgcn_permlane32_swap(acc[1], acc[3], false, false);
    const uint2_t s01 = __builtin_amdgcn_permlane16_swap(s02[0], s13[0], false, false);
    const uint2_t s23 = __builtin_amdgcn_permlane16_swap(s02[1], s13[1], false, false);
    const unsigned int step = 4u * nt;
    return static_cast<unsigned long long>(s01[0] | (s01[1] << step))
           | (static_cast<unsigned long long>(s23[0] | (s23[1] << step)) << (2u * step));
    }

//! The FP64 definition for the batch's values within `band` of zero: their bits of acc set anew.
//! leaf: the leaf of batch slot `lane`; cd, R2: this lane's query in the batch's image.
template<class SrcT>
__device__ __forceinline__ void batch_decide(const FrontWave& W, const float B[4], const floatx4 C[4], const unsigned int nt,
                                             const unsigned int groups, const float band, const SrcT& src, const ExactSphereQueryOp& query,
                                             const unsigned int leaf, const double3& cd, const double R2, uint32_t acc[4])
    {
    const unsigned int lane = anew(threadIdx.x & 63u);
    const float* a = W.leaf + (lane >> 4) * kLeafStride + ((lane >> 2) & 3u) * (4u * nt) + (lane & 3u);
    #pragma unroll
    for (unsigned int g = 0; g < 4; ++g)
        {
        if (!((groups >> g) & 1u)) continue;
        const int owner = static_cast<int>(16u * g + (lane & 15u));
        for (unsigned int t = 0; t < nt; ++t)
            {
            const floatx4 d = __builtin_amdgcn_mfma_f32_16x16x4f32(a[4u * t], B[g], C[g], 0, 0, 0);
            for (unsigned int v = 0; v < 4; ++v)
                {
                const float s = v == 0u ? d[0] : v == 1u ? d[1] : v == 2u ? d[2] : d[3];
                const bool close = fabsf(s) <= band;
                if (!wave::vote(close)) continue;
                const unsigned int bit = 4u * t + v;
                const unsigned int at = static_cast<unsigned int>(__shfl(static_cast<int>(leaf), static_cast<int>((lane >> 4) * (4u * nt) + bit), 64));
                const double cx = __shfl(cd.x, owner, 64), cy = __shfl(cd.y, owner, 64), cz = __shfl(cd.z, owner, 64);
                const double rr = __shfl(R2, owner, 64);
                if (close)
                    {
                    const float4 p = src.point(query, at);
                    const double dx = cx - static_cast<double>(p.x);
                    const double dy = cy - static_cast<double>(p.y);
                    const double dz = cz - static_cast<double>(p.z);
                    const bool in = (dx * dx + dy * dy) + dz * dz <= rr;
                    acc[g] = in ? acc[g] | (1u << bit) : acc[g] & ~(1u << bit);
                    }
                }
            }
        }
    }

//! Rows that the walk writes itself: the library's pair rows and fixed-stride lists.  Any other op,
//! also one derived from these, gets its hits through process().
template<class OutputOpT>
struct Rows
    {
    static constexpr bool kOn = false;
    };
template<class OutputOpT>
struct PairRows
    {
    static constexpr bool kOn = true;
    typedef typename OutputOpT::ThreadData ThreadData;
    __device__ static __forceinline__ unsigned long long at(const OutputOpT&, const ThreadData& t) { return t.pos; }
    __device__ static __forceinline__ unsigned long long end(const OutputOpT&, const ThreadData& t) { return t.end; }
    __device__ static __forceinline__ void add(ThreadData& t, const uint32_t n)
        {
        t.pos += n;
        t.num_neigh += n;
        }
    __device__ static __forceinline__ unsigned int* neigh(const OutputOpT& o) { return o.neigh; }
    __device__ static __forceinline__ unsigned char* image(const OutputOpT& o) { return o.image; }
    };
template<> struct Rows<PairListOp> : PairRows<PairListOp> {};
template<> struct Rows<RowPairOp> : PairRows<RowPairOp> {};
template<> struct Rows<PlacedRowPairOp> : PairRows<PlacedRowPairOp> {};
template<>
struct Rows<NeighborListOp>
    {
    static constexpr bool kOn = true;
    typedef NeighborListOp::ThreadData ThreadData;
    __device__ static __forceinline__ unsigned long long at(const NeighborListOp& o, const ThreadData& t)
        {
        return static_cast<unsigned long long>(o.max_neigh) * t.idx + t.num_neigh;
        }
    __device__ static __forceinline__ unsigned long long end(const NeighborListOp& o, const ThreadData& t)
        {
        return static_cast<unsigned long long>(o.max_neigh) * t.idx + o.max_neigh;
        }
    __device__ static __forceinline__ void add(ThreadData& t, const uint32_t n) { t.num_neigh += n; }
    __device__ static __forceinline__ unsigned int* neigh(const NeighborListOp& o) { return o.neigh_list; }
    __device__ static __forceinline__ unsigned char* image(const NeighborListOp&) { return nullptr; }
    };

//! Writes the hits (bit s: batch leaf s) of each lane's query at its row position: `at`, before
//! `end`.  Lists the hits in LDS, query by query, so that the stores of the lanes are runs.
__device__ __forceinline__ void write_hits(unsigned int* __restrict__ neigh, unsigned char* __restrict__ image, FrontPairs& P,
                                           unsigned long long hits, unsigned long long at, const unsigned long long end,
                                           const unsigned int k)
    {
    const unsigned int lane = threadIdx.x & 63u;
    uint32_t n = static_cast<uint32_t>(__popcll(hits));
    if (wave::vote(at + n > end))
        {
        // hits past the row's end are counted, not written
        const uint32_t fits = at >= end ? 0u : static_cast<uint32_t>(min(static_cast<unsigned long long>(n), end - at));
        for (; n > fits; --n) hits &= ~(1ull << (63 - __builtin_clzll(hits)));
        }
    uint32_t incl = wave_sum_inclusive(n);
    uint32_t total = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(incl), 63));
    // at most kHits listed at once: all 64 leaves, or 16 leaves at a time
    const unsigned int parts = total <= kHits ? 1u : 4u;
    for (unsigned int part = 0; part < parts; ++part)
        {
        unsigned long long mine = hits;
        if (parts != 1u)
            {
            mine = hits & (0xffffull << (16u * part));
            n = static_cast<uint32_t>(__popcll(mine));
            incl = wave_sum_inclusive(n);
            total = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(incl), 63));
            }
        const uint32_t first = incl - n;
        P.row[lane] = at - first;
        at += n;
        // each lane lists its query's hits, from both ends of each half at once
        uint16_t* low = P.hit + first;
        #pragma unroll
        for (unsigned int half = 0; half < 2; ++half)
            {
            uint32_t m = static_cast<uint32_t>(mine >> (32u * half));
            const uint32_t tag = (lane << 6) | (32u * half);
            uint16_t* const next = low + __popc(m);
            uint16_t* high = next;
            while (m)
                {
                const uint32_t b = 31u - static_cast<uint32_t>(__builtin_clz(m));
                *low++ = static_cast<uint16_t>(tag + static_cast<uint32_t>(__builtin_ctz(m)));
                *--high = static_cast<uint16_t>(tag + b);
                m &= (m - 1u) & ~(1u << b);
                }
            low = next;
            }
        wave::lds_order();
        for (uint32_t s = lane; s < total; s += 64u)
            {
            const unsigned int h = P.hit[s];
            const unsigned long long to_pos = P.row[h >> 6] + s;
            neigh[to_pos] = P.prim[h & 63u];
            if (image) image[to_pos] = static_cast<unsigned char>(k);
            }
        wave::lds_order();
        }
    }

//! The thread data of an output op.  A set-up runs once for each query, in a lane that serves it: an
//! op of a program's own may clear or reserve there what it writes to later.
template<class ThreadDataT>
union Slot
    {
    char none;
    ThreadDataT data;
    __device__ Slot() : none(0) {}
    __device__ ~Slot() {}
    };

//! Boxes around each quad of lanes' queries, and their largest radius (in all of its lanes).
struct Quad
    {
    float3 lo, hi;
    float r;
    };
__device__ __forceinline__ Quad quad_of(const bool act, const float4& q)
    {
    return Quad{make_float3(quad_min(act ? q.x : kNever), quad_min(act ? q.y : kNever), quad_min(act ? q.z : kNever)),
                make_float3(-quad_min(act ? -q.x : kNever), -quad_min(act ? -q.y : kNever), -quad_min(act ? -q.z : kNever)),
                -quad_min(act ? -fabsf(q.w) : 0.0f)};
    }
__device__ __forceinline__ float volume(const BoundingBox& b)
    {
    return fmaxf(b.hi.x - b.lo.x, 0.0f) * fmaxf(b.hi.y - b.lo.y, 0.0f) * fmaxf(b.hi.z - b.lo.z, 0.0f);
    }
//! Side of the cube that holds one of the tree's leaves on average.
__device__ __forceinline__ float mean_cell(const BoundingBox& root_box, const unsigned int n_nodes)
    {
    const float leaves = 0.5f * static_cast<float>(n_nodes + 1u);
    return exp2f(log2f(volume(root_box) / leaves) * (1.0f / 3.0f));
    }
//! Lanes of the groups or quads whose box is mostly empty.
__device__ __forceinline__ unsigned long long mostly_empty(const float3& lo, const float3& hi, const float radius, const float cell)
    {
    return wave::vote(fmaxf(fmaxf(hi.x - lo.x, hi.y - lo.y), hi.z - lo.z) > fmaxf(kSpreadRadii * radius, kSpreadCells * cell));
    }
//! Queries all over the tree (qwide: mostly_empty of the quads): a front, or one path for the wave,
//! would walk the union of their paths.
__device__ __forceinline__ bool scattered(const unsigned long long act, const unsigned long long qwide, const unsigned int n_nodes)
    {
    return n_nodes > kSmallTree && 8u * static_cast<unsigned int>(__popcll(qwide)) > kScattered * static_cast<unsigned int>(__popcll(act));
    }

//! True when few leaves are expected within the radius of the launch's first query (fewer than limit).
template<class QueryOpT>
__device__ __forceinline__ bool sparse(const QueryOpT& query, const unsigned int* __restrict__ order, const BoundingBox& root_box,
                                       const unsigned int n_nodes, const float limit)
    {
    const float R = fabsf(query.spheres[order ? order[0] : 0u].w);
    return 4.18879f * R * R * R * (0.5f * static_cast<float>(n_nodes + 1u)) < limit * volume(root_box);
    }

//! The walk over the subtree of `root` (n_nodes nodes) for one query per lane, by one wave or, TEAM,
//! by the four waves of a block for the same queries; false: not walked (queries too scattered).
/*!
 * Front: a stack of (node, image) entries, the first of the traversal order on top.  A step
 * takes up to 64 entries off the top, tests them, and puts the children of the inner nodes
 * that any group reaches and the reached buckets (runs of at most kRun leaves, where the source
 * has no buckets) back in their places; the buckets before the first inner node go to the list
 * instead, which therefore grows in traversal order.  The right child of an inner node follows
 * from its record alone: Karras's split gamma names the left child (node gamma or leaf gamma),
 * and the right one is leaf gamma + 1 when the node's range, which the rope ends, ends there,
 * else node gamma + 1.  A left child starts where its parent does, a right child at gamma + 1.
 *
 * Box tests: a group's box (or a query's center) and the node box, moved by the image vector
 * in float, against the radius padded by R 2^-20 + 2^-20 (largest coordinate + largest image
 * component) + twice the boxes' own error: each of the three roundings per axis errs by at most
 * 2^-24 of a magnitude below that sum (and the reference query's directed roundings admit at
 * most 15 2^-24 more of R^2; 2^-120 covers squares below the range of float), so a box with a
 * hit always passes.
 *
 * Leaf tests, exact query: with o the wave's origin of the image (float), q' = fl((q + t) - o)
 * and p' = fl(p - o), the value s = |p'|^2 - 2 p'.q' + (|q'|^2 - R^2) computed in float differs
 * from d^2 - R^2 by at most 50 2^-24 B^2 for leaves with |p'| <= B = max |q'| + max R (three
 * roundings of |p'|^2, five sums of terms that stay below 4 B^2, taken as truncated, and the
 * roundings of p' and q' times 2 R); farther leaves have s > 0 by more than their own error.
 * |s| > band = 2^-18 B^2 is therefore decided by the sign; the others by the FP64 definition.
 *
 * Rope and quantized records hold a leaf's value only, and the exact query its own point of it.
 * A point in the leaf's box and the root's is decided as above (its boxes' conservative tests
 * pass where the point is a hit); any other point by the query's box and point tests, which
 * admit boxes up to R 2^-20 + 2^-21 (largest coordinate) and roundings farther than R: such
 * walks pad by 2^-18 in place of 2^-20.
 *
 * Reference query: p is the center of the leaf's box, h a bound of the batch's half diagonals.
 * The box is a hit if the center is (distance <= R) and a miss if the center is farther than
 * R + h; s is taken about the middle of these two, R^2 + R h + h^2 / 2, and values within
 * R h + h^2 / 2 + band of zero (band = 2^-17 B^2: the errors above, and the directed roundings'
 * share of R^2) are decided by the query's own test against the leaf's box.
 *
 * TEAM: every wave walks the front (the same for all), wave w tests the batches w, w + 4, ...
 * Counts are added up at the end; for rows the waves exchange their hits per query after each
 * round of four batches, which places every wave's hits in the rows.
 */
template<bool TEAM, class SrcT, class OutputOpT, class QueryOpT, class TranslateOpT>
__device__ __forceinline__ bool walk(const OutputOpT& out, const SrcT& src, const int root, const BoundingBox& root_box,
                                     const QueryOpT& query, const TranslateOpT& images, const bool valid, const unsigned int idx,
                                     const float4& q, const unsigned int n_nodes, FrontWave& W, FrontPairs& P, Team* team)
    {
    constexpr bool kExact = std::is_same<QueryOpT, ExactSphereQueryOp>::value;
    constexpr bool kCount = std::is_same<OutputOpT, CountNeighborsOp>::value;
    constexpr bool kRows = Rows<OutputOpT>::kOn;
    constexpr bool kChecked = kExact && SrcT::kFirst;   // points come from the query: any may lie outside of its leaf's box
    constexpr float kPad = kChecked ? 0x1p-18f : 0x1p-20f;
    static_assert(!TEAM || kCount || kRows, "teams count or write rows");
    const unsigned int lane = threadIdx.x & 63u;
    const unsigned int member = TEAM ? static_cast<unsigned int>(__builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6))) : 0u;
    const unsigned int n_internal = src.n_internal;
    const unsigned int nimg = images.size() < 32u ? images.size() : 32u;
    Slot<typename OutputOpT::ThreadData> slot;
    typename OutputOpT::ThreadData& result = slot.data;
    // counts and rows only read in their set-ups: all lanes, before the loops (spills otherwise)
    if constexpr (kCount || kRows) new (&slot.data) typename OutputOpT::ThreadData(out.setup(idx, q));
    const float r = fabsf(q.w);

    // image vectors in float and their largest component
    float tmax = 0.0f;
    if (lane < nimg)
        {
        const double3 t = as_double3(images.get(lane));
        W.image[lane] = make_float4(static_cast<float>(t.x), static_cast<float>(t.y), static_cast<float>(t.z), 0.0f);
        tmax = static_cast<float>(fmax(fmax(fabs(t.x), fabs(t.y)), fabs(t.z)));
        }
    tmax = -over_rows_min(over_quads_min(quad_min(-tmax)));

    bool act = valid;
    for (int pass = 0; pass < 2; ++pass)
        {
        // ------------------------------------------------ groups
        const unsigned long long actm = wave::vote(act);
        unsigned int active = 0u, spread = 0u;
        float band;                             // error bound of the leaf tests
        float rmax;
        float3 center;                          // of the wave's queries: its origin before the image vector
        {
        const Quad quad = quad_of(act, q);
        const float3 qlo = quad.lo, qhi = quad.hi;
        const float qrr = quad.r;
        const float3 glo = make_float3(over_quads_min(qlo.x), over_quads_min(qlo.y), over_quads_min(qlo.z));
        const float3 ghi = make_float3(-over_quads_min(-qhi.x), -over_quads_min(-qhi.y), -over_quads_min(-qhi.z));
        const float grr = -over_quads_min(-qrr);
        const float3 ulo = make_float3(over_rows_min(glo.x), over_rows_min(glo.y), over_rows_min(glo.z));
        const float3 uhi = make_float3(-over_rows_min(-ghi.x), -over_rows_min(-ghi.y), -over_rows_min(-ghi.z));
        const float cmax = fmaxf(fmaxf(fmaxf(fabsf(ulo.x), fabsf(uhi.x)), fmaxf(fabsf(ulo.y), fabsf(uhi.y))),
                                 fmaxf(fabsf(ulo.z), fabsf(uhi.z)));
        const float pad = kPad * (cmax + tmax) + 2.0f * src.error();
        const auto padded = [&](const float radius) {
            const float R = radius * (1.0f + kPad) + pad;
            return R * R * (1.0f + 0x1p-19f) + 0x1p-120f;
        };
        W.sphere[lane] = make_float4(q.x, q.y, q.z, act ? padded(r) : -1.0f);
        if ((lane & 3u) == 0u)
            {
            W.lo[4u + (lane >> 2)] = make_float4(qlo.x, qlo.y, qlo.z, padded(qrr));
            W.hi[4u + (lane >> 2)] = make_float4(qhi.x, qhi.y, qhi.z, 0.0f);
            }
        if ((lane & 15u) == 0u)
            {
            W.lo[lane >> 4] = make_float4(glo.x, glo.y, glo.z, padded(grr));
            W.hi[lane >> 4] = make_float4(ghi.x, ghi.y, ghi.z, 0.0f);
            }
        const float cell = mean_cell(root_box, n_nodes);
        const unsigned long long wide = mostly_empty(glo, ghi, grr, cell), qwide = mostly_empty(qlo, qhi, qrr, cell);
        #pragma unroll
        for (unsigned int g = 0; g < 4; ++g)
            {
            if ((actm >> (16u * g)) & 0xffffull) active |= 1u << g;
            if ((wide >> (16u * g)) & 1ull) spread |= 1u << g;
            }
        // the few queries of a team are walked faster by its four waves than one per lane also where
        // they are scattered: 4000 spheres of radius 5.9 in a tree of 396,000 points, 16 per team, 123
        // us against 185
        if (pass == 0 && (!TEAM || __popcll(actm) > 16) && scattered(actm, qwide, n_nodes)) return false;
        if constexpr (!kCount && !kRows)
            if (pass == 0 && valid) new (&slot.data) typename OutputOpT::ThreadData(out.setup(idx, q));
        if (spread && qwide)
            {
            #pragma unroll
            for (unsigned int c = 0; c < 16; ++c)
                if ((qwide >> (4u * c)) & 1ull) spread |= 1u << (4u + c);
            }
        const float hx = 0.5f * (uhi.x - ulo.x), hy = 0.5f * (uhi.y - ulo.y), hz = 0.5f * (uhi.z - ulo.z);
        rmax = uniform(-over_rows_min(-grr));
        const float reach = (sqrtf(hx * hx + hy * hy + hz * hz) + rmax) * (1.0f + 0x1p-10f) + pad;
        band = uniform((kExact ? 0x1p-18f : 0x1p-17f) * reach * reach + 0x1p-110f);
        center = make_float3(uniform(0.5f * (ulo.x + uhi.x)), uniform(0.5f * (ulo.y + uhi.y)), uniform(0.5f * (ulo.z + uhi.z)));
        }

        // ------------------------------------------------ walk
        unsigned int sp = nimg, ln = 0u;        // front entries, listed buckets
        if (lane < nimg)
            {
            W.node[nimg - 1u - lane] = static_cast<uint32_t>(root);
            W.img[nimg - 1u - lane] = static_cast<uint8_t>(lane);
            if constexpr (SrcT::kFirst) W.first[nimg - 1u - lane] = 0u;
            }
        wave::lds_order();
        unsigned int cur = ~0u;                 // image of the open batch operands
        float half = 0.0f;                      // their bound of the leaf boxes' half diagonals
        float3 o = make_float3(0.0f, 0.0f, 0.0f);
        uint32_t cnt[4] = {0u, 0u, 0u, 0u};
        uint32_t odd_hits = 0u;                 // kChecked, counts: hits outside of their leaves' boxes
        unsigned long long run0 = 0ull;
        unsigned int round = 0u;
        // each step settles at least its first entry, and every image visits a node at most once
        unsigned long long budget = static_cast<unsigned long long>(n_nodes) * nimg;
        while (sp | ln)
            {
            if (sp && ln <= kList - 64u)
                {
                // ---- one step of the front
                if (budget-- == 0ull) return true;  // never for a tree's own records
                const unsigned int room = sp + kReserve < kStack ? kStack - kReserve - sp : 1u;
                const unsigned int m = min(min(sp, 64u), room);
                const bool have = lane < m;
                const unsigned int at = have ? sp - 1u - lane : 0u;
                const uint32_t node = have ? W.node[at] : static_cast<uint32_t>(root);
                const unsigned int k = have ? W.img[at] : 0u;
                const Node rec = src.node(node);
                const float4 t = W.image[k];
                const unsigned int g = groups_in_reach(W, active, spread, make_float3(rec.lo.x - t.x, rec.lo.y - t.y, rec.lo.z - t.z),
                                                       make_float3(rec.hi.x - t.x, rec.hi.y - t.y, rec.hi.z - t.z));
                const bool reached = have && g != 0u;
                const unsigned int end = bucket_end(rec.rope, n_internal);                // one past the node's last leaf
                unsigned int first;
                bool inner;
                if constexpr (SrcT::kFirst)
                    {
                    first = W.first[at];
                    inner = end - first > kRun;
                    }
                else
                    {
                    first = ~static_cast<unsigned int>(rec.lf);
                    inner = rec.lf >= 0;
                    }
                const unsigned long long bm = wave::vote(reached && !inner);
                const unsigned long long im = wave::vote(reached && inner);
                const unsigned long long lead = bm & (im ? (im & -im) - 1ull : ~0ull);    // buckets before the first inner node
                const unsigned long long later = bm & ~lead;
                wave::lds_order();
                if (wave::lane_in(lead))
                    W.list[ln + wave::count_below(lead)] = make_uint2(first, (end - first) | (k << 8) | (g << 16));
                ln += static_cast<unsigned int>(__popcll(lead));
                const unsigned int put = 2u * wave::count_below(im) + wave::count_below(later);
                sp = sp - m + 2u * static_cast<unsigned int>(__popcll(im)) + static_cast<unsigned int>(__popcll(later));
                if (sp > kStack) return true;   // never for a tree's own records
                const unsigned int to = sp - 1u - put;
                if (wave::lane_in(im))
                    {
                    const unsigned int left = static_cast<unsigned int>(rec.lf);
                    const unsigned int split = left < n_internal ? left : left - n_internal;
                    W.node[to] = left;
                    W.node[to - 1u] = split + 1u + (end == split + 2u ? n_internal : 0u);
                    W.img[to] = static_cast<uint8_t>(k);
                    W.img[to - 1u] = static_cast<uint8_t>(k);
                    if constexpr (SrcT::kFirst)
                        {
                        W.first[to] = first;
                        W.first[to - 1u] = split + 1u;
                        }
                    }
                else if (wave::lane_in(later))
                    {
                    W.node[to] = node;
                    W.img[to] = static_cast<uint8_t>(k);
                    if constexpr (SrcT::kFirst) W.first[to] = first;
                    }
                wave::lds_order();
                continue;
                }

            // ---- the listed buckets, in batches of up to 64 leaves of one image
            const uint2 l0 = W.list[lane], l1 = W.list[64u + lane];
            unsigned int e = 0u, off = 0u;      // next entry, leaves of it already taken
            const auto entry = [&](const unsigned int i) {
                const int l = static_cast<int>(i & 63u);
                return i < 64u ? make_uint2(__builtin_amdgcn_readlane(l0.x, l), __builtin_amdgcn_readlane(l0.y, l))
                               : make_uint2(__builtin_amdgcn_readlane(l1.x, l), __builtin_amdgcn_readlane(l1.y, l));
            };
            // the next batch: its image, leaves (slot `lane` holds `leaf`) and groups; fill 0: none left
            unsigned int bk = 0u, bfill = 0u, bgroups = 0u, bleaf = 0u;
            const auto take_batch = [&]() {
                bfill = 0u;
                bgroups = 0u;
                if (e == ln) return;
                uint2 en = entry(e);
                bk = (en.y >> 8) & 31u;
                for (;;)
                    {
                    const unsigned int n = en.y & 0xffu;
                    const unsigned int take = min(n - off, 64u - bfill);
                    if (lane >= bfill) bleaf = en.x + off + (lane - bfill);
                    bgroups |= en.y >> 16;
                    bfill += take;
                    off += take;
                    if (off == n)
                        {
                        off = 0u;
                        if (++e == ln) break;
                        en = entry(e);
                        if (((en.y >> 8) & 31u) != bk) break;
                        }
                    if (bfill == 64u) break;
                    }
            };
            // operands of the open image (again after a part of the walk)
            float B[4];
            floatx4 C[4];
            const auto operands = [&]() {
                const float* loc = reinterpret_cast<const float*>(W.local);
                #pragma unroll
                for (unsigned int g = 0; g < 4; ++g)
                    {
                    const unsigned int base = 4u * (16u * g + (lane & 15u));
                    const float b = loc[base + (lane >> 4)];
                    const float c = loc[base + 3u];
                    C[g] = floatx4{c, c, c, c};
                    B[g] = lane < 48u ? b : 1.0f;
                    }
            };
            // image k's queries about its origin, and |q'|^2 less the middle of the decision's bounds
            const auto open = [&](const unsigned int k) {
                const float4 qq = anew(q);
                const double3 t = as_double3(images.get(k));
                o = make_float3(uniform(static_cast<float>(center.x + t.x)), uniform(static_cast<float>(center.y + t.y)),
                                uniform(static_cast<float>(center.z + t.z)));
                double cx, cy, cz;
                bool takes_part = act;
                if constexpr (kExact)
                    {
                    cx = static_cast<double>(qq.x) + t.x;
                    cy = static_cast<double>(qq.y) + t.y;
                    cz = static_cast<double>(qq.z) + t.z;
                    }
                else
                    {
                    const BoundingSphere v = query.get(qq, images.get(k));
                    takes_part = act && query.overlap(v, root_box);     // the reference's image test
                    cx = v.origin.x;
                    cy = v.origin.y;
                    cz = v.origin.z;
                    }
                const float x = static_cast<float>(cx - o.x), y = static_cast<float>(cy - o.y), z = static_cast<float>(cz - o.z);
                const double q2 = (static_cast<double>(x) * x + static_cast<double>(y) * y) + static_cast<double>(z) * z;
                const double R = fabs(static_cast<double>(qq.w));
                const double mid = kExact ? R * R : R * R + (R + 0.5 * half) * half;
                wave::lds_order();
                W.local[lane] = takes_part ? make_float4(-2.0f * x, -2.0f * y, -2.0f * z, static_cast<float>(q2 - mid))
                                           : make_float4(0.0f, 0.0f, 0.0f, kNever);
                wave::lds_order();
                operands();
            };
            operands();
            for (;;)
                {
                bool some = false;
                if constexpr (!TEAM)
                    {
                    take_batch();
                    some = bfill != 0u;
                    }
                else
                    {
                    // of the next four batches, the member's
                    unsigned int ok = 0u, ofill = 0u, ogroups = 0u, oleaf = 0u;
                    for (unsigned int w = 0; w < kTeam; ++w)
                        {
                        take_batch();
                        some = some || bfill != 0u;
                        if (w == member)
                            {
                            ok = bk;
                            ofill = bfill;
                            ogroups = bgroups;
                            oleaf = bleaf;
                            }
                        }
                    bk = ok;
                    bfill = ofill;
                    bgroups = ogroups;
                    bleaf = oleaf;
                    }
                if (!some) break;
                const unsigned int k = bk, fill = bfill, groups = bgroups, leaf = bleaf;
                unsigned long long hits = 0ull;
                if (fill)
                    {
                    const bool has = lane < fill;
                    const unsigned int nt = (fill + 15u) / 16u;
                    // the batch's leaves: points, or box centers with a bound of the half diagonals
                    float px = 0.0f, py = 0.0f, pz = 0.0f;
                    uint32_t value = 0u;
                    float reach2 = 0.0f;
                    bool inside = true;
                    if (has)
                        {
                        if constexpr (kExact)
                            {
                            const float4 p = src.point(query, leaf, root_box, inside);
                            px = p.x;
                            py = p.y;
                            pz = p.z;
                            if constexpr (!kCount) value = src.point_value(p);
                            }
                        else
                            {
                            const Node b = src.leaf(leaf);
                            px = 0.5f * (b.lo.x + b.hi.x);
                            py = 0.5f * (b.lo.y + b.hi.y);
                            pz = 0.5f * (b.lo.z + b.hi.z);
                            const float ex = fmaxf(b.hi.x - px, px - b.lo.x), ey = fmaxf(b.hi.y - py, py - b.lo.y),
                                        ez = fmaxf(b.hi.z - pz, pz - b.lo.z);
                            reach2 = fmaf(ex, ex, fmaf(ey, ey, ez * ez));
                            if constexpr (!kCount) value = src.value(leaf, b);
                            }
                        }
                    if constexpr (!kExact)
                        {
                        const float h = sqrtf(-over_rows_min(over_quads_min(quad_min(-reach2)))) * (1.0f + 0x1p-20f) + 2.0f * src.error();
                        if (h > half)
                            {
                            half = uniform(1.25f * h);      // a little more: boxes of about one size open an image once
                            if (cur != ~0u && k == cur) open(k);
                            }
                        }
                    if (k != cur)
                        {
                        if constexpr (kRows && !TEAM)
                            {
                            if (cur != ~0u && Rows<OutputOpT>::image(out))
                                {
                                const unsigned long long at = Rows<OutputOpT>::at(out, result), end = Rows<OutputOpT>::end(out, result);
                                wave::image_run(Rows<OutputOpT>::image(out), run0, at < end ? at : end, cur);
                                }
                            run0 = Rows<OutputOpT>::at(out, result);
                            }
                        cur = k;
                        open(k);
                        }
                    float x = px - o.x, y = py - o.y, z = pz - o.z;
                    float w = fmaf(z, z, fmaf(y, y, x * x));
                    if (!has || !inside || !(w < kFarLeaf))
                        {
                        x = y = z = 0.0f;
                        w = kNever;
                        }
                    W.leaf[lane] = x;
                    W.leaf[kLeafStride + lane] = y;
                    W.leaf[2u * kLeafStride + lane] = z;
                    W.leaf[3u * kLeafStride + lane] = w;
                    if constexpr (!kCount) P.prim[lane] = value;
                    wave::lds_order();
                    uint32_t acc[4];
                    if constexpr (kExact)
                        {
                        const float least = batch_signs<false>(W, B, C, nt, groups, band, acc, acc);
                        if (wave::vote(least <= band))
                            {
                            const float4 qq = anew(q);
                            const double3 t = as_double3(images.get(k));
                            batch_decide(W, B, C, nt, groups, band, src, query, leaf,
                                         make_double3(static_cast<double>(qq.x) + t.x, static_cast<double>(qq.y) + t.y,
                                                      static_cast<double>(qq.z) + t.z),
                                         static_cast<double>(qq.w) * static_cast<double>(qq.w), acc);
                            }
                        if constexpr (!kCount) hits = by_query(acc, nt);
                        else
                            {
                            #pragma unroll
                            for (unsigned int g = 0; g < 4; ++g) cnt[g] += static_cast<uint32_t>(__popc(acc[g]));
                            }
                        if constexpr (kChecked)
                            {
                            // the others by the query's own tests
                            for (unsigned long long odd = wave::vote(has && !inside); odd; odd &= odd - 1ull)
                                {
                                const unsigned int b = static_cast<unsigned int>(__builtin_ctzll(odd));
                                const unsigned int l = static_cast<unsigned int>(__builtin_amdgcn_readlane(static_cast<int>(leaf), static_cast<int>(b)));
                                const ExactSphere v = query.get(anew(q), images.get(k));
                                const bool in = act && query.overlap(v, root_box) && query.overlap(v, src.box(n_internal + l))
                                                && ExactSphereQueryOp::refine_point(v, src.point(query, l));
                                if constexpr (kCount) odd_hits += in ? 1u : 0u;
                                else hits |= in ? 1ull << b : 0ull;
                                }
                            }
                        }
                    else
                        {
                        uint32_t am[4];
                        batch_signs<true>(W, B, C, nt, groups, (rmax + 0.5f * half) * half * (1.0f + 0x1p-18f) + band, acc, am);
                        hits = by_query(acc, nt);
                        unsigned long long open_hits = by_query(am, nt);
                        hits &= ~open_hits;
                        if (wave::vote(open_hits != 0ull))
                            {
                            const float4 qq = anew(q);
                            const BoundingSphere v = query.get(qq, images.get(k));
                            const float eb = src.error();
                            const float slack = 4.0f * eb * (fabsf(qq.w) + 2.0f * eb);
                            const bool tiny = !(v.Rsq > 0x1p-90f);      // below the reach of the relative bounds
                            const float r_lo = tiny ? -1.0f : v.Rsq * (1.0f - 0x1p-19f) - slack;
                            const float r_hi = tiny ? kNever : v.Rsq * (1.0f + 0x1p-19f) + slack;
                            while (wave::vote(open_hits != 0ull))
                                {
                                const bool one = open_hits != 0ull;
                                const unsigned int b = one ? static_cast<unsigned int>(__builtin_ctzll(open_hits)) : 0u;
                                const uint32_t l = static_cast<uint32_t>(__shfl(static_cast<int>(leaf), static_cast<int>(b), 64));
                                if (one)
                                    {
                                    const Node bx = src.leaf(l);
                                    const float d2 = wave::box_distance2(v.origin, make_float4(bx.lo.x, bx.lo.y, bx.lo.z, 0.0f),
                                                                         make_float4(bx.hi.x, bx.hi.y, bx.hi.z, 0.0f));
                                    bool in = d2 <= r_lo;
                                    if (!in && d2 <= r_hi) in = query.overlap(v, src.box(n_internal + l));
                                    if (in) hits |= 1ull << b;
                                    open_hits &= open_hits - 1ull;
                                    }
                                }
                            }
                        if constexpr (kCount) cnt[0] += static_cast<uint32_t>(__popcll(hits));
                        }
                    }
                if constexpr (kRows)
                    {
                    const uint32_t n = static_cast<uint32_t>(__popcll(hits));
                    if constexpr (!TEAM)
                        {
                        write_hits(Rows<OutputOpT>::neigh(out), nullptr, P, hits, Rows<OutputOpT>::at(out, result),
                                   Rows<OutputOpT>::end(out, result), k);
                        Rows<OutputOpT>::add(result, n);
                        }
                    else
                        {
                        // the members' hits in turn: this wave's follow those of the members before it
                        uint32_t (&counts)[kTeam][64] = team->count[round & 1u];
                        counts[member][lane] = n;
                        __syncthreads();
                        uint32_t before = 0u, all = 0u;
                        #pragma unroll
                        for (unsigned int w = 0; w < kTeam; ++w)
                            {
                            const uint32_t c = counts[w][lane];
                            if (w < member) before += c;
                            all += c;
                            }
                        write_hits(Rows<OutputOpT>::neigh(out), Rows<OutputOpT>::image(out), P, hits,
                                   Rows<OutputOpT>::at(out, result) + before, Rows<OutputOpT>::end(out, result), k);
                        Rows<OutputOpT>::add(result, all);
                        ++round;
                        }
                    }
                else if constexpr (!kCount)
                    {
                    // any other output op takes its hits one by one
                    while (hits)
                        {
                        detail::emit_hit(out, result, static_cast<int>(P.prim[__builtin_ctzll(hits)]), k, 0);
                        hits &= hits - 1ull;
                        }
                    }
                wave::lds_order();
                }
            ln = 0u;
            }

        if constexpr (kRows && !TEAM)
            {
            if (cur != ~0u && Rows<OutputOpT>::image(out))
                {
                const unsigned long long at = Rows<OutputOpT>::at(out, result), end = Rows<OutputOpT>::end(out, result);
                wave::image_run(Rows<OutputOpT>::image(out), run0, at < end ? at : end, cur);
                }
            }
        if constexpr (kCount)
            {
            uint32_t mine = cnt[0];
            if constexpr (kExact)
                {
                // each query's counts lie in four lanes (one per row), by group
                #pragma unroll
                for (unsigned int g = 0; g < 4; ++g)
                    {
                    uint32_t c = cnt[g];
                    c += static_cast<uint32_t>(__shfl_xor(static_cast<int>(c), 16, 64));
                    c += static_cast<uint32_t>(__shfl_xor(static_cast<int>(c), 32, 64));
                    if ((lane >> 4) == g) mine = c;
                    }
                if constexpr (kChecked) mine += odd_hits;
                }
            if constexpr (TEAM)
                {
                team->count[0][member][lane] = mine;
                __syncthreads();
                mine = 0u;
                #pragma unroll
                for (unsigned int w = 0; w < kTeam; ++w) mine += team->count[0][w][lane];
                }
            result.num_neigh += mine;
            }
        if constexpr (!detail::relocates<OutputOpT>::value) break;
        else if constexpr (!TEAM)
            {
            const bool again = valid && out.relocate(result);
            if (!wave::vote(again)) break;
            act = again;
            }
        else
            {
            // one member moves the rows; the others take its new positions
            if (member == 0u)
                {
                const bool again = valid && out.relocate(result);
                team->pos[lane] = result.pos;
                team->end[lane] = again ? result.end : 0ull;
                team->count[round & 1u][0][lane] = again ? 1u : 0u;
                }
            __syncthreads();
            act = team->count[round & 1u][0][lane] != 0u;
            if (act)
                {
                result.pos = team->pos[lane];
                result.end = team->end[lane];
                result.num_neigh = 0u;
                }
            ++round;
            if (!wave::vote(act)) break;
            }
        }
    if (valid && member == 0u) out.finalize(result);
    return true;
    }

__device__ __forceinline__ bool small(const float x, const float y, const float z)
    {
    return fabsf(x) < kMaxCoordinate && fabsf(y) < kMaxCoordinate && fabsf(z) < kMaxCoordinate;
    }
//! True when a query takes the walk above.
__device__ __forceinline__ bool takes(const float4& q) { return small(q.x, q.y, q.z) && fabsf(q.w) < kMaxCoordinate; }

//! True when the image vectors (reference query, quantized boxes: and the root box, which holds every
//! box) let queries take the walk above (wave-uniform).
template<class SrcT, class QueryOpT, class TranslateOpT>
__device__ __forceinline__ bool takes(const TranslateOpT& images, const BoundingBox& root_box)
    {
    const unsigned int lane = threadIdx.x & 63u;
    const unsigned int nimg = images.size() < 32u ? images.size() : 32u;
    bool ok = true;
    if (lane < nimg)
        {
        const double3 t = as_double3(images.get(lane));
        ok = small(static_cast<float>(t.x), static_cast<float>(t.y), static_cast<float>(t.z));
        }
    if constexpr (SrcT::kFirst || !std::is_same<QueryOpT, ExactSphereQueryOp>::value)
        ok = ok && small(root_box.lo.x, root_box.lo.y, root_box.lo.z) && small(root_box.hi.x, root_box.hi.y, root_box.hi.z);
    return wave::vote(!ok) == 0ull;
    }

//! The walk of the queries that the front walk does not take: one rope path per lane, the query's
//! own tests.
template<class SrcT, class OutputOpT, class QueryOpT, class TranslateOpT>
__device__ __forceinline__ void lane_walk(const OutputOpT& out, const SrcT& src, const int root, const int stop, const BoundingBox& root_box,
                                          const QueryOpT& query, const TranslateOpT& images, const unsigned int idx, const float4& q,
                                          const unsigned int n_nodes)
    {
    constexpr bool kExact = std::is_same<QueryOpT, ExactSphereQueryOp>::value;
    typename OutputOpT::ThreadData result = out.setup(idx, q);
    // each lane goes from one of its own images to the next: the lanes walk different ones together
    // (image by image for all lanes, counts of 10^6 in random order 7859 us instead of 6698)
    uint32_t reached = 0u;
    unsigned int nimg = images.size() < 32u ? images.size() : 32u;
    if constexpr (kExact)
        if (!wave::can_hit(q)) nimg = 0u;
    for (unsigned int k = 0; k < nimg; ++k)
        if (query.overlap(query.get(q, images.get(k)), root_box)) reached |= 1u << k;
    for (int pass = 0; pass < 2; ++pass)
        {
        uint32_t flags = reached;
        while (flags)
            {
            const unsigned int k = __builtin_ctz(flags);
            flags &= flags - 1u;
            const typename QueryOpT::Volume v = query.get(q, images.get(k));
            int node = root;
            for (int budget = 2 * static_cast<int>(n_nodes); node != stop && budget > 0; --budget)
                {
                const Node rec = src.node(static_cast<uint32_t>(node));
                int next = rec.rope;
                if (query.overlap(v, src.box(static_cast<uint32_t>(node))))
                    {
                    if (rec.lf >= 0) next = rec.lf;
                    else if constexpr (SrcT::kFirst)
                        {
                        if (detail::refine_hit(query, q, v, ~rec.lf, 0)) detail::emit_hit(out, result, ~rec.lf, k, 0);
                        }
                    else
                        {
                        const unsigned int end = bucket_end(next, src.n_internal);
                        for (unsigned int leaf = ~static_cast<unsigned int>(rec.lf); leaf < end; ++leaf)
                            {
                            if constexpr (kExact)
                                {
                                const float4 p = src.point(query, leaf);
                                if (ExactSphereQueryOp::refine_point(v, p))
                                    detail::emit_hit(out, result, static_cast<int>(src.point_value(p)), k, 0);
                                }
                            else
                                {
                                if (query.overlap(v, src.box(src.n_internal + leaf)))
                                    detail::emit_hit(out, result, static_cast<int>(src.value(leaf, rec)), k, 0);
                                }
                            }
                        }
                    }
                node = next;
                }
            }
        if constexpr (!detail::relocates<OutputOpT>::value) break;
        else if (!out.relocate(result)) break;
        }
    out.finalize(result);
    }

//! Launches that the walk by one rope path per wave can serve, too.
template<class SrcT, class OutputOpT, class QueryOpT>
struct waves
    : std::integral_constant<bool, !SrcT::kFirst && std::is_same<QueryOpT, ExactSphereQueryOp>::value && wave::walks<OutputOpT>::value>
    {};

//! The walk of a wave's unusual queries, before that of the others (nothing of them is held in
//! registers then).  lds: the wave's part.
template<class SrcT, class OutputOpT, class QueryOpT, class TranslateOpT>
__device__ __forceinline__ void walk_alone(const OutputOpT& out, const SrcT& src, const int root, const int stop, const BoundingBox& root_box,
                                           const QueryOpT& query, const TranslateOpT& images, const bool mine, const unsigned int idx,
                                           const float4& q, const unsigned int n_nodes, unsigned char* lds)
    {
    if constexpr (waves<SrcT, OutputOpT, QueryOpT>::value)
        {
        // a radius that reaches every point: 64 of a bucket's leaves at a time
        static_assert(sizeof(wave::CompactWave) <= sizeof(FrontWave), "in the wave's part");
        wave::walk(out, src.nodes, src.points, root_box, root, stop, query, images, src.transform, mine, idx, q, src.n_internal, n_nodes,
                   *reinterpret_cast<wave::CompactWave*>(lds));
        wave::lds_order();
        }
    else if (mine) lane_walk(out, src, root, stop, root_box, query, images, idx, q, n_nodes);
    }

//! LDS of the front kernels: one part per wave, the second struct (not for counts) behind the first.
template<class OutputOpT>
struct FrontLds
    {
    static constexpr size_t kPart = sizeof(FrontWave) + (std::is_same<OutputOpT, CountNeighborsOp>::value ? 0 : sizeof(FrontPairs));
    static_assert(sizeof(FrontWave) % 16 == 0 && kPart % 16 == 0, "aligned parts");
    };
} // end namespace front

//! Morton code (its first `bits` bits) of a query's center in the tree's root box.
struct QueryCode
    {
    const float4* spheres;
    float3 lo, L;
    unsigned int bits;

    __device__ __forceinline__ uint32_t operator()(const uint32_t i) const
        {
        const float4 c = spheres[i];
        return morton3(fraction_to_bin((c.x - lo.x) / L.x), fraction_to_bin((c.y - lo.y) / L.y), fraction_to_bin((c.z - lo.z) / L.z)) >> (30u - bits);
        }
    };
__device__ __forceinline__ QueryCode query_code(const float4* spheres, const float3* root_lo, const float3* root_hi, const unsigned int bits)
    {
    const float3 lo = *root_lo, hi = *root_hi;
    return {spheres, lo, make_float3(hi.x - lo.x, hi.y - lo.y, hi.z - lo.z), bits};
    }

//! Morton codes of query centers in the tree's root box, their digit histograms, and the clearing
//! of the sort's status words: the order in which a launch serves queries given without one.
__global__ void __launch_bounds__(256) query_codes(const float4* __restrict__ spheres, const uint32_t n,
                                                   const float3* __restrict__ root_lo, const float3* __restrict__ root_hi,
                                                   const unsigned int bits, uint32_t* __restrict__ codes, uint32_t* __restrict__ hist,
                                                   const unsigned int passes, uint32_t* __restrict__ clear, const size_t clear_words)
    {
    __shared__ uint32_t s_hist[4 * radix::kRadix];
    for (unsigned int j = threadIdx.x; j < passes * radix::kRadix; j += blockDim.x) s_hist[j] = 0u;
    __syncthreads();
    const QueryCode code_of = query_code(spheres, root_lo, root_hi, bits);
    const size_t stride = static_cast<size_t>(gridDim.x) * blockDim.x;
    const size_t first = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    for (size_t i = first; i < n; i += stride)
        {
        const uint32_t code = code_of(static_cast<uint32_t>(i));
        codes[i] = code;
        for (unsigned int p = 0; p < passes; ++p)
            radix::count_digit(s_hist + p * radix::kRadix, (code >> (p * radix::kBits)) & (radix::kRadix - 1));
        }
    for (size_t i = first; i < clear_words; i += stride) clear[i] = 0u;
    __syncthreads();
    uint32_t* part = radix::hist_part(hist, passes);
    for (unsigned int j = threadIdx.x; j < passes * radix::kRadix; j += blockDim.x)
        if (s_hist[j]) atomicAdd(&part[j], s_hist[j]);
    }

//! The order of few queries in one launch (radix::kernel::rank_sort).
__global__ void __launch_bounds__(radix::kernel::kRankBlock) query_order_ranked(const float4* __restrict__ spheres, const uint32_t n,
                                                                                const float3* __restrict__ root_lo,
                                                                                const float3* __restrict__ root_hi, const unsigned int bits,
                                                                                uint32_t* __restrict__ order)
    {
    __shared__ radix::kernel::RankSort lds;
    uint32_t code;
    const uint32_t place = radix::kernel::rank_sort(lds, query_code(spheres, root_lo, root_hi, bits), n, blockIdx.x, code);
    const uint32_t i = blockIdx.x * 64u + threadIdx.x;
    if (threadIdx.x < 64u && i < n) order[place] = i;
    }

//! Traversal by node fronts, one wave per 64 consecutive queries of the traversal order.  Blocks
//! map to queries by wave::tail_block.  BESIDE: launched beside lbvh_traverse_wave, which serves the
//! queries when few leaves (fewer than limit) are within their radius.
template<bool BESIDE, class SrcT, class OutputOpT, class QueryOpT, class TranslateOpT>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4, 8)))
lbvh_traverse_front(const OutputOpT out,
                    SrcT src,
                    const float3* __restrict__ root_lo,
                    const float3* __restrict__ root_hi,
                    const float3* __restrict__ bins,
                    const int root,
                    const QueryOpT query,
                    const TranslateOpT images,
                    const unsigned int* __restrict__ order,
                    const unsigned int n_nodes,
                    const unsigned int tail_groups,
                    const unsigned int tail_split,
                    const float limit)
    {
    typedef front::FrontLds<OutputOpT> Lds;
    __shared__ alignas(16) unsigned char lds[4][Lds::kPart];
    const unsigned int n = query.size();
    const wave::BlockSpan span = wave::tail_block(blockIdx.x, (n + 255u) / 256u, tail_groups, tail_split);
    if (!span.live) return;
    const unsigned int lane = threadIdx.x & 63u;
    const unsigned int wid = static_cast<unsigned int>(__builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6)));
    const unsigned int t = span.first + wid * span.per_wave + lane;
    bool valid = lane < span.per_wave && t < n;
    const unsigned int idx = valid ? (order ? order[t] : t) : 0u;
    const BoundingBox root_box(*root_lo, *root_hi);
    if constexpr (BESIDE)
        if (front::sparse(query, order, root_box, n_nodes, limit)) return;
    wave::place_rows(out, t, idx, valid);
    const float4 q = valid ? query.setup(idx) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    front::bind(src, root_box, bins);
    front::FrontWave& W = *reinterpret_cast<front::FrontWave*>(lds[wid]);
    front::FrontPairs& P = *reinterpret_cast<front::FrontPairs*>(lds[wid] + sizeof(front::FrontWave));
    const bool odd = valid && !(front::takes(q) && front::takes<SrcT, QueryOpT>(images, root_box));
    if (__builtin_expect(wave::vote(odd) != 0ull, 0))
        {
        front::walk_alone(out, src, root, LBVHSentinel, root_box, query, images, odd, idx, q, n_nodes, lds[wid]);
        valid = valid && !odd;
        }
    if (front::walk<false>(out, src, root, root_box, query, images, valid, idx, q, n_nodes, W, P, nullptr)) return;
    if (valid)
        front::lane_walk(out, src, root, LBVHSentinel, root_box, query, images, idx, q, n_nodes);
    }

//! Exact counts and pair rows by one rope path per wave for 64 consecutive queries (wave::walk).
//! Blocks map to queries by wave::tail_block.  A finite limit: launched beside lbvh_traverse_front,
//! which serves the queries unless fewer leaves than limit are within their radius.
template<class OutputOpT, class TranslateOpT, class TransformOpT>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8, 8)))
lbvh_traverse_wave(const OutputOpT out,
                   const front::BucketSource<TransformOpT> src,
                   const float3* __restrict__ root_lo,
                   const float3* __restrict__ root_hi,
                   const int root,
                   const ExactSphereQueryOp query,
                   const TranslateOpT images,
                   const unsigned int* __restrict__ order,
                   const unsigned int n_nodes,
                   const unsigned int tail_groups,
                   const unsigned int tail_split,
                   const float limit)
    {
    __shared__ wave::CompactWave lds[4];
    const unsigned int n = query.size();
    const wave::BlockSpan span = wave::tail_block(blockIdx.x, (n + 255u) / 256u, tail_groups, tail_split);
    if (!span.live) return;
    const unsigned int lane = threadIdx.x & 63u;
    const unsigned int t = span.first + (threadIdx.x >> 6) * span.per_wave + lane;
    const bool valid = lane < span.per_wave && t < n;
    const unsigned int idx = valid ? (order ? order[t] : t) : 0u;
    const BoundingBox root_box(*root_lo, *root_hi);
    if (limit < __builtin_huge_valf() && !front::sparse(query, order, root_box, n_nodes, limit)) return;
    wave::place_rows(out, t, idx, valid);
    const float4 q = valid ? query.setup(idx) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    const front::Quad quad = front::quad_of(valid, q);
    const unsigned long long qwide = front::mostly_empty(quad.lo, quad.hi, quad.r, front::mean_cell(root_box, n_nodes));
    if (__builtin_expect(front::scattered(wave::vote(valid), qwide, n_nodes), 0))
        {
        if (valid) front::lane_walk(out, src, root, LBVHSentinel, root_box, query, images, idx, q, n_nodes);
        return;
        }
    wave::walk(out, src.nodes, src.points, root_box, root, LBVHSentinel, query, images, src.transform, valid, idx, q, src.n_internal,
               n_nodes, lds[threadIdx.x >> 6]);
    }

//! lbvh_traverse_front with the four waves of a block for the same `per` (4, 16, 32 or 64) queries:
//! launches of few queries, whose time is that of one wave's own chain of steps.
template<class SrcT, class OutputOpT, class QueryOpT, class TranslateOpT>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(std::is_same<OutputOpT, CountNeighborsOp>::value ? 4 : 3, 8)))
lbvh_traverse_team(const OutputOpT out,
                   SrcT src,
                   const float3* __restrict__ root_lo,
                   const float3* __restrict__ root_hi,
                   const float3* __restrict__ bins,
                   const int root,
                   const QueryOpT query,
                   const TranslateOpT images,
                   const unsigned int* __restrict__ order,
                   const unsigned int n_nodes,
                   const unsigned int per)
    {
    typedef front::FrontLds<OutputOpT> Lds;
    __shared__ alignas(16) unsigned char lds[4][Lds::kPart];
    __shared__ front::Team team;
    static_assert(!wave::places_rows<OutputOpT>::value, "rows are placed by blocks that serve whole groups");
    const unsigned int n = query.size();
    const unsigned int lane = threadIdx.x & 63u;
    const unsigned int wid = static_cast<unsigned int>(__builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6)));
    const unsigned int t = per * wave::xcd_block(blockIdx.x, gridDim.x) + lane;
    bool valid = lane < per && t < n;
    const unsigned int idx = valid ? (order ? order[t] : t) : 0u;
    const float4 q = valid ? query.setup(idx) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    const BoundingBox root_box(*root_lo, *root_hi);
    front::bind(src, root_box, bins);
    front::FrontWave& W = *reinterpret_cast<front::FrontWave*>(lds[wid]);
    front::FrontPairs& P = *reinterpret_cast<front::FrontPairs*>(lds[wid] + sizeof(front::FrontWave));
    const bool odd = valid && !(front::takes(q) && front::takes<SrcT, QueryOpT>(images, root_box));
    if (__builtin_expect(wave::vote(odd) != 0ull, 0))
        {
        if (wid == 0u) front::walk_alone(out, src, root, LBVHSentinel, root_box, query, images, odd, idx, q, n_nodes, lds[wid]);
        valid = valid && !odd;
        }
    if (front::walk<true>(out, src, root, root_box, query, images, valid, idx, q, n_nodes, W, P, &team)) return;
    // scattered (more than 16 queries, so 32 or 64): a quarter to each wave, which takes the longest
    // paths from one wave; short ones, over rope records without images, are bound by the waves'
    // instructions and stay in one (counts of 65,536 in random order, one wave and four: bucket records
    // 389 and 305 us, with images 697 and 487; quantized records 579 and 847, with images 2260 and 2090)
    const bool quarters = !SrcT::kFirst || images.size() > 1u;
    if (valid && (quarters ? lane / (per / 4u) : 0u) == wid)
        front::lane_walk(out, src, root, LBVHSentinel, root_box, query, images, idx, q, n_nodes);
    }

} // end namespace kernel
} // end namespace gpu
} // end namespace neighbor

#endif // NEIGHBOR_KERNELS_FRONT_WALK_H_
