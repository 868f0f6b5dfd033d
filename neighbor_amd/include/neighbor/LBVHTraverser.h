// LBVHTraverser.h -- stackless rope traversal of an LBVH.
//
// Public interface of the reference (include/neighbor/LBVHTraverser.h:60-355):
// setup() compresses once and arms replay, reset() disarms it, traverse() with
// LaunchParameters / stream / default overloads and optional translate and
// transform ops, getData() for the compressed records; Tunable block size.
// traverse() silently returns for an empty tree, no queries or no images and
// throws std::runtime_error for more than 32 images (LBVHTraverser.h:423-432).
//
// Variants (this library): Quantized holds the reference's 16-B records; FloatRope 32-B records
// with the decoded quantized boxes (same results); FloatRopeExact the exact node boxes, meant for
// ExactSphereQueryOp (with the float SphereQueryOp it reports fewer, tighter hits than the
// reference); Wave (ExactSphereQueryOp only) exact-box records with bucket leaves; WaveQuantized
// the same over decoded quantized boxes, for SphereQueryOp (results identical to Quantized) and
// ExactSphereQueryOp.  Both queries walk by node fronts (kernels/FrontWalk.h), many exact queries over
// bucket records by one rope path per wave (kernels/WaveWalk.h, sparseLimit); other query ops, and
// many exact queries over float rope records (kRopeFronts), take one rope path per query.
#ifndef NEIGHBOR_LBVH_TRAVERSER_H_
#define NEIGHBOR_LBVH_TRAVERSER_H_

#include "LBVH.h"
#include "LBVHTraverserData.h"
#include "Memory.h"
#include "OutputOps.h"
#include "QueryOps.h"
#include "TransformOps.h"
#include "TranslateOps.h"
#include "Tunable.h"
#include "kernels/FrontWalk.h"
#include "kernels/LBVHTraverse.h"

#include <algorithm>
#include <limits>
#include <memory>
#include <mutex>
#include <stdexcept>
#include <type_traits>
#include <vector>

namespace neighbor
{

//! Raised by traverse() for more than 32 images.
class image_limit_error : public std::runtime_error
    {
    public:
        image_limit_error() : std::runtime_error("A maximum of 32 image vectors are supported by LBVH traversers.") {}
    };

enum class TraversalVariant { Quantized = 0, FloatRope = 1, FloatRopeExact = 2, Wave = 3, WaveQuantized = 4 };

class LBVHTraverser : public Tunable<unsigned int>
    {
    public:
        static constexpr unsigned int kDefaultBlock = 256;

        LBVHTraverser()
            : Tunable<unsigned int>(32, 1024, 32),
              m_root(LBVHSentinel),
              m_lbvh_lo(1, MemoryKind::Device), m_lbvh_hi(1, MemoryKind::Device), m_bins(1, MemoryKind::Device),
              m_replay(false), m_variant(TraversalVariant::Quantized), m_order(nullptr), m_order_n(0)
            {}

        template<class TransformOpT>
        void setup(const LaunchParameters& params, const LBVH& lbvh, const TransformOpT& transform)
            {
            reset();
            if (lbvh.getN() != 0)
                {
                compress(params, lbvh, transform);
                m_replay = true;
                }
            }
        void setup(const LaunchParameters& params, const LBVH& lbvh) { setup(params, lbvh, NullTransformOp()); }
        template<class TransformOpT>
        void setup(stream_t stream, const LBVH& lbvh, const TransformOpT& transform)
            {
            setup(LaunchParameters(kDefaultBlock, stream), lbvh, transform);
            }
        void setup(stream_t stream, const LBVH& lbvh) { setup(stream, lbvh, NullTransformOp()); }
        template<class TransformOpT>
        void setup(const LBVH& lbvh, const TransformOpT& transform) { setup(stream_t(0), lbvh, transform); }
        void setup(const LBVH& lbvh) { setup(stream_t(0), lbvh, NullTransformOp()); }

        void reset() { m_replay = false; }

        template<class QueryOpT, class OutputOpT, class TranslateOpT, class TransformOpT>
        void traverse(const LaunchParameters& params, const LBVH& lbvh, const QueryOpT& query,
                      const OutputOpT& out, const TranslateOpT& images, const TransformOpT& transform);

        template<class QueryOpT, class OutputOpT, class TranslateOpT>
        void traverse(const LaunchParameters& params, const LBVH& lbvh, const QueryOpT& query,
                      const OutputOpT& out, const TranslateOpT& images)
            {
            traverse(params, lbvh, query, out, images, NullTransformOp());
            }
        template<class QueryOpT, class OutputOpT>
        void traverse(const LaunchParameters& params, const LBVH& lbvh, const QueryOpT& query, const OutputOpT& out)
            {
            traverse(params, lbvh, query, out, SelfOp(), NullTransformOp());
            }
        template<class QueryOpT, class OutputOpT, class TranslateOpT, class TransformOpT>
        void traverse(stream_t stream, const LBVH& lbvh, const QueryOpT& query, const OutputOpT& out,
                      const TranslateOpT& images, const TransformOpT& transform)
            {
            traverse(LaunchParameters(kDefaultBlock, stream), lbvh, query, out, images, transform);
            }
        template<class QueryOpT, class OutputOpT, class TranslateOpT>
        void traverse(stream_t stream, const LBVH& lbvh, const QueryOpT& query, const OutputOpT& out,
                      const TranslateOpT& images)
            {
            traverse(stream, lbvh, query, out, images, NullTransformOp());
            }
        template<class QueryOpT, class OutputOpT>
        void traverse(stream_t stream, const LBVH& lbvh, const QueryOpT& query, const OutputOpT& out)
            {
            traverse(stream, lbvh, query, out, SelfOp(), NullTransformOp());
            }
        template<class QueryOpT, class OutputOpT, class TranslateOpT, class TransformOpT>
        void traverse(const LBVH& lbvh, const QueryOpT& query, const OutputOpT& out, const TranslateOpT& images,
                      const TransformOpT& transform)
            {
            traverse(stream_t(0), lbvh, query, out, images, transform);
            }
        template<class QueryOpT, class OutputOpT, class TranslateOpT>
        void traverse(const LBVH& lbvh, const QueryOpT& query, const OutputOpT& out, const TranslateOpT& images)
            {
            traverse(stream_t(0), lbvh, query, out, images, NullTransformOp());
            }
        template<class QueryOpT, class OutputOpT>
        void traverse(const LBVH& lbvh, const QueryOpT& query, const OutputOpT& out)
            {
            traverse(stream_t(0), lbvh, query, out, SelfOp(), NullTransformOp());
            }

        //! Quantized rope records (reference layout); not produced by the Wave variant.
        const shared_array<int4>& getData() const { return m_data; }
        //! Float rope records (FloatRope variants) or bucket records (wave variants); the Wave
        //! variant does not write the records of nodes below a bucket (never visited).
        const shared_array<float4>& getFloatRopeData() const { return m_float; }
        const shared_array<float3>& getRootLower() const { return m_lbvh_lo; }
        const shared_array<float3>& getRootUpper() const { return m_lbvh_hi; }
        const shared_array<float3>& getBins() const { return m_bins; }

        //! Select the node record walked by traverse(); takes effect at the next compression.
        void setVariant(TraversalVariant v)
            {
            if (v != m_variant) m_replay = false;
            m_variant = v;
            }
        TraversalVariant getVariant() const { return m_variant; }

        //! Thread t serves query order[t] (order must hold a permutation of [0, n)); null clears.
        void setQueryOrder(const unsigned int* order, unsigned int n)
            {
            m_order = order;
            m_order_n = n;
            }

        //! Wave-walk statistics (wave variants, count traversals): each launched wave w writes
        //! its node records loaded, buckets tested and leaves in those buckets to log[3w ..
        //! 3w+2].  words: the log's size; a traversal launching more waves than it holds, or
        //! another output op while the log is set, throws.  null clears.
        void setVisitLog(unsigned int* log, size_t words)
            {
            m_visits = log;
            m_visit_words = log ? words : 0;
            }
        //! Words of visit log a wave traversal of n queries writes.
        static size_t visitLogWords(unsigned int n) { return 3 * static_cast<size_t>(div_up(n, 256)) * 4; }

    private:
        int m_root;
        shared_array<int4> m_data;
        shared_array<float4> m_float;
        shared_array<float3> m_lbvh_lo;
        shared_array<float3> m_lbvh_hi;
        shared_array<float3> m_bins;
        bool m_replay;
        TraversalVariant m_variant;
        const unsigned int* m_order;
        unsigned int m_order_n;
        unsigned int* m_visits = nullptr;
        size_t m_visit_words = 0;

        LBVHCompressedData data()
            {
            LBVHCompressedData c;
            c.root = m_root;
            c.data = m_data.get();
            c.lo = m_lbvh_lo.get();
            c.hi = m_lbvh_hi.get();
            c.bins = m_bins.get();
            return c;
            }

        template<class TransformOpT>
        void compress(const LaunchParameters& params, const LBVH& lbvh, const TransformOpT& transform);

        //! Workspace that sorts the queries of one launch (done: the last launch that reads it).
        struct QuerySort
            {
            shared_array<unsigned int> keys[2], vals[2], work;
            stream_t stream = nullptr;
            std::shared_ptr<void> done;     //!< hipEvent_t
            };
        //! Bounded: a launch takes the workspace last used with its stream's handle, a free one, a new
        //! one or the oldest, and waits on the device for the workspace's last launch: equal handles
        //! may be different streams (each thread's hipStreamPerThread, a new stream at a destroyed
        //! one's address).  Only the null stream is always itself (the call costs 1.5 us of a list of
        //! 1000 points' 80).  The lock is held from the sort to the record of `done` (several threads
        //! may traverse at once); a copy of the traverser starts with none.
        struct QuerySorts
            {
            static constexpr size_t kMost = 4;
            std::vector<QuerySort> all;
            size_t oldest = 0;
            std::mutex lock;

            QuerySorts() = default;
            QuerySorts(const QuerySorts&) {}
            QuerySorts& operator=(const QuerySorts&) { return *this; }
            } m_sorts;

        //! Calls in its scope are not those that another thread's capture (global mode) forbids: they
        //! allocate, free and ask events, on nothing that a capture uses.
        struct BesideCaptures
            {
            hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
            BesideCaptures() { NEIGHBOR_HIP_CHECK(hipThreadExchangeStreamCaptureMode(&mode)); }
            ~BesideCaptures() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
            BesideCaptures(const BesideCaptures&) = delete;
            BesideCaptures& operator=(const BesideCaptures&) = delete;
            };

        //! Room for n queries in s: all of it or none.
        static void grow(QuerySort& s, const unsigned int n, const size_t words, const bool both)
            {
            const auto room = [](shared_array<unsigned int>& kept, const size_t size) {
                return size > kept.size() ? shared_array<unsigned int>(size, MemoryKind::Device) : shared_array<unsigned int>();
            };
            shared_array<unsigned int> keys[2], vals[2], work;
            for (int i = 0; i < 2; ++i)
                {
                if (both) keys[i] = room(s.keys[i], n);
                if (both || i == 0) vals[i] = room(s.vals[i], n);
                }
            work = room(s.work, words);
            for (int i = 0; i < 2; ++i)
                {
                if (keys[i].size()) s.keys[i].swap(keys[i]);
                if (vals[i].size()) s.vals[i].swap(vals[i]);
                }
            if (work.size()) s.work.swap(work);
            }

        QuerySort& query_sort(stream_t stream)
            {
            QuerySort& s = pick_sort(stream);
            #ifdef HIP_API_PER_THREAD_DEFAULT_STREAM
            const bool same = false;
            #else
            const bool same = !stream && !s.stream;
            #endif
            if (!same) NEIGHBOR_HIP_CHECK(hipStreamWaitEvent(stream, static_cast<hipEvent_t>(s.done.get()), 0));
            s.stream = stream;
            return s;
            }
        QuerySort& pick_sort(stream_t stream)
            {
            for (QuerySort& s : m_sorts.all)
                if (s.stream == stream) return s;
            for (QuerySort& s : m_sorts.all)
                {
                if (hipEventQuery(static_cast<hipEvent_t>(s.done.get())) == hipSuccess) return s;
                (void)hipGetLastError();    // not ready
                }
            if (m_sorts.all.size() == QuerySorts::kMost) return m_sorts.all[m_sorts.oldest++ % QuerySorts::kMost];
            hipEvent_t e;
            NEIGHBOR_HIP_CHECK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
            QuerySort s;
            s.done = std::shared_ptr<void>(static_cast<void*>(e), [](void* p) { (void)hipEventDestroy(static_cast<hipEvent_t>(p)); });
            m_sorts.all.push_back(s);
            return m_sorts.all.back();
            }

        static bool capturing(stream_t stream)
            {
            hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
            const hipError_t e = hipStreamIsCapturing(stream, &status);
            if (e != hipSuccess) (void)hipGetLastError();
            return e != hipSuccess || status != hipStreamCaptureStatusNone;
            }

        //! Queries in the Morton order of their centers in the root box (16 or 24 bits of code).
        const unsigned int* sorted_queries(QuerySort& s, const float4* spheres, const unsigned int n, stream_t stream)
            {
            const unsigned int bits = n <= (1u << 20) ? 16u : 24u;
            if (n <= gpu::radix::kernel::kRankSort)
                {
                grow(s, n, 0, false);
                hipLaunchKernelGGL(gpu::kernel::query_order_ranked, dim3(div_up(n, 64)), dim3(gpu::radix::kernel::kRankBlock), 0, stream,
                                   spheres, n, m_lbvh_lo.get(), m_lbvh_hi.get(), bits, s.vals[0].get());
                return s.vals[0].get();
                }
            grow(s, n, gpu::radix::Workspace::words(n, bits), true);
            const gpu::radix::Workspace ws = gpu::radix::Workspace::carve(s.work.get(), n, bits);
            const size_t header = gpu::radix::Workspace::header_words(ws.passes);
            hipLaunchKernelGGL(gpu::radix::kernel::fill_zero, dim3(div_up(header, 256)), dim3(256), 0, stream, ws.hist, header);
            hipLaunchKernelGGL(gpu::kernel::query_codes, dim3(std::min<unsigned int>(div_up(n, 1024), 2048u)), dim3(256), 0, stream,
                               spheres, n, m_lbvh_lo.get(), m_lbvh_hi.get(), bits, s.keys[0].get(), ws.hist, ws.passes, ws.status,
                               static_cast<size_t>(ws.passes) * ws.tiles * gpu::radix::kRadix);
            const bool alt = gpu::radix::sort_passes(s.keys[0].get(), s.vals[0].get(), s.keys[1].get(), s.vals[1].get(), n, true, ws, stream);
            return s.vals[alt ? 1 : 0].get();
            }

        //! The front walk's launch: few queries by teams of four waves, others by one wave per 64.
        template<class QueryOpT, class OutputOpT, class TranslateOpT, class SourceT>
        void launch_front(const LaunchParameters& params, const QueryOpT& query, const OutputOpT& out, const TranslateOpT& images,
                          const unsigned int* order, const unsigned int n_nodes, const SourceT& src)
            {
            constexpr bool placed = gpu::kernel::wave::places_rows<OutputOpT>::value;    // whole groups per block
            // queries in no given order are sorted first: a wave's queries must lie close together
            if constexpr (!placed)
                if (!order && query.size() > kSortQueries && !capturing(params.stream))
                    {
                    const std::lock_guard<std::mutex> guard(m_sorts.lock);
                    const BesideCaptures beside;
                    QuerySort* sort = nullptr;
                    const unsigned int* sorted = nullptr;
                    try
                        {
                        sort = &query_sort(params.stream);
                        sorted = sorted_queries(*sort, query.spheres, query.size(), params.stream);
                        }
                    catch (const hip_error& e)
                        {
                        if (e.code() != hipErrorOutOfMemory) throw;     // no room for the sort: served as they come
                        }
                    launch_front_in_order(params, query, out, images, sorted, n_nodes, src);
                    if (sorted) NEIGHBOR_HIP_CHECK(hipEventRecord(static_cast<hipEvent_t>(sort->done.get()), params.stream));
                    return;
                    }
            launch_front_in_order(params, query, out, images, order, n_nodes, src);
            }

        template<class QueryOpT, class OutputOpT, class TranslateOpT, class SourceT>
        void launch_front_in_order(const LaunchParameters& params, const QueryOpT& query, const OutputOpT& out, const TranslateOpT& images,
                                   const unsigned int* order, const unsigned int n_nodes, const SourceT& src)
            {
            constexpr bool placed = gpu::kernel::wave::places_rows<OutputOpT>::value;
            constexpr bool teams = !placed && (gpu::kernel::front::Rows<OutputOpT>::kOn || std::is_same<OutputOpT, CountNeighborsOp>::value);
            const unsigned int n = query.size();
            if constexpr (teams)
                if (const unsigned int per = teamSize(std::is_same<OutputOpT, CountNeighborsOp>::value, n))
                    {
                    hipLaunchKernelGGL((gpu::kernel::lbvh_traverse_team<SourceT, OutputOpT, QueryOpT, TranslateOpT>),
                                       dim3(div_up(n, per)), dim3(256), 0, params.stream, out, src, m_lbvh_lo.get(), m_lbvh_hi.get(),
                                       m_bins.get(), m_root, query, images, order, n_nodes, per);
                    return;
                    }
            // tail-split map (wave::tail_block): XCD 0 holds the most groups; the other XCDs'
            // blocks past their own count exit at once
            const unsigned int tail = placed ? 0u : m_tail_set || (n > kAllSplit && n <= kHalfSplit) ? m_tail_groups : n <= kAllSplit ? kAllSplitGroups : kTailGroups;
            const unsigned int G = div_up(n, 256);
            const unsigned int x0 = G / 8u + (G % 8u ? 1u : 0u);
            const dim3 grid = tail ? dim3(8u * (x0 + (m_tail_split - 1u) * std::min(x0, tail))) : dim3(G);
            const auto fronts = [&](auto beside, const float limit) {
                hipLaunchKernelGGL((gpu::kernel::lbvh_traverse_front<decltype(beside)::value, SourceT, OutputOpT, QueryOpT, TranslateOpT>),
                                   grid, dim3(256), 0, params.stream, out, src, m_lbvh_lo.get(), m_lbvh_hi.get(), m_bins.get(), m_root, query,
                                   images, order, n_nodes, tail, m_tail_split, limit);
            };
            if constexpr (gpu::kernel::front::waves<SourceT, OutputOpT, QueryOpT>::value)
                {
                constexpr bool count = std::is_same<OutputOpT, CountNeighborsOp>::value;
                const float limit = sparseLimit(!count, n, m_bucket, images.size());
                if (limit > 0.0f)
                    {
                    launch_wave(params, query, out, images, order, n_nodes, src, limit);
                    if constexpr (count) fronts(std::true_type(), limit);
                    return;
                    }
                }
            fronts(std::false_type(), 0.0f);
            }

        //! Exact counts and pair rows by one rope path per wave.
        template<class OutputOpT, class TranslateOpT, class TransformOpT>
        void launch_wave(const LaunchParameters& params, const ExactSphereQueryOp& query, const OutputOpT& out, const TranslateOpT& images,
                         const unsigned int* order, const unsigned int n_nodes, const gpu::kernel::front::BucketSource<TransformOpT>& src,
                         const float limit)
            {
            // the last wave that each SIMD of an XCD receives, in halves
            const unsigned int tail = gpu::kernel::wave::places_rows<OutputOpT>::value ? 0u : m_tail_groups;
            const unsigned int G = div_up(query.size(), 256);
            const unsigned int x0 = G / 8u + (G % 8u ? 1u : 0u);
            const dim3 grid = tail ? dim3(8u * (x0 + (m_tail_split - 1u) * std::min(x0, tail))) : dim3(G);
            hipLaunchKernelGGL((gpu::kernel::lbvh_traverse_wave<OutputOpT, TranslateOpT, TransformOpT>), grid, dim3(256), 0, params.stream,
                               out, src, m_lbvh_lo.get(), m_lbvh_hi.get(), m_root, query, images, order, n_nodes, tail, m_tail_split, limit);
            }

        //! Exact queries over bucket records: the walk by node fronts serves those with more leaves within
        //! their radius than this, one rope path per wave the others (0: fronts only; infinite, rows: never).
        /*!
         * Fronts take a third of the dependent steps with half the waves on the chip: they win where one
         * wave's chain is long (dense neighbors, images, small buckets), lose where the launch is many
         * rounds of short walks.  Measured with uniform points at density 0.85 and radii 1.5, 2 and 2.8
         * (13, 29 and 79 neighbors), one rope path per wave against fronts in us:
         *  - Counts, no images, 64 leaves per bucket: 300,000 points 111/114, 135/123, 184/159; 10^6
         *    249/306, 302/325, 423/345; 4 10^6 862/1185, 1074/1230, 1542/1563.  16 leaves: 10^6 333/306,
         *    394/366, 514/427.  27 images, 64 leaves: 10^6 308/327, 371/351, 483/374; 2 10^6 532/639,
         *    630/656, 874/814.  The radius decides, and only the device knows it: both kernels are launched
         *    and one leaves at once (5 to 9 us), where the limit is not below 8 (about the fewest leaves
         *    per radius in use) and, with images, above 2^20 queries.
         *  - Rows depend less on it.  No images, 64 leaves: 200,000 108/120, 127/126, 173/159; 300,000
         *    128/159, 151/177, 217/251; 10^6 289/408, 350/458, 506/557; 32 leaves: 300,000 138/148,
         *    164/164, 237/259, 10^6 306/384, 370/442, 531/550; 16 leaves: 10^6 366/386, 452/484, 666/634.
         *    27 images, 64 leaves: 700,000 295/311, 343/349, 442/418, 10^6 374/433, 453/487, 611/601; 32
         *    leaves: 10^6 398/403, 469/472, 641/586, 2 10^6 683/773, 842/849, 1268/1380.
         * Left, with images: sparse queries (5 neighbors, 10^6: rows with 48 leaves 326/380, counts with
         * 64 leaves 263/317), and rows of 300,000 dense ones (64 leaves 254/278).
         */
        static float sparseLimit(const bool rows, const unsigned int n, const unsigned int bucket, const unsigned int images)
            {
            const float size = static_cast<float>(n) * 0x1p-20f, leaves = static_cast<float>(bucket);
            constexpr float never = std::numeric_limits<float>::infinity();
            if (n <= kFrontsOnly) return 0.0f;
            if (rows) return bucket >= 24u && (images == 1u || size * leaves > 48.0f) ? never : 0.0f;
            if (images > 1u && n <= 4u * kFrontsOnly) return 0.0f;
            const float limit = (images == 1u ? 0.6f : 0.3f) * leaves * std::min(leaves * 0x1p-5f, 1.0f) * size;
            return limit < 8.0f ? 0.0f : limit;
            }

        //! Rope and quantized records by node fronts; false: not this query op, or too many exact queries.
        template<class QueryOpT, class OutputOpT, class TranslateOpT>
        bool traverse_rope_fronts(const LaunchParameters& params, const LBVH& lbvh, const QueryOpT& query, const OutputOpT& out,
                                  const TranslateOpT& images, const unsigned int* order)
            {
            constexpr bool exact = std::is_same<QueryOpT, ExactSphereQueryOp>::value;
            constexpr bool reference = std::is_same<QueryOpT, SphereQueryOp>::value;
            if constexpr (exact || reference)
                {
                if (exact && m_variant != TraversalVariant::Quantized && query.size() > kRopeFronts) return false;
                if (m_variant == TraversalVariant::Quantized)
                    launch_front(params, query, out, images, order, lbvh.getNNodes(),
                                 gpu::kernel::front::QuantizedSource{m_data.get(), float3(), float3(), float3(), lbvh.getNInternal()});
                else
                    launch_front(params, query, out, images, order, lbvh.getNNodes(),
                                 gpu::kernel::front::RopeSource{m_float.get(), lbvh.getNInternal()});
                return true;
                }
            return false;
            }

        //! One rope path per query: other query ops, and more exact queries than kRopeFronts.
        template<class QueryOpT, class OutputOpT, class TranslateOpT>
        void traverse_rope_paths(const LaunchParameters& params, const LBVH& lbvh, const QueryOpT& query, const OutputOpT& out,
                                 const TranslateOpT& images, const unsigned int* order)
            {
            if constexpr (!std::is_same<QueryOpT, SphereQueryOp>::value)
                {
                const unsigned int block = checkParameter(params);
                const dim3 grid(div_up(query.size(), block));
                if (m_variant == TraversalVariant::Quantized)
                    {
                    hipLaunchKernelGGL((gpu::kernel::lbvh_traverse_ropes<OutputOpT, QueryOpT, TranslateOpT>), grid, dim3(block), 0,
                                       params.stream, out, data(), query, images, order, lbvh.getNNodes());
                    }
                else
                    {
                    LBVHFloatRopeData f;
                    f.root = m_root;
                    f.data = m_float.get();
                    // the image bits use the unquantized root box stored by the compression
                    hipLaunchKernelGGL((gpu::kernel::lbvh_traverse_float_ropes<OutputOpT, QueryOpT, TranslateOpT>), grid, dim3(block), 0,
                                       params.stream, out, f, m_lbvh_lo.get(), m_lbvh_hi.get(), query, images, order, lbvh.getNNodes());
                    }
                }
            }

        //! Bucket records: both sphere queries (exact boxes, the Wave variant: ExactSphereQueryOp only).
        template<class QueryOpT, class OutputOpT, class TranslateOpT, class TransformOpT>
        void traverse_wave(const LaunchParameters& params, const LBVH& lbvh, const QueryOpT& query, const OutputOpT& out,
                           const TranslateOpT& images, const TransformOpT& transform, const unsigned int* order)
            {
            constexpr bool exact = std::is_same<QueryOpT, ExactSphereQueryOp>::value;
            constexpr bool reference = std::is_same<QueryOpT, SphereQueryOp>::value;
            if constexpr (exact || reference)
                {
                // exact node boxes are only conservative for the exact query's FP64 test
                if (!exact && m_variant == TraversalVariant::Wave)
                    throw std::runtime_error("the Wave variant needs ExactSphereQueryOp; use WaveQuantized");
                // whole waves: 256-thread blocks regardless of the tunable block size
                const dim3 grid(div_up(query.size(), 256));
                if (m_visits)
                    {
                    if constexpr (std::is_same<OutputOpT, CountNeighborsOp>::value)
                        {
                        if (m_visit_words < visitLogWords(query.size()))
                            throw std::invalid_argument("the visit log holds fewer words than the traversal's waves write");
                        hipLaunchKernelGGL((gpu::kernel::lbvh_visit_log<QueryOpT, TranslateOpT>), grid, dim3(256), 0, params.stream,
                                           out, m_float.get(), lbvh.getSortedPoints().get(), m_lbvh_lo.get(), m_lbvh_hi.get(), m_root,
                                           query, images, order, lbvh.getNNodes(), m_visits);
                        return;
                        }
                    else
                        {
                        throw std::invalid_argument("the visit log records count traversals only");
                        }
                    }
                typedef gpu::kernel::front::BucketSource<TransformOpT> Source;
                launch_front(params, query, out, images, order, lbvh.getNNodes(),
                             Source{m_float.get(), lbvh.getSortedPoints().get(), lbvh.getPrimitives().get(), transform, lbvh.getNInternal()});
                }
            else
                {
                throw std::runtime_error("the wave traversal variants need SphereQueryOp or ExactSphereQueryOp");
                }
            }

        unsigned int m_bucket = 16;
        //! Queries given without an order above which they are sorted first.  The sort takes about
        //! 10 us for few queries and 70 us for 10^6.  Counts in random order and sorted here, with 27
        //! images: 256 queries 44 us and 44, 512 71 and 54, 1000 89 and 44; without images 14 and 24,
        //! 21 and 30, 34 and 33; 10^6 (one rope path per lane) 8.2 ms and 0.7.
        static constexpr unsigned int kSortQueries = 256;
        //! Exact queries over float rope records up to which they walk by fronts (quantized ones: any
        //! number).  These records are the choice for few neighbors per query, where a walk is one short
        //! path down from the root.  Exact counts by a path per lane and by fronts, uniform points: 262,144
        //! queries of 2.5 neighbors 100/114 us, of 5 126/118; 330,000 106/133, 124/142 (3.6), 150/146 (5),
        //! 263/148 (13); 524,288 167/185, 213/194, 269/199, 498/208; 990,000 275/339, 340/351, 424/359,
        //! 836/371: the lines cross near 4 neighbors at any size above.  Quantized, whose decoding a path
        //! repeats at every node: 330,000 299/148, 326/154, 337/163, 423/165; 990,000 617/373, 675/387,
        //! 726/397, 998/409.
        static constexpr unsigned int kRopeFronts = 1u << 18;
        //! Queries that a team of four waves serves together (0: one wave per 64).
        /*!
         * One wave's chain of steps takes longer than the chip needs for few queries.  Exact count and fill
         * of 10,000 points (27 images): 82 and 115 us with a wave per 64 queries, 48 and 61 with teams for
         * 16; of 131,071 points (no images) 90 and 125 us with waves, 201 and 229 with teams.  Teams for 16
         * and for 4: 1000 points 35 and 47 us, 29 and 38; 4000 points 56 and 72, 45 and 56; 8000 points 48
         * and 65, 62 and 77.
         * The lines lie where a launch fills the chip's round: 1024 blocks that count, 768 of 42 KB of LDS
         * that write rows; a second round that is nearly empty takes as long as the first.  Fills (27 images,
         * 79 neighbors, 48 leaves per bucket) by the smaller team and by the next: 12,288 at most in one
         * round: 13,000 63/53 us, 16,384 76/55; 24,576: 25,000 117/133 (16 leaves; 87/82), 28,000 136/142
         * (102/88), 32,768 169/155 (115/94): up to 28,672; 49,152: 50,000 145/128, 56,000 151/121, 65,536
         * 148/108 (no images 125/93; a rope path per wave took 105).  For 4 and 16: 4096 points 60/62, with
         * 16 leaves 74/108.
         */
        static unsigned int teamSize(const bool count, const unsigned int n)
            {
            if (n <= (1u << 12)) return 4u;
            if (n <= (count ? 4u << 12 : 3u << 12)) return 16u;
            if (n <= (count ? 8u << 12 : 7u << 12)) return 32u;
            return n <= (count ? 16u << 12 : 12u << 12) ? 64u : 0u;
            }
        static constexpr unsigned int kFrontsOnly = 1u << 18;
        //! Tail split (wave::tail_block): per XCD, the last groups of 256 queries run as m_tail_split
        //! blocks each, so that the waves that start last are shorter.  An XCD holds 128 of the front
        //! walk's blocks at once: all groups are split while that leaves slots free (up to kAllSplit
        //! queries), 32 of each XCD as long as the launch is one round then, too (96 + 32 blocks:
        //! kHalfSplit), above it 16.  Sums of five kinds of count, fill and float count (two radii, with
        //! and without images, 16 to 48 leaves) in us with 16, 32 and 64 groups: 85,000 points 1365, 1335 and
        //! 1196; 110,000 1560, 1469, 1442; 120,000 1555, 1471, 1513; 131,072 1645, 1521, 1584; 140,000 1709,
        //! 1705, 1976; 165,000 1876, 1811, 2211; 180,000 1997, 1890, 2310; 200,000 2032, 2306, 2477; 230,000
        //! 2386, 2608, 2742; 262,144 2792, 2900, 2964.  Exact count and fill, 500,000 points, with 0, 16 and
        //! 32: 257/374, 236/359, 247/377; 10^6 356/594, 348/581, 358/597.
        //! The walk by one rope path per wave (256 blocks per XCD) takes 32 for any number: 10^6 points
        //! 452 us without, 438 with them.
        unsigned int m_tail_groups = 32;
        unsigned int m_tail_split = 2;
        bool m_tail_set = false;        //!< by setTailSplit: kept for any number of queries
        static constexpr unsigned int kAllSplit = 7u << 14, kAllSplitGroups = 64, kHalfSplit = 3u << 16, kTailGroups = 16;

    public:
        //! Leaves per bucket of the wave variant (1..64); takes effect at the next compression.
        void setBucketSize(unsigned int b)
            {
            if (b < 1 || b > 64) throw std::runtime_error("bucket size must be in [1, 64]");
            if (b != m_bucket) m_replay = false;
            m_bucket = b;
            }
        unsigned int getBucketSize() const { return m_bucket; }

        //! Tail split of launches without teams (teamSize: more than 65,536 counts, 49,152 rows): per XCD, the last `groups` groups of
        //! 256 queries run as `split` blocks of 256/split queries each, so the waves that start last are
        //! shorter (groups = 0: one block per group).  Kept for any number of queries from then on; before,
        //! the front walk splits by the number of queries and getTailGroups() is what the other walk takes.
        void setTailSplit(unsigned int groups, unsigned int split)
            {
            if (split != 1 && split != 2 && split != 4) throw std::invalid_argument("the tail split must be 1, 2 or 4");
            m_tail_groups = groups;
            m_tail_split = split;
            m_tail_set = true;
            }
        unsigned int getTailGroups() const { return m_tail_groups; }
        unsigned int getTailSplit() const { return m_tail_split; }
    };

template<class TransformOpT>
void LBVHTraverser::compress(const LaunchParameters& params, const LBVH& lbvh, const TransformOpT& transform)
    {
    const unsigned int block = checkParameter(params);
    const unsigned int nodes = lbvh.getNNodes();
    if (nodes > m_data.size()) shared_array<int4>(nodes, MemoryKind::Device).swap(m_data);
    m_root = lbvh.getRoot();
    const ConstLBVHData tree = lbvh.data();
    const LBVHCompressedData c = data();
    // the Wave variant walks its own exact bucket records (and the root box they also write):
    // the quantized records are made for the other variants only
    if (m_variant != TraversalVariant::Wave)
        {
        hipLaunchKernelGGL(gpu::kernel::lbvh_compress<TransformOpT>, dim3(div_up(nodes, block)), dim3(block), 0, params.stream,
                           c, transform, tree, lbvh.getNInternal(), nodes);
        check_launch("lbvh_compress");
        }
    if (m_variant != TraversalVariant::Quantized)
        {
        if (2 * static_cast<size_t>(nodes) > m_float.size()) shared_array<float4>(2 * static_cast<size_t>(nodes), MemoryKind::Device).swap(m_float);
        if (m_variant == TraversalVariant::Wave)
            hipLaunchKernelGGL((gpu::kernel::lbvh_bucket_records<false, true>), dim3(div_up(nodes, block)), dim3(block), 0,
                               params.stream, m_float.get(), c, tree, lbvh.getNInternal(), nodes, m_bucket);
        else if (m_variant == TraversalVariant::WaveQuantized)
            hipLaunchKernelGGL(gpu::kernel::lbvh_bucket_records<true>, dim3(div_up(nodes, block)), dim3(block), 0, params.stream,
                               m_float.get(), c, tree, lbvh.getNInternal(), nodes, m_bucket);
        else if (m_variant == TraversalVariant::FloatRope)
            hipLaunchKernelGGL(gpu::kernel::lbvh_float_ropes<true>, dim3(div_up(nodes, block)), dim3(block), 0, params.stream,
                               m_float.get(), c, tree, nodes);
        else
            hipLaunchKernelGGL(gpu::kernel::lbvh_float_ropes<false>, dim3(div_up(nodes, block)), dim3(block), 0, params.stream,
                               m_float.get(), c, tree, nodes);
        check_launch("lbvh_float_ropes");
        }
    }

template<class QueryOpT, class OutputOpT, class TranslateOpT, class TransformOpT>
void LBVHTraverser::traverse(const LaunchParameters& params, const LBVH& lbvh, const QueryOpT& query,
                             const OutputOpT& out, const TranslateOpT& images, const TransformOpT& transform)
    {
    constexpr bool placed = gpu::kernel::wave::places_rows<OutputOpT>::value;
    if constexpr (placed)
        if (m_variant != TraversalVariant::Wave && m_variant != TraversalVariant::WaveQuantized)
            throw std::invalid_argument("PlacedRowPairOp: rows are placed by the wave traversal variants only");
    if (lbvh.getN() == 0) return;
    if (query.size() == 0 || images.size() == 0) return;
    if (images.size() > 32) throw image_limit_error();
    (void)checkParameter(params);
    if (!m_replay) compress(params, lbvh, transform);

    const unsigned int* order = (m_order && m_order_n == query.size()) ? m_order : nullptr;
    if (m_variant == TraversalVariant::Wave || m_variant == TraversalVariant::WaveQuantized)
        {
        traverse_wave(params, lbvh, query, out, images, transform, order);
        }
    else
        {
        // refused above: placed rows
        if constexpr (!placed)
            if (!traverse_rope_fronts(params, lbvh, query, out, images, order)) traverse_rope_paths(params, lbvh, query, out, images, order);
        }
    check_launch("lbvh_traverse");
    }

} // end namespace neighbor

#endif // NEIGHBOR_LBVH_TRAVERSER_H_
