// custom_output.hip -- traversals with output ops of a program's own, run by
// tests/test_gpu_custom_output.py.
//
// Usage: custom_output.bin MODE in out
//   in : n, nq, variant, bucket, order (0 none, 1 the tree's, 2 given), nimg, exact (u32 each), the
//        box side (float), points (n float3), spheres (nq float4), images (nimg double3), order (nq u32)
//        and, mode half, the row starts (nq + 1 u64)
//   out: per query, sums, set-ups and finalizes (mode log); counts of the hits kept, then the pairs
//        (mode half)
#include "neighbor/neighbor.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <stdexcept>
#include <string>
#include <vector>

using namespace neighbor;

// Counts its own calls; setup clears the query's sum, process adds to it in memory.
struct LogOp
    {
    struct ThreadData
        {
        unsigned int idx;
        };
    template<class QueryDataT>
    __device__ ThreadData setup(const unsigned int idx, const QueryDataT&) const
        {
        atomicAdd(&setups[idx], 1u);
        sums[idx] = 0u;
        return ThreadData{idx};
        }
    __device__ void process(ThreadData& t, const int primitive, const unsigned int image) const
        {
        sums[t.idx] += 31u * static_cast<unsigned int>(primitive) + 7u * image + 1u;
        }
    __device__ void finalize(const ThreadData& t) const { atomicAdd(&finals[t.idx], 1u); }

    unsigned int* sums;
    unsigned int* setups;
    unsigned int* finals;
    };

// Pair rows of the hits whose primitive is not below the query's index.
struct HalfPairsOp : public PairListOp
    {
    using PairListOp::PairListOp;
    __device__ void process(ThreadData& t, const int primitive, const unsigned int image) const
        {
        if (static_cast<unsigned int>(primitive) >= t.idx) PairListOp::process(t, primitive, image);
        }
    };

namespace
{
template<class T>
T* upload(const std::vector<T>& v)
    {
    T* p = nullptr;
    NEIGHBOR_HIP_CHECK(hipMalloc(&p, std::max<size_t>(v.size(), 1) * sizeof(T)));
    NEIGHBOR_HIP_CHECK(hipMemcpy(p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
    return p;
    }
template<class T>
void download(FILE* f, const T* p, size_t n)
    {
    std::vector<T> v(n);
    NEIGHBOR_HIP_CHECK(hipMemcpy(v.data(), p, n * sizeof(T), hipMemcpyDeviceToHost));
    if (std::fwrite(v.data(), sizeof(T), n, f) != n) throw std::runtime_error("short write");
    }
template<class T>
std::vector<T> take(FILE* f, size_t n)
    {
    std::vector<T> v(n);
    if (n && std::fread(v.data(), sizeof(T), n, f) != n) throw std::runtime_error("short read");
    return v;
    }

int run(const std::string& mode, const char* in, const char* out)
    {
    FILE* f = std::fopen(in, "rb");
    if (!f) throw std::runtime_error("no input");
    const std::vector<unsigned int> head = take<unsigned int>(f, 7);
    const unsigned int n = head[0], nq = head[1], nimg = head[5];
    const float L = take<float>(f, 1)[0];
    const std::vector<float3> points = take<float3>(f, n);
    const std::vector<float4> spheres = take<float4>(f, nq);
    const std::vector<double3> images = take<double3>(f, nimg);
    const std::vector<unsigned int> order = take<unsigned int>(f, head[4] == 2u ? nq : 0u);
    const std::vector<unsigned long long> starts = take<unsigned long long>(f, mode == "half" ? nq + 1u : 0u);
    std::fclose(f);
    std::vector<float3> images_f;
    for (const double3& t : images)
        images_f.push_back(make_float3(static_cast<float>(t.x), static_cast<float>(t.y), static_cast<float>(t.z)));
    const float3* d_points = upload(points);
    const float4* d_spheres = upload(spheres);
    const double3* d_images = upload(images);
    const float3* d_images_f = upload(images_f);
    const unsigned int* d_order = upload(order);

    LBVH lbvh;
    lbvh.build(PointInsertOp(d_points, n), make_float3(0.f, 0.f, 0.f), make_float3(L, L, L));
    LBVHTraverser trav;
    trav.setVariant(static_cast<TraversalVariant>(head[2]));
    trav.setBucketSize(head[3]);
    trav.setup(lbvh);
    if (head[4]) trav.setQueryOrder(head[4] == 1u ? lbvh.getPrimitives().get() : d_order, nq);
    const auto traverse = [&](const auto& op) {
        if (head[6])
            trav.traverse(lbvh, ExactSphereQueryOp(d_spheres, nq, d_points), op, ImageListOp<double3>(d_images, nimg));
        else
            trav.traverse(lbvh, SphereQueryOp(d_spheres, nq), op, ImageListOp<float3>(d_images_f, nimg));
        NEIGHBOR_HIP_CHECK(hipDeviceSynchronize());
    };

    FILE* o = std::fopen(out, "wb");
    if (!o) throw std::runtime_error("no output");
    if (mode == "log")
        {
        const std::vector<unsigned int> zero(nq, 0u);
        const LogOp op{upload(zero), upload(zero), upload(zero)};
        traverse(op);
        download(o, op.sums, nq);
        download(o, op.setups, nq);
        download(o, op.finals, nq);
        }
    else if (mode == "half")
        {
        const size_t total = starts[nq];
        const HalfPairsOp op(upload(starts), upload(std::vector<unsigned int>(total, ~0u)), nullptr,
                             upload(std::vector<unsigned int>(nq, 0u)), total);
        traverse(op);
        download(o, op.nneigh, nq);
        download(o, op.neigh, total);
        }
    else throw std::runtime_error("unknown mode");
    std::fclose(o);
    return 0;
    }
} // end anonymous namespace

int main(int argc, char** argv)
    {
    if (argc != 4) return 2;
    try
        {
        return run(argv[1], argv[2], argv[3]);
        }
    catch (const std::exception& e)
        {
        std::fprintf(stderr, "%s\n", e.what());
        return 1;
        }
    }
