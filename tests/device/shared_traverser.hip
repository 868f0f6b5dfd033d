// shared_traverser.hip -- one traverser's unordered queries (sorted in its own workspaces) from several
// host threads, run by tests/test_gpu_shared_traverser.py.
//
// Usage: shared_traverser.bin MODE    prints OK and exits 0 on success
//   threads  two host threads, each on its per-thread stream (one handle value for both)
//   memory   the workspaces' allocations fail, one after the other
//   capture  beside another thread's capture in global mode
#include <hip/hip_runtime.h>

#include <atomic>

// The library's allocations, of which the one that counts the number down to zero fails.
static std::atomic<int> g_fails_in{-1};
template<class T>
static hipError_t counted_malloc(T** p, const size_t size)
    {
    if (g_fails_in > 0 && --g_fails_in == 0) return hipErrorOutOfMemory;
    return hipMalloc(p, size);
    }
#define hipMalloc(p, size) counted_malloc(p, size)
#include "neighbor/neighbor.h"

#include <cmath>
#include <cstdio>
#include <exception>
#include <memory>
#include <random>
#include <stdexcept>
#include <string>
#include <thread>
#include <vector>

using namespace neighbor;

namespace
{
template<class T>
std::shared_ptr<T> device(size_t n)
    {
    T* p = nullptr;
    NEIGHBOR_HIP_CHECK(hipMalloc(&p, n * sizeof(T)));
    return std::shared_ptr<T>(p, [](T* q) { (void)hipFree(q); });
    }

//! Points in a cube and as many queries, in random order; their counts in the tree's order.
struct System
    {
    unsigned int n;
    std::shared_ptr<float3> points;
    std::shared_ptr<float4> spheres;
    LBVH lbvh;
    std::vector<unsigned int> counts;

    System(const unsigned int n_, const unsigned int seed) : n(n_)
        {
        const float L = std::cbrt(static_cast<float>(n) / 0.85f);
        std::mt19937 gen(seed);
        std::uniform_real_distribution<float> u(0.0f, L);
        std::vector<float3> p(n);
        std::vector<float4> s(n);
        for (unsigned int i = 0; i < n; ++i)
            {
            p[i] = make_float3(u(gen), u(gen), u(gen));
            s[i] = make_float4(p[i].x, p[i].y, p[i].z, 1.3f);
            }
        points = device<float3>(n);
        spheres = device<float4>(n);
        NEIGHBOR_HIP_CHECK(hipMemcpy(points.get(), p.data(), n * sizeof(float3), hipMemcpyHostToDevice));
        NEIGHBOR_HIP_CHECK(hipMemcpy(spheres.get(), s.data(), n * sizeof(float4), hipMemcpyHostToDevice));
        lbvh.build(PointInsertOp(points.get(), n), make_float3(0.f, 0.f, 0.f), make_float3(L, L, L));
        LBVHTraverser trav;
        trav.setup(lbvh);
        trav.setQueryOrder(lbvh.getPrimitives().get(), n);
        const std::shared_ptr<unsigned int> c = device<unsigned int>(n);
        trav.traverse(lbvh, SphereQueryOp(spheres.get(), n), CountNeighborsOp(c.get()));
        counts.resize(n);
        NEIGHBOR_HIP_CHECK(hipMemcpy(counts.data(), c.get(), n * sizeof(unsigned int), hipMemcpyDeviceToHost));
        }
    };

//! Counts of the first nq queries on a stream, with no order given.
void count(const System& sys, LBVHTraverser& trav, unsigned int* out, const unsigned int nq, const stream_t stream)
    {
    trav.traverse(stream, sys.lbvh, SphereQueryOp(sys.spheres.get(), nq), CountNeighborsOp(out));
    }
void check(const System& sys, const unsigned int* out, const unsigned int nq, const std::string& what)
    {
    std::vector<unsigned int> got(nq);
    NEIGHBOR_HIP_CHECK(hipMemcpy(got.data(), out, nq * sizeof(unsigned int), hipMemcpyDeviceToHost));
    for (unsigned int i = 0; i < nq; ++i)
        if (got[i] != sys.counts[i]) throw std::runtime_error(what + ": count " + std::to_string(i) + " is wrong");
    }

//! Runs f in a thread and hands on what it throws.
template<class F>
class Thread
    {
    public:
        explicit Thread(F f) : m_thread([this, f] {
            try { f(); } catch (...) { m_error = std::current_exception(); }
        }) {}
        void join()
            {
            m_thread.join();
            if (m_error) std::rethrow_exception(m_error);
            }
    private:
        std::exception_ptr m_error;
        std::thread m_thread;
    };

//! Sizes on both sides of the sorts' limits (one launch, short tiles, long tiles), in turn.
const unsigned int kSizes[] = {2000, 20000, 400000, 30000, 16384, 16385, 393216, 393217};

void threads()
    {
    const System sys(420000, 3);
    LBVHTraverser trav;
    trav.setup(sys.lbvh);
    NEIGHBOR_HIP_CHECK(hipDeviceSynchronize());
    const auto work = [&](const unsigned int first) {
        std::vector<std::shared_ptr<unsigned int>> outs;
        std::vector<unsigned int> sizes;
        for (unsigned int k = 0; k < 24; ++k)
            {
            sizes.push_back(kSizes[(first + k) % 8u]);
            outs.push_back(device<unsigned int>(sizes.back()));
            count(sys, trav, outs.back().get(), sizes.back(), hipStreamPerThread);
            }
        NEIGHBOR_HIP_CHECK(hipStreamSynchronize(hipStreamPerThread));
        for (unsigned int k = 0; k < outs.size(); ++k) check(sys, outs[k].get(), sizes[k], "thread " + std::to_string(first));
    };
    const auto a = [&] { work(0); };
    const auto b = [&] { work(3); };
    Thread<decltype(a)> ta(a);
    Thread<decltype(b)> tb(b);
    ta.join();
    tb.join();
    }

void memory()
    {
    const System sys(30000, 4);
    const std::shared_ptr<unsigned int> out = device<unsigned int>(sys.n);
    const unsigned int sizes[] = {3000, 20000, 30000};
    for (int fails_in = 1; fails_in <= 12; ++fails_in)
        {
        LBVHTraverser trav;
        trav.setup(sys.lbvh);
        g_fails_in = fails_in;
        for (unsigned int k = 0; k < 9; ++k)
            {
            NEIGHBOR_HIP_CHECK(hipMemset(out.get(), 0xff, sys.n * sizeof(unsigned int)));
            count(sys, trav, out.get(), sizes[k % 3u], 0);
            check(sys, out.get(), sizes[k % 3u], "allocation " + std::to_string(fails_in) + " fails, call " + std::to_string(k));
            }
        g_fails_in = -1;
        }
    }

__global__ void mark(unsigned int* p)
    {
    *p = 7u;
    }

void capture()
    {
    const System sys(30000, 5);
    LBVHTraverser trav;
    trav.setup(sys.lbvh);
    const std::shared_ptr<unsigned int> out = device<unsigned int>(sys.n), word = device<unsigned int>(1);
    NEIGHBOR_HIP_CHECK(hipMemset(word.get(), 0, sizeof(unsigned int)));
    hipStream_t captured, other;
    NEIGHBOR_HIP_CHECK(hipStreamCreateWithFlags(&captured, hipStreamNonBlocking));
    NEIGHBOR_HIP_CHECK(hipStreamCreateWithFlags(&other, hipStreamNonBlocking));
    NEIGHBOR_HIP_CHECK(hipDeviceSynchronize());
    NEIGHBOR_HIP_CHECK(hipStreamBeginCapture(captured, hipStreamCaptureModeGlobal));
    std::string error;
    try
        {
        // first uses, growth and a size that fits, beside the capture
        const auto work = [&] {
            for (const unsigned int nq : {3000u, 20000u, 30000u, 10000u}) count(sys, trav, out.get(), nq, other);
        };
        Thread<decltype(work)> t(work);
        t.join();
        }
    catch (const std::exception& e) { error = e.what(); }
    hipLaunchKernelGGL(mark, dim3(1), dim3(1), 0, captured, word.get());
    hipGraph_t graph = nullptr;
    const hipError_t ended = hipStreamEndCapture(captured, &graph);
    if (!error.empty()) throw std::runtime_error("traversal beside a capture: " + error);
    NEIGHBOR_HIP_CHECK(ended);
    hipGraphExec_t exec;
    NEIGHBOR_HIP_CHECK(hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0));
    NEIGHBOR_HIP_CHECK(hipGraphLaunch(exec, captured));
    NEIGHBOR_HIP_CHECK(hipDeviceSynchronize());
    unsigned int got = 0;
    NEIGHBOR_HIP_CHECK(hipMemcpy(&got, word.get(), sizeof(got), hipMemcpyDeviceToHost));
    if (got != 7u) throw std::runtime_error("the captured kernel did not run");
    check(sys, out.get(), 30000, "beside a capture");
    NEIGHBOR_HIP_CHECK(hipGraphExecDestroy(exec));
    NEIGHBOR_HIP_CHECK(hipGraphDestroy(graph));
    NEIGHBOR_HIP_CHECK(hipStreamDestroy(captured));
    NEIGHBOR_HIP_CHECK(hipStreamDestroy(other));
    }
} // end anonymous namespace

int main(int argc, char** argv)
    {
    const std::string mode = argc == 2 ? argv[1] : "";
    try
        {
        if (mode == "threads") threads();
        else if (mode == "memory") memory();
        else if (mode == "capture") capture();
        else return 2;
        }
    catch (const std::exception& e)
        {
        std::fprintf(stderr, "%s\n", e.what());
        return 1;
        }
    std::printf("OK\n");
    return 0;
    }
