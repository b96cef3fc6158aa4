// A CPU model of workgroups for tests: kernels compiled as C++ run with their wavefronts
// in an order that the test chooses.  Lanes are fibers; a barrier waits for the lanes that
// have not returned, a shuffle for those of its width (as on the GPU, where a wave's end
// also releases the barriers that it has not reached).  A workgroup may wait for another
// one between two of its waves.  Every workgroup that does so has a thread of its own, so
// that its LDS (thread-local statics, which keep what the last workgroup left) is its own.
#pragma once
#include <ucontext.h>

#include <cmath>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <future>
#include <memory>
#include <thread>
#include <vector>

#define __global__
#define __device__
#define __host__
#define __forceinline__ inline
#define __launch_bounds__(...)
#define __shared__ static thread_local

typedef void* hipStream_t;
typedef int hipError_t;
constexpr hipError_t hipSuccess = 0;
inline const char* hipGetErrorString(hipError_t) { return ""; }
using std::isfinite;

struct dim3 {
    unsigned x, y, z;
    dim3(unsigned a = 1, unsigned b = 1, unsigned c = 1) : x(a), y(b), z(c) {}
};

namespace model {

constexpr int kWave = 64, kBarrier = 1;
inline thread_local dim3 block_idx, thread_idx, grid_dim, block_dim;

struct Workgroup {
    struct Lane {
        ucontext_t ctx;
        std::vector<char> stack = std::vector<char>(32 << 10);
        int wait = 0;   // 0 running, kBarrier, or the width of the shuffle it is at
        bool ended = false;
    };
    std::vector<Lane> lanes;
    std::vector<double> exchange;
    ucontext_t scheduler;
    int at = 0;
    const std::function<void()>* kernel = nullptr;
};
inline thread_local Workgroup* current = nullptr;

inline void wait(int what) {
    Workgroup& g = *current;
    g.lanes[g.at].wait = what;
    swapcontext(&g.lanes[g.at].ctx, &g.scheduler);
}

inline void enter() {
    (*current->kernel)();
    Workgroup& g = *current;
    g.lanes[g.at].ended = true;
    swapcontext(&g.lanes[g.at].ctx, &g.scheduler);
}

// one workgroup; its waves start in the order of `waves`, and before(w) is called as wave w starts
inline void run(dim3 block, dim3 index, dim3 grid, unsigned threads, const std::function<void()>& kernel,
                const std::vector<int>& waves, const std::function<void(int)>& before) {
    Workgroup g;
    current = &g;
    g.lanes.resize(threads);
    g.exchange.resize(threads);
    g.kernel = &kernel;
    block_idx = index;
    block_dim = block;
    grid_dim = grid;
    auto step = [&](unsigned t) {   // runs lane t until it waits or ends
        g.at = (int)t;
        thread_idx = dim3(t, 0, 0);
        swapcontext(&g.scheduler, &g.lanes[t].ctx);
    };
    std::vector<bool> started(threads / kWave, false);
    // runs wave w until all its lanes wait at a barrier or have ended; a shuffle goes on when the
    // lanes of its group that have not ended are all there
    auto settle = [&](int w) {
        const unsigned t0 = (unsigned)w * kWave, t1 = t0 + kWave;
        for (bool again = true; again;) {
            again = false;
            for (unsigned t = t0; t < t1; t++)
                if (!g.lanes[t].ended && g.lanes[t].wait == 0) step(t);
            for (unsigned t = t0; t < t1; t++) {
                const unsigned width = (unsigned)g.lanes[t].wait;
                if (g.lanes[t].ended || width <= kBarrier || t % width) continue;
                bool all = true;
                for (unsigned u = t; u < t + width; u++) all = all && (g.lanes[u].ended || g.lanes[u].wait == (int)width);
                if (!all) continue;
                for (unsigned u = t; u < t + width; u++) g.lanes[u].wait = 0;
                again = true;
            }
        }
    };
    for (int w : waves) {
        before(w);
        for (unsigned t = w * kWave; t < (unsigned)(w + 1) * kWave; t++) {
            getcontext(&g.lanes[t].ctx);
            g.lanes[t].ctx.uc_stack.ss_sp = g.lanes[t].stack.data();
            g.lanes[t].ctx.uc_stack.ss_size = g.lanes[t].stack.size();
            g.lanes[t].ctx.uc_link = nullptr;
            makecontext(&g.lanes[t].ctx, enter, 0);
        }
        settle(w);
    }
    for (bool left = true; left;) {   // every wave waits at a barrier or has ended: on to the next barrier
        left = false;
        for (auto& l : g.lanes)
            if (!l.ended) {
                l.wait = 0;
                left = true;
            }
        if (left)
            for (int w : waves) settle(w);
    }
    current = nullptr;
}

// Launches run workgroup by workgroup, unless `late` names one of them (its launch counted from
// the last reset, and its index): that one's wave `late_wave` then starts after all others
// of the workgroup wait at their first barrier and workgroup (0, y) has ended.
struct Plan {
    int launch = -1;
    dim3 late;
    int late_wave = 0;
    int count = 0;
};
inline Plan plan;

inline void launch(dim3 grid, dim3 block, const std::function<void()>& kernel) {
    const int waves = (int)block.x / kWave;
    std::vector<int> order(waves);
    for (int w = 0; w < waves; w++) order[w] = w;
    const bool planned = plan.count++ == plan.launch;
    for (unsigned y = 0; y < grid.y; y++) {
        if (!planned || y != plan.late.y) {
            for (unsigned x = 0; x < grid.x; x++)
                run(block, dim3(x, y), grid, block.x, kernel, order, [](int) {});
            continue;
        }
        std::promise<void> others_wait, first_ended;
        std::thread first([&] {
            others_wait.get_future().wait();
            run(block, dim3(0, y), grid, block.x, kernel, order, [](int) {});
            first_ended.set_value();
        });
        std::vector<int> last;
        for (int w : order)
            if (w != plan.late_wave) last.push_back(w);
        last.push_back(plan.late_wave);
        run(block, dim3(plan.late.x, y), grid, block.x, kernel, last, [&](int w) {
            if (w != plan.late_wave) return;
            others_wait.set_value();
            first_ended.get_future().wait();
        });
        first.join();
        for (unsigned x = 1; x < grid.x; x++)
            if (x != plan.late.x) run(block, dim3(x, y), grid, block.x, kernel, order, [](int) {});
    }
}

// launches between the begin and the end of a capture
typedef std::vector<std::function<void()>> Graph;
inline Graph* recording = nullptr;

}  // namespace model

typedef model::Graph *hipGraph_t, *hipGraphExec_t;
constexpr hipError_t hipErrorNotReady = 600;
constexpr int hipStreamCaptureModeThreadLocal = 1, hipHostMallocCoherent = 1, hipHostMallocMapped = 2;
constexpr int hipMemcpyHostToDevice = 1;
#define __HIP_MEMORY_SCOPE_SYSTEM 0
#define __hip_atomic_store(p, v, order, scope) __atomic_store_n(p, v, order)
inline hipError_t hipMalloc(void** p, size_t n) { return (*p = aligned_alloc(256, (n + 255) / 256 * 256)) ? 0 : 2; }
inline hipError_t hipHostMalloc(void** p, size_t n, int) { return hipMalloc(p, n); }
inline hipError_t hipMemcpyAsync(void* to, const void* from, size_t n, int, hipStream_t) { return memcpy(to, from, n), 0; }
inline hipError_t hipFree(void* p) { return free(p), 0; }
inline hipError_t hipGetLastError() { return 0; }
inline hipError_t hipStreamQuery(hipStream_t) { return 0; }
inline hipError_t hipStreamBeginCapture(hipStream_t, int) { return model::recording = new model::Graph, 0; }
inline hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
    *g = model::recording;
    model::recording = nullptr;
    return 0;
}
inline hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t g, void*, void*, size_t) {
    return *e = new model::Graph(*g), 0;
}
inline hipError_t hipGraphDestroy(hipGraph_t g) { return delete g, 0; }
inline hipError_t hipGraphExecDestroy(hipGraphExec_t g) { return delete g, 0; }
inline hipError_t hipGraphLaunch(hipGraphExec_t g, hipStream_t) {
    for (auto& f : *g) f();
    return 0;
}
struct double2 {
    double x, y;
};
inline int min(int a, int b) { return a < b ? a : b; }
inline void __threadfence_system() {}

#define blockIdx model::block_idx
#define threadIdx model::thread_idx
#define gridDim model::grid_dim
#define blockDim model::block_dim
// arguments are evaluated at the launch, so that a captured one can run later
template <typename F, typename... A>
void launch_kernel(dim3 grid, dim3 block, F kernel, A... args) {
    std::function<void()> f = [=] { kernel(args...); };
    if (model::recording)
        model::recording->push_back([=] { model::launch(grid, block, f); });
    else
        model::launch(grid, block, f);
}
#define hipLaunchKernelGGL(kernel, grid, block, lds, stream, ...) \
    launch_kernel(grid, block, [](auto... a) { kernel(a...); }, __VA_ARGS__)

inline void __syncthreads() { model::wait(model::kBarrier); }

template <typename T>
T shuffle(T v, int to, int width) {
    static_assert(sizeof(T) <= sizeof(double), "one exchange slot per lane");
    model::Workgroup& g = *model::current;
    const int t = g.at;
    g.exchange[t] = v;
    model::wait(width);   // the others' values are there when this wave comes round again
    const T r = (T)g.exchange[to];
    model::wait(width);
    return r;
}

template <typename T>
T __shfl_xor(T v, int mask, int width) {
    const int t = model::current->at;
    return shuffle(v, t - t % width + ((t % width) ^ mask), width);
}

template <typename T>
T __shfl_down(T v, int by, int width) {
    const int t = model::current->at;
    return shuffle(v, t % width + by < width ? t + by : t, width);
}
