// sse_persist.h -- one persistent, work-queue-driven launch for a whole call.
//
// Walkers are independent Markov chains: Carlo.sweep! of one walker
// (sse.jl:62-68) needs nothing from any other walker.  The per-sweep kernels
// hold every walker of a launch to the pace of the launch's slowest worm
// update; here each walker advances on its own.  The launch has as many
// workgroups (one wave each) as the device holds at the launch's LDS size.
// A workgroup takes the next task from an atomic counter and runs that task's
// sweeps back to back, each the fused diagonal update + vertex list (K1
// phase), worm update (K2 phase) and, once thermalized, measurement (K3 phase,
// accumulated), until the counter passes the task count.  A task is one walker
// and, where the device holds all of a call's walkers, its whole sweep budget.
// With more walkers than that, a walker's budget is cut into up to
// kPersistSegments tasks, all walkers' first ones before any second one: whole
// budgets would end the launch in a last round of workgroups that is nearly
// empty (4096 walkers on 1792 places: 3 rounds for the work of 2.3).
//
// Ownership, and why nothing waits: due[w] counts the sweeps of walker w that
// tasks have handed out and nobody has finished.  A workgroup adds its task's
// sweeps to it.  If it was 0, the walker is this workgroup's: it alone reads and
// writes the walker's DevWalker, slab, spins and accumulator row until it has
// brought due[w] back to 0.  If not, the sweeps are left to the owner, who finds
// them when it takes its own off, and the workgroup takes the next task.  A
// fence on both sides of the hand-over makes one owner's stores visible to the
// next, which may run on another XCD.  No workgroup ever waits for another;
// the only other shared state is the task counter and the slab pool's bump
// pointer (both atomics) and the pool's error/maximum words (atomicOr /
// atomicMax).  Between the phases of one walker the workgroup passes a barrier
// (which orders its own global and LDS accesses), and every global record a
// phase reads was written by vector stores and is read with vector loads, never
// through the scalar cache.  Tasks run largest expected work first (the schedule
// order), so the launch ends with the small ones.
#pragma once
#include "sse_wave.h"

constexpr int kPersistSegments = 16;

// Makes the workgroup's stores visible to the other XCDs: the L2's write-back has to
// be over before the walker is given away.  The fence alone does not ensure that: the
// compiler drops the wait behind buffer_wbl2 where it knows of no other access in
// flight, as it does after a sweep.
__device__ __forceinline__ void persist_release()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// Runs the tasks of a launch: task t is segment t / n_walkers of the budget of
// walker order[t % n_walkers] (budgets[w] sweeps, or n_sweeps when budgets is
// null).  queue[0] is the task counter and due = queue + 1 (segments > 1), all 0
// at launch (persist_reset_kernel).  sweep(w) runs one sweep of walker w.
template <class Sweep>
__device__ __forceinline__ void persist_tasks(int32_t *queue, const int32_t *order, int n_walkers,
                                              const int32_t *budgets, int n_sweeps, int segments,
                                              const Sweep &sweep)
{
    const int lane = threadIdx.x;
    int32_t *due = queue + 1;
    const int total = n_walkers * segments;
    for (;;) {
        int t = 0;
        if (lane == 0)
            t = atomicAdd(queue, 1);
        t = (int)uni((uint32_t)__shfl(t, 0));
        if (t >= total)
            break;
        const int seg = t / n_walkers;
        const int wi = walker_at(order, t - seg * n_walkers);
        const int64_t ns = budgets ? budgets[wi] : n_sweeps;
        // sweeps [ceil(ns seg / segments), ceil(ns (seg + 1) / segments)): the
        // first segments hold the larger shares, a single sweep is in the first
        int todo = (int)((ns * (seg + 1) + segments - 1) / segments - (ns * seg + segments - 1) / segments);
        todo = (int)uni((uint32_t)todo);
        if (todo <= 0)
            continue;
        if (segments > 1) {
            int was = 0;
            if (lane == 0)
                was = atomicAdd(due + wi, todo);
            if (uni((uint32_t)__shfl(was, 0)) != 0u)
                continue;  // its owner runs them
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        }
        while (todo > 0) {
            for (int s = 0; s < todo; ++s)
                if (!sweep(wi))
                    break;
            if (segments == 1)
                break;
            persist_release();
            int left = 0;
            if (lane == 0)
                left = atomicSub(due + wi, todo) - todo;
            todo = (int)uni((uint32_t)__shfl(left, 0));
        }
    }
}

// a walker that stopped (error, retired budget, inactive) ends its task
__device__ __forceinline__ bool persist_stopped(const DevWalker &w)
{
    return uni((uint32_t)(w.error | !w.active | w.retire)) != 0u;
}

// The measurement as a call, with registers to itself: with all three phases inlined
// the work-queue kernels spill more of the other two (31 and 20 vector registers,
// now 9 and 9).  14x10 squares 10.76 -> 10.48 ms, trimers 20.62 -> 20.48 ms, 32x32
// walkers 78 -> 73 ms per sweep.  The diagonal update as a call too: two-site bonds
// the same, but 33.5 instead of 33.2 ms for 4096 16x16 walkers and trimers 2 % slower.
// Arguments are wave-uniform, pointers global.
template <class T>
__device__ __forceinline__ T *arg_global(T *p)
{
    return (T *)(gmem<T> *)uni64((uint64_t)p);
}
template <int NS>  // 0: the two-site kernels' measurement
__device__ __noinline__ void persist_measure(DevWalker *W, const DevModel *models, double *out, double *sum,
                                             double *sumsq, int64_t *count, double *wlf, int wi, int32_t *done)
{
    W = arg_global(W);
    models = arg_global(models);
    out = arg_global(out);
    sum = arg_global(sum);
    sumsq = arg_global(sumsq);
    count = arg_global(count);
    wlf = arg_global(wlf);
    done = arg_global(done);
    wi = (int)uni((uint32_t)wi);
    if constexpr (NS == 0)
        k3_walker(W, models, out, sum, sumsq, count, wlf, wi, 1, done);
    else
        k3n_walker<NS>(W, models, out, sum, sumsq, count, wlf, wi, 1, done);
}

// measure 1 runs the measurement after every thermalized sweep (sse_run), 0
// leaves it out (sse_sweep).
__global__ __launch_bounds__(64, 2) void wave_persist_kernel(DevWalker *W, const DevModel *models,
                                                             DevPool *pool, double *out, double *sum,
                                                             double *sumsq, int64_t *count,
                                                             double *wlf, int32_t *done,
                                                             const int32_t *order, int n_walkers,
                                                             const int32_t *budgets, int n_sweeps,
                                                             int segments, int measure, int lds_bytes,
                                                             int rec_mode, int32_t *queue)
{
    extern __shared__ __align__(16) char lds[];
    persist_tasks(queue, order, n_walkers, budgets, n_sweeps, segments, [&](int wi) __attribute__((always_inline)) {
        if (persist_stopped(W[wi]))
            return false;
        k1_walker(W, models, pool, wi, 3, -1, lds, lds_bytes, 7);
        __syncthreads();
        worm_walker<2>(W, models, pool, wi, 1, lds_bytes, rec_mode, lds);
        __syncthreads();
        if (measure) {
            persist_measure<0>(W, models, out, sum, sumsq, count, wlf, wi, done);
            __syncthreads();
        }
        return true;
    });
}

// The same for bonds of any site count.  1024 walkers on rings of three- and
// four-site bonds: 28.0 -> 22.4 ms (8 sweeps) and 9.4 -> 6.3 ms (10) against stream
// groups, which wait for their slowest worm each sweep.
__global__ __launch_bounds__(64, 2) void waven_persist_kernel(DevWalker *W, const DevModel *models,
                                                              DevPool *pool, double *out, double *sum,
                                                              double *sumsq, int64_t *count,
                                                              double *wlf, int32_t *done,
                                                              const int32_t *order, int n_walkers,
                                                              const int32_t *budgets, int n_sweeps,
                                                              int segments, int measure, int lds_bytes,
                                                              int rec_mode, int32_t *queue)
{
    extern __shared__ __align__(16) char lds[];
    persist_tasks(queue, order, n_walkers, budgets, n_sweeps, segments, [&](int wi) __attribute__((always_inline)) {
        if (persist_stopped(W[wi]))
            return false;
        const int ns = (int)uni((uint32_t)models[W[wi].model].nsb);
#define PERSIST_CALL(K)                                                             \
    k1n_walker_sel<K>(W, models, pool, wi, 3, -1, lds, 7, lds_bytes);               \
    __syncthreads();                                                                \
    worm_walker<K>(W, models, pool, wi, 1, lds_bytes, rec_mode, lds);               \
    __syncthreads();                                                                \
    if (measure)                                                                    \
        persist_measure<K>(W, models, out, sum, sumsq, count, wlf, wi, done);
        SSE_NS_DISPATCH(ns, PERSIST_CALL)
#undef PERSIST_CALL
        __syncthreads();
        return true;
    });
}

__global__ void persist_reset_kernel(int32_t *queue, int n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n)
        queue[i] = 0;
}

// LDS bytes of a persistent launch: the diagonal-update phase's (model tables
// staged) and the worm phase's record size, whichever is larger
static inline size_t persist_lds_bytes(const WaveConfig &c)
{
    return std::max(c.generic ? c.lds_k1n : c.lds_k1, c.lds_k2);
}

// Workgroups the device holds at once at lds bytes per workgroup
static inline int persist_resident(size_t lds, int n_cu)
{
    return (int)lds_walkers(lds) * n_cu;
}

// Segments of a launch: 1 where every walker has a workgroup of its own for the
// whole call, else enough that the walkers advance together.  most is the
// largest budget.
static inline int persist_segments(const WaveConfig &c, int n_walkers, int64_t most, int n_cu)
{
    if (n_walkers <= persist_resident(persist_lds_bytes(c), n_cu) || n_walkers > (1 << 26))
        return 1;
    return (int)std::max<int64_t>(1, std::min<int64_t>(most, kPersistSegments));
}

// queue: n_walkers + 1 words (n_walkers over all of the batch's walkers)
static inline int wave_launch_persist(WaveConfig &c, hipStream_t s, DevWalker *W, const DevModel *M,
                                      DevPool *pool, double *out, double *sum, double *sumsq,
                                      int64_t *count, double *wlf, int32_t *done,
                                      const int32_t *order, int n_walkers, const int32_t *budgets,
                                      int n_sweeps, int segments, int measure, int32_t *queue,
                                      int n_queue, int n_cu)
{
    if (n_walkers <= 0)
        return SSE_OK;
    const size_t lds = persist_lds_bytes(c);
    const int grid = std::min(n_walkers, persist_resident(lds, n_cu));
    const int nq = segments > 1 ? n_queue : 1;
    hipLaunchKernelGGL(persist_reset_kernel, dim3((nq + 255) / 256), dim3(256), 0, s, queue, nq);
    auto kernel = c.generic ? waven_persist_kernel : wave_persist_kernel;
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(64), lds, s, W, M, pool, out, sum, sumsq, count, wlf, done,
                       order, n_walkers, budgets, n_sweeps, segments, measure, (int)lds, c.rec_mode, queue);
    return hipGetLastError() == hipSuccess ? SSE_OK : SSE_ERR_HIP;
}
