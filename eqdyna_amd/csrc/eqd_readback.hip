// Readback of the evolved state (eqd_get) and of other large results: pack
// kernels that write the reference's layouts, and the pinned staging slots
// they go through (eqd_readback.h).
#include "eqd_readback.h"

#include <omp.h>
#include <unistd.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

namespace eqd {
namespace {

__device__ __forceinline__ double bf16_value(uint16_t h) { return (double)__uint_as_float((uint32_t)h << 16); }

// One thread per output value, so a wavefront writes 512 consecutive bytes
// over the host link and reads three short runs of a node block.  Bound by
// that link: 3.55 M nodes (85 MB) leave the device at 55 GB/s, the rate of a
// copy between device and pinned memory.  A device-to-host copy of the
// blocked arrays followed by a serial transposition on the host took 38 ms
// for these nodes' velocities in the FP32 bulk mode; through this kernel and
// the staging slots it takes 4.
// FP32 bulk mode: the FP32 velocity, the displacement hi + lo, and for split
// nodes the fault's FP64 state.
template <bool kF32>
__global__ void __launch_bounds__(256) pack_nodes_kernel(NodeState N, FaultState F, int vel, int64_t first,
                                                         int64_t count, double *__restrict__ out)
{
    const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= 3 * count) return;
    const int64_t node = N.at ? N.at[first + j / 3] : first + j / 3;
    const int k = (int)(j % 3);
    const int64_t at = blk_at<3>(node, k);
    double x;
    if constexpr (kF32) {
        const int ps = N.pair_slot[node];
        if (ps >= 0) x = (vel ? F.sv : F.su)[((ps & 1) * 3 + k) * F.ld + (ps >> 1)];
        else if (vel) x = (double)N.vel32[at];
        else x = (double)N.dhi[at] + bf16_value(N.dlo[at]);
    } else {
        x = (vel ? N.vel : N.disp)[at];
    }
    out[j] = x;
}

// fric from [slot][pair] to the reference's [pair][slot]: a block transposes
// 64 pairs in LDS (rows of 65 values: both passes hit all banks), reading and
// writing whole lines.  100 slots of 24,090 pairs: 5.5 -> 1.2 ms on the host
// side of the call, again bound by the host link and the caller's pages.
constexpr int kPackPairs = 64, kFricSlots = 100;
__global__ void __launch_bounds__(256) pack_fric_kernel(const double *__restrict__ fric, int64_t ld, int64_t first,
                                                        int64_t count, double *__restrict__ out)
{
    __shared__ double tile[kFricSlots * (kPackPairs + 1)];
    const int64_t p0 = (int64_t)blockIdx.x * kPackPairs;
    const int np = (int)(count - p0 < kPackPairs ? count - p0 : kPackPairs);
    for (int j = threadIdx.x; j < kFricSlots * kPackPairs; j += blockDim.x) {
        const int k = j / kPackPairs, i = j % kPackPairs;
        if (i < np) tile[k * (kPackPairs + 1) + i] = fric[k * ld + first + p0 + i];
    }
    __syncthreads();
    for (int j = threadIdx.x; j < np * kFricSlots; j += blockDim.x) {
        const int i = j / kFricSlots, k = j % kFricSlots;
        out[p0 * kFricSlots + j] = tile[k * (kPackPairs + 1) + i];
    }
}

// ---------------- staging slots

// From a slot into the caller's memory, which is often not yet backed by
// pages: a few threads share the page faults (83 MB into new memory: 19 ms
// with one thread, 5.4 with four, 3.5 with eight, 2.5 with sixteen).  They
// belong to the lease and sleep between calls.  An OpenMP team spins on for
// 200 ms after its last loop and slows what the caller does next (the inputs
// and the commit of the next scenario, 161,500 elements: 202 -> 229 ms); threads
// made in each call cost it 0.05 to 0.14 ms, waking these 0.02 (8 MB: 0.36, 0.25;
// an OpenMP team still spinning 0.23).
class Crew {
   public:
    Crew() : pid_(getpid())
    {
        try {
            for (int k = std::min(8, omp_get_max_threads()) - 1; k > 0; k--) helpers_.emplace_back([this] { help(); });
        } catch (...) {  // as many as there are
        }
    }
    ~Crew()
    {
        {
            std::lock_guard<std::mutex> lk(mu_);
            stop_ = true;
        }
        wake_.notify_all();
        for (std::thread &t : helpers_) t.join();
    }
    bool here() const { return pid_ == getpid(); }  // not in a child of the process that made it
    // a call begins: the helpers wake while its first slot is being filled
    void begin()
    {
        {
            std::lock_guard<std::mutex> lk(mu_);
            active_.store(true, std::memory_order_relaxed);
        }
        wake_.notify_all();
    }
    void end() { active_.store(false, std::memory_order_relaxed); }
    // The caller copies too and waits for pieces, not for helpers: one that
    // wakes late, or not at all, costs nothing.
    void copy(char *dst, const char *src, size_t bytes)
    {
        if (bytes <= kCrewMin) {
            memcpy(dst, src, bytes);
            return;
        }
        const uint64_t pieces = (bytes + kPiece - 1) / kPiece, job = ++jobs_ << 32;
        dst_ = dst;
        src_ = src;
        bytes_ = bytes;
        done_.store(0, std::memory_order_relaxed);
        next_.store(job, std::memory_order_release);
        limit_.store(job | pieces, std::memory_order_release);
        while (piece()) {}
        for (int k = 0; done_.load(std::memory_order_acquire) != pieces; k++)
            if (k >= 100) std::this_thread::yield();
    }
    static constexpr size_t kPiece = (size_t)1 << 20, kCrewMin = 2 * kPiece;

   private:
    const pid_t pid_;
    std::mutex mu_;
    std::condition_variable wake_;
    bool stop_ = false;
    std::atomic<bool> active_{false};
    // the job's number above, the next piece or the number of pieces below
    std::atomic<uint64_t> next_{0}, limit_{0}, done_{0};
    uint64_t jobs_ = 0;
    char *dst_ = nullptr;
    const char *src_ = nullptr;
    size_t bytes_ = 0;
    std::vector<std::thread> helpers_;

    // Copy one piece; false when there is none.  A piece that was taken is of the
    // current job, since a job ends only when all its pieces are copied.
    bool piece()
    {
        uint64_t at = next_.load(std::memory_order_acquire);
        for (;;) {
            const uint64_t end = limit_.load(std::memory_order_acquire);
            if (at >> 32 != end >> 32 || at >= end) return false;
            if (next_.compare_exchange_weak(at, at + 1, std::memory_order_acq_rel, std::memory_order_acquire)) break;
        }
        const size_t b = (size_t)(at & 0xFFFFFFFFu) * kPiece;
        memcpy(dst_ + b, src_ + b, std::min(kPiece, bytes_ - b));
        done_.fetch_add(1, std::memory_order_release);
        return true;
    }
    void help()
    {
        for (;;) {
            for (int k = 0; active_.load(std::memory_order_relaxed); k++) {
                if (piece()) k = 0;
                else if (k >= 100) std::this_thread::yield();
            }
            std::unique_lock<std::mutex> lk(mu_);
            wake_.wait(lk, [this] { return stop_ || active_.load(std::memory_order_relaxed); });
            if (stop_) return;
        }
    }
};

struct Lease {
    void *slot[kStageSlots] = {};
    Crew *crew = nullptr;
    bool busy = false;
};

std::mutex g_mu;
std::condition_variable g_free;
Lease g_lease[kStageLeases];
int64_t g_users = 0;

Lease *take()
{
    std::unique_lock<std::mutex> lk(g_mu);
    for (;;) {
        // one that has slots already, else an empty one
        Lease *best = nullptr;
        for (Lease &l : g_lease)
            if (!l.busy && (!best || (l.slot[0] && !best->slot[0]))) best = &l;
        if (best) {
            best->busy = true;
            return best;
        }
        g_free.wait(lk);
    }
}

void drop(Lease &l)
{
    for (void *&p : l.slot) {
        if (p) (void)hipHostFree(p);
        p = nullptr;
    }
    if (l.crew && l.crew->here()) delete l.crew;
    l.crew = nullptr;
}

void give(Lease *l)
{
    std::lock_guard<std::mutex> lk(g_mu);
    l->busy = false;
    if (g_users == 0) drop(*l);
    g_free.notify_one();
}

}  // namespace

void stage_retain()
{
    std::lock_guard<std::mutex> lk(g_mu);
    g_users++;
}

void stage_release()
{
    std::lock_guard<std::mutex> lk(g_mu);
    if (--g_users > 0) return;
    for (Lease &l : g_lease)
        if (!l.busy) drop(l);
}

hipError_t stage_out(void *out, size_t bytes, size_t unit, hipStream_t s, const StageFill &fill)
{
    if (bytes == 0) return hipSuccess;
    if (unit == 0 || unit > kStageSlot) return hipErrorInvalidValue;
    const size_t step = kStageSlot / unit * unit;
    Lease *l = take();
    if (bytes > Crew::kCrewMin) {
        if (!l->crew) l->crew = new (std::nothrow) Crew();
        if (l->crew) l->crew->begin();
    }
    hipEvent_t ev[kStageSlots] = {};
    hipError_t rc = hipSuccess;
    auto start = [&](size_t first) {  // fill the slot of the piece at `first`
        const int k = (int)(first / step % kStageSlots);
        if (!l->slot[k]) rc = hipHostMalloc(&l->slot[k], kStageSlot, hipHostMallocPortable);
        if (rc == hipSuccess) rc = fill(l->slot[k], first, std::min(step, bytes - first), s);
        if (rc == hipSuccess && bytes > step) {
            if (!ev[k]) rc = hipEventCreateWithFlags(&ev[k], hipEventDisableTiming);
            if (rc == hipSuccess) rc = hipEventRecord(ev[k], s);
        }
    };
    start(0);
    for (size_t b = 0; b < bytes && rc == hipSuccess; b += step) {
        const int k = (int)(b / step % kStageSlots);
        if (b + step < bytes) start(b + step);
        const hipError_t w = bytes > step ? hipEventSynchronize(ev[k]) : hipStreamSynchronize(s);
        if (rc == hipSuccess) rc = w;
        if (rc != hipSuccess) break;
        char *dst = (char *)out + b;
        if (l->crew) l->crew->copy(dst, (const char *)l->slot[k], std::min(step, bytes - b));
        else memcpy(dst, l->slot[k], std::min(step, bytes - b));
    }
    if (l->crew) l->crew->end();
    if (rc != hipSuccess) (void)hipStreamSynchronize(s);  // nothing writes a slot that is given back
    for (hipEvent_t e : ev)
        if (e) (void)hipEventDestroy(e);
    give(l);
    return rc;
}

hipError_t stage_copy(void *out, const void *dev, size_t bytes, hipStream_t s)
{
    return stage_out(out, bytes, 1, s, [dev](void *slot, size_t first, size_t count, hipStream_t st) {
        return hipMemcpyAsync(slot, (const char *)dev + first, count, hipMemcpyDeviceToHost, st);
    });
}

hipError_t launch_pack_nodes(const NodeState &N, const FaultState &F, bool vel, int64_t first, int64_t count,
                             double *out, hipStream_t s)
{
    if (count <= 0) return hipSuccess;
    const int64_t grid = (3 * count + 255) / 256;
    if (grid > 0x7fffffff) return hipErrorInvalidValue;
    if (N.vel32) pack_nodes_kernel<true><<<(unsigned)grid, 256, 0, s>>>(N, F, vel, first, count, out);
    else pack_nodes_kernel<false><<<(unsigned)grid, 256, 0, s>>>(N, F, vel, first, count, out);
    return hipGetLastError();
}

hipError_t launch_pack_fric(const FaultState &F, int64_t first, int64_t count, double *out, hipStream_t s)
{
    if (count <= 0) return hipSuccess;
    const int64_t grid = (count + kPackPairs - 1) / kPackPairs;
    if (grid > 0x7fffffff) return hipErrorInvalidValue;
    pack_fric_kernel<<<(unsigned)grid, 256, 0, s>>>(F.fric, F.ld, first, count, out);
    return hipGetLastError();
}

}  // namespace eqd
