// axs_transfer.hip -- bulk transfers between the device arrays and a caller's
// pageable arrays: host threads that (de)interleave, and the chunk pipeline
// that keeps the link to the host and the threads busy together.
//
// A transfer is a list of segments (one device array each).  It is cut into
// chunks that pass through a ring of pinned slots: to the host, a chunk is
// copied into its slot and then unpacked by the threads while the following
// chunks travel; to the device, the threads pack chunks ahead of the copies.
// The pinned memory is the ring (24 MiB at most), whatever the lattice's
// size, where a staging copy of a whole array per field took as long to pin
// as to send.  In ms, a staging copy per array and the runtime's copies / now:
// six arrays of 128^3 up 3.5 / 2.1, back 4.6-6.5 / 2.6; of 256^3 22 / 16 and 24 /
// 18; two of 1000^2 back 1.9 / 0.7 (slots of 1 or 2 MiB, or eight threads: up to
// 20% more; of 8 MiB 2-5% less, but more to pin on a first call).
#include <string.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <memory>
#include <mutex>
#include <optional>
#include <thread>
#include <vector>

#include "axs_internal.hpp"

namespace axs {

// host threads for the bulk work of all contexts, started by the first large
// transfer and ended with the last context that used them
struct HostPool {
    std::mutex job_mu;                     // one job at a time
    std::mutex mu;
    std::condition_variable cv, idle;
    std::vector<std::thread> threads;
    void (*fn)(void *) = nullptr;
    void *arg = nullptr;
    uint64_t gen = 0;
    unsigned running = 0;
    bool stop = false;

    explicit HostPool(unsigned n)
    {
        for (unsigned t = 0; t < n; ++t) {
            try {
                threads.emplace_back([this] { work(); });
            } catch (...) {
                break;                     // fewer threads; none: the caller works alone
            }
        }
    }
    ~HostPool()
    {
        {
            std::lock_guard<std::mutex> lk(mu);
            stop = true;
        }
        cv.notify_all();
        for (auto &t : threads) t.join();
    }
    void work()
    {
        uint64_t seen = 0;
        std::unique_lock<std::mutex> lk(mu);
        for (;;) {
            cv.wait(lk, [&] { return stop || gen != seen; });
            if (stop) return;
            seen = gen;
            lk.unlock();
            fn(arg);
            lk.lock();
            if (--running == 0) idle.notify_all();
        }
    }
    // start f(arg) on every thread; wait() returns when all have finished
    void start(void (*f)(void *), void *a)
    {
        {
            std::lock_guard<std::mutex> lk(mu);
            fn = f;
            arg = a;
            running = (unsigned)threads.size();
            ++gen;
        }
        cv.notify_all();
    }
    void wait()
    {
        std::unique_lock<std::mutex> lk(mu);
        idle.wait(lk, [&] { return running == 0; });
    }
};

static std::mutex g_pool_mu;
static HostPool *g_pool = nullptr;
static int g_pool_users = 0;               // contexts with pool_user set

void release_pool(Context *c)
{
    HostPool *last = nullptr;
    {
        std::lock_guard<std::mutex> lk(g_pool_mu);
        if (c->pool_user && --g_pool_users == 0) {
            last = g_pool;
            g_pool = nullptr;
        }
        c->pool_user = false;
    }
    delete last;
}

// Threads for one job: the shared ones, or, while they are at work for another
// caller (a read-back beside axs_snapshot_end, another context), some of its own
// for as long as it lasts.  p is null where none could be started.
struct PoolLease {
    HostPool *p = nullptr;
    explicit PoolLease(Context *c)
    {
        const unsigned hw = std::thread::hardware_concurrency(), n = hw ? std::min(hw, 12u) : 4u;
        {
            std::lock_guard<std::mutex> lk(g_pool_mu);
            if (!g_pool) g_pool = new (std::nothrow) HostPool(n);
            if (g_pool && !c->pool_user) {
                c->pool_user = true;
                ++g_pool_users;
            }
            p = g_pool;
        }
        if (p && !p->threads.empty()) {
            job = std::unique_lock<std::mutex>(p->job_mu, std::try_to_lock);
            if (!job.owns_lock()) {
                own.reset(new (std::nothrow) HostPool(n));
                p = own.get();
            }
        }
        if (p && p->threads.empty()) p = nullptr;
    }

private:
    std::unique_lock<std::mutex> job;
    std::unique_ptr<HostPool> own;
};

namespace {

// loops shorter than this run on the calling thread (waking the others takes
// as long)
constexpr size_t kForAlone = (size_t)1 << 18;

struct ForJob {
    size_t n, grain;
    void (*fn)(size_t, size_t, void *);
    void *arg;
    std::atomic<size_t> next{0};
};

void for_worker(void *p)
{
    ForJob *j = (ForJob *)p;
    for (;;) {
        const size_t b = j->next.fetch_add(j->grain);
        if (b >= j->n) return;
        j->fn(b, std::min(j->n, b + j->grain), j->arg);
    }
}

}  // namespace

void parallel_for(Context *c, size_t n, void (*fn)(size_t, size_t, void *), void *arg)
{
    if (n < kForAlone) {
        fn(0, n, arg);
        return;
    }
    PoolLease lease(c);
    HostPool *p = lease.p;
    if (!p) {
        fn(0, n, arg);
        return;
    }
    ForJob j;
    j.n = n;
    j.grain = std::max<size_t>((size_t)1 << 14, n / (4 * p->threads.size()));
    j.fn = fn;
    j.arg = arg;
    p->start(for_worker, &j);
    for_worker(&j);
    p->wait();
}

namespace {

// One chunk between a slot and its device array, 16 bytes a work-item and
// round; n16 of them, then the last bytes one by one.  64 groups keep the link
// full (52 GB/s either way at 4 MiB, as 256 do).  A kernel rather than a copy
// command: in many contexts the runtime's copies of a chunk cost 130 us each
// beside their transfer once both directions have been used, whatever the
// host's load (a list of 743 MB 44 ms, against 30 in 64 MiB chunks and 19 now;
// six arrays of 128^3, upload / read-back: 5.5 / 5.5 ms, 2.1 / 2.6 now).  Small
// transfers, a chunk at a time, keep the copy command: 10 to 20 us less.
__global__ void __launch_bounds__(256)
chunk_copy_kernel(const uint4 *__restrict__ src, uint4 *__restrict__ dst, uint32_t n16,
                  uint32_t tail)
{
    // one contiguous eighth per XCD (work-groups are dealt to the eight in
    // turn): each translates the host pages of its own part only
    const uint32_t part = (n16 + 7) / 8, x = blockIdx.x & 7u;
    const uint32_t lo = x * part, hi = lo + part < n16 ? lo + part : n16;
    const uint32_t step = (gridDim.x / 8) * 256u;
    for (uint32_t i = lo + (blockIdx.x >> 3) * 256u + threadIdx.x; i < hi; i += step)
        dst[i] = src[i];
    if (blockIdx.x == 0 && threadIdx.x < tail)
        ((unsigned char *)(dst + n16))[threadIdx.x] =
            ((const unsigned char *)(src + n16))[threadIdx.x];
}

// both ends on 16-byte boundaries (whole arrays, slots, whole slots into them)
hipError_t copy_chunk(Context *c, void *dst, const void *src, size_t bytes)
{
    const uint32_t n16 = (uint32_t)(bytes / 16);
    const uint32_t groups = 8 * std::max(1u, std::min(8u, (n16 + 2047) / 2048));
    hipLaunchKernelGGL(chunk_copy_kernel, dim3(groups), dim3(256), 0, c->stream,
                       (const uint4 *)src, (uint4 *)dst, n16, (uint32_t)(bytes % 16));
    return hipGetLastError();
}

constexpr size_t kSlotBytes = (size_t)4 << 20;
constexpr int kSlots = 6;
constexpr int kSlices = 16;                // pieces of a chunk that threads take
// below this the calling thread works alone through one slot: starting the
// threads and pinning the ring costs a new context more (0.7 ms) than they save
constexpr size_t kPipeBytes = (size_t)8 << 20;

struct Chunk {
    const Segment *seg;
    size_t lo, n;                          // sites
};

struct Pipe {
    std::vector<Chunk> chunks;
    char *ring = nullptr;
    size_t slot_bytes = 0;
    int slots = 0;
    // to the host: chunks whose copies have landed; to the device: chunks
    // whose slot is free to be packed
    std::atomic<size_t> open{0};
    std::atomic<size_t> next{0};           // piece to take
    std::atomic<bool> stop{false};
    std::vector<std::atomic<int>> done;    // pieces finished per chunk
    explicit Pipe(size_t n) : done(n) {}

    char *slot(size_t q) const { return ring + (q % (size_t)slots) * slot_bytes; }
    void piece(size_t u)
    {
        const size_t q = u / kSlices, s = u % kSlices;
        const Chunk &k = chunks[q];
        const size_t b = k.n * s / kSlices, e = k.n * (s + 1) / kSlices;
        if (e > b) k.seg->fn(slot(q) + b * k.seg->site_bytes, k.lo + b, e - b, k.seg->arg);
        done[q].fetch_add(1, std::memory_order_release);
    }
    bool finished(size_t q) const { return done[q].load(std::memory_order_acquire) == kSlices; }
};

void pipe_worker(void *p)
{
    Pipe *w = (Pipe *)p;
    const size_t total = w->chunks.size() * kSlices;
    for (;;) {
        const size_t u = w->next.fetch_add(1);
        if (u >= total) return;
        while (w->open.load(std::memory_order_acquire) <= u / kSlices) {
            if (w->stop.load()) return;
            std::this_thread::yield();
        }
        w->piece(u);
    }
}

}  // namespace

int transfer(Context *c, const Segment *segs, int nsegs, bool to_host)
{
    size_t nchunks = 0, most = 0;
    for (int s = 0; s < nsegs; ++s) {
        const size_t per = kSlotBytes / segs[s].site_bytes;
        nchunks += (segs[s].L + per - 1) / per;
        most = std::max(most, std::min(segs[s].L, per) * segs[s].site_bytes);
    }
    if (nchunks == 0) return AXS_OK;
    Pipe w(nchunks);
    w.slot_bytes = (most + 255) & ~(size_t)255;
    w.slots = (int)std::min<size_t>(nchunks, kSlots);
    for (int s = 0; s < nsegs; ++s) {
        const size_t per = kSlotBytes / segs[s].site_bytes;
        for (size_t lo = 0; lo < segs[s].L; lo += per)
            w.chunks.push_back(Chunk{&segs[s], lo, std::min(per, segs[s].L - lo)});
    }
    size_t bytes = 0;
    for (const Chunk &k : w.chunks) bytes += k.n * k.seg->site_bytes;
    std::optional<PoolLease> lease;
    if (bytes >= kPipeBytes) lease.emplace(c);
    HostPool *p = lease ? lease->p : nullptr;
    if (!p) {
        // one slot, this thread alone
        AXS_TRY(ensure_pinned(c, w.slot_bytes));
        for (const Chunk &k : w.chunks) {
            char *dev = (char *)k.seg->dev + k.lo * k.seg->site_bytes, *st = (char *)c->pinned;
            const size_t nb = k.n * k.seg->site_bytes;
            if (to_host) {
                AXS_HIP_TRY(hipMemcpyAsync(st, dev, nb, hipMemcpyDeviceToHost, c->stream));
                AXS_HIP_TRY(hipStreamSynchronize(c->stream));
                k.seg->fn(st, k.lo, k.n, k.seg->arg);
            } else {
                k.seg->fn(st, k.lo, k.n, k.seg->arg);
                AXS_HIP_TRY(hipMemcpyAsync(dev, st, nb, hipMemcpyHostToDevice, c->stream));
                AXS_HIP_TRY(hipStreamSynchronize(c->stream));
            }
        }
        return AXS_OK;
    }
    AXS_TRY(ensure_pinned(c, w.slot_bytes * (size_t)w.slots));
    w.ring = (char *)c->pinned;
    for (int h = 0; h < w.slots; ++h)
        if (!c->stage_ev[h])
            AXS_HIP_TRY(hipEventCreateWithFlags(
                &c->stage_ev[h], hipEventDisableTiming | hipEventReleaseToSystem));
    p->start(pipe_worker, &w);

    auto copy = [&](size_t q) -> hipError_t {
        const Chunk &k = w.chunks[q];
        char *dev = (char *)k.seg->dev + k.lo * k.seg->site_bytes;
        const size_t nb = k.n * k.seg->site_bytes;
        hipError_t e = to_host ? copy_chunk(c, w.slot(q), dev, nb)
                               : copy_chunk(c, dev, w.slot(q), nb);
        if (e == hipSuccess) e = hipEventRecord(c->stage_ev[q % (size_t)w.slots], c->stream);
        return e;
    };
    auto settle = [&](size_t q) {
        while (!w.finished(q)) std::this_thread::yield();
    };
    const size_t slots = (size_t)w.slots, lag = std::min<size_t>(2, slots - 1);
    hipError_t e = hipSuccess;
    if (to_host) {
        for (size_t q = 0; q < slots && e == hipSuccess; ++q) e = copy(q);
        for (size_t q = 0; q < nchunks && e == hipSuccess; ++q) {
            e = hipEventSynchronize(c->stage_ev[q % slots]);
            if (e != hipSuccess) break;
            w.open.store(q + 1, std::memory_order_release);
            // a slot is refilled `lag` chunks after its copy landed, when the
            // threads are usually through with it
            if (q >= lag && q - lag + slots < nchunks) {
                settle(q - lag);
                e = copy(q - lag + slots);
            }
        }
    } else {
        w.open.store(slots, std::memory_order_release);
        for (size_t q = 0; q < nchunks && e == hipSuccess; ++q) {
            settle(q);
            e = copy(q);
            // a slot is packed again once its chunk has been sent; the copies
            // of the `lag` chunks after it stay queued meanwhile
            if (e == hipSuccess && q >= lag && q - lag + slots < nchunks) {
                e = hipEventSynchronize(c->stage_ev[(q - lag) % slots]);
                if (e == hipSuccess)
                    w.open.store(q - lag + slots + 1, std::memory_order_release);
            }
        }
        if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
    }
    if (e != hipSuccess) w.stop.store(true);
    p->wait();
    if (e != hipSuccess) {
        (void)hipStreamSynchronize(c->stream);      // nothing reads the ring any more
        set_error("transfer of %zu bytes failed: %s", bytes, hipGetErrorString(e));
        return AXS_ERR_HIP;
    }
    return AXS_OK;
}

static void bytes_out(char *stage, size_t lo, size_t n, void *arg)
{
    memcpy((char *)arg + lo, stage, n);
}

int copy_to_host(Context *c, void *dst, const void *src, size_t bytes)
{
    const Segment s{const_cast<void *>(src), 1, bytes, bytes_out, dst};
    return transfer(c, &s, 1, true);
}

}  // namespace axs
