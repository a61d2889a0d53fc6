// egx_xfer.hip -- host arrays to and from the device through pinned chunks.
//
// The callers' arrays are pageable (numpy), and usually fresh: a result of
// 16.7M doubles took 9 ms of a 19.5 ms solve, one thread touching 134 MB of new
// pages (16.8 GB/s) after a 67 MB copy, and 112 MB of CSR arrays went up at
// 27 GB/s.  Both directions now run in chunks of kChunkBytes through a ring
// of pinned chunks: queued kernels move one chunk over the link while up to
// kThreads threads fill or empty others (PCIe carries 57 GB/s from pinned
// memory).  Chunks and threads are kept for the process and shared by all
// callers: a caller takes what is free (it always makes progress alone) and
// gives it back before it returns; until its values are due it holds two chunks
// and waits by itself.  Transfers down of at most kInlineBytes use one
// chunk and no threads, those up of at most kUploadSmall too.
#include <sched.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <deque>
#include <functional>
#include <memory>
#include <mutex>
#include <new>
#include <system_error>
#include <thread>

#include "egx_xfer.h"

namespace egx {
namespace {

// Measured (112 MB up with the checks around it / 77 MB of packed columns down
// and finished, with the solve): chunks of 1 MiB 3.95 / 7.57 ms, 2 MiB 3.07 / 6.77, 4 MiB
// 2.76 / 6.74, 8 MiB 2.69 / 6.68; 4 threads 2.71 / 7.27, 16 threads 2.82 / 6.68.
constexpr size_t kChunkBytes = (size_t)4 << 20;
constexpr size_t kInlineBytes = (size_t)256 << 10;
// Uploads up to here go through one chunk, by the calling thread: no threads
// to wake.
constexpr size_t kUploadSmall = (size_t)2 << 20;
constexpr int kMaxChunks = 24;    // pinned chunks the process keeps, at most
constexpr int kCallChunks = 12;   // of them for one transfer
constexpr int kAheadChunks = 2;   // of them for one whose values are not due yet
constexpr int kThreads = 8;       // the calling thread among them

struct Chunk {
    char* p = nullptr;           // `bytes`, and the flag behind them
    size_t bytes = 0;            // kChunkBytes, or kInlineBytes for those that need no more (making either takes 0.05 ms)
    uint32_t* count = nullptr;   // device: workgroups that have written their share
    hipEvent_t ev = nullptr;     // the chunk's last upload
    int dev = -1;                // of count and ev
    uint32_t* flag() const { return reinterpret_cast<uint32_t*>(p + bytes); }
};

// Device memory to a pinned chunk, and 1 to *flag once all of it is there.
// Bound by the link.  A copy call and an event for each part left 10 us between
// parts of 512 KB, which the link carries in 9.7; queued kernels follow each
// other at once, and the host reads the flag (a solve of 1,048,576 nodes,
// 20 iterations: 1.22 ms -> 1.16; 64 columns of 300,007 6.5 -> 6.3).
constexpr int kFetchThreads = 256;
constexpr int kFetchBlocks = 64;
__device__ __forceinline__ void copy_words(const char* __restrict__ from, char* __restrict__ to, int64_t bytes) {
    const int64_t t = (int64_t)blockIdx.x * kFetchThreads + threadIdx.x;
    const int64_t stride = (int64_t)gridDim.x * kFetchThreads;
    int64_t words = 0;  // 4-byte words already taken by 16-byte copies
    if ((reinterpret_cast<uintptr_t>(from) | reinterpret_cast<uintptr_t>(to)) % 16 == 0) {  // (uniform) results of a set may begin at any float
        const uint4* f = reinterpret_cast<const uint4*>(from);
        uint4* o = reinterpret_cast<uint4*>(to);
        const int64_t n = bytes / 16;
#pragma unroll 4
        for (int64_t i = t; i < n; i += stride) o[i] = f[i];
        words = n * 4;
    }
    for (int64_t i = words + t; i < bytes / 4; i += stride)
        reinterpret_cast<uint32_t*>(to)[i] = reinterpret_cast<const uint32_t*>(from)[i];
}

__global__ __launch_bounds__(kFetchThreads) void k_fetch_part(const char* __restrict__ from, char* __restrict__ to,
                                                              int64_t bytes, uint32_t* count, uint32_t* flag) {
    copy_words(from, to, bytes);
    raise_flag(count, flag);
}

// The other way, from a pinned chunk.  The copy engine reaches the same rate,
// but the first copy it makes for a process takes 6 ms to set up: the first
// graph built from host arrays took 6.9 ms, and 1.1 so (16,384 nodes); later
// builds 377 -> 361 us there, 4.98 -> 4.80 ms with 112 MB of weighted arcs.
__global__ __launch_bounds__(kFetchThreads) void k_upload_part(const char* __restrict__ from, char* __restrict__ to,
                                                               int64_t bytes) {
    copy_words(from, to, bytes);
}

unsigned copy_blocks(size_t bytes) {
    const int64_t blocks = ((int64_t)bytes + kFetchThreads * 16 - 1) / (kFetchThreads * 16);
    return (unsigned)std::min<int64_t>(kFetchBlocks, std::max<int64_t>(blocks, 1));
}

__global__ void k_fetch_reset(uint32_t* count) { *count = 0; }

struct ChunkPool {
    std::mutex mu;
    std::vector<Chunk> idle;
    int made[2] = {0, 0};  // small, large
};
ChunkPool& chunk_pool() {
    static ChunkPool* p = new ChunkPool();  // kept until the process ends
    return *p;
}

// Up to `want` chunks that hold `bytes`, usable on device dev (for work on s), at least one unless nothing is
// free and no more may be made (then none).
std::vector<Chunk> take_chunks(int want, size_t bytes, int dev, hipStream_t s) {
    ChunkPool& pool = chunk_pool();
    bytes = bytes <= kInlineBytes ? kInlineBytes : kChunkBytes;
    int& made = pool.made[bytes == kChunkBytes ? 1 : 0];
    std::vector<Chunk> got;
    got.reserve((size_t)want);
    std::lock_guard<std::mutex> lk(pool.mu);
    pool.idle.reserve((size_t)kMaxChunks * 2);  // so that giving back never allocates
    for (size_t i = pool.idle.size(); i-- > 0 && (int)got.size() < want;) {
        if (pool.idle[i].dev != dev || pool.idle[i].bytes != bytes) continue;
        got.push_back(pool.idle[i]);
        pool.idle.erase(pool.idle.begin() + (std::ptrdiff_t)i);
    }
    while ((int)got.size() < want && made < kMaxChunks) {
        Chunk c;
        c.dev = dev;
        c.bytes = bytes;
        if (hipHostMalloc(reinterpret_cast<void**>(&c.p), bytes + 64) != hipSuccess) {
            (void)hipGetLastError();
            break;
        }
        hipError_t e = hipMalloc(reinterpret_cast<void**>(&c.count), 64);
        if (e != hipSuccess) {
            (void)hipGetLastError();
            pool_trim();  // idle blocks may be what is missing
            e = hipMalloc(reinterpret_cast<void**>(&c.count), 64);
        }
        if (e != hipSuccess) {
            (void)hipGetLastError();
            (void)hipHostFree(c.p);
            break;
        }
        k_fetch_reset<<<1, 1, 0, s>>>(c.count);  // s has passed it before the chunk is given back
        if (hipEventCreateWithFlags(&c.ev, hipEventDisableTiming) != hipSuccess) {
            (void)hipGetLastError();
            (void)hipFree(c.count);
            (void)hipHostFree(c.p);
            break;
        }
        made += 1;
        got.push_back(c);
    }
    return got;
}

void give_chunks(const std::vector<Chunk>& chunks) {
    ChunkPool& pool = chunk_pool();
    std::lock_guard<std::mutex> lk(pool.mu);
    for (const Chunk& c : chunks) pool.idle.push_back(c);
}

// Helper threads, started with the first transfer that wants them.
struct Helpers {
    std::mutex mu;
    std::condition_variable work;
    struct Task {
        const void* owner;
        const std::function<void()>* fn;
        int* running;
        std::condition_variable* done;
    };
    std::deque<Task> tasks;
    int threads = 0;

    void loop() {
        std::unique_lock<std::mutex> lk(mu);
        for (;;) {
            work.wait(lk, [&] { return !tasks.empty(); });
            const Task t = tasks.front();
            tasks.pop_front();
            *t.running += 1;
            lk.unlock();
            (*t.fn)();
            lk.lock();
            if (--*t.running == 0) t.done->notify_all();
        }
    }
};
Helpers& helpers() {
    static Helpers* h = new Helpers();  // its threads run until the process ends
    return *h;
}

int helper_count() {
    static const int n = [] {
        cpu_set_t set;
        CPU_ZERO(&set);
        const int cpus = sched_getaffinity(0, sizeof(set), &set) == 0 ? CPU_COUNT(&set) : 1;
        return std::max(0, std::min(kThreads, cpus) - 1);
    }();
    return n;
}

// fn on the calling thread and on up to `more` helpers; returns when all
// that started have ended.  fn must not throw.
void run_together(const std::function<void()>& fn, int more) {
    Helpers& h = helpers();
    int running = 0;
    std::condition_variable done;
    more = std::min(more, helper_count());
    {
        std::lock_guard<std::mutex> lk(h.mu);
        try {
            while (h.threads < helper_count() && h.threads < more) {
                std::thread([&h] { h.loop(); }).detach();
                h.threads += 1;
            }
            for (int i = 0; i < std::min(more, h.threads); ++i)
                h.tasks.push_back(Helpers::Task{&running, &fn, &running, &done});
        } catch (const std::system_error&) {  // no thread to be had: fewer, or this one alone
        } catch (const std::bad_alloc&) {
        }
    }
    h.work.notify_all();
    fn();
    std::unique_lock<std::mutex> lk(h.mu);
    // tasks that no helper has begun are not needed any more
    h.tasks.erase(std::remove_if(h.tasks.begin(), h.tasks.end(),
                                 [&](const Helpers::Task& t) { return t.owner == &running; }),
                  h.tasks.end());
    done.wait(lk, [&] { return running == 0; });
}

// values [i0, i0 + n) of a job, from a chunk
void finish_values(const Fetch& f, int64_t i0, int64_t n, const char* from) {
    if (f.words) {
        std::memcpy(f.words + i0, from, (size_t)n * 4);
        return;
    }
    double* out = f.host + i0;
    if (!f.packed) {
        std::memcpy(out, from, (size_t)n * 8);
        return;
    }
    const float* x = reinterpret_cast<const float*>(from);
    const double sum = f.sum_at ? *f.sum_at : f.sum;
    if (sum > 0.0) {
        const double inv = 1.0 / sum;
        for (int64_t i = 0; i < n; ++i) out[i] = (double)x[i] * inv;
    } else {
        const double u = 1.0 / (double)f.n;
        for (int64_t i = 0; i < n; ++i) out[i] = u;
    }
}

// Bytes per part: whole chunks, or less where the threads would otherwise
// have none to share (one 4 MB result by one thread: 0.25 ms).
size_t part_bytes(size_t total) {
    const size_t even = (total / kThreads + 4095) / 4096 * 4096;
    return std::min(kChunkBytes, std::max(kInlineBytes, even));
}

// Values [i0, i0 + n) of a job, `at` bytes into the part that carries them.
struct Piece {
    const Fetch* f;
    int64_t i0, n;
    size_t at;
};

struct Part {
    const char* host;      // source (upload)
    char* dev;
    size_t bytes;
    size_t first, pieces;  // of the run's pieces (fetch): one job's values, or those of jobs that follow each other
};

// The transfer's parts, taken in order by several threads; part k uses
// chunk k % chunks, after part k - chunks is through with it.  Chunks that it
// still holds when it ends (finish_run has given them back, unless something
// failed on the way) go back once its stream is through with them.
struct Run {
    Run() = default;
    Run(const Run&) = delete;
    Run& operator=(const Run&) = delete;
    ~Run() {
        if (chunks.empty()) return;
        (void)hipStreamSynchronize(s);
        give_chunks(chunks);
    }
    std::vector<Part> parts;
    std::vector<Piece> pieces;
    std::vector<Chunk> chunks;
    std::unique_ptr<std::atomic<int>[]> stage;  // per part: 1 queued (fetch), 2 through
    std::atomic<int64_t> next{0};
    std::atomic<int> err{0};  // first hipError_t
    hipStream_t s = nullptr;
    int dev = -1;

    bool ok(hipError_t e) {
        if (e == hipSuccess) return true;
        int none = 0;
        err.compare_exchange_strong(none, (int)e);
        return false;
    }
    // Waits until part k has reached a stage; false once the run has failed.
    bool reached(int64_t k, int st) {
        while (stage[(size_t)k].load(std::memory_order_acquire) < st) {
            if (err.load(std::memory_order_relaxed)) return false;
            std::this_thread::yield();
        }
        return true;
    }
    void finish(const Part& p, const char* from) const {
        for (size_t q = p.first; q < p.first + p.pieces; ++q)
            finish_values(*pieces[q].f, pieces[q].i0, pieces[q].n, from + pieces[q].at);
    }
    void queue_fetch(int64_t k) {
        const Part& p = parts[(size_t)k];
        const Chunk& c = chunks[(size_t)k % chunks.size()];
        __atomic_store_n(c.flag(), 0u, __ATOMIC_RELEASE);
        k_fetch_part<<<copy_blocks(p.bytes), kFetchThreads, 0, s>>>(p.dev, c.p, (int64_t)p.bytes, c.count, c.flag());
        if (ok(hipGetLastError())) stage[(size_t)k].store(1, std::memory_order_release);
    }
    // Waits until the part in chunk c has landed, or is about to; false when its stream failed.
    bool landed(const Chunk& c, const Due& due = Due{}) {
        for (uint32_t spins = 1;; ++spins) {
            if (__atomic_load_n(c.flag(), __ATOMIC_ACQUIRE) != 0u || (due.soon && due.soon(due.of))) return true;
            if (spins % 4096 == 0) {
                const hipError_t e = hipStreamQuery(s);
                if (e == hipErrorNotReady) (void)hipGetLastError();  // not an error: clear it
                else if (__atomic_load_n(c.flag(), __ATOMIC_ACQUIRE) == 0u) return ok(e == hipSuccess ? hipErrorUnknown : e);
            }
            std::this_thread::yield();
        }
    }
    void fetch_parts() {
        const int64_t total = (int64_t)parts.size(), ring = (int64_t)chunks.size();
        if (!ok(hipSetDevice(dev))) return;
        for (;;) {
            const int64_t k = next.fetch_add(1);
            if (k >= total || !reached(k, 1)) return;
            const Part& p = parts[(size_t)k];
            const Chunk& c = chunks[(size_t)k % chunks.size()];
            if (!landed(c)) return;
            finish(p, c.p);
            stage[(size_t)k].store(2, std::memory_order_release);
            if (k + ring < total) queue_fetch(k + ring);
        }
    }
    void upload_parts() {
        const int64_t total = (int64_t)parts.size(), ring = (int64_t)chunks.size();
        if (!ok(hipSetDevice(dev))) return;
        for (;;) {
            const int64_t k = next.fetch_add(1);
            if (k >= total) return;
            const Part& p = parts[(size_t)k];
            const Chunk& c = chunks[(size_t)k % chunks.size()];
            // the ring's previous part has been queued from this chunk, and its copy has ended
            if (k >= ring && (!reached(k - ring, 2) || !ok(hipEventSynchronize(c.ev)))) return;
            std::memcpy(c.p, p.host, p.bytes);
            k_upload_part<<<copy_blocks(p.bytes), kFetchThreads, 0, s>>>(c.p, p.dev, (int64_t)p.bytes);
            if (!ok(hipGetLastError()) || !ok(hipEventRecord(c.ev, s))) return;
            stage[(size_t)k].store(2, std::memory_order_release);
        }
    }
};

int finish_run(Run& r) {
    // no copy may still use a chunk when another caller gets it
    const hipError_t e = hipStreamSynchronize(r.s);
    give_chunks(r.chunks);
    r.chunks.clear();
    const hipError_t first = (hipError_t)r.err.load();
    if (first != hipSuccess || e != hipSuccess) {
        set_last_error(std::string("host transfer: ") + hipGetErrorString(first != hipSuccess ? first : e));
        return EGX_DEVICE_ERR;
    }
    return EGX_SUCC;
}

size_t largest(const std::vector<Part>& parts) {
    size_t most = 0;
    for (const Part& p : parts) most = std::max(most, p.bytes);
    return most;
}

// Up to `want` chunks that hold `bytes` for the run, kCallChunks with those it has.
void add_chunks(Run& r, size_t want, size_t bytes) {
    for (const Chunk& c : take_chunks((int)want, bytes, r.dev, r.s)) r.chunks.push_back(c);  // begin_run has reserved them
}

// Chunks for `parts` parts of at most `bytes`, at most `most` of them; -1 when there are none to be had.
int begin_run(Run& r, size_t parts, size_t bytes, hipStream_t s, int most = kCallChunks) {
    r.s = s;
    if (hipGetDevice(&r.dev) != hipSuccess) return -1;
    r.stage.reset(new std::atomic<int>[std::max<size_t>(parts, 1)]);
    for (size_t i = 0; i < parts; ++i) r.stage[i].store(0);
    r.chunks.reserve(kCallChunks);
    add_chunks(r, std::min<size_t>(parts, (size_t)most), bytes);
    return r.chunks.empty() ? -1 : 0;
}

int upload_plain(const std::vector<Upload>& jobs, hipStream_t s) {
    for (const Upload& u : jobs)
        if (u.bytes)
            EGX_HIP_TRY(hipMemcpyWithStream(u.dev, u.host, u.bytes, hipMemcpyHostToDevice, s), EGX_DEVICE_ERR);
    return EGX_SUCC;
}

// All in one chunk, by the calling thread.
int upload_small(const std::vector<Upload>& jobs, size_t total_bytes, hipStream_t s) {
    Run r;
    if (begin_run(r, 1, total_bytes + 16 * jobs.size(), s) != 0) return upload_plain(jobs, s);
    size_t at = 0;
    for (const Upload& u : jobs) {
        if (u.bytes == 0) continue;
        char* from = r.chunks[0].p + at;
        std::memcpy(from, u.host, u.bytes);
        k_upload_part<<<copy_blocks(u.bytes), kFetchThreads, 0, s>>>(from, static_cast<char*>(u.dev), (int64_t)u.bytes);
        if (!r.ok(hipGetLastError())) break;
        at += (u.bytes + 15) / 16 * 16;
    }
    return finish_run(r);
}

int upload_chunked(const std::vector<Upload>& jobs, size_t total_bytes, hipStream_t s) {
    Run r;
    const size_t step = part_bytes(total_bytes);
    for (const Upload& u : jobs)
        for (size_t at = 0; at < u.bytes; at += step)
            r.parts.push_back(Part{static_cast<const char*>(u.host) + at, static_cast<char*>(u.dev) + at,
                                   std::min(step, u.bytes - at), 0, 0});
    const std::function<void()> work = [&] { r.upload_parts(); };
    if (begin_run(r, r.parts.size(), largest(r.parts), s) != 0) return upload_plain(jobs, s);  // no pinned memory
    run_together(work, (int)std::min<size_t>(r.parts.size(), kThreads) - 1);
    return finish_run(r);
}

int fetch_chunked(const std::vector<Fetch>& jobs, size_t total_bytes, hipStream_t s, const Due& due) {
    Run r;
    const size_t step = part_bytes(total_bytes);
    for (const Fetch& f : jobs) {
        const size_t elem = f.packed ? 4 : 8;
        char* dev = static_cast<char*>(const_cast<void*>(f.dev));
        for (int64_t i = 0; i < f.n;) {
            char* at = dev + (size_t)i * elem;
            if (r.parts.empty() || r.pieces.back().f->packed != f.packed ||
                r.parts.back().dev + r.parts.back().bytes != at || r.parts.back().bytes + elem > step)
                r.parts.push_back(Part{nullptr, at, 0, r.pieces.size(), 0});
            Part& p = r.parts.back();
            const int64_t k = std::min((int64_t)((step - p.bytes) / elem), f.n - i);
            r.pieces.push_back(Piece{&f, i, k, p.bytes});
            p.bytes += (size_t)k * elem;
            p.pieces += 1;
            i += k;
        }
    }
    if (r.parts.empty()) return EGX_SUCC;
    const std::function<void()> work = [&] { r.fetch_parts(); };
    // Values behind a whole solve: until they are due the call holds
    // kAheadChunks chunks, and one thread waits.  (With all of them and the
    // helpers from the start, a solve of 4.2M nodes and 300 iterations kept 8.0
    // cores spinning, and half of the process's chunks from others.)
    const size_t part = largest(r.parts);
    if (begin_run(r, r.parts.size(), part, s, due.soon ? kAheadChunks : kCallChunks) != 0) {
        // no pinned memory: through a pageable buffer
        std::vector<char> buf(kChunkBytes);
        for (const Part& p : r.parts) {
            EGX_HIP_TRY(hipMemcpyWithStream(buf.data(), p.dev, p.bytes, hipMemcpyDeviceToHost, s), EGX_DEVICE_ERR);
            r.finish(p, buf.data());
        }
        return EGX_SUCC;
    }
    size_t queued = 0;
    for (; queued < r.chunks.size(); ++queued) r.queue_fetch((int64_t)queued);
    if (r.parts.size() == 1) {
        work();
        return finish_run(r);
    }
    if (due.soon) {
        if (!r.landed(r.chunks[0], due)) return finish_run(r);
        const size_t all = std::min<size_t>(r.parts.size(), kCallChunks);
        if (all > queued) add_chunks(r, all - queued, part);
        for (; queued < r.chunks.size(); ++queued) r.queue_fetch((int64_t)queued);
    }
    run_together(work, (int)std::min<size_t>(r.parts.size(), kThreads) - 1);
    return finish_run(r);
}

}  // namespace

int upload(const std::vector<Upload>& jobs, hipStream_t s) {
    size_t total = 0;
    for (const Upload& u : jobs) total += u.bytes;
    if (total == 0) return EGX_SUCC;
    try {
        if (total <= kUploadSmall) return upload_small(jobs, total, s);
        return upload_chunked(jobs, total, s);
    } catch (const std::bad_alloc&) {
        set_last_error("host transfer: out of host memory");
        return EGX_FAILED_TO_ALLOCATE_HOST_MEM;
    }
}

struct DirectFetch::State {
    Run r;
};

DirectFetch::DirectFetch() = default;

DirectFetch::~DirectFetch() {
    if (st_) (void)finish_run(st_->r);  // the kernel may still write
}

bool DirectFetch::begin(size_t bytes, hipStream_t s) {
    if (bytes > kInlineBytes) return false;
    try {
        std::unique_ptr<State> st(new State());
        if (begin_run(st->r, 1, bytes, s) != 0) return false;
        st_ = std::move(st);
    } catch (const std::bad_alloc&) {
        return false;
    }
    const Chunk& c = st_->r.chunks[0];
    __atomic_store_n(c.flag(), 0u, __ATOMIC_RELEASE);
    to = c.p;
    count = c.count;
    flag = c.flag();
    return true;
}

int DirectFetch::finish(const Fetch& f) {
    Run& r = st_->r;
    if (r.landed(r.chunks[0])) finish_values(f, 0, f.n, r.chunks[0].p);
    const int rc = finish_run(r);
    st_.reset();
    return rc;
}

int fetch(const std::vector<Fetch>& jobs, hipStream_t s, const Due& due) {
    size_t total = 0;
    for (const Fetch& f : jobs) total += (size_t)f.n * (f.packed ? 4 : 8);
    try {
        return fetch_chunked(jobs, total, s, due);
    } catch (const std::bad_alloc&) {
        set_last_error("host transfer: out of host memory");
        return EGX_FAILED_TO_ALLOCATE_HOST_MEM;
    }
}

int download(const void* dev, int32_t* host, int64_t n, hipStream_t s) {
    return fetch({Fetch{dev, nullptr, n, true, 0.0, nullptr, host}}, s);
}

}  // namespace egx
