// egx_prim.hip -- device primitives for the graph build: exclusive scan,
// stable LSD radix sort (8-bit digits) and lower-bound probes.
//
// Written for gfx950 wave64: the radix rank uses 64-lane ballots to find the
// lanes that share a digit, so one tile needs no per-thread digit counters.
#include <algorithm>
#include <mutex>
#include <new>
#include <vector>

#include "egx_common.h"

namespace egx {

namespace {

// Device blocks of released buffers, kept for the next ones of their size.
// A graph build allocates and frees some 70 buffers; hipMalloc and hipFree
// took 13 ms of a 21 ms build and solve of an 11M-arc weighted graph (hipFree
// waits for the device, 120 us at a time) and 6 ms at 5M arcs.
//
// A block that its stream may still be working on (tagged with that
// stream) goes to a buffer of the same stream only, whose work is queued
// behind it; once the stream is known to be idle the tag is dropped and any
// stream may have it.  The allocator itself never waits.  At most kPoolBytes
// (and kPoolBlocks blocks) stay idle per process (the oldest blocks are freed first, a larger block
// at once); a failed hipMalloc gives all of them back and tries again, and so
// does egx_pagerank_cache_reset.
constexpr size_t kPoolBytes = (size_t)4 << 30;
constexpr size_t kPoolBlocks = 4096;

struct PoolBlock {
    void* p;
    size_t cap;
    int dev;
    hipStream_t stream;  // null: idle
};

struct DevPool {
    std::mutex mu;
    std::vector<PoolBlock> idle;  // oldest first
    size_t bytes = 0;
};

DevPool& dev_pool() {
    static DevPool* p = new DevPool();  // never destroyed: buffers may outlive static objects
    return *p;
}

thread_local hipStream_t t_alloc_stream = nullptr;

// Block sizes: eight steps per power of two, at least 512 bytes, so that
// builds of nearly equal graphs share blocks.
size_t block_size(size_t n) {
    if (n <= 512) return 512;
    size_t top = 512;
    while (top <= n / 2) top *= 2;
    const size_t step = top / 8;
    return (n + step - 1) / step * step;
}

// The smallest fitting block that stream s may use, at most a quarter larger.
bool pool_take(size_t need, int dev, hipStream_t s, PoolBlock* out) {
    DevPool& pool = dev_pool();
    std::lock_guard<std::mutex> lk(pool.mu);
    size_t best = pool.idle.size();
    for (size_t i = pool.idle.size(); i-- > 0;) {
        const PoolBlock& b = pool.idle[i];
        if (b.dev != dev || b.cap < need || b.cap - need > need / 4 || (b.stream && b.stream != s)) continue;
        if (best == pool.idle.size() || b.cap < pool.idle[best].cap) best = i;
        if (b.cap == need) break;
    }
    if (best == pool.idle.size()) return false;
    *out = pool.idle[best];
    pool.bytes -= out->cap;
    pool.idle.erase(pool.idle.begin() + (std::ptrdiff_t)best);
    return true;
}

void pool_give(const PoolBlock& b) {
    DevPool& pool = dev_pool();
    if (b.cap > kPoolBytes / 4) {
        (void)hipFree(b.p);
        return;
    }
    PoolBlock add = b;
    for (;;) {
        PoolBlock drop;  // freed outside the lock: hipFree waits for the device
        {
            std::lock_guard<std::mutex> lk(pool.mu);
            if (add.p && pool.bytes + add.cap <= kPoolBytes && pool.idle.size() < kPoolBlocks) {
                try {
                    pool.idle.push_back(add);
                    pool.bytes += add.cap;
                    return;
                } catch (const std::bad_alloc&) {
                    drop = add;
                    add.p = nullptr;
                }
            } else {
                // the new block fits once older ones have gone
                drop = pool.idle.front();
                pool.bytes -= drop.cap;
                pool.idle.erase(pool.idle.begin());
            }
        }
        (void)hipFree(drop.p);
        if (!add.p) return;
    }
}

}  // namespace

StreamScope::StreamScope(hipStream_t s) : prev(t_alloc_stream) { t_alloc_stream = s; }
StreamScope::~StreamScope() { t_alloc_stream = prev; }

void pool_stream_idle(hipStream_t s) {
    if (!s) return;
    DevPool& pool = dev_pool();
    std::lock_guard<std::mutex> lk(pool.mu);
    for (PoolBlock& b : pool.idle)
        if (b.stream == s) b.stream = nullptr;
}

size_t pool_idle_bytes(int dev) {
    DevPool& pool = dev_pool();
    std::lock_guard<std::mutex> lk(pool.mu);
    size_t n = 0;
    for (const PoolBlock& b : pool.idle) n += b.dev == dev ? b.cap : 0;
    return n;
}

void pool_trim() {
    std::vector<PoolBlock> out;
    {
        DevPool& pool = dev_pool();
        std::lock_guard<std::mutex> lk(pool.mu);
        out.swap(pool.idle);
        pool.bytes = 0;
    }
    for (const PoolBlock& b : out) (void)hipFree(b.p);
}

int DevBuf::alloc(size_t nbytes) { return alloc(nbytes, t_alloc_stream); }

int DevBuf::alloc(size_t nbytes, hipStream_t s) {
    release();
    if (nbytes == 0) nbytes = 16;
    size_t need = nbytes;
    if (s) {
        int d = -1;
        EGX_HIP_TRY(hipGetDevice(&d), EGX_DEVICE_ERR);
        need = block_size(nbytes);
        PoolBlock b;
        if (pool_take(need, d, s, &b)) {
            p = b.p;
            bytes = nbytes;
            cap = b.cap;
            dev = d;
            stream = s;
            return EGX_SUCC;
        }
        dev = d;
    }
    hipError_t e = hipMalloc(&p, need);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        pool_trim();  // idle blocks may be what is missing
        e = hipMalloc(&p, need);
    }
    if (e != hipSuccess) {
        p = nullptr;
        dev = -1;
        set_last_error(std::string("hipMalloc(") + std::to_string(nbytes) + "): " + hipGetErrorString(e));
        // the failure is reported here; clear HIP's sticky last error so the
        // next launch check does not report it again (a caller that falls
        // back, such as the blocked-layout build, then goes on cleanly)
        (void)hipGetLastError();
        return EGX_FAILED_TO_ALLOCATE_DEVICE_MEM;
    }
    bytes = nbytes;
    cap = s ? need : 0;
    stream = s;
    return EGX_SUCC;
}

void DevBuf::release() {
    if (p) {
        if (cap) pool_give(PoolBlock{p, cap, dev, stream});
        else (void)hipFree(p);
    }
    p = nullptr;
    bytes = 0;
    cap = 0;
    dev = -1;
    stream = nullptr;
}

namespace {

constexpr int kScanThreads = 256;
constexpr int kScanItems = 8;
constexpr int kScanTile = kScanThreads * kScanItems;

template <typename T>
__device__ __forceinline__ T block_reduce_sum(T v, T* sh_w) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, kWave);
    if (lane_id() == 0) sh_w[wave_id()] = v;
    __syncthreads();
    T total = 0;
    if (threadIdx.x == 0) {
        for (int w = 0; w < kScanThreads / kWave; ++w) total += sh_w[w];
    }
    return total;
}

// Exclusive scan of one value per thread across the block.
template <typename T>
__device__ __forceinline__ T block_exclusive_scan(T v, T* sh_w) {
    const int lane = lane_id();
    T inc = v;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
        T o = __shfl_up(inc, off, kWave);
        if (lane >= off) inc += o;
    }
    if (lane == kWave - 1) sh_w[wave_id()] = inc;
    __syncthreads();
    T wbase = 0;
    for (int w = 0; w < wave_id(); ++w) wbase += sh_w[w];
    __syncthreads();
    return wbase + inc - v;
}

template <typename T>
__global__ __launch_bounds__(kScanThreads) void k_scan_reduce(const T* __restrict__ in, int64_t n,
                                                              T* __restrict__ partial) {
    __shared__ T sh_w[kScanThreads / kWave];
    const int64_t base = (int64_t)blockIdx.x * kScanTile;
    T sum = 0;
#pragma unroll
    for (int i = 0; i < kScanItems; ++i) {
        int64_t idx = base + (int64_t)i * kScanThreads + threadIdx.x;
        if (idx < n) sum += in[idx];
    }
    T total = block_reduce_sum(sum, sh_w);
    if (threadIdx.x == 0) partial[blockIdx.x] = total;
}

template <typename T>
__global__ __launch_bounds__(kScanThreads) void k_scan_tile(const T* in, T* out, int64_t n,
                                                            const T* __restrict__ offsets) {
    __shared__ T sh[kScanTile];
    __shared__ T sh_w[kScanThreads / kWave];
    const int64_t base = (int64_t)blockIdx.x * kScanTile;
#pragma unroll
    for (int i = 0; i < kScanItems; ++i) {
        int64_t idx = base + (int64_t)i * kScanThreads + threadIdx.x;
        sh[i * kScanThreads + threadIdx.x] = (idx < n) ? in[idx] : (T)0;
    }
    __syncthreads();
    T local[kScanItems];
    T tsum = 0;
#pragma unroll
    for (int i = 0; i < kScanItems; ++i) {
        local[i] = sh[threadIdx.x * kScanItems + i];
        tsum += local[i];
    }
    T run = block_exclusive_scan(tsum, sh_w);
    if (offsets) run += offsets[blockIdx.x];
#pragma unroll
    for (int i = 0; i < kScanItems; ++i) {
        sh[threadIdx.x * kScanItems + i] = run;
        run += local[i];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kScanItems; ++i) {
        int64_t idx = base + (int64_t)i * kScanThreads + threadIdx.x;
        if (idx < n) out[idx] = sh[i * kScanThreads + threadIdx.x];
    }
}

template <typename T>
int scan_impl(const T* in, T* out, int64_t n, hipStream_t s) {
    if (n <= 0) return EGX_SUCC;
    const int64_t nb = (n + kScanTile - 1) / kScanTile;
    if (nb == 1) {
        k_scan_tile<T><<<1, kScanThreads, 0, s>>>(in, out, n, nullptr);
        EGX_CHECK_LAUNCH(EGX_DEVICE_ERR);
        return EGX_SUCC;
    }
    DevBuf part;
    EGX_TRY(part.alloc((size_t)nb * sizeof(T), s));  // released in s's order: no wait
    k_scan_reduce<T><<<(unsigned)nb, kScanThreads, 0, s>>>(in, n, part.as<T>());
    EGX_CHECK_LAUNCH(EGX_DEVICE_ERR);
    EGX_TRY(scan_impl<T>(part.as<T>(), part.as<T>(), nb, s));
    k_scan_tile<T><<<(unsigned)nb, kScanThreads, 0, s>>>(in, out, n, part.as<T>());
    EGX_CHECK_LAUNCH(EGX_DEVICE_ERR);
    return EGX_SUCC;
}

// ---------------------------------------------------------------------------
// radix sort
// ---------------------------------------------------------------------------
constexpr int kSortThreads = 256;
constexpr int kSortItems = 16;
constexpr int kSortTile = kSortThreads * kSortItems;
constexpr int kSortWaves = kSortThreads / kWave;

template <typename K>
__global__ __launch_bounds__(kSortThreads) void k_radix_upsweep(const K* __restrict__ keys, int64_t n,
                                                                int shift, uint32_t* __restrict__ counts,
                                                                uint32_t nblocks) {
    __shared__ uint32_t hist[256];
    hist[threadIdx.x] = 0;
    __syncthreads();
    const int64_t base = (int64_t)blockIdx.x * kSortTile;
#pragma unroll 4
    for (int i = 0; i < kSortItems; ++i) {
        int64_t idx = base + (int64_t)i * kSortThreads + threadIdx.x;
        if (idx < n) {
            uint32_t d = (uint32_t)(keys[idx] >> shift) & 255u;
            atomicAdd(&hist[d], 1u);
        }
    }
    __syncthreads();
    counts[(size_t)threadIdx.x * nblocks + blockIdx.x] = hist[threadIdx.x];
}

// Stable scatter: within the tile, key i*256+t precedes key (i+1)*256+t' and
// key i*256+t precedes i*256+t+1, which is the tile's input order.
template <typename K, bool HAS_VAL>
__global__ __launch_bounds__(kSortThreads) void k_radix_downsweep(
    const K* __restrict__ keys_in, const uint32_t* __restrict__ vals_in, K* __restrict__ keys_out,
    uint32_t* __restrict__ vals_out, int64_t n, int shift, const uint32_t* __restrict__ offsets,
    uint32_t nblocks) {
    __shared__ uint32_t gbase[256];
    __shared__ uint32_t run[256];
    __shared__ uint32_t wcnt[kSortWaves][256];
    const int t = threadIdx.x;
    const int lane = lane_id();
    const int w = wave_id();
    gbase[t] = offsets[(size_t)t * nblocks + blockIdx.x];
    run[t] = 0;
    const uint64_t lt_mask = (lane == 0) ? 0ull : ((1ull << lane) - 1ull);
    const int64_t base = (int64_t)blockIdx.x * kSortTile;
    for (int r = 0; r < kSortItems; ++r) {
        const int64_t idx = base + (int64_t)r * kSortThreads + t;
        const bool valid = idx < n;
        K key = valid ? keys_in[idx] : (K)0;
        uint32_t val = 0;
        if (HAS_VAL && valid) val = vals_in[idx];
        const uint32_t d = (uint32_t)(key >> shift) & 255u;
#pragma unroll
        for (int ww = 0; ww < kSortWaves; ++ww) wcnt[ww][t] = 0;
        __syncthreads();
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int bit = 0; bit < 8; ++bit) {
            const bool set = (d >> bit) & 1u;
            const uint64_t b = __ballot(set);
            peers &= set ? b : ~b;
        }
        const uint32_t rank = (uint32_t)__popcll(peers & lt_mask);
        if (valid && rank == 0) wcnt[w][d] = (uint32_t)__popcll(peers);
        __syncthreads();
        {
            uint32_t acc = run[t];
#pragma unroll
            for (int ww = 0; ww < kSortWaves; ++ww) {
                uint32_t c = wcnt[ww][t];
                wcnt[ww][t] = acc;
                acc += c;
            }
            run[t] = acc;
        }
        __syncthreads();
        if (valid) {
            const uint32_t dest = gbase[d] + wcnt[w][d] + rank;
            keys_out[dest] = key;
            if (HAS_VAL) vals_out[dest] = val;
        }
        __syncthreads();
    }
}

template <typename K>
int radix_sort_impl(K* keys, K* keys_alt, uint32_t* vals, uint32_t* vals_alt, int64_t n, int nbits,
                    hipStream_t s) {
    if (n <= 1 || nbits <= 0) return EGX_SUCC;
    if (n > (int64_t)0xFFFFFFFFll) {
        set_last_error("radix sort: more than 2^32-1 keys");
        return EGX_UNSUPPORTED_GRAPH;
    }
    const int64_t nb64 = (n + kSortTile - 1) / kSortTile;
    const uint32_t nb = (uint32_t)nb64;
    DevBuf counts;
    EGX_TRY(counts.alloc((size_t)256 * nb * sizeof(uint32_t), s));
    const bool has_val = vals != nullptr;
    K* kin = keys;
    K* kout = keys_alt;
    uint32_t* vin = vals;
    uint32_t* vout = vals_alt;
    int passes = 0;
    for (int shift = 0; shift < nbits; shift += 8, ++passes) {
        k_radix_upsweep<K><<<nb, kSortThreads, 0, s>>>(kin, n, shift, counts.as<uint32_t>(), nb);
        EGX_CHECK_LAUNCH(EGX_DEVICE_ERR);
        EGX_TRY(scan_impl<uint32_t>(counts.as<uint32_t>(), counts.as<uint32_t>(), (int64_t)256 * nb, s));
        if (has_val)
            k_radix_downsweep<K, true><<<nb, kSortThreads, 0, s>>>(kin, vin, kout, vout, n, shift,
                                                                   counts.as<uint32_t>(), nb);
        else
            k_radix_downsweep<K, false><<<nb, kSortThreads, 0, s>>>(kin, nullptr, kout, nullptr, n,
                                                                    shift, counts.as<uint32_t>(), nb);
        EGX_CHECK_LAUNCH(EGX_DEVICE_ERR);
        K* tk = kin; kin = kout; kout = tk;
        uint32_t* tv = vin; vin = vout; vout = tv;
    }
    if (passes & 1) {
        EGX_HIP_TRY(hipMemcpyAsync(keys, kin, (size_t)n * sizeof(K), hipMemcpyDeviceToDevice, s), EGX_DEVICE_ERR);
        if (has_val)
            EGX_HIP_TRY(hipMemcpyAsync(vals, vin, (size_t)n * sizeof(uint32_t), hipMemcpyDeviceToDevice, s),
                        EGX_DEVICE_ERR);
    }
    return EGX_SUCC;
}

template <typename K>
__global__ void k_lower_bound_iota(const K* __restrict__ sorted, int64_t n, int shift,
                                   int32_t* __restrict__ out, int64_t nprobe) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nprobe) return;
    const K target = (K)((uint64_t)i << shift);
    int64_t lo = 0, hi = n;
    while (lo < hi) {
        int64_t mid = (lo + hi) >> 1;
        if (sorted[mid] < target) lo = mid + 1;
        else hi = mid;
    }
    out[i] = (int32_t)lo;
}

}  // namespace

int exclusive_scan_u32(const uint32_t* in, uint32_t* out, int64_t n, hipStream_t s) {
    return scan_impl<uint32_t>(in, out, n, s);
}
int exclusive_scan_i64(const int64_t* in, int64_t* out, int64_t n, hipStream_t s) {
    return scan_impl<int64_t>(in, out, n, s);
}

int radix_sort_u32(uint32_t* keys, uint32_t* keys_alt, uint32_t* vals, uint32_t* vals_alt, int64_t n,
                   int nbits, hipStream_t s) {
    return radix_sort_impl<uint32_t>(keys, keys_alt, vals, vals_alt, n, nbits, s);
}
int radix_sort_u64(uint64_t* keys, uint64_t* keys_alt, uint32_t* vals, uint32_t* vals_alt, int64_t n,
                   int nbits, hipStream_t s) {
    return radix_sort_impl<uint64_t>(keys, keys_alt, vals, vals_alt, n, nbits, s);
}

int lower_bound_iota_u32(const uint32_t* sorted, int64_t n, int32_t* out, int64_t nprobe, hipStream_t s) {
    if (nprobe <= 0) return EGX_SUCC;
    const unsigned blocks = (unsigned)((nprobe + 255) / 256);
    k_lower_bound_iota<uint32_t><<<blocks, 256, 0, s>>>(sorted, n, 0, out, nprobe);
    EGX_CHECK_LAUNCH(EGX_DEVICE_ERR);
    return EGX_SUCC;
}
int lower_bound_iota_u64(const uint64_t* sorted, int64_t n, int shift, int32_t* out, int64_t nprobe,
                         hipStream_t s) {
    if (nprobe <= 0) return EGX_SUCC;
    const unsigned blocks = (unsigned)((nprobe + 255) / 256);
    k_lower_bound_iota<uint64_t><<<blocks, 256, 0, s>>>(sorted, n, shift, out, nprobe);
    EGX_CHECK_LAUNCH(EGX_DEVICE_ERR);
    return EGX_SUCC;
}

}  // namespace egx
