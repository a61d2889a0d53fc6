// egx_prim.hip -- device blocks, and device primitives for the graph build:
// exclusive scan, stable LSD radix sort and lower-bound probes.
//
// Written for gfx950 wave64: the radix rank uses 64-lane ballots to find the
// lanes that share a digit, so one tile needs no per-thread digit counters.
#include <algorithm>
#include <mutex>
#include <new>
#include <utility>
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
// at once); a failed hipMalloc gives all of them back and tries again, and
// egx_device_trim and egx_pagerank_cache_reset give them back.
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

// Scan of one tile.  What comes before it is offsets[tile], or, with each > 0,
// the sum of before[0, tile * each): the tiles' sums (each 1), or the input
// itself (each kScanTile; not in place).
template <typename T>
__global__ __launch_bounds__(kScanThreads) void k_scan_tile(const T* in, T* out, int64_t n,
                                                            const T* __restrict__ offsets, const T* before,
                                                            int32_t each) {
    __shared__ T sh[kScanTile];
    __shared__ T sh_w[kScanThreads / kWave];
    T start = 0;
    if (each > 0) {
        const int64_t k = (int64_t)blockIdx.x * each;
        T sum = 0;
#pragma unroll 8
        for (int64_t i = threadIdx.x; i < k; i += kScanThreads) sum += before[i];
        __shared__ T total;
        const T got = block_reduce_sum(sum, sh_w);
        if (threadIdx.x == 0) total = got;
        __syncthreads();
        start = total;
    } else if (offsets) {
        start = offsets[blockIdx.x];
    }
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
    run += start;
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

// Up to kScanDirect tiles out of place, each adds up all before it (one
// launch: 16,384 elements took three, 10 us and the gaps between them); up to kScanSelf
// tiles, each adds up the tiles' sums; above, those are scanned first.
constexpr int64_t kScanDirect = 16;
constexpr int64_t kScanSelf = 1024;
template <typename T>
int scan_impl(const T* in, T* out, int64_t n, hipStream_t s) {
    if (n <= 0) return EGX_SUCC;
    const int64_t nb = (n + kScanTile - 1) / kScanTile;
    if (nb == 1 || (nb <= kScanDirect && in != out)) {
        k_scan_tile<T><<<(unsigned)nb, kScanThreads, 0, s>>>(in, out, n, nullptr, in, nb == 1 ? 0 : kScanTile);
        EGX_CHECK_LAUNCH(EGX_DEVICE_ERR);
        return EGX_SUCC;
    }
    DevBuf part;
    EGX_TRY(part.alloc((size_t)nb * sizeof(T), s));  // released in s's order: no wait
    k_scan_reduce<T><<<(unsigned)nb, kScanThreads, 0, s>>>(in, n, part.as<T>());
    EGX_CHECK_LAUNCH(EGX_DEVICE_ERR);
    if (nb > kScanSelf) EGX_TRY(scan_impl<T>(part.as<T>(), part.as<T>(), nb, s));
    k_scan_tile<T><<<(unsigned)nb, kScanThreads, 0, s>>>(in, out, n, part.as<T>(), part.as<T>(),
                                                         nb > kScanSelf ? 0 : 1);
    EGX_CHECK_LAUNCH(EGX_DEVICE_ERR);
    return EGX_SUCC;
}

// ---------------------------------------------------------------------------
// radix sort
// ---------------------------------------------------------------------------
// Stable LSD, up to kDigitBits bits per pass (the passes share the key bits
// evenly, so 17 or 18 bits take two passes and 25 bits three).  One
// workgroup takes a tile of kSortThreads * ITEMS keys; counts holds the
// tiles' digit counts.
constexpr int kSortThreads = 512;
constexpr int kSortWaves = kSortThreads / kWave;
constexpr int kDigitBits = 9;
constexpr int kBins = 1 << kDigitBits;
static_assert(kBins == kSortThreads, "thread t owns digit t");
constexpr int kItemsSmall = 4;   // tiles of 2048 keys: R-MAT 14's 228K arcs fill 112 workgroups
constexpr int kItemsLarge = 16;  // tiles of 8192 keys (4096 of 64 bits): runs of 64 bytes and more per digit
// Up to this many tiles, counts stay tile-major and each tile adds up the
// ones before it itself (one launch less than three scan launches: 57K
// counters took 10 us to scan); above, a digit-major scan.
constexpr uint32_t kSelfScanTiles = 128;

template <typename K, int ITEMS>
__global__ __launch_bounds__(kSortThreads) void k_radix_upsweep(const K* __restrict__ keys, int64_t n, int shift,
                                                                uint32_t mask, uint32_t* __restrict__ counts,
                                                                uint32_t nblocks, int tile_major) {
    // two copies, by wavefront parity: fewer lanes meet on one hot digit
    __shared__ uint32_t hist[2][kBins];
    hist[0][threadIdx.x] = 0;
    hist[1][threadIdx.x] = 0;
    __syncthreads();
    const int64_t base = (int64_t)blockIdx.x * (kSortThreads * ITEMS);
    uint32_t* h = hist[wave_id() & 1];
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        const int64_t idx = base + (int64_t)i * kSortThreads + threadIdx.x;
        if (idx < n) atomicAdd(&h[(uint32_t)(keys[idx] >> shift) & mask], 1u);
    }
    __syncthreads();
    if (threadIdx.x <= mask) {
        const uint32_t c = hist[0][threadIdx.x] + hist[1][threadIdx.x];
        if (tile_major) counts[(size_t)blockIdx.x * kBins + threadIdx.x] = c;
        else counts[(size_t)threadIdx.x * nblocks + blockIdx.x] = c;
    }
}

// Exclusive sum over the workgroup of one value per thread.
__device__ __forceinline__ uint32_t sort_block_scan(uint32_t v, uint32_t* sh_w) {
    uint32_t inc = v;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
        const uint32_t o = __shfl_up(inc, off, kWave);
        if (lane_id() >= off) inc += o;
    }
    if (lane_id() == kWave - 1) sh_w[wave_id()] = inc;
    __syncthreads();
    uint32_t base = 0;
    for (int w = 0; w < wave_id(); ++w) base += sh_w[w];
    __syncthreads();
    return base + inc - v;
}

// Stable scatter of one tile.  Wavefront w holds the tile's keys [w * 64 *
// ITEMS, ...), 64 consecutive ones per step, and ranks them by itself: the
// lanes that share a digit find each other by ballots, and a counter per
// (wavefront, digit) in LDS carries the count over the steps, so the ranking
// needs no barrier.  The tile is then put in digit order in LDS and written
// out by consecutive threads, so that each digit's run is stored in
// consecutive addresses.  The form with four barriers per 256 keys and
// stores in key order took 2.05 ms per pass over 263M pairs and 15 us over
// 228K.
template <typename K, bool HAS_VAL, int ITEMS>
__global__ __launch_bounds__(kSortThreads) void k_radix_downsweep(
    const K* __restrict__ keys_in, const uint32_t* __restrict__ vals_in, K* __restrict__ keys_out,
    uint32_t* __restrict__ vals_out, int64_t n, int shift, uint32_t mask, int bits,
    const uint32_t* __restrict__ offsets, uint32_t nblocks, int tile_major) {
    constexpr int kTile = kSortThreads * ITEMS;
    __shared__ K stage[kTile];
    __shared__ uint32_t wcnt[kSortWaves][kBins];
    __shared__ uint32_t start[kBins];   // first position of the digit in the tile
    __shared__ uint32_t gbase[kBins];   // its first position in the output
    __shared__ uint32_t sh_w[kSortWaves];
    const int t = threadIdx.x;
    const int lane = lane_id();
    const int w = wave_id();
    const int64_t base = (int64_t)blockIdx.x * kTile;
    const int32_t count = (int32_t)min((int64_t)kTile, n - base);  // keys of this tile
    const int32_t wbase = w * (kWave * ITEMS) + lane;
    K key[ITEMS];
    uint32_t val[HAS_VAL ? ITEMS : 1];
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const int32_t i = wbase + r * kWave;
        const int64_t at = base + (i < count ? i : 0);
        key[r] = keys_in[at];
        if (HAS_VAL) val[r] = vals_in[at];
    }
#pragma unroll
    for (int ww = 0; ww < kSortWaves; ++ww) wcnt[ww][t] = 0;
    // this tile's first output position of every digit
    uint32_t tot = 0, before = 0;
    if (tile_major) {
        if ((uint32_t)t <= mask) {
#pragma unroll 8
            for (uint32_t b = 0; b < nblocks; ++b) {
                const uint32_t c = offsets[(size_t)b * kBins + t];
                tot += c;
                before += b < blockIdx.x ? c : 0u;
            }
        }
    } else if ((uint32_t)t <= mask) {
        before = offsets[(size_t)t * nblocks + blockIdx.x];
    }
    __syncthreads();
    if (tile_major) before += sort_block_scan(tot, sh_w);
    gbase[t] = before;
    const uint64_t lt_mask = (1ull << lane) - 1ull;
    uint32_t rank[ITEMS];
    volatile uint32_t* cnt = wcnt[w];
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const bool valid = wbase + r * kWave < count;
        // keys past the end take the last digit: they rank behind its keys
        const uint32_t d = valid ? (uint32_t)(key[r] >> shift) & mask : mask;
        uint64_t peers = ~0ull;
#pragma unroll
        for (int bit = 0; bit < kDigitBits; ++bit) {
            if (bit < bits) {
                const bool set = (d >> bit) & 1u;
                const uint64_t b = __ballot(set);
                peers &= set ? b : ~b;
            }
        }
        const uint32_t pre = cnt[d];
        const uint32_t mine = (uint32_t)__popcll(peers & lt_mask);
        __builtin_amdgcn_wave_barrier();
        if (mine == 0) cnt[d] = pre + (uint32_t)__popcll(peers);
        __builtin_amdgcn_wave_barrier();
        rank[r] = pre + mine;
    }
    __syncthreads();
    {
        uint32_t acc = 0;
#pragma unroll
        for (int ww = 0; ww < kSortWaves; ++ww) {
            const uint32_t c = wcnt[ww][t];
            wcnt[ww][t] = acc;
            acc += c;
        }
        start[t] = sort_block_scan(acc, sh_w);
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const bool valid = wbase + r * kWave < count;
        const uint32_t d = valid ? (uint32_t)(key[r] >> shift) & mask : mask;
        rank[r] += start[d] + wcnt[w][d];
        stage[rank[r]] = key[r];
    }
    __syncthreads();
    uint32_t dest[ITEMS];
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const int32_t i = r * kSortThreads + t;
        if (i < count) {
            const K k = stage[i];
            const uint32_t d = (uint32_t)(k >> shift) & mask;
            dest[r] = gbase[d] + ((uint32_t)i - start[d]);
            keys_out[dest[r]] = k;
        }
    }
    if (HAS_VAL) {
        __syncthreads();
        uint32_t* vstage = reinterpret_cast<uint32_t*>(stage);
#pragma unroll
        for (int r = 0; r < ITEMS; ++r) vstage[rank[r]] = val[HAS_VAL ? r : 0];
        __syncthreads();
#pragma unroll
        for (int r = 0; r < ITEMS; ++r) {
            const int32_t i = r * kSortThreads + t;
            if (i < count) vals_out[dest[r]] = vstage[i];
        }
    }
}

template <typename K, int ITEMS>
int radix_passes(DevBuf& keys, DevBuf& keys_alt, DevBuf* vals, DevBuf* vals_alt, int64_t n, int nbits,
                 hipStream_t s) {
    const uint32_t nb = (uint32_t)((n + kSortThreads * ITEMS - 1) / (kSortThreads * ITEMS));
    const int passes = (nbits + kDigitBits - 1) / kDigitBits;
    const int tile_major = nb <= kSelfScanTiles ? 1 : 0;
    DevBuf counts;
    EGX_TRY(counts.alloc((size_t)kBins * nb * sizeof(uint32_t), s));
    for (int q = 0, shift = 0; q < passes; ++q) {
        const int bits = (nbits - shift + passes - q - 1) / (passes - q);
        const uint32_t mask = (1u << bits) - 1u;
        k_radix_upsweep<K, ITEMS><<<nb, kSortThreads, 0, s>>>(keys.as<K>(), n, shift, mask, counts.as<uint32_t>(), nb,
                                                              tile_major);
        EGX_CHECK_LAUNCH(EGX_DEVICE_ERR);
        if (!tile_major)
            EGX_TRY(scan_impl<uint32_t>(counts.as<uint32_t>(), counts.as<uint32_t>(), (int64_t)(mask + 1) * nb, s));
        if (vals)
            k_radix_downsweep<K, true, ITEMS><<<nb, kSortThreads, 0, s>>>(
                keys.as<K>(), vals->as<uint32_t>(), keys_alt.as<K>(), vals_alt->as<uint32_t>(), n, shift, mask, bits,
                counts.as<uint32_t>(), nb, tile_major);
        else
            k_radix_downsweep<K, false, ITEMS><<<nb, kSortThreads, 0, s>>>(keys.as<K>(), nullptr, keys_alt.as<K>(),
                                                                           nullptr, n, shift, mask, bits,
                                                                           counts.as<uint32_t>(), nb, tile_major);
        EGX_CHECK_LAUNCH(EGX_DEVICE_ERR);
        std::swap(keys, keys_alt);
        if (vals) std::swap(*vals, *vals_alt);
        shift += bits;
    }
    return EGX_SUCC;
}

template <typename K>
int radix_sort_impl(DevBuf& keys, DevBuf& keys_alt, DevBuf* vals, DevBuf* vals_alt, int64_t n, int nbits,
                    hipStream_t s) {
    if (n <= 1 || nbits <= 0) return EGX_SUCC;
    if (n > (int64_t)0xFFFFFFFFll) {
        set_last_error("radix sort: more than 2^32-1 keys");
        return EGX_UNSUPPORTED_GRAPH;
    }
    if (n <= (int64_t)kSelfScanTiles * kSortThreads * kItemsSmall)
        return radix_passes<K, kItemsSmall>(keys, keys_alt, vals, vals_alt, n, nbits, s);
    constexpr int kItems = sizeof(K) == 8 ? kItemsLarge / 2 : kItemsLarge;
    return radix_passes<K, kItems>(keys, keys_alt, vals, vals_alt, n, nbits, s);
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

int radix_sort_u32(DevBuf& keys, DevBuf& keys_alt, DevBuf* vals, DevBuf* vals_alt, int64_t n, int nbits,
                   hipStream_t s) {
    return radix_sort_impl<uint32_t>(keys, keys_alt, vals, vals_alt, n, nbits, s);
}
int radix_sort_u64(DevBuf& keys, DevBuf& keys_alt, DevBuf* vals, DevBuf* vals_alt, int64_t n, int nbits,
                   hipStream_t s) {
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
