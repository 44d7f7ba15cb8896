// prims.hip -- reduce-then-scan exclusive scans and a stable LSD radix sort.
//
// Both are deterministic (integer only).  They serve the CSR -> ABHSF
// conversion, which replaces the reference's parallel sort + linear block scan
// (preprocessing/test.cpp:237-368).
#include "prims.hpp"

#include <algorithm>
#include <mutex>
#include <utility>

namespace abhsf {
namespace {

// Scratch kept between operations, or (owner) idle within one: its earlier use
// may not have finished on the owner's stream.
struct KeptBuf {
    int device;
    uint64_t at;  // when it was given back (Kept::now)
    DevBuf buf;
    const Arena *owner = nullptr;
    hipStream_t stream = nullptr;  // the owner's
};
struct Kept {
    std::mutex m;
    uint64_t now = 0;
    std::vector<KeptBuf> bufs;
};
Kept &kept()
{
    static Kept *k = new Kept;  // (not destroyed: the HIP runtime may end before static objects do)
    return *k;
}

constexpr int kThreads = 256;
constexpr int kItems = 8;
constexpr int kTile = kThreads * kItems;  // 2048 elements per workgroup

template <typename T>
__device__ inline T shfl_up_t(T v, int o) { return __shfl_up(v, o, kWave); }

// Workgroup exclusive scan of one value per thread; also returns the total.
template <typename T>
__device__ inline T block_excl_scan(T v, T *lds, T &total)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    T incl = v;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        T t = shfl_up_t(incl, o);
        if (lane >= o) incl += t;
    }
    if (lane == kWave - 1) lds[wave] = incl;
    __syncthreads();
    T woff = 0, tot = 0;
#pragma unroll
    for (int w = 0; w < kThreads / kWave; w++) {
        T c = lds[w];
        if (w < wave) woff += c;
        tot += c;
    }
    __syncthreads();
    total = tot;
    return woff + incl - v;
}

template <typename T>
__global__ __launch_bounds__(kThreads) void k_tile_reduce(const T *__restrict__ in, uint64_t n,
                                                          T *__restrict__ sums)
{
    __shared__ T lds[kThreads / kWave];
    const uint64_t base = (uint64_t)blockIdx.x * kTile;
    T acc = 0;
#pragma unroll
    for (int i = 0; i < kItems; i++) {
        uint64_t g = base + (uint64_t)i * kThreads + threadIdx.x;
        if (g < n) acc += in[g];
    }
    T tot;
    (void)block_excl_scan(acc, lds, tot);
    if (threadIdx.x == 0) sums[blockIdx.x] = tot;
}

// Exclusive scan of one tile; each thread owns kItems consecutive elements.
template <typename T>
__global__ __launch_bounds__(kThreads) void k_tile_scan(const T *in, T *out, uint64_t n,
                                                        const T *__restrict__ tile_off,
                                                        T *__restrict__ total)
{
    __shared__ T lds[kThreads / kWave];
    __shared__ T stage[kTile];
    const uint64_t base = (uint64_t)blockIdx.x * kTile;
    // coalesced load into LDS, then each thread scans its kItems run
#pragma unroll
    for (int i = 0; i < kItems; i++) {
        uint64_t g = base + (uint64_t)i * kThreads + threadIdx.x;
        stage[i * kThreads + threadIdx.x] = (g < n) ? in[g] : T(0);
    }
    __syncthreads();
    T v[kItems];
    T acc = 0;
#pragma unroll
    for (int i = 0; i < kItems; i++) {
        v[i] = stage[threadIdx.x * kItems + i];
        acc += v[i];
    }
    T tot;
    T off = block_excl_scan(acc, lds, tot);
    if (tile_off) off += tile_off[blockIdx.x];
#pragma unroll
    for (int i = 0; i < kItems; i++) {
        stage[threadIdx.x * kItems + i] = off;
        off += v[i];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kItems; i++) {
        uint64_t g = base + (uint64_t)i * kThreads + threadIdx.x;
        if (g < n) out[g] = stage[i * kThreads + threadIdx.x];
    }
    if (total && threadIdx.x == 0 && gridDim.x == 1) *total = tot;
}

template <typename T>
void exclusive_scan_impl(const T *in, T *out, uint64_t n, T *total, hipStream_t st, Arena &tmp)
{
    if (n == 0) {
        if (total) ABHSF_HIP(hipMemsetAsync(total, 0, sizeof(T), st));
        return;
    }
    const uint64_t ntiles = (n + kTile - 1) / kTile;
    if (ntiles == 1) {
        k_tile_scan<T><<<1, kThreads, 0, st>>>(in, out, n, nullptr, total);
        ABHSF_HIP(hipGetLastError());
        return;
    }
    T *sums = tmp.take<T>(ntiles);
    k_tile_reduce<T><<<(unsigned)ntiles, kThreads, 0, st>>>(in, n, sums);
    ABHSF_HIP(hipGetLastError());
    exclusive_scan_impl<T>(sums, sums, ntiles, total, st, tmp);
    k_tile_scan<T><<<(unsigned)ntiles, kThreads, 0, st>>>(in, out, n, sums, nullptr);
    ABHSF_HIP(hipGetLastError());
}

// ---- radix sort --------------------------------------------------------------

constexpr int kRadixBits = 8;
constexpr int kRadix = 1 << kRadixBits;

__global__ __launch_bounds__(kThreads) void k_radix_hist(const uint64_t *__restrict__ keys, uint64_t n,
                                                         int shift, uint32_t *__restrict__ hist,
                                                         uint32_t ntiles)
{
    __shared__ uint32_t cnt[kRadix];
    cnt[threadIdx.x] = 0;
    __syncthreads();
    const uint64_t base = (uint64_t)blockIdx.x * kTile;
#pragma unroll
    for (int i = 0; i < kItems; i++) {
        uint64_t g = base + (uint64_t)i * kThreads + threadIdx.x;
        if (g < n) atomicAdd(&cnt[(keys[g] >> shift) & (kRadix - 1)], 1u);
    }
    __syncthreads();
    hist[(uint64_t)threadIdx.x * ntiles + blockIdx.x] = cnt[threadIdx.x];
}

__global__ __launch_bounds__(kThreads) void k_radix_scatter(const uint64_t *__restrict__ kin,
                                                            const uint32_t *__restrict__ vin,
                                                            uint64_t *__restrict__ kout,
                                                            uint32_t *__restrict__ vout, uint64_t n,
                                                            int shift, const uint32_t *__restrict__ offs,
                                                            uint32_t ntiles)
{
    static_assert(kThreads == kRadix, "one thread per digit");
    __shared__ uint32_t run[kRadix];
    __shared__ uint32_t wc[kThreads / kWave][kRadix];
    const int wave = threadIdx.x >> 6;
    run[threadIdx.x] = offs[(uint64_t)threadIdx.x * ntiles + blockIdx.x];
    const uint64_t base = (uint64_t)blockIdx.x * kTile;
    for (int r = 0; r < kItems; r++) {
#pragma unroll
        for (int w = 0; w < kThreads / kWave; w++) wc[w][threadIdx.x] = 0;
        __syncthreads();
        const uint64_t g = base + (uint64_t)r * kThreads + threadIdx.x;
        const bool valid = g < n;
        const uint64_t key = valid ? kin[g] : 0;
        const uint32_t val = valid ? vin[g] : 0;
        const uint32_t d = (uint32_t)(key >> shift) & (kRadix - 1);
        // lanes of this wave holding the same digit
        uint64_t mask = __ballot(valid);
#pragma unroll
        for (int b = 0; b < kRadixBits; b++) {
            const bool bit = (d >> b) & 1;
            const uint64_t bal = __ballot(bit);
            mask &= bit ? bal : ~bal;
        }
        const uint32_t rank = __popcll(mask & lanemask_lt());
        if (valid && rank == 0) wc[wave][d] = __popcll(mask);
        __syncthreads();
        if (valid) {
            uint32_t pos = run[d] + rank;
            for (int w = 0; w < wave; w++) pos += wc[w][d];
            kout[pos] = key;
            vout[pos] = val;
        }
        __syncthreads();
        uint32_t add = 0;
#pragma unroll
        for (int w = 0; w < kThreads / kWave; w++) add += wc[w][threadIdx.x];
        run[threadIdx.x] += add;
        __syncthreads();
    }
}

}  // namespace

size_t scratch_trim()
{
    std::vector<KeptBuf> out;
    {
        std::lock_guard<std::mutex> l(kept().m);
        for (const auto &q : kept().bufs)  // (under the lock: the owner cannot end meanwhile)
            if (q.owner) (void)hipStreamSynchronize(q.stream);
        out.swap(kept().bufs);
    }
    size_t bytes = 0;
    for (const auto &q : out) bytes += q.buf.bytes();
    return bytes;  // freed here
}

Arena::Arena(hipStream_t st) : st_(st)
{
    ABHSF_HIP(hipGetDevice(&device_));
    std::lock_guard<std::mutex> l(kept().m);
    from_ = kept().now++;
}

Arena::~Arena()
{
    // nothing on the stream uses the buffers any more; after an error they go
    // back to the runtime
    const bool done = hipStreamSynchronize(st_) == hipSuccess;
    std::lock_guard<std::mutex> l(kept().m);
    auto &b = kept().bufs;
    const uint64_t at = ++kept().now;
    size_t total = 0;
    for (const auto &q : b)
        if (q.device == device_ && !q.owner && q.at > from_) total += q.buf.bytes();
    for (size_t i = 0; i < b.size();) {
        KeptBuf &q = b[i];
        const bool mine = q.owner == this;
        // what lay there all the while goes too: this operation had no use for it
        const bool drop = mine ? !done || total + q.buf.bytes() > kScratchKeep
                               : q.device == device_ && !q.owner && q.at <= from_;
        if (drop) {
            b.erase(b.begin() + (std::ptrdiff_t)i);
            continue;
        }
        if (mine) {
            q.owner = nullptr;
            q.at = at;
            total += q.buf.bytes();
        }
        i++;
    }
    if (!done) return;
    try {
        for (auto &q : used_)
            if (total + q.bytes() <= kScratchKeep) {
                b.push_back({device_, at, std::move(q)});
                total += b.back().buf.bytes();
            }
    } catch (...) {  // out of host memory: what is left is freed
    }
}

void *Arena::fresh(size_t bytes)
{
    used_.reserve(used_.size() + 1);
    // a kept buffer of at most 1/8 more: the builds of one matrix size ask for
    // the same sizes, and more would be memory that nothing can give back
    const size_t most = bytes + bytes / 8;
    {
        std::lock_guard<std::mutex> l(kept().m);
        auto &b = kept().bufs;
        size_t best = b.size();
        for (size_t i = 0; i < b.size(); i++)
            if (b[i].device == device_ && (!b[i].owner || b[i].owner == this) && b[i].buf.bytes() >= bytes &&
                b[i].buf.bytes() <= most && (best == b.size() || b[i].buf.bytes() < b[best].buf.bytes()))
                best = i;
        if (best < b.size()) {
            used_.push_back(std::move(b[best].buf));
            b.erase(b.begin() + (std::ptrdiff_t)best);
            return used_.back().get();
        }
    }
    used_.emplace_back(bytes);
    return used_.back().get();
}

void Arena::to_idle(size_t first)
{
    try {
        std::lock_guard<std::mutex> l(kept().m);
        auto &b = kept().bufs;
        b.reserve(b.size() + used_.size() - first);
        for (size_t i = first; i < used_.size(); i++)
            b.push_back({device_, kept().now, std::move(used_[i]), this, st_});
        used_.resize(first);
    } catch (...) {  // out of host memory: they stay in use to the end
    }
}

void *Arena::take_bytes(size_t bytes)
{
    bytes = (bytes + 255) & ~(size_t)255;
    if (bytes == 0) return nullptr;
    if (bytes > kChunk) return fresh(bytes);
    if (!chunk_ || at_ + bytes > kChunk) {
        chunk_ = static_cast<char *>(fresh(kChunk));
        at_ = 0;
    }
    void *p = chunk_ + at_;
    at_ += bytes;
    return p;
}

void exclusive_scan_u32(const uint32_t *in, uint32_t *out, uint64_t n, uint32_t *total, hipStream_t st, Arena &tmp)
{
    exclusive_scan_impl<uint32_t>(in, out, n, total, st, tmp);
}

void exclusive_scan_u64(const uint64_t *in, uint64_t *out, uint64_t n, uint64_t *total, hipStream_t st, Arena &tmp)
{
    exclusive_scan_impl<uint64_t>(in, out, n, total, st, tmp);
}

void radix_sort_pairs(uint64_t *keys, uint32_t *vals, uint64_t n, int key_bits, hipStream_t st, Arena &tmp)
{
    if (n < 2 || key_bits <= 0) return;
    ABHSF_REQUIRE(n < (1ull << 32), ABHSF_ERR_UNSUPPORTED, "radix sort limited to 2^32 elements");
    const uint64_t ntiles = (n + kTile - 1) / kTile;
    ABHSF_REQUIRE(ntiles * kRadix < (1ull << 32), ABHSF_ERR_UNSUPPORTED, "radix histogram too large");
    const Arena::Scope scope(tmp);
    uint64_t *ka = keys, *kb = tmp.take<uint64_t>(n);
    uint32_t *va = vals, *vb = tmp.take<uint32_t>(n);
    uint32_t *hist = tmp.take<uint32_t>(ntiles * kRadix);
    for (int shift = 0; shift < key_bits; shift += kRadixBits) {
        k_radix_hist<<<(unsigned)ntiles, kThreads, 0, st>>>(ka, n, shift, hist, (uint32_t)ntiles);
        ABHSF_HIP(hipGetLastError());
        exclusive_scan_impl<uint32_t>(hist, hist, ntiles * kRadix, nullptr, st, tmp);
        k_radix_scatter<<<(unsigned)ntiles, kThreads, 0, st>>>(ka, va, kb, vb, n, shift, hist, (uint32_t)ntiles);
        ABHSF_HIP(hipGetLastError());
        std::swap(ka, kb);
        std::swap(va, vb);
    }
    if (ka != keys) {
        ABHSF_HIP(hipMemcpyAsync(keys, ka, n * sizeof(uint64_t), hipMemcpyDeviceToDevice, st));
        ABHSF_HIP(hipMemcpyAsync(vals, va, n * sizeof(uint32_t), hipMemcpyDeviceToDevice, st));
    }
}

}  // namespace abhsf
