// prims.hpp -- device buffers, scans and a stable LSD radix sort (gfx950).
#pragma once

#include "common.hpp"

#include <vector>

namespace abhsf {

// Frees the scratch kept between operations (Arena); its bytes.
size_t scratch_trim();

// RAII device buffer.
class DevBuf {
  public:
    DevBuf() = default;
    explicit DevBuf(size_t bytes) { alloc(bytes); }
    ~DevBuf() { release(); }
    DevBuf(const DevBuf &) = delete;
    DevBuf &operator=(const DevBuf &) = delete;
    DevBuf(DevBuf &&o) noexcept : p_(o.p_), n_(o.n_) { o.p_ = nullptr; o.n_ = 0; }
    DevBuf &operator=(DevBuf &&o) noexcept
    {
        if (this != &o) { release(); p_ = o.p_; n_ = o.n_; o.p_ = nullptr; o.n_ = 0; }
        return *this;
    }
    void alloc(size_t bytes)
    {
        release();
        n_ = bytes;
        if (bytes == 0) return;
        // a failed call's error stays with the thread, past calls that succeed,
        // until it is read: the next launch check would report it
        auto get = [&] {
            const hipError_t r = hipMalloc(&p_, bytes);
            if (r != hipSuccess) (void)hipGetLastError();
            return r;
        };
        hipError_t e = get();
        if (e != hipSuccess && scratch_trim()) e = get();
        if (e != hipSuccess) {
            p_ = nullptr;
            n_ = 0;
            throw Error(ABHSF_ERR_ALLOC, "hipMalloc of " + std::to_string(bytes) + " bytes failed: " +
                                             hipGetErrorString(e));
        }
    }
    void release()
    {
        if (p_) (void)hipFree(p_);
        p_ = nullptr;
        n_ = 0;
    }
    template <typename T = void>
    T *get() const { return static_cast<T *>(p_); }
    size_t bytes() const { return n_; }

  private:
    void *p_ = nullptr;
    size_t n_ = 0;
};

// Device scratch of one operation on a stream, handed out piece by piece.  A
// conversion needs some thirty pieces (24 bytes an entry and 45 a block, and
// the sort's 12.5 an entry, which are idle after it), and allocating and freeing them every time cost more than its kernels: a free
// waits for the device, and freed memory is cleared before it is given out
// again (converting R-MAT scale 20, 0.9 GB of scratch, again and again: 12 ms
// at first, 28 ms once the clearing lags behind).  Small pieces share chunks;
// the buffers of the last operation stay for the next one: at most
// kScratchKeep bytes per device, no others than that operation used, and none
// if an allocation fails: an operation takes a kept buffer when it needs one of
// its size, and the others stay where scratch_trim finds them.  An Arena owns
// what it took until it is destroyed, after the stream has finished, so
// operations of several threads or streams never share a buffer.  Pieces are
// 256-byte aligned.
constexpr size_t kScratchKeep = (size_t)1 << 30;

class Arena {
  public:
    explicit Arena(hipStream_t st);
    ~Arena();
    Arena(const Arena &) = delete;
    Arena &operator=(const Arena &) = delete;
    void *take_bytes(size_t bytes);
    template <typename T>
    T *take(uint64_t n) { return static_cast<T *>(take_bytes((size_t)n * sizeof(T))); }

    // Pieces taken in a scope are idle after it: later pieces of the Arena
    // (on the same stream, so in order) take their place, and they are freed
    // if an allocation fails.
    class Scope {
      public:
        explicit Scope(Arena &a) : a_(a), first_(a.used_.size()), chunk_(a.chunk_), at_(a.at_) {}
        ~Scope()
        {
            a_.chunk_ = chunk_;
            a_.at_ = at_;
            a_.to_idle(first_);
        }
        Scope(const Scope &) = delete;
        Scope &operator=(const Scope &) = delete;

      private:
        Arena &a_;
        size_t first_;
        char *chunk_;
        size_t at_;
    };

  private:
    static constexpr size_t kChunk = (size_t)16 << 20;
    void *fresh(size_t bytes);  // a kept buffer that fits, or a new one
    void to_idle(size_t first);  // used_[first ..]
    std::vector<DevBuf> used_;
    uint64_t from_ = 0;  // when the operation began (Kept::now)
    char *chunk_ = nullptr;
    size_t at_ = 0;
    int device_ = 0;
    hipStream_t st_;
};

// Exclusive scan out[i] = sum_{j<i} in[j]; out may alias in.  If total is
// non-null the sum of all n inputs is written there (device pointer).  The
// scratch stays in `tmp`; the calls only enqueue.
void exclusive_scan_u32(const uint32_t *in, uint32_t *out, uint64_t n, uint32_t *total, hipStream_t st, Arena &tmp);
void exclusive_scan_u64(const uint64_t *in, uint64_t *out, uint64_t n, uint64_t *total, hipStream_t st, Arena &tmp);

// Stable LSD radix sort of (key, value) pairs by the low key_bits of key.
// keys/vals are sorted in place (scratch of the same sizes comes from tmp).
void radix_sort_pairs(uint64_t *keys, uint32_t *vals, uint64_t n, int key_bits, hipStream_t st, Arena &tmp);

}  // namespace abhsf
